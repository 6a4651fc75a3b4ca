"""Where the launcher's lines between the small tiles, the larger ones, split K, stream-K and the streaming kernels lie: problems
timed on both sides (us beside them), which a line drawn elsewhere had made slower."""
import pytest

S8, BF16F32, BF16, F16, F32, E4M3, E5M2 = range(7)


def kind(p, capi):
    if p.streamk_tiles:
        return "stream-K"
    if p.split_k > 1 and p.tile_m == 64:
        return "split K"
    if p.rung == capi.RUNG_SKINNY and p.variant == 1:
        return "stream"
    if (p.tile_m, p.tile_n) == (64, 64):   # four waves of the whole tile each, or the register-staged kernel
        return "64 own slabs" if (p.wave_m, p.wave_n, p.threads) == (64, 64, 256) else "64 staged"
    return p.tile_m


@pytest.mark.parametrize("types,m,n,k,la,lb,want", [
    # 64 x 64 tiles: slabs of the waves' own from as many as earn the sums in LDS back (own slabs / staged)
    (BF16F32, 896, 1408, 128, 0, 1, "64 staged"),        # 5.3 / 4.3
    (BF16F32, 816, 1296, 64, 0, 1, "64 staged"),         # 6.0 / 4.5
    (BF16, 1152, 1280, 128, 0, 1, "64 staged"),          # 5.3 / 4.3
    (E4M3, 960, 960, 960, 0, 1, "64 staged"),            # 6.9 / 5.9
    (S8, 1024, 1024, 1024, 0, 0, "64 own slabs"),        # 6.3 / 7.2
    (BF16F32, 1024, 1024, 1024, 0, 0, "64 own slabs"),
    (S8, 1024, 1024, 2048, 0, 1, "64 own slabs"),
    # decode, 65 rows and more with a short K: 32 x 32 tiles instead of 64 x 64 that leave compute units idle
    (E4M3, 113, 857, 640, 0, 1, 32),                     # 7.8 on 64 x 64 own slabs, 5.6 staged, 3.3
    (BF16, 69, 314, 384, 0, 1, 32),                      # 8.0, 5.2, 3.4
    (BF16F32, 96, 1024, 128, 0, 1, 32),                  # 4.1, 3.3, 2.8
    # ... with a last stage that the end of K cuts
    (BF16, 124, 768, 1424, 0, 1, 32),                    # 13.0 on the tile kernel
    (E4M3, 112, 128, 2784, 0, 1, 32),                    # 8.8
    # few rows and a long K: in parts, or 32 x 32 tiles, not the tile kernel
    (BF16F32, 30, 1280, 4224, 0, 1, "split K"),          # 10.9 on the tile kernel, 8.4
    (BF16F32, 36, 7296, 7168, 0, 1, "split K"),          # 29.3 on the tile kernel, 21.5
    (F16, 56, 7168, 8472, 0, 1, "split K"),              # 41.7 on the tile kernel, 27.8
    # 32 x 32 tiles of rows that begin inside a line (from memory: rows of whole and half lines)
    (BF16F32, 89, 1856, 7632, 0, 1, "split K"),          # 23.9 on 32 x 32 tiles, 18.5
    (BF16F32, 37, 2248, 5088, 0, 1, 32),                 # 13.1, 13.6 in parts
    (BF16, 960, 32, 5424, 0, 1, "split K"),              # 20.1 on 32 x 32 tiles, 10.7
    # fp32: a 128 x 128 tile's products take the compute unit that has two of them twice as long
    (F32, 2112, 2112, 2112, 0, 0, "small"),              # 238 on 128 x 128, 186 on 64 x 64
    (F32, 2240, 2240, 2240, 0, 1, "small"),              # 250, 207, 196 on 32 x 32
    (F32, 1600, 2457, 1024, 0, 0, "small"),              # 137 on 128 x 128 staged, 78 on 64 x 64
    (F32, 1938, 2092, 1999, 0, 0, "small"),              # 262, 152
    (F32, 2048, 2048, 2048, 0, 0, 128),                  # 120, 138 on 64 x 64
    # stream-K against the small tiles as they are
    (BF16F32, 456, 1536, 5504, 0, 1, "64 own slabs"),    # 40 on stream-K, 21
    (F16, 289, 2776, 7424, 0, 1, "64 own slabs"),        # 47, 29
    (BF16F32, 640, 640, 16384, 0, 1, "split K"),         # 52, 27
    (BF16F32, 1024, 1024, 16384, 0, 1, "stream-K"),      # 53, 55 in parts
])
def test_line(capi, types, m, n, k, la, lb, want):
    p = capi.plan(types, m, n, k, la, lb)
    assert p.tile_m <= 64 if want == "small" else kind(p, capi) == want, (kind(p, capi), p.as_dict())


def test_waves_of_the_8_bit_floats(capi):
    """A K-contiguous B from memory: four waves where M or N is ragged (1500 x 8192 x 4096 48.0 us on four, 54.7 on eight), eight
    on whole tiles (4608^3 101.8 / 96.5, 4096 x 8192 x 4096 103.4 / 99.7)."""
    for types in (E4M3, E5M2):
        assert capi.plan(types, 1000, 14336, 4096, 0, 1).threads == 256
        assert capi.plan(types, 2000, 8192, 4096, 0, 1).threads == 256
        for m, n, k in [(4608, 4608, 4608), (4864, 4864, 4864), (4096, 8192, 4096)]:
            assert capi.plan(types, m, n, k, 0, 1).threads == 512, (m, n, k)


def test_short_parts_of_a_split_k_run_on_the_staged_kernel(capi):
    short, long = capi.plan(BF16F32, 62, 256, 8320, 0, 1), capi.plan(BF16F32, 36, 7296, 7168, 0, 1)
    assert short.split_k > 1 and short.wave_m == 32      # 9.2 us staged, 10.2 on slabs of the waves' own
    assert long.split_k > 1 and long.wave_m == 64


@pytest.mark.parametrize("types,m,n,k,la,lb,tile,ring", [
    (E5M2, 6736, 6944, 160, 0, 1, 128, False),     # 44 on the ring kernel's 256 x 256, 37
    (E4M3, 4160, 4928, 368, 0, 0, 128, False),     # past a round, the last one less than half full
    (E4M3, 3520, 3520, 368, 0, 0, 256, True),      # one round
    (S8, 3328, 2944, 240, 0, 1, 256, False),       # 1.08 of the staged kernel's time on the ring kernel
    (BF16F32, 4096, 2240, 120, 1, 1, 256, False),  # 14.4 on the ring kernel, 13.1
    (BF16F32, 4096, 2240, 120, 1, 0, 256, True),
    (BF16F32, 4096, 2240, 248, 0, 0, 256, True),   # four slabs
])
def test_a_short_k_tail(capi, types, m, n, k, la, lb, tile, ring):
    p = capi.plan(types, m, n, k, la, lb)
    assert p.tile_m == tile and (p.variant in (5, 6, 11)) == ring, p.as_dict()


def test_waves_of_the_8_bit_floats_with_a_k_tail(capi):
    """Eight, but for a K-contiguous B past 24 slabs (eight / four 0.92 - 1.00 up to 24 slabs, 0.97 - 1.05 at 32; a row-major
    B 0.77 - 1.01)."""
    for types in (E4M3, E5M2):
        assert capi.plan(types, 3520, 3520, 1040, 0, 0).threads == 512
        assert capi.plan(types, 3520, 3520, 4000, 0, 0).threads == 512
        assert capi.plan(types, 3520, 3520, 1040, 0, 1).threads == 512
        assert capi.plan(types, 3520, 3520, 4000, 0, 1).threads == 256
