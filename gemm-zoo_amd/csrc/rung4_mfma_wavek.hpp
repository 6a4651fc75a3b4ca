// MFMA rung, small tiles: K dealt to the waves of a work-group.
//
// For grids that 128 x 128 tiles leave mostly empty.  Such a work-group is alone on its compute unit, and what it waits
// for is operands: a compute unit takes in 120 - 150 bytes per ns from its L2, so a 128-byte slab of a 64 x 64 tile
// (16 KiB) could come in 0.13 us, but a tile whose waves share every slab - one barrier per slab, two slabs on their
// way - took 0.45 - 0.55.  Here every wave multiplies the WHOLE tile over slabs of its own (wave w takes slabs w, w + W,
// ...), through a part of the LDS that no other wave touches.  There is no barrier in the main loop, up to eight slabs
// are on their way, and each fragment is read once per tile and not once per wave (16 KiB of LDS reads per slab instead
// of 32).  The waves' sums meet in LDS at the end, added in the order of the waves, so the result does not depend on
// timing.  A slab of a 64 x 64 tile takes 0.2 - 0.3 us now, of a 32 x 32 tile 0.1 (us, before / after, operands rotating
// through 300 MB: bf16 row/row 256^3 4.2 / 3.0, 512^3 5.5 / 3.7, 1024^3 10.1 / 8.7; row/col 512^2 x 2048 10.5 / 5.9, 640 x
// 1024 x 4096 column-major A 22.9 / 17.6; int8 512^2 x 8192 15.0 / 8.6; fp32 256^3 7.5 / 3.9, 512^3 10.3 / 5.6).
//
// Two ways in, chosen per launch:
//   FEED_DMA  lines that are whole 16-byte pieces: global_load_lds_dwordx4 into the wave's stages, rows past the end clamped,
//             pieces past the end of K fetched from inside it and zeroed in LDS.  The copies of slab i + NST go out
//             between the matrix instructions of slab i, into the stage whose fragments have just been read.
//   FEED_REG  any alignment: through registers (Stager, one wave wide).  32 x 32 tiles only: on 64 x 64 ones the staged
//             kernel, whose four waves share the loads of a slab, is 2 - 15 % faster (bf16 487 x 1283 x 1099 11.0 / 13.3).
#pragma once
#include "rung4_mfma.hpp"

namespace gz {

enum { FEED_DMA = 0, FEED_REG = 1 };

// K part `part` of `parts`: the first slab and the number of slabs (struct SplitK)
__device__ inline void splitk_range(const SplitK& sk, int part, int& first, int& count) {
  first = part * sk.q + min(part, sk.rem);
  count = sk.q + (part < sk.rem ? 1 : 0);
}

// LDS row of K line r of a line operand within its copy, and the piece swizzle there.  A transposing read takes 4
// (16-bit) or 8 (8-bit) K lines x 64 (32) bytes per half wave, an fp32 read one line per half wave, four lines apart:
// without this, lines of 128 bytes (64 rows of 16 bits) two apart, of 64 bytes (64 rows of 8 bits) four apart would meet
// in the same banks.
template <int ES, int R> __device__ inline int wavek_line_swz(int r) {
  if constexpr (R == 64) return ES == 2 ? ((r >> 1) & 1) << 2 : ES == 1 ? ((r >> 2) & 1) << 1 : ((r >> 2) & 1) << 3;
  else return 0;
}
// (fp32 with 32 rows: lines of 128 bytes, r and r + 4 side by side)
template <int ES, int R> __host__ __device__ constexpr int wavek_line_at(int p) {   // line held by LDS row p
  return (ES == 4 && R == 32) ? (p & ~7) | ((p >> 1) & 3) | ((p & 1) << 2) : p;
}
template <int ES, int R> __host__ __device__ constexpr int wavek_row_of(int r) {    // LDS row of line r
  return (ES == 4 && R == 32) ? (r & ~7) | ((r & 3) << 1) | ((r >> 2) & 1) : r;
}

// One operand, R tile rows (or columns), fed by copies into the wave's own stages.
template <typename in_t, int R, bool KC> struct DmaFeed {
  static constexpr int ES = (int)sizeof(in_t), EPV = 16 / ES, BK = SLAB_BYTES / ES;
  static constexpr int COPIES = R / 8;                        // 1 KiB each
  static constexpr int BYTES = R * SLAB_BYTES;
  static constexpr int LINE_BYTES = R * ES, KRC = 1024 / LINE_BYTES, LPR = 64 / KRC;   // K lines per copy, lanes per line
  static constexpr uint32_t BIAS = 4096;                      // keeps offset - immediate non-negative
  const char* base;   // the tile's first row at K line / element 0 of this work-group's range
  size_t pitch;       // bytes between lines
  int rows_left;      // rows of the operand from the tile's first
  uint32_t voff[COPIES];

  __device__ __forceinline__ int row_of(int t, int lane) const { return 8 * t + (lane >> 3); }                    // KC
  __device__ __forceinline__ int piece_of(int t, int lane) const {
    if constexpr (KC) return (lane & 7) ^ dtl_swz(row_of(t, lane));
    else return (lane % LPR) ^ wavek_line_swz<ES, R>(line_of(t, lane));
  }
  __device__ __forceinline__ int line_of(int t, int lane) const { return wavek_line_at<ES, R>(t * KRC + lane / LPR); }   // !KC
  // byte offset from the slab's base (KC: row 0 at its first k; lines: its first line) of what the lane fetches in copy t;
  // k_left: k lines from the slab's first to the end of K
  __device__ __forceinline__ uint32_t offset(int t, int lane, int k_left) const {
    if constexpr (KC) {
      const int row = min(row_of(t, lane), rows_left - 1), k = min(piece_of(t, lane) * EPV, k_left - EPV);
      return (uint32_t)((size_t)row * pitch) + (uint32_t)(k * ES);
    } else {
      const int line = min(line_of(t, lane), k_left - 1), piece = min(piece_of(t, lane), rows_left / EPV - 1);
      return (uint32_t)((size_t)line * pitch) + (uint32_t)(piece * 16);
    }
  }
  __device__ __forceinline__ void init(const in_t* p, size_t ld, int row0, int rows, int lane) {
    pitch = ld * ES;
    rows_left = rows - row0;
    base = reinterpret_cast<const char*>(p) + (KC ? (size_t)row0 * pitch : (size_t)row0 * ES);
#pragma unroll
    for (int t = 0; t < COPIES; t++) voff[t] = offset(t, lane, BK) + BIAS - (uint32_t)((t - COPIES / 2) * 1024);
  }
  __device__ __forceinline__ const char* slab_base(int slab) const {
    return KC ? base + (size_t)slab * SLAB_BYTES : base + (size_t)slab * BK * pitch;
  }
  // LDS destination of the copies that follow; `st`: this operand's part of a stage
  __device__ __forceinline__ void aim(uint32_t st) const { asm_set_m0(st + (COPIES / 2) * 1024); }
  template <int T> __device__ __forceinline__ void copy(const char* src_minus_bias) const {
    asm_copy16<(T - COPIES / 2) * 1024>(voff[T], src_minus_bias);
  }
  // a slab that the end of K cuts: addresses clamped into the operand
  // (the lane number made opaque: what is computed from it here would otherwise be kept in registers through the loop)
  __device__ __forceinline__ void copy_cut(uint32_t st, int slab, int k_left, int lane) const {
    asm volatile("" : "+v"(lane));
    const char* const src = slab_base(slab) - BIAS;
    aim(st);
    static_for<COPIES>([&](auto t_c) {
      constexpr int T = decltype(t_c)::value;
      asm_copy16<(T - COPIES / 2) * 1024>(offset(T, lane, k_left) + BIAS - (uint32_t)((T - COPIES / 2) * 1024), src);
    });
  }
  // ... and zeros for what lies past it, once it has landed
  __device__ __forceinline__ void zero_cut(char* st, int k_left, int lane) const {
    asm volatile("" : "+v"(lane));
    const u32x4_t z = {0, 0, 0, 0};
#pragma unroll
    for (int t = 0; t < COPIES; t++) {
      const int k = KC ? piece_of(t, lane) * EPV : line_of(t, lane);
      if (k >= k_left) *reinterpret_cast<u32x4_t*>(st + t * 1024 + lane * 16) = z;
    }
  }
  // fragment of 32-row block `blk`, K step `ks` (32 bytes of K): row lane % 32, 16 bytes at (lane / 32) * 16
  __device__ static __forceinline__ u32x4_t fragment(const char* st, int blk, int ks, int lane) {
    if constexpr (KC) {
      const int row = lane & 31;
      return *reinterpret_cast<const u32x4_t*>(st + (blk * 32 + row) * SLAB_BYTES + (((ks * 2 + (lane >> 5)) ^ dtl_swz(row)) * 16));
    } else if constexpr (ES == 4) {
      u32x4_t v;
#pragma unroll
      for (int e = 0; e < 4; e++) {
        const int line = ks * 8 + (lane >> 5) * 4 + e, col = blk * 32 + (lane & 31);
        v[e] = *reinterpret_cast<const uint32_t*>(st + wavek_row_of<ES, R>(line) * LINE_BYTES +
                                                  (((col / EPV) ^ wavek_line_swz<ES, R>(line)) * 16) + (col % EPV) * ES);
      }
      return v;
    } else {
      constexpr int TR_LPR = ES == 2 ? 4 : 2;        // lanes per K line of a [4 x 16] / [8 x 16] block
      constexpr int HALF = 16 / TR_LPR;              // K lines per transposing read
      const int i16 = lane & 15, ti = i16 / TR_LPR;
      const int col = blk * 32 + ((lane >> 4) & 1) * 16 + (i16 % TR_LPR) * (8 / ES);
      const int line = ks * (32 / ES) + (lane >> 5) * (16 / ES) + ti;
      // (the second read is HALF lines further: for 16 bits bit 2 of the line, for 8 bits bit 3, outside the swizzle)
      const char* const p = st + line * LINE_BYTES + (((col / EPV) ^ wavek_line_swz<ES, R>(line)) * 16) + (col % EPV) * ES;
      const u32x2_t lo = lds_read_tr<ES>(p), hi = lds_read_tr<ES>(p + HALF * LINE_BYTES);
      return u32x4_t{lo[0], lo[1], hi[0], hi[1]};
    }
  }
};

// The same operand through registers: Stager as one wave uses it, with its padded LDS rows.
template <typename in_t, int R, bool KC> struct RegFeed {
  using S = Stager<in_t, R, 64, KC, true>;
  static constexpr int ES = (int)sizeof(in_t);
  static constexpr bool NAT = ES == 4 && !KC;   // k lines kept whole in LDS
  static constexpr int BYTES = S::LDS_BYTES;
  __device__ static __forceinline__ u32x4_t fragment(const char* st, int blk, int ks, int lane) {
    if constexpr (NAT) {
      const char* const p = st + (ks * 8 + (lane >> 5) * 4) * S::NAT_PITCH + (blk * 32 + (lane & 31)) * 4;
      return u32x4_t{*reinterpret_cast<const uint32_t*>(p), *reinterpret_cast<const uint32_t*>(p + S::NAT_PITCH),
                     *reinterpret_cast<const uint32_t*>(p + 2 * S::NAT_PITCH), *reinterpret_cast<const uint32_t*>(p + 3 * S::NAT_PITCH)};
    } else {
      return *reinterpret_cast<const u32x4_t*>(st + (blk * 32 + (lane & 31)) * PITCH + ks * 32 + (lane >> 5) * 16);
    }
  }
};

template <int TYPES, int TM, int TN, int W, int NST, int FEED, bool A_KC, bool B_KC> struct WaveK {
  using in_t = typename Traits<TYPES>::in_t;
  using FA = std::conditional_t<FEED == FEED_DMA, DmaFeed<in_t, TM, A_KC>, RegFeed<in_t, TM, A_KC>>;
  using FB = std::conditional_t<FEED == FEED_DMA, DmaFeed<in_t, TN, B_KC>, RegFeed<in_t, TN, B_KC>>;
  static constexpr int STAGE = FA::BYTES + FB::BYTES;
  // stages of a wave in LDS (FEED_REG: NST slabs are on their way in registers, one is in LDS), and room for its sums
  static constexpr int STAGES = FEED == FEED_DMA ? NST : 1;
  static constexpr int WAVE_BYTES = STAGE * STAGES > TM * TN * 4 ? STAGE * STAGES : TM * TN * 4;
  static constexpr int LDS_BYTES = W * WAVE_BYTES;
};

// RES: work-groups per compute unit that the registers must leave room for
template <int TYPES, int TM, int TN, int W, int NST, int RES, int FEED, bool A_KC, bool B_KC>
__global__ void __launch_bounds__(W * 64, RES * W / 4) mfma_wavek_kernel(GemmArgs<TYPES> g, int tiles_m, int tiles_n, SplitK sk) {
  using T = Traits<TYPES>;
  using in_t = typename T::in_t;
  using out_t = typename T::out_t;
  using acc_t = typename T::acc_t;
  using acc_v = typename AccVec<TYPES>::type;
  using P = WaveK<TYPES, TM, TN, W, NST, FEED, A_KC, B_KC>;
  using FA = typename P::FA;
  using FB = typename P::FB;
  constexpr int ES = (int)sizeof(in_t), BK = SLAB_BYTES / ES;
  constexpr int FM = TM / 32, FN = TN / 32;
  constexpr bool F8 = is_fp8(TYPES);
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  int tm, tn, slot = 0, slab0 = 0, ktiles = (g.K + BK - 1) / BK;
  const int tiles = tiles_m * tiles_n;
  if (sk.parts > 1) {
    // (the tiles of one K part side by side: the work-groups of an XCD share their operands)
    const int lid = lid_of_block(blockIdx.x, tiles * sk.parts), part = lid / tiles;
    tile_of_lid(lid - part * tiles, tiles_m, tiles_n, tm, tn);
    splitk_range(sk, part, slab0, ktiles);
    slot = part * tiles + tm * tiles_n + tn;
  } else {
    tile_of_block(blockIdx.x, tiles_m, tiles_n, tm, tn);
  }
  const int m0 = tm * TM, n0 = tn * TN;
  const int end = slab0 + ktiles;                          // slabs [slab0, end) of K, this wave's: slab0 + wave + W i
  const int first = slab0 + wave, mine = first < end ? (end - first + W - 1) / W : 0;
  char* const own = lds + wave * P::WAVE_BYTES;

  acc_v acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; i++)
#pragma unroll
    for (int j = 0; j < FN; j++)
#pragma unroll
      for (int v = 0; v < 16; v++) acc[i][j][v] = 0;

  u32x4_t af[KSTEPS][FM], bf[KSTEPS][FN];
  auto read_step = [&](const char* st, int ks) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < FM; i++) af[ks][i] = FA::fragment(st, i, ks, lane);
#pragma unroll
    for (int j = 0; j < FN; j++) bf[ks][j] = FB::fragment(st + FA::BYTES, j, ks, lane);
  };
  auto read_slab = [&](const char* st) __attribute__((always_inline)) {
#pragma unroll
    for (int ks = 0; ks < KSTEPS; ks++) read_step(st, ks);
  };
  // block products of the slab in the fragments, one at a time: NPROD of them, product Q
  constexpr int STEPS = F8 ? KSTEPS / 2 : KSTEPS, NPROD = STEPS * FM * FN;
  auto product = [&](auto q_c) __attribute__((always_inline)) {
    constexpr int Q = decltype(q_c)::value, KS = Q / (FM * FN), I = Q / FN % FM, J = Q % FN;
    if constexpr (F8) acc[I][J] = mfma_f8_pair<TYPES>(bf[2 * KS][J], bf[2 * KS + 1][J], af[2 * KS][I], af[2 * KS + 1][I], acc[I][J]);
    else acc[I][J] = mfma32<TYPES>(bf[KS][J], af[KS][I], acc[I][J]);
  };

  if constexpr (FEED == FEED_DMA) {
    FA fa;
    FB fb;
    fa.init(g.A, (size_t)g.lda, m0, g.M, lane);
    fb.init(g.B, (size_t)g.ldb, n0, g.N, lane);
    const uint32_t own_addr = (uint32_t)(uintptr_t)own;
    const int cut_slab = g.K % BK ? g.K / BK : -1;   // the slab that the end of K cuts
    constexpr int NC = FA::COPIES + FB::COPIES;
    static_assert((NST - 1) * NC < 64, "vmcnt is a 6-bit counter");
    // copy C of the slab's NC, with the destination set before the first of each operand
    auto one_copy = [&](auto c_c, uint32_t st, const char* sa, const char* sb) __attribute__((always_inline)) {
      constexpr int C = decltype(c_c)::value;
      if constexpr (C == 0) fa.aim(st);
      if constexpr (C == FA::COPIES) fb.aim(st + FA::BYTES);
      if constexpr (C < FA::COPIES) fa.template copy<C>(sa);
      else fb.template copy<C - FA::COPIES>(sb);
    };
    auto copy_slab = [&](uint32_t st, int slab) __attribute__((always_inline)) {
      if (slab == cut_slab) {
        fa.copy_cut(st, slab, g.K - slab * BK, lane);
        fb.copy_cut(st + FA::BYTES, slab, g.K - slab * BK, lane);
      } else {
        const char* const sa = fa.slab_base(slab) - FA::BIAS;
        const char* const sb = fb.slab_base(slab) - FB::BIAS;
        static_for<NC>([&](auto c) { one_copy(c, st, sa, sb); });
      }
    };
    static_for<NST>([&](auto i_c) {
      constexpr int I = decltype(i_c)::value;
      if (I < mine) copy_slab(own_addr + I * P::STAGE, first + I * W);
    });
    int st = 0;
    for (int i = 0; i < mine; i++) {
      const int slab = first + i * W;
      // the slab has landed; those of the stages after it may still be on their way (loads return in order)
      if (NST > 1 && i + NST <= mine) asm volatile("s_waitcnt vmcnt(%0)" : : "i"((NST - 1) * NC) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      char* const stage = own + st * P::STAGE;
      if (slab == cut_slab) {
        fa.zero_cut(stage, g.K - slab * BK, lane);
        fb.zero_cut(stage + FA::BYTES, g.K - slab * BK, lane);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
      }
      const int next = slab + NST * W;
      if constexpr (TYPES == GZ_F32F32F32) {
        // bound by the matrix instructions (64 cycles each, 4 KSTEPS FM FN of them): the reads of a K step pass behind the
        // products of the one before, and the copies go out behind the last read
        read_step(stage, 0);
        static_for<KSTEPS>([&](auto k_c) {
          constexpr int KS = decltype(k_c)::value;
          if constexpr (KS + 1 < KSTEPS) read_step(stage, KS + 1);
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (KS + 1 == KSTEPS) {
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (i + NST < mine) copy_slab(own_addr + st * P::STAGE, next);
          }
          static_for<FM * FN>([&](auto q_c) { product(std::integral_constant<int, KS * FM * FN + decltype(q_c)::value>{}); });
          __builtin_amdgcn_sched_barrier(0);
        });
        st = st + 1 < NST ? st + 1 : 0;
        continue;
      }
      read_slab(stage);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the stage is free: its fragments are in registers
      __builtin_amdgcn_sched_barrier(0);
      if (i + NST < mine && next != cut_slab) {
        const char* const sa = fa.slab_base(next) - FA::BIAS;
        const char* const sb = fb.slab_base(next) - FB::BIAS;
        constexpr int STEP = NPROD > NC ? NPROD / NC : 1, PER = NPROD > NC ? 1 : NC / NPROD;
        static_for<NPROD>([&](auto q_c) {
          constexpr int Q = decltype(q_c)::value;
          product(q_c);
          if constexpr (Q % STEP == 0)
            static_for<PER>([&](auto p_c) {
              constexpr int C = Q / STEP * PER + decltype(p_c)::value;
              if constexpr (C < NC) one_copy(std::integral_constant<int, C>{}, own_addr + st * P::STAGE, sa, sb);
            });
          __builtin_amdgcn_sched_barrier(0);
        });
      } else {
        if (i + NST < mine) copy_slab(own_addr + st * P::STAGE, next);
        static_for<NPROD>([&](auto q_c) { product(q_c); });
      }
      st = st + 1 < NST ? st + 1 : 0;
    }
  } else {
    typename FA::S sa[NST];
    typename FB::S sb[NST];
    const int K = g.K;   // (32 x 32 tiles: never a K part)
    const bool ragged_lines = (!A_KC && m0 + TM > g.M) || (!B_KC && n0 + TN > g.N);
    // (lines shorter than one 16-byte piece are loaded element by element, and a piece of lines shorter than two could
    // reach further than the next line: no slab of those is loaded unconditionally)
    const bool tiny_lines = (A_KC ? g.K : g.M) < 16 / ES || (B_KC ? g.K : g.N) < 16 / ES;
    const bool short_lines = (!A_KC && g.lda < 16) || (!B_KC && g.ldb < 16);
    const int full_slabs = ragged_lines ? (short_lines ? 0 : min((g.K - 1) / BK, K / BK)) : K / BK;
    // this wave's slabs that are loaded unconditionally: its first n_inside.  Their loop knows nothing of the others, whose
    // loads end in merges that wait for them.
    const int n_inside = first < full_slabs ? min(mine, (full_slabs - first + W - 1) / W) : 0;
    auto load_inside = [&](auto s_c, int slab) __attribute__((always_inline)) {
      constexpr int X = decltype(s_c)::value;
      sa[X].load_inside(g.A, g.M, K, m0, slab * BK, lane, (size_t)g.lda);
      sb[X].load_inside(g.B, g.N, K, n0, slab * BK, lane, (size_t)g.ldb);
    };
    auto load_any = [&](auto s_c, int slab) __attribute__((always_inline)) {
      constexpr int X = decltype(s_c)::value;
      if (slab < full_slabs) {
        load_inside(s_c, slab);
      } else if (!tiny_lines) {
        sa[X].load_clamped(g.A, g.M, K, m0, slab * BK, lane, (size_t)g.lda);
        sb[X].load_clamped(g.B, g.N, K, n0, slab * BK, lane, (size_t)g.ldb);
        sa[X].fix(g.M, K, m0, slab * BK, lane);
        sb[X].fix(g.N, K, n0, slab * BK, lane);
      } else {
        sa[X].load(g.A, g.M, K, m0, slab * BK, lane, (size_t)g.lda);
        sb[X].load(g.B, g.N, K, n0, slab * BK, lane, (size_t)g.ldb);
      }
    };
    // (the LDS executes a wave's instructions in order: these stores come behind the reads of the slab before)
    auto park = [&](auto s_c) __attribute__((always_inline)) {
      constexpr int X = decltype(s_c)::value;
      sa[X].store(own, lane);
      sb[X].store(own + FA::BYTES, lane);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    };
    auto multiply = [&]() __attribute__((always_inline)) {
      read_slab(own);
      static_for<NPROD>([&](auto q_c) { product(q_c); });
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    };
    if (n_inside >= NST) {
      static_for<NST>([&](auto x_c) { load_inside(x_c, first + decltype(x_c)::value * W); });
    } else {
      static_for<NST>([&](auto x_c) {
        constexpr int X = decltype(x_c)::value;
        if (X < mine) load_any(x_c, first + X * W);
      });
    }
    int i = 0;
    for (; i + 2 * NST <= n_inside; i += NST)
      static_for<NST>([&](auto x_c) {
        park(x_c);
        load_inside(x_c, first + (i + decltype(x_c)::value + NST) * W);
        multiply();
      });
    for (; i < mine; i += NST)
      static_for<NST>([&](auto x_c) {
        constexpr int X = decltype(x_c)::value;
        if (i + X < mine) {
          park(x_c);
          if (i + X + NST < mine) load_any(x_c, first + (i + X + NST) * W);
          multiply();
        }
      });
  }

  // ---- the waves' sums: each parks its own, unpadded rows of TN values with the 16-byte pieces of row r at p ^ r ----
  typedef acc_t raw4_t __attribute__((ext_vector_type(4)));
  constexpr int PPR = TN / 4, SWZ = PPR - 1;   // pieces per row: 16 or 8
#pragma unroll
  for (int i = 0; i < FM; i++)
#pragma unroll
    for (int j = 0; j < FN; j++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const int row = 32 * i + (lane & 31), piece = 8 * j + 2 * q + (lane >> 5);
        *reinterpret_cast<raw4_t*>(own + row * (TN * 4) + ((piece ^ (row & SWZ)) * 16)) =
            raw4_t{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2], acc[i][j][4 * q + 3]};
      }
  constexpr int PIECES = TM * TN / 4, NT = W * 64, PER = (PIECES + NT - 1) / NT;
  static_assert(PIECES % NT == 0 || PIECES < NT, "the pieces divide over the lanes");
  // (All waves', also those that had no slab and parked zeros: asking first whether a wave had one put a branch and a wait
  // into every LDS read.  us, with / without: bf16 512^2 x 256 64 x 64 tiles 4.7 / 4.3, x 768 6.6 / 6.2, 32 x 32 3.9 / 3.7)
  auto sum_of = [&](int row, int piece) -> raw4_t {
    const char* const p = lds + row * (TN * 4) + ((piece ^ (row & SWZ)) * 16);
    raw4_t s = *reinterpret_cast<const raw4_t*>(p);
#pragma unroll
    for (int w = 1; w < W; w++) {
      const raw4_t v = *reinterpret_cast<const raw4_t*>(p + w * P::WAVE_BYTES);
#pragma unroll
      for (int e = 0; e < 4; e++) s[e] += v[e];
    }
    return s;
  };
  if (sk.parts > 1) {
    // 32 x 32 blocks of a tile in row order, a block's pieces in the order [column group of 8][half][row]: whole lines
    __syncthreads();
    raw4_t* const out = reinterpret_cast<raw4_t*>(sk.ws) + (size_t)slot * PIECES;
#pragma unroll
    for (int it = 0; it < PER; it++) {
      const int p = it * NT + tid;
      if (PIECES < NT && p >= PIECES) break;
      const int blk = p / 256, r = p % 32, c = p % 256 / 32;   // c: column group of four within the block
      const int row = blk / FN * 32 + r, piece = blk % FN * 8 + c;
      if (m0 + blk / FN * 32 < g.M && n0 + blk % FN * 32 < g.N) out[p] = sum_of(row, piece);
    }
    return;
  }
  const size_t LDC = (size_t)g.ldc, LDD = (size_t)g.ldd;
  const bool use_c = g.beta != 0;
  constexpr uintptr_t VEC_ALIGN = 4 * sizeof(out_t) - 1;
  // rows of C and D that are whole aligned groups of four: vectors; otherwise the lanes take one column each
  const bool vec = (g.N & 3) == 0 && (LDD & 3) == 0 && (!use_c || (LDC & 3) == 0) &&
                   ((reinterpret_cast<uintptr_t>(g.D) | (use_c ? reinterpret_cast<uintptr_t>(g.C) : 0)) & VEC_ALIGN) == 0;
  if (vec) {
    out_t cv[PER][4];
#pragma unroll
    for (int it = 0; it < PER; it++) {   // C before the barrier, from clamped addresses
      const int p = it * NT + tid, m = min(m0 + p / PPR % TM, g.M - 1), n = min(n0 + p % PPR * 4, g.N - 4);
#pragma unroll
      for (int e = 0; e < 4; e++) cv[it][e] = 0;
      if (use_c) __builtin_memcpy(cv[it], g.C + (size_t)m * LDC + n, sizeof(cv[it]));
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < PER; it++) {
      const int p = it * NT + tid, row = p / PPR, m = m0 + row, n = n0 + p % PPR * 4;
      if (PIECES < NT && p >= PIECES) break;
      const raw4_t s = sum_of(row, p % PPR);
      out_t dv[4];
#pragma unroll
      for (int e = 0; e < 4; e++) dv[e] = epilogue<TYPES>(s[e], g.alpha, g.beta, &cv[it][e]);
      if (m < g.M && n < g.N) __builtin_memcpy(g.D + (size_t)m * LDD + n, dv, sizeof(dv));
    }
  } else {
    // Four values of a lane at a time, LDS reads and loads of C from clamped places before the guarded stores.  (One value after
    // the other, bf16 512 x 514 x 256: 64 x 64 tiles 7.1 us, now 5.4, 32 x 32 3.7 and 3.6; 1000 x 1030 x 768 10.3 and 8.6, 10.6 and
    // 9.1.)
    __syncthreads();
    constexpr int VALUES = TM * TN, PASS = VALUES / NT < 4 ? VALUES / NT : 4;
    static_assert(VALUES % (NT * PASS) == 0, "the values divide over the lanes");
    for (int v0 = tid; v0 < VALUES; v0 += NT * PASS) {
      acc_t sums[PASS];
      out_t c[PASS];
#pragma unroll
      for (int e = 0; e < PASS; e++) {
        const int row = (v0 + e * NT) / TN, col = (v0 + e * NT) % TN;
        const char* const p = lds + row * (TN * 4) + (((col / 4) ^ (row & SWZ)) * 16) + col % 4 * 4;
        sums[e] = *reinterpret_cast<const acc_t*>(p);
#pragma unroll
        for (int w = 1; w < W; w++) sums[e] += *reinterpret_cast<const acc_t*>(p + w * P::WAVE_BYTES);
        c[e] = 0;
        if (use_c) c[e] = g.C[(size_t)min(m0 + row, g.M - 1) * LDC + min(n0 + col, g.N - 1)];
      }
#pragma unroll
      for (int e = 0; e < PASS; e++) {
        const int m = m0 + (v0 + e * NT) / TN, n = n0 + (v0 + e * NT) % TN;
        const out_t d = epilogue<TYPES>(sums[e], g.alpha, g.beta, &c[e]);
        if (m < g.M && n < g.N) g.D[(size_t)m * LDD + n] = d;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Launchers
// ---------------------------------------------------------------------------
template <int TYPES, int TM, int TN, int W, int NST, int RES, int FEED>
static int launch_wavek_as(const GemmArgs<TYPES>& g, const SplitK& sk, hipStream_t s) {
  const int tiles_m = ceil_div(g.M, TM), tiles_n = ceil_div(g.N, TN);
  const dim3 grid((unsigned)(tiles_m * tiles_n * sk.parts)), block(W * 64);
  const bool a_kc = g.layoutA == GZ_ROW_MAJOR, b_kc = g.layoutB == GZ_COL_MAJOR;
#define GZ_LAUNCH_WAVEK(AKC, BKC)                                                        \
  do {                                                                                   \
    constexpr size_t lds = (size_t)WaveK<TYPES, TM, TN, W, NST, FEED, AKC, BKC>::LDS_BYTES; \
    auto kern = mfma_wavek_kernel<TYPES, TM, TN, W, NST, RES, FEED, AKC, BKC>;           \
    GZ_SET_LDS_LIMIT(kern, lds);                                                         \
    hipLaunchKernelGGL(kern, grid, block, lds, s, g, tiles_m, tiles_n, sk);              \
  } while (0)
  if (a_kc && b_kc) GZ_LAUNCH_WAVEK(true, true);
  else if (a_kc) GZ_LAUNCH_WAVEK(true, false);
  else if (b_kc) GZ_LAUNCH_WAVEK(false, true);
  else GZ_LAUNCH_WAVEK(false, false);
#undef GZ_LAUNCH_WAVEK
  GZ_HIP_TRY(hipGetLastError());
  return GZ_OK;
}

// Tiles of 64 x 64 (four waves, aligned lines; mfma_wavek_stages) or 32 x 32 (eight).
template <int TYPES> int launch_wavek(const GemmArgs<TYPES>& g, int tile, const SplitK& sk, hipStream_t s) {
  if (tile == 32)
    return wavek_dma_ok<TYPES>(g) ? launch_wavek_as<TYPES, 32, 32, 8, 1, 2, FEED_DMA>(g, sk, s)
                                  : launch_wavek_as<TYPES, 32, 32, 8, 1, 2, FEED_REG>(g, sk, s);
  if constexpr (TYPES != GZ_F32F32F32) {
    const long long groups = (long long)ceil_div(g.M, 64) * ceil_div(g.N, 64) * sk.parts;
    return mfma_wavek_stages(groups, device_compute_units(), MFMA_LDS_PER_CU) == 1 ? launch_wavek_as<TYPES, 64, 64, 4, 1, 2, FEED_DMA>(g, sk, s)
                                                                                   : launch_wavek_as<TYPES, 64, 64, 4, 2, 1, FEED_DMA>(g, sk, s);
  }
  set_error("mfma rung: no 64 x 64 tile with its K dealt to the waves for this type bundle");
  return GZ_ERR_UNSUPPORTED;
}

}  // namespace gz
