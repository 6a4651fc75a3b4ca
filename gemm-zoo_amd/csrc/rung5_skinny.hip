// Rung 5: weight-streaming kernels for decode-shaped problems (M <= 128).
//
// The weight matrix B (N x K, K contiguous) is read exactly once and nothing about it is reused by another
// wave, so the kernel is a streaming read of B with a little matrix-core work attached.  What decides its
// speed on MI355X (measured):
//   * a compute unit sustains only a limited number of outstanding memory requests, so the chip's bandwidth is
//     reached only when every compute unit streams its equal share: the columns are dealt out in equal
//     groups of at most 32, 4-column granular, one or two groups per compute unit (cols_per_wg);
//   * rows of B are a multiple of 4 KiB apart for the usual K, so work-groups that walk K in step all hit the
//     same L2 / memory channel at the same moment: every work-group starts at a different K chunk (rot);
//   * each byte is used once: the copies carry the non-temporal hint.
//
// Element types: the 16-bit floats, int8 and the 8-bit floats.  The kernels work on bytes of K - a fragment is 16 bytes
// per lane whatever the type - and take any K that is whole 16-byte pieces: the last chunk or stage of a row moves the
// pieces that exist, and the rest counts as zeros on both operands.
//
// skinny_dtl_kernel (M <= 16): a work-group of KS waves owns up to 32 columns; its waves take the 256-byte
// K chunks round-robin.  A wave moves its chunk of the 4 NCP rows from global memory straight
// into a private LDS ring with global_load_lds_dwordx4 -- every instruction moves four 256-byte row pieces --
// and reads the MFMA fragments back with ds_read_b128; the 16-byte pieces of a row are XOR-swizzled with the
// row number on the way in, so the reads are bank-conflict free.  There is no barrier in the main loop and
// S stages are in flight per wave; the waits are hand-counted (the compiler does not see LDS-DMA).  The K
// partial sums of the KS waves meet in LDS at the end.  Activations (at most 16 rows) come from L2 into
// registers with the same depth.  A narrow share of columns moves little per stage, so it gets more waves and more
// stages (skinny_dtl_shape): what a compute unit has in flight stays near 128 KiB.
//
// stream_wide_kernel + stream_wide_reduce_kernel (16-bit types, 64 < M <= 128, K >= 8192, K % 64 == 0): stream_tile_kernel with column blocks of
// up to 256 columns and K split in two or four parts, so that a compute unit pulls a part of A instead of all of it;
// the parts meet in a workspace and a second launch adds them in a fixed order (gz_skinny_cfg.hpp says when).
//
// stream_tile_kernel (16 < M <= 128): here the activations no longer fit a wave's registers and every
// compute unit needs all of them, so they are shared through LDS.  One work-group per compute unit owns up to 64
// columns.  Four producer waves move stage after stage (128 bytes of K: A rows and B rows, swizzled)
// into a ring with direct-to-LDS copies; four consumer waves read the fragments and run the 32x32 instructions.
// Splitting the roles matters: a copy instruction occupies its wave for about 55 cycles however many lanes it
// moves, and with one wave per SIMD doing both jobs the copy issue, the LDS reads and the MFMAs of a stage ran
// back to back.  One barrier per stage says both "stage i has landed" and "stage i - 1 may be overwritten".
//
// (both kernels: the weight fragment is the first operand, so a lane ends with 4 consecutive
// columns of one output row.)
#include "gz_common.hpp"
#include <type_traits>
#include <utility>

#include "gz_skinny_cfg.hpp"

namespace gz {

typedef __bf16 sk_bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 sk_f16x8_t __attribute__((ext_vector_type(8)));
typedef float sk_f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t sk_u32x4_t __attribute__((ext_vector_type(4)));
typedef float sk_f32x16_t __attribute__((ext_vector_type(16)));

typedef int sk_i32x4_t __attribute__((ext_vector_type(4)));
typedef int sk_i32x8_t __attribute__((ext_vector_type(8)));
typedef int sk_i32x16_t __attribute__((ext_vector_type(16)));

template <int TYPES> struct SkAcc { using v4 = sk_f32x4_t; using v16 = sk_f32x16_t; };
template <> struct SkAcc<GZ_S8S8S32> { using v4 = sk_i32x4_t; using v16 = sk_i32x16_t; };

// `n` consecutive 16-byte K fragments of the weights (first operand) and of the activations.  A lane's 16 bytes are 8 or
// 16 elements of K, and which k they stand for is the same on both operands, which is all a dot product needs: so the
// 8-bit floats put two fragments side by side for v_mfma_f32_*_f8f6f4, which takes 32 bytes per lane.
template <int TYPES, int NF>
__device__ __forceinline__ void mfma16_run(const sk_u32x4_t (&first)[NF], const sk_u32x4_t (&second)[NF], typename SkAcc<TYPES>::v4& acc) {
  if constexpr (is_fp8(TYPES)) {
    constexpr int FMT = TYPES == GZ_E5M2E5M2F16 ? 1 : 0;
    static_assert(NF % 2 == 0, "fragments in pairs");
#pragma unroll
    for (int t = 0; t < NF; t += 2) {
      const sk_i32x8_t f = __builtin_shufflevector(__builtin_bit_cast(sk_i32x4_t, first[t]), __builtin_bit_cast(sk_i32x4_t, first[t + 1]), 0, 1, 2, 3, 4, 5, 6, 7);
      const sk_i32x8_t s = __builtin_shufflevector(__builtin_bit_cast(sk_i32x4_t, second[t]), __builtin_bit_cast(sk_i32x4_t, second[t + 1]), 0, 1, 2, 3, 4, 5, 6, 7);
      acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(f, s, acc, FMT, FMT, 0, 0, 0, 0);
    }
  } else {
#pragma unroll
    for (int t = 0; t < NF; t++) {
      if constexpr (TYPES == GZ_S8S8S32)
        acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(sk_i32x4_t, first[t]), __builtin_bit_cast(sk_i32x4_t, second[t]), acc, 0, 0, 0);
      else if constexpr (TYPES == GZ_F16F16F16)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(sk_f16x8_t, first[t]), __builtin_bit_cast(sk_f16x8_t, second[t]), acc, 0, 0, 0);
      else
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(sk_bf16x8_t, first[t]), __builtin_bit_cast(sk_bf16x8_t, second[t]), acc, 0, 0, 0);
    }
  }
}

// one fragment pair of 32 rows each (not the 8-bit floats)
template <int TYPES>
__device__ inline typename SkAcc<TYPES>::v16 mfma32x16(sk_u32x4_t first, sk_u32x4_t second, typename SkAcc<TYPES>::v16 acc) {
  if constexpr (TYPES == GZ_S8S8S32)
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(sk_i32x4_t, first), __builtin_bit_cast(sk_i32x4_t, second), acc, 0, 0, 0);
  else if constexpr (TYPES == GZ_F16F16F16)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(sk_f16x8_t, first), __builtin_bit_cast(sk_f16x8_t, second), acc, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(sk_bf16x8_t, first), __builtin_bit_cast(sk_bf16x8_t, second), acc, 0, 0, 0);
}
template <int TYPES>
__device__ inline sk_f32x16_t mfma32x64_f8(sk_u32x4_t f0, sk_u32x4_t f1, sk_u32x4_t s0, sk_u32x4_t s1, sk_f32x16_t acc) {
  constexpr int FMT = TYPES == GZ_E5M2E5M2F16 ? 1 : 0;
  const sk_i32x8_t f = __builtin_shufflevector(__builtin_bit_cast(sk_i32x4_t, f0), __builtin_bit_cast(sk_i32x4_t, f1), 0, 1, 2, 3, 4, 5, 6, 7);
  const sk_i32x8_t s = __builtin_shufflevector(__builtin_bit_cast(sk_i32x4_t, s0), __builtin_bit_cast(sk_i32x4_t, s1), 0, 1, 2, 3, 4, 5, 6, 7);
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(f, s, acc, FMT, FMT, 0, 0, 0, 0);
}

// ---------------------------------------------------------------------------------------------------------
// Direct-to-LDS streaming kernel
// ---------------------------------------------------------------------------------------------------------
template <class F, int... I> __device__ __forceinline__ void sk_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F> __device__ __forceinline__ void sk_for(F&& f) {
  sk_for_impl(f, std::make_integer_sequence<int, N>{});
}
template <int OFF> __device__ __forceinline__ void sk_ds_read16(sk_u32x4_t& dst, uint32_t addr) {
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "i"(OFF));
}
template <int OFF> __device__ __forceinline__ void sk_ds_zero16(uint32_t addr) {
  const sk_u32x4_t z = {0, 0, 0, 0};
  asm volatile("ds_write_b128 %0, %1 offset:%2" : : "v"(addr), "v"(z), "i"(OFF) : "memory");
}
__device__ __forceinline__ void sk_set_m0(uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" : : "s"(lds_addr) : "memory");
}
// 64 lanes x 16 bytes, global (sbase + voff + OFF) -> LDS (M0 + OFF + 16 * lane); lanes outside `mask` move nothing
// but the instruction still takes its place in the vmcnt order
template <int OFF> __device__ __forceinline__ void sk_copy16(uint32_t voff, const void* sbase_minus_off, uint64_t mask) {
  static_assert(OFF >= -4096 && OFF <= 4095, "13-bit signed immediate");
  asm volatile("s_mov_b64 exec, %3\n\tglobal_load_lds_dwordx4 %0, %1 offset:%2 nt\n\ts_mov_b64 exec, -1"
               :
               : "v"(voff), "s"(sbase_minus_off), "i"(OFF), "s"(mask)
               : "memory");
}
// the same without the non-temporal hint (activations are re-read by every compute unit: keep them in L2)
template <int OFF>
__device__ __forceinline__ void sk_copy16_keep(uint32_t voff, const void* sbase_minus_off, uint64_t mask) {
  static_assert(OFF >= -4096 && OFF <= 4095, "13-bit signed immediate");
  asm volatile("s_mov_b64 exec, %3\n\tglobal_load_lds_dwordx4 %0, %1 offset:%2\n\ts_mov_b64 exec, -1"
               :
               : "v"(voff), "s"(sbase_minus_off), "i"(OFF), "s"(mask)
               : "memory");
}
// every lane
template <int OFF> __device__ __forceinline__ void sk_copy16_all(uint32_t voff, const void* sbase) {
  static_assert(OFF >= -4096 && OFF <= 4095, "13-bit signed immediate");
  asm volatile("global_load_lds_dwordx4 %0, %1 offset:%2" : : "v"(voff), "s"(sbase), "i"(OFF) : "memory");
}
template <int OFF> __device__ __forceinline__ void sk_load16(sk_u32x4_t& dst, uint32_t voff, const void* sbase) {
  asm volatile("global_load_dwordx4 %0, %1, %2 offset:%3" : "=&v"(dst) : "v"(voff), "s"(sbase), "i"(OFF) : "memory");
}
template <int N> __device__ __forceinline__ void sk_wait_vm() { asm volatile("s_waitcnt vmcnt(%0)" : : "i"(N) : "memory"); }
__device__ __forceinline__ void sk_wait_lgkm0() { asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory"); }
template <int N> __device__ __forceinline__ void sk_wait_lgkm() {
  static_assert(N >= 0 && N <= 15, "lgkmcnt is a 4-bit counter");
  asm volatile("s_waitcnt lgkmcnt(%0)" : : "i"(N) : "memory");
}
// orders later uses of a register after the asm statements that precede this one
__device__ __forceinline__ void sk_touch(sk_u32x4_t& v) { asm volatile("" : "+v"(v)); }

// SHORT: K is not whole chunks, the last one moves the pieces that exist.  An instance of its own: asking in every chunk
// cost 1 - 3 % (bf16 13 x 4224 x 6144 12.7 / 13.1 us), and two forms of the copies in one loop a quarter.
template <int TYPES, int NCP, int KS, int S, bool SHORT>
__global__ void __launch_bounds__(KS * 64) skinny_dtl_kernel(GemmArgs<TYPES> g, int cols_per_wg) {
  using T = Traits<TYPES>;
  using out_t = typename T::out_t;
  using acc_t = typename T::acc_t;
  extern __shared__ __attribute__((aligned(1024))) char sk_lds[];
  constexpr int ES = sizeof(typename T::in_t);
  constexpr int MBLK = 1;
  constexpr int CB = NCP > 4 ? 2 : 1;            // 16-column MFMA blocks per work-group
  constexpr int STAGE = NCP * 1024;              // 4 NCP rows x 256 bytes, NCP copies of 4 rows each
  constexpr int PER = NCP + 4 * MBLK;            // vector-memory instructions per stage
  constexpr int NA = MBLK * CB;
  static_assert((S - 1) * PER < 64, "vmcnt is a 6-bit counter");
  const uint32_t lds_base = (uint32_t)(uintptr_t)sk_lds;
  const int lane = threadIdx.x & 63;
  const int ks = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n_base = blockIdx.x * cols_per_wg;
  const int N = g.N, M = g.M;
  const uint32_t Kb = (uint32_t)g.K * ES;        // a multiple of 16 (the launcher checks)
  const uint32_t ring = lds_base + ks * (S * STAGE);
  const size_t rowb = (size_t)g.ldb * ES, rowb_a = (size_t)g.lda * ES;   // bytes between the columns of B and the rows of A

  // copy j moves rows 4j .. 4j+3 of the group: 16 lanes per row; the lane that fills position p of the LDS row
  // fetches piece p ^ (row & 15) of the 256-byte chunk.  The offsets stay below 2^32: a work-group's columns times
  // the pitch of B, the rows of A times its pitch (the launcher checks both).
  uint32_t voff[NCP];
#pragma unroll
  for (int j = 0; j < NCP; j++) {
    const int row = 4 * j + (lane >> 4), p = lane & 15;
    const int n = min(n_base + row, N - 1);
    voff[j] = (uint32_t)((size_t)(n - n_base) * rowb) + (uint32_t)((p ^ (row & 15)) * 16);
  }
  const char* sb = reinterpret_cast<const char*>(g.B) + (size_t)n_base * rowb;
  const int r16 = lane & 15, grp = lane >> 4;
  uint32_t a_row[MBLK];
#pragma unroll
  for (int mb = 0; mb < MBLK; mb++) a_row[mb] = (uint32_t)((size_t)min(mb * 16 + r16, M - 1) * rowb_a) + (SHORT ? 0 : grp * 16);
  const char* sa = reinterpret_cast<const char*>(g.A);
  // fragment of MFMA step t: row r16 of a column block, K piece 4t + grp.  (Fewer than 16 columns: the rows past the
  // stage are whatever lies behind it in LDS; they only reach columns that are not stored.)
  uint32_t b_addr[4];
#pragma unroll
  for (int t = 0; t < 4; t++) b_addr[t] = ring + r16 * 256 + (((t * 4 + grp) ^ r16) * 16);

  typename SkAcc<TYPES>::v4 acc[MBLK][CB];
#pragma unroll
  for (int mb = 0; mb < MBLK; mb++)
#pragma unroll
    for (int cb = 0; cb < CB; cb++)
#pragma unroll
      for (int e = 0; e < 4; e++) acc[mb][cb][e] = 0;
  sk_u32x4_t aq[S][MBLK][4];

  const int chunks = (int)((Kb + 255) / 256);
  const int mine = (chunks - ks + KS - 1) / KS;          // this wave's chunks: ks, ks + KS, ... (before rotation)
  const int rot = (int)(blockIdx.x % (unsigned)chunks);

  auto chunk_byte = [&](int i) {
    int c = i * KS + ks + rot;
    if (c >= chunks) c -= chunks;
    return (uint32_t)c * 256;
  };
  auto issue_copies = [&](auto slot_c, int i) {
    constexpr int SL = decltype(slot_c)::value;
    const uint32_t kbyte = chunk_byte(i);
    sk_for<(NCP + 3) / 4>([&](auto q_c) {
      constexpr int Q = decltype(q_c)::value;  // four copies share one M0
      sk_set_m0(ring + SL * STAGE + Q * 4096 + 2048);
      sk_for<(NCP < 4 ? NCP : 4)>([&](auto j_c) {
        constexpr int J = decltype(j_c)::value;
        // cols_per_wg is a multiple of 4: a copy moves four whole rows or nothing; of a last, shorter chunk only the
        // pieces that exist
        const uint32_t on = (uint32_t)__builtin_amdgcn_readfirstlane(4 * (Q * 4 + J) < cols_per_wg ? -1 : 0);
        uint64_t mask = ((uint64_t)on << 32) | on;
        if constexpr (SHORT)
          mask &= __builtin_amdgcn_ballot_w64((uint32_t)(((lane & 15) ^ ((4 * J + (lane >> 4)) & 15)) * 16) < Kb - kbyte);
        sk_copy16<(J - 2) * 1024>(voff[Q * 4 + J], sb + kbyte - (J - 2) * 1024, mask);
      });
    });
  };
  auto issue_a = [&](auto slot_c, int i) {
    constexpr int SL = decltype(slot_c)::value;
    const uint32_t kbyte = chunk_byte(i);
    sk_for<MBLK>([&](auto mb_c) {
      constexpr int MB = decltype(mb_c)::value;
      sk_for<4>([&](auto t_c) {
        constexpr int TT = decltype(t_c)::value;
        if constexpr (SHORT) {   // (a piece past the end: the row's first, zeroed below)
          const uint32_t k = kbyte + TT * 64 + grp * 16;
          sk_load16<0>(aq[SL][MB][TT], a_row[MB] + (k < Kb ? k : 0u), sa);
        } else {
          sk_load16<TT * 64>(aq[SL][MB][TT], a_row[MB], sa + kbyte);
        }
      });
    });
  };

  sk_for<S>([&](auto sl) {
    if (decltype(sl)::value < mine) {
      issue_copies(sl, decltype(sl)::value);
      issue_a(sl, decltype(sl)::value);
    }
  });

  for (int i0 = 0; i0 < mine; i0 += S) {
    sk_for<S>([&](auto sl) {
      constexpr int SL = decltype(sl)::value;
      const int i = i0 + SL;
      if (i < mine) {
        // stage i has landed once at most the S - 1 younger stages are outstanding
        if (i + S - 1 < mine) sk_wait_vm<(S - 1) * PER>();
        else sk_wait_vm<0>();
        sk_u32x4_t bf[CB][4];
        sk_for<CB>([&](auto cb_c) {
          constexpr int CBI = decltype(cb_c)::value;
          sk_for<4>([&](auto t_c) {
            constexpr int TT = decltype(t_c)::value;
            sk_ds_read16<SL * STAGE + CBI * 4096>(bf[CBI][TT], b_addr[TT]);
          });
        });
        sk_wait_lgkm0();
#pragma unroll
        for (int cb = 0; cb < CB; cb++)
#pragma unroll
          for (int t = 0; t < 4; t++) sk_touch(bf[cb][t]);
#pragma unroll
        for (int mb = 0; mb < MBLK; mb++)
#pragma unroll
          for (int t = 0; t < 4; t++) sk_touch(aq[SL][mb][t]);
        const bool more = i + S < mine;
        if (more) issue_copies(sl, i + S);  // the fragments are in registers: the stage buffer is free
        const uint32_t left = Kb - chunk_byte(i);
        if (SHORT && left < 256) {
          // pieces past the end of K count as zeros on both sides (what is left in LDS may be NaN or infinite)
#pragma unroll
          for (int t = 0; t < 4; t++) {
            const bool exists = (uint32_t)((t * 4 + grp) * 16) < left;
#pragma unroll
            for (int e = 0; e < 4; e++) {
#pragma unroll
              for (int mb = 0; mb < MBLK; mb++) aq[SL][mb][t][e] = exists ? aq[SL][mb][t][e] : 0u;
#pragma unroll
              for (int cb = 0; cb < CB; cb++) bf[cb][t][e] = exists ? bf[cb][t][e] : 0u;
            }
          }
        }
#pragma unroll
        for (int mb = 0; mb < MBLK; mb++)
#pragma unroll
          for (int cb = 0; cb < CB; cb++) mfma16_run<TYPES, 4>(bf[cb], aq[SL][mb], acc[mb][cb]);
        if (more) issue_a(sl, i + S);
      }
    });
  }

  // every wave has waited for all of its copies (the last stages wait with vmcnt(0)): the rings can be reused
  acc_t* red = reinterpret_cast<acc_t*>(sk_lds);
  if constexpr (KS > 1) {
    __syncthreads();
#pragma unroll
    for (int mb = 0; mb < MBLK; mb++)
#pragma unroll
      for (int cb = 0; cb < CB; cb++)
#pragma unroll
        for (int e = 0; e < 4; e++) red[((ks * NA + mb * CB + cb) * 4 + e) * 64 + lane] = acc[mb][cb][e];
    __syncthreads();
    if (ks != 0) return;
#pragma unroll
    for (int w = 1; w < KS; w++)
#pragma unroll
      for (int mb = 0; mb < MBLK; mb++)
#pragma unroll
        for (int cb = 0; cb < CB; cb++)
#pragma unroll
          for (int e = 0; e < 4; e++) acc[mb][cb][e] += red[((w * NA + mb * CB + cb) * 4 + e) * 64 + lane];
  }

  // acc[mb][cb][v] = D(16 mb + r16, n_base + 16 cb + 4 grp + v)
  const int n_end = min(n_base + cols_per_wg, N);
  const bool vec_ok = (g.ldd % 4 == 0) && (g.beta == 0 || g.ldc % 4 == 0) && ((reinterpret_cast<uintptr_t>(g.D) & 15u) == 0) &&
                      (g.beta == 0 || (reinterpret_cast<uintptr_t>(g.C) & 15u) == 0);
#pragma unroll
  for (int mb = 0; mb < MBLK; mb++) {
    const int m = mb * 16 + r16;
    if (m >= M) continue;
#pragma unroll
    for (int cb = 0; cb < CB; cb++) {
      const int n = n_base + cb * 16 + 4 * grp;
      const size_t o = (size_t)m * (size_t)g.ldd + n, oc = (size_t)m * (size_t)g.ldc + n;
      if (vec_ok && n + 3 < n_end) {
        out_t cv[4] = {0, 0, 0, 0}, dv[4];
        if (g.beta != 0) __builtin_memcpy(cv, g.C + oc, sizeof(cv));
#pragma unroll
        for (int e = 0; e < 4; e++) dv[e] = epilogue<TYPES>(acc[mb][cb][e], g.alpha, g.beta, &cv[e]);
        __builtin_memcpy(g.D + o, dv, sizeof(dv));
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (n + e < n_end) g.D[o + e] = epilogue<TYPES>(acc[mb][cb][e], g.alpha, g.beta, g.C + oc + e);
      }
    }
  }
}


// ---------------------------------------------------------------------------------------------------------
// Producer / consumer streaming tile kernel, 16 < M <= 128
//   LDS ring: S stages of [A: 32 MB32 rows | B: 64 rows] x 128 bytes; piece p (16 bytes) of tile row r sits at
//   position p ^ ((r >> 1) & 7), which makes the 32-row fragment reads bank-conflict free.
//   Consumer wave w: column block w & 1; MB32 >= 2: row group w >> 1 (MB32 / 2 blocks of 32 rows), all four
//   k-steps of a stage; MB32 == 1: the wave pairs split the k-steps and add their sums through LDS at the end.
// ---------------------------------------------------------------------------------------------------------
template <int TYPES, int MB32, int S>
__global__ void __launch_bounds__(STREAM_TILE_THREADS) stream_tile_kernel(GemmArgs<TYPES> g, int cols_per_wg) {
  constexpr int NCW = 4;  // consumer waves; the four producer waves follow
  using T = Traits<TYPES>;
  using out_t = typename T::out_t;
  using acc_t = typename T::acc_t;
  constexpr int ES = sizeof(typename T::in_t);
  extern __shared__ __attribute__((aligned(1024))) char sk_lds[];
  constexpr int RB = STREAM_TILE_ROW_BYTES, B_BYTES = STREAM_TILE_COLS * RB, A_ROWS = MB32 * 32, A_BYTES = A_ROWS * RB, STAGE = A_BYTES + B_BYTES;
  constexpr int NA = MB32, NB = 2, NCP = NA + NB;      // copies per producer wave and stage
  // NCW consumer waves: 2 column blocks x NRG row groups x KSPLIT shares of the 4 MFMA k-steps of a stage
  constexpr int NRG = MB32 >= 2 ? 2 : 1, NRB = MB32 / NRG, KSPLIT = NCW / (2 * NRG), NT = 4 / KSPLIT;
  static_assert(KSPLIT >= 1 && NT >= 1, "");
  static_assert(MB32 == 1 || MB32 == 2 || MB32 == 4, "");
  static_assert((S - 2) * NCP < 64, "vmcnt");
  const uint32_t lds_base = (uint32_t)(uintptr_t)sk_lds;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int N = g.N, M = g.M;
  const int n_base = blockIdx.x * cols_per_wg;
  const int n_end = min(n_base + cols_per_wg, N);
  const size_t rowb = (size_t)g.ldb * ES, rowb_a = (size_t)g.lda * ES;   // bytes between the columns of B and the rows of A
  const uint32_t Kb = (uint32_t)g.K * ES;                       // a multiple of 16 (the launcher checks)
  const int nst = (int)((Kb + RB - 1) / RB);
  const uint32_t last = Kb - (uint32_t)(nst - 1) * RB;           // bytes per row of the last stage
  const int rot = (int)(blockIdx.x % (unsigned)nst);

  if (wave >= NCW) {
    // ---------------- producers: wave p moves A rows [8 NA p, 8 NA (p+1)) and B rows [16 (3 - p), 16 (3 - p) + 16) of every stage,
    // eight rows per copy.  Copies of rows that do not exist - past M, past the work-group's columns - are not issued
    // at all: a copy occupies its wave and the compute unit's address path whether or not its lanes move anything.
    const int p = wave - NCW;
    const int row_in = lane >> 3, pos = lane & 7;
    const int a_row0 = p * NA * 8, b_row0 = (NCW - 1 - p) * NB * 8;
    // per-lane offsets with the copy's own share of the immediate taken off and a bias, taken off the base, that keeps
    // them non-negative: the copies of an operand in a stage share one scalar base
    constexpr uint32_t BIAS = 4096;
    uint32_t voffA[NA], voffB[NB];
    uint64_t maskB[NB], lastA[NA], lastB[NB];   // lanes that move something: of any stage, and of the last one (shorter rows)
#pragma unroll
    for (int j = 0; j < NA; j++) {
      const int row = a_row0 + j * 8 + row_in;
      const uint32_t piece = (uint32_t)((pos ^ ((row >> 1) & 7)) * 16);
      voffA[j] = (uint32_t)((size_t)min(row, M - 1) * rowb_a) + piece + BIAS - (j - 2) * 1024;
      lastA[j] = __builtin_amdgcn_ballot_w64(piece < last);
    }
#pragma unroll
    for (int j = 0; j < NB; j++) {
      const int row = b_row0 + j * 8 + row_in;
      const int n = min(n_base + row, N - 1);
      const uint32_t piece = (uint32_t)((pos ^ ((row >> 1) & 7)) * 16);
      voffB[j] = (uint32_t)((size_t)(n - n_base) * rowb) + piece + BIAS - (j - 2) * 1024;
      maskB[j] = __builtin_amdgcn_ballot_w64(n_base + row < n_end);
      lastB[j] = maskB[j] & __builtin_amdgcn_ballot_w64(piece < last);
    }
    const char* sA = reinterpret_cast<const char*>(g.A) - BIAS;
    const char* sB = reinterpret_cast<const char*>(g.B) + (size_t)n_base * rowb - BIAS;
    const uint32_t dstA = lds_base + a_row0 * RB + 2048, dstB = lds_base + A_BYTES + b_row0 * RB + 2048;
    const int na = __builtin_amdgcn_readfirstlane(max(0, min(NA, (M - a_row0 + 7) / 8)));
    const int nb = __builtin_amdgcn_readfirstlane(max(0, min(NB, (n_end - n_base - b_row0 + 7) / 8)));
    auto produce = [&](auto na_c, auto nb_c) {
      constexpr int CA = decltype(na_c)::value, CB = decltype(nb_c)::value;   // copies of this wave per stage
      uint32_t so = 0;
      int s = 0, c = rot;
      auto issue = [&]() {
        const char *pa = sA + (size_t)c * RB, *pb = sB + (size_t)c * RB;
        if (s < nst && (c < nst - 1 || last == RB)) {
          if constexpr (CA > 0) sk_set_m0(dstA + so);
          sk_for<CA>([&](auto j_c) {
            constexpr int J = decltype(j_c)::value;
            sk_copy16_all<(J - 2) * 1024>(voffA[J], pa);
          });
          if constexpr (CB > 0) sk_set_m0(dstB + so);
          sk_for<CB>([&](auto j_c) {
            constexpr int J = decltype(j_c)::value;
            sk_copy16<(J - 2) * 1024>(voffB[J], pb, maskB[J]);
          });
        } else {   // the shorter last chunk of the rows, or a stage past the end: every copy masked off but still counted
          const uint64_t any = __builtin_amdgcn_ballot_w64(s < nst);
          if constexpr (CA > 0) sk_set_m0(dstA + so);
          sk_for<CA>([&](auto j_c) {
            constexpr int J = decltype(j_c)::value;
            sk_copy16_keep<(J - 2) * 1024>(voffA[J], pa, any & lastA[J]);
          });
          if constexpr (CB > 0) sk_set_m0(dstB + so);
          sk_for<CB>([&](auto j_c) {
            constexpr int J = decltype(j_c)::value;
            sk_copy16<(J - 2) * 1024>(voffB[J], pb, any & lastB[J]);
          });
        }
        so = so + STAGE == S * STAGE ? 0 : so + STAGE;
        s++;
        c = c + 1 == nst ? 0 : c + 1;
      };
      for (int i = 0; i < S - 1; i++) issue();
      for (int i = 0; i < nst; i++) {
        sk_wait_vm<(S - 2) * (CA + CB)>();           // stage i has landed
        asm volatile("s_barrier" ::: "memory");     // consumers are done with stage i - 1
        issue();
      }
      sk_wait_vm<0>();
    };
    auto with_a = [&](auto na_c) {
      if (nb == 0) produce(na_c, std::integral_constant<int, 0>{});
      else if (nb == 1) produce(na_c, std::integral_constant<int, 1>{});
      else produce(na_c, std::integral_constant<int, 2>{});
    };
    sk_for<NA + 1>([&](auto na_c) {
      if (na == decltype(na_c)::value) with_a(na_c);
    });
    if constexpr (KSPLIT > 1) { __syncthreads(); __syncthreads(); }
    return;
  }

  // ------------------------------------------- consumers: waves 0..3 -------------------------------------------
  const int r32 = lane & 31, g2 = lane >> 5;
  const int cbw = wave & 1, rb0 = ((wave >> 1) % NRG) * NRB;
  const int kq = (wave >> 1) / NRG, t0 = kq * NT;
  uint32_t b_addr[NT], a_addr[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) {
    const int pp = ((2 * (t + t0) + g2) ^ ((r32 >> 1) & 7)) * 16;
    a_addr[t] = lds_base + (rb0 * 32 + r32) * RB + pp;
    b_addr[t] = lds_base + A_BYTES + (cbw * 32 + r32) * RB + pp;
  }
  typename SkAcc<TYPES>::v16 acc[NRB];
#pragma unroll
  for (int r = 0; r < NRB; r++)
#pragma unroll
    for (int e = 0; e < 16; e++) acc[r][e] = 0;

  const bool has_cols = n_base + cbw * 32 < n_end;   // a wave whose column block is empty only keeps the barriers company
  uint32_t so = 0;
  for (int i = 0, c = rot; i < nst; i++, c = c + 1 == nst ? 0 : c + 1) {
    asm volatile("s_barrier" ::: "memory");
    if (!has_cols) continue;
    if (c == nst - 1 && last < (uint32_t)RB) {
      // Pieces past the end of K count as zeros on both sides (what is left in LDS may be NaN or infinite): the wave
      // clears the ones that it is about to read.  (Its LDS accesses execute in order.  Clearing the fragments in
      // registers instead cost every stage of the loop: bf16 M = 128, N = 14336, K = 4096 33.1 us against 31.)
      sk_for<NT>([&](auto t_c) {
        constexpr int TT = decltype(t_c)::value;
        if ((uint32_t)((2 * (TT + t0) + g2) * 16) >= last) {
          sk_ds_zero16<0>(b_addr[TT] + so);
          sk_for<NRB>([&](auto r_c) {
            constexpr int R = decltype(r_c)::value;
            sk_ds_zero16<R * 32 * RB>(a_addr[TT] + so);
          });
        }
      });
    }
    // All fragment reads of the stage are requested at once, k-step by k-step, and the MFMAs of a k-step start as
    // soon as its own fragments are there (LDS reads return in order), instead of one wait for all of them.
    sk_u32x4_t bf[NT], af[NRB][NT];
    sk_for<NT>([&](auto t_c) {
      constexpr int TT = decltype(t_c)::value;
      sk_ds_read16<0>(bf[TT], b_addr[TT] + so);
      sk_for<NRB>([&](auto r_c) {
        constexpr int R = decltype(r_c)::value;
        sk_ds_read16<R * 32 * RB>(af[R][TT], a_addr[TT] + so);
      });
    });
    so = so + STAGE == S * STAGE ? 0 : so + STAGE;
    sk_for<NT>([&](auto t_c) {
      constexpr int TT = decltype(t_c)::value;
      sk_wait_lgkm<(NT - 1 - TT) * (1 + NRB)>();
      sk_touch(bf[TT]);
#pragma unroll
      for (int r = 0; r < NRB; r++) sk_touch(af[r][TT]);
#pragma unroll
      for (int r = 0; r < NRB; r++) {
        if constexpr (!is_fp8(TYPES)) acc[r] = mfma32x16<TYPES>(bf[TT], af[r][TT], acc[r]);
        else if constexpr (TT % 2 == 1) acc[r] = mfma32x64_f8<TYPES>(bf[TT - 1], bf[TT], af[r][TT - 1], af[r][TT], acc[r]);
      }
    });
  }
  if constexpr (KSPLIT > 1) {
    acc_t* red = reinterpret_cast<acc_t*>(sk_lds);
    __syncthreads();   // every copy has landed and every fragment has been read: the rings are free
    const int tile = wave % (2 * NRG);
    if (kq > 0) {
#pragma unroll
      for (int r = 0; r < NRB; r++)
#pragma unroll
        for (int e = 0; e < 16; e++) red[((((kq - 1) * 2 * NRG + tile) * NRB + r) * 16 + e) * 64 + lane] = acc[r][e];
    }
    __syncthreads();
    if (kq > 0) return;
#pragma unroll
    for (int q = 1; q < KSPLIT; q++)
#pragma unroll
      for (int r = 0; r < NRB; r++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[r][e] += red[((((q - 1) * 2 * NRG + tile) * NRB + r) * 16 + e) * 64 + lane];
  }

  const bool vec_ok = (g.ldd % 4 == 0) && (g.beta == 0 || g.ldc % 4 == 0) && ((reinterpret_cast<uintptr_t>(g.D) & 15u) == 0) &&
                      (g.beta == 0 || (reinterpret_cast<uintptr_t>(g.C) & 15u) == 0);
#pragma unroll
  for (int r = 0; r < NRB; r++) {
    const int m = (rb0 + r) * 32 + r32;
    if (m >= M) continue;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int n = n_base + cbw * 32 + q * 8 + g2 * 4;
      const size_t o = (size_t)m * (size_t)g.ldd + n, oc = (size_t)m * (size_t)g.ldc + n;
      if (vec_ok && n + 3 < n_end) {
        out_t cv[4] = {0, 0, 0, 0}, dv[4];
        if (g.beta != 0) __builtin_memcpy(cv, g.C + oc, sizeof(cv));
#pragma unroll
        for (int e = 0; e < 4; e++) dv[e] = epilogue<TYPES>(acc[r][4 * q + e], g.alpha, g.beta, &cv[e]);
        __builtin_memcpy(g.D + o, dv, sizeof(dv));
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++)
          if (n + e < n_end) g.D[o + e] = epilogue<TYPES>(acc[r][4 * q + e], g.alpha, g.beta, g.C + oc + e);
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------------------
// The producer / consumer kernel with wide column blocks and a split K, 64 < M <= 128 (see skinny_resolve_wide)
//   Work-group b serves K part ks = (b % 8) % KS of column group (b / 8) * (8 / KS) + (b % 8) / KS: work-groups go
//   to the XCDs in turn, so the work-groups of one XCD share a K part of A and its L2 holds that part only.
//   LDS ring: S stages of [A: 128 rows | B: 64 CB rows] x 128 bytes, swizzled as above.  Producer wave p moves A rows
//   [32 p, 32 p + 32) and B rows [16 CB p, 16 CB (p + 1)) of every stage.  Consumer wave w: row blocks 2 (w >> 1) and
//   2 (w >> 1) + 1, the 32-column blocks (w & 1) + 2 c for c < CB, all four k-steps of a stage; the fragments of
//   k-step t + 1 are requested before the MFMAs of k-step t.
//   The sums leave as the waves hold them: slot (ks, group) of the workspace, float4 index
//   (((wave * 2 + r) * CB + c) * 4 + q) * 64 + lane - whole 1 KiB stores; stream_wide_reduce_kernel reads them back in
//   the same order.
// ---------------------------------------------------------------------------------------------------------
template <int TYPES, int CB, int S>
__global__ void __launch_bounds__(STREAM_TILE_THREADS) stream_wide_kernel(GemmArgs<TYPES> g, int cols_per_wg, int groups, int KS,
                                                                          float* ws) {
  constexpr int NCW = 4;
  extern __shared__ __attribute__((aligned(1024))) char sk_lds[];
  constexpr int RB = STREAM_TILE_ROW_BYTES, A_ROWS = 128, A_BYTES = A_ROWS * RB, B_ROWS = STREAM_TILE_COLS * CB;
  constexpr int B_BYTES = B_ROWS * RB, STAGE = A_BYTES + B_BYTES;
  constexpr int NA = 4, NB = 2 * CB, NCP = NA + NB;   // copies per producer wave and stage
  constexpr int NRB = 2, NT = 4;
  static_assert(CB >= 2 && CB <= STREAM_WIDE_MAX_CB, "two to four 64-column blocks");
  static_assert((S - 2) * NCP < 64, "vmcnt");
  static_assert(S * STAGE <= 160 * 1024, "LDS");
  const uint32_t lds_base = (uint32_t)(uintptr_t)sk_lds;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int N = g.N, M = g.M;
  const int xcd = blockIdx.x % 8;
  const int ks = xcd % KS, cg = ((int)blockIdx.x / 8) * (8 / KS) + xcd / KS;
  if (cg >= groups) return;   // the grid is rounded up to whole rounds of the XCDs; before any barrier
  const int n_base = cg * cols_per_wg;
  const int n_end = min(n_base + cols_per_wg, N);
  const size_t rowb = (size_t)g.ldb * 2, rowb_a = (size_t)g.lda * 2;
  const int nst_all = g.K / STREAM_WIDE_K_STEP;
  const int st_q = nst_all / KS, st_r = nst_all % KS;
  const int st0 = ks * st_q + min(ks, st_r), nst = st_q + (ks < st_r ? 1 : 0);
  const int rot = (int)((unsigned)cg % (unsigned)nst);

  if (wave >= NCW) {
    const int p = wave - NCW;
    uint32_t voffA[NA], voffB[NB];
    uint64_t maskB[NB];
    const int row_in = lane >> 3, pos = lane & 7;
#pragma unroll
    for (int j = 0; j < NA; j++) {
      const int row = (p * NA + j) * 8 + row_in;
      voffA[j] = (uint32_t)((size_t)min(row, M - 1) * rowb_a) + (pos ^ ((row >> 1) & 7)) * 16;
    }
#pragma unroll
    for (int j = 0; j < NB; j++) {
      const int row = (p * NB + j) * 8 + row_in;
      const int n = min(n_base + row, N - 1);
      voffB[j] = (uint32_t)((size_t)(n - n_base) * rowb) + (pos ^ ((row >> 1) & 7)) * 16;
      maskB[j] = __builtin_amdgcn_ballot_w64(n_base + row < n_end);
    }
    const char* sA = reinterpret_cast<const char*>(g.A) + (size_t)st0 * RB;
    const char* sB = reinterpret_cast<const char*>(g.B) + (size_t)n_base * rowb + (size_t)st0 * RB;
    int slot = 0;
    auto issue = [&](int s) {   // a stage past the end: every copy masked off but still counted
      const bool exists = s < nst;
      int c = s + rot;
      if (c >= nst) c -= nst;
      if (!exists) c = 0;
      const uint32_t dst = lds_base + (uint32_t)slot * STAGE;
      slot = slot + 1 == S ? 0 : slot + 1;
      sk_set_m0(dst + p * (NA * 1024) + 2048);
      sk_for<NA>([&](auto j_c) {
        constexpr int J = decltype(j_c)::value;
        sk_copy16_keep<(J - 2) * 1024>(voffA[J], sA + (size_t)c * RB - (J - 2) * 1024, __builtin_amdgcn_ballot_w64(exists));
      });
      sk_set_m0(dst + A_BYTES + p * (NB * 1024) + (NB / 2) * 1024);
      sk_for<NB>([&](auto j_c) {
        constexpr int J = decltype(j_c)::value;
        const uint64_t m = maskB[J] & __builtin_amdgcn_ballot_w64(exists);
        sk_copy16<(J - NB / 2) * 1024>(voffB[J], sB + (size_t)c * RB - (J - NB / 2) * 1024, m);
      });
    };
    for (int s = 0; s < S - 1; s++) issue(s);
    for (int i = 0; i < nst; i++) {
      sk_wait_vm<(S - 2) * NCP>();                 // stage i has landed
      asm volatile("s_barrier" ::: "memory");     // consumers are done with stage i - 1
      issue(i + S - 1);
    }
    sk_wait_vm<0>();
    return;
  }

  // consumers
  const int r32 = lane & 31, g2 = lane >> 5;
  const int cbw = wave & 1, rb0 = (wave >> 1) * NRB;
  uint32_t b_addr[NT], a_addr[NT];
#pragma unroll
  for (int t = 0; t < NT; t++) {
    const int pp = ((2 * t + g2) ^ ((r32 >> 1) & 7)) * 16;
    a_addr[t] = lds_base + (rb0 * 32 + r32) * RB + pp;
    b_addr[t] = lds_base + A_BYTES + (cbw * 32 + r32) * RB + pp;
  }
  sk_f32x16_t acc[NRB][CB];
#pragma unroll
  for (int r = 0; r < NRB; r++)
#pragma unroll
    for (int c = 0; c < CB; c++)
#pragma unroll
      for (int e = 0; e < 16; e++) acc[r][c][e] = 0.f;

  uint32_t so = 0;
  for (int i = 0; i < nst; i++) {
    asm volatile("s_barrier" ::: "memory");
    sk_u32x4_t bf[2][CB], af[2][NRB];
    auto request = [&](auto t_c) {
      constexpr int TT = decltype(t_c)::value;
      sk_for<NRB>([&](auto r_c) {
        constexpr int R = decltype(r_c)::value;
        sk_ds_read16<R * 32 * RB>(af[TT & 1][R], a_addr[TT] + so);
      });
      sk_for<CB>([&](auto c_c) {
        constexpr int C = decltype(c_c)::value;
        sk_ds_read16<C * 64 * RB>(bf[TT & 1][C], b_addr[TT] + so);
      });
    };
    request(std::integral_constant<int, 0>{});
    sk_for<NT>([&](auto t_c) {
      constexpr int TT = decltype(t_c)::value;
      if constexpr (TT + 1 < NT) {
        request(std::integral_constant<int, TT + 1>{});
        sk_wait_lgkm<NRB + CB>();
      } else {
        sk_wait_lgkm0();
      }
#pragma unroll
      for (int r = 0; r < NRB; r++) sk_touch(af[TT & 1][r]);
#pragma unroll
      for (int c = 0; c < CB; c++) sk_touch(bf[TT & 1][c]);
#pragma unroll
      for (int r = 0; r < NRB; r++)
#pragma unroll
        for (int c = 0; c < CB; c++) acc[r][c] = mfma32x16<TYPES>(bf[TT & 1][c], af[TT & 1][r], acc[r][c]);
    });
    so = so + STAGE == S * STAGE ? 0 : so + STAGE;
  }

  sk_f32x4_t* out = reinterpret_cast<sk_f32x4_t*>(ws) +
                    ((size_t)ks * groups + cg) * (size_t)(NCW * NRB * CB * 4 * 64) + (size_t)wave * (NRB * CB * 4 * 64) + lane;
#pragma unroll
  for (int r = 0; r < NRB; r++)
#pragma unroll
    for (int c = 0; c < CB; c++)
#pragma unroll
      for (int q = 0; q < 4; q++)
        out[((r * CB + c) * 4 + q) * 64] = sk_f32x4_t{acc[r][c][4 * q], acc[r][c][4 * q + 1], acc[r][c][4 * q + 2], acc[r][c][4 * q + 3]};
}

// Second launch of the split: a work-group per 32 x 32 block of the output.  Its 256 lanes read the block's sums in
// the order the first launch stored them (whole lines), add the K parts in their order, turn the block through LDS
// and write it row by row - eight lanes per row, 128 contiguous bytes of an fp32 D - with alpha, beta and the rounding.
// (One lane per four outputs in storage order, each lane writing its own 16 bytes, took 10 us at M = 128, N = 14336:
// a wave's store then touched 32 rows.)
template <int TYPES>
__global__ void __launch_bounds__(256) stream_wide_reduce_kernel(GemmArgs<TYPES> g, int cols_per_wg, int groups, int KS, int CB,
                                                                 const float* ws) {
  using out_t = typename Traits<TYPES>::out_t;
  __shared__ float tile[32][36];
  const int per_slot = 4 * 2 * CB * 4 * 64;   // float4 per slot
  const int blocks_per_slot = 4 * 2 * CB;
  const int cg = (int)blockIdx.x / blocks_per_slot, blk = (int)blockIdx.x % blocks_per_slot;
  const int c = blk % CB, r = (blk / CB) % 2, wave = blk / (2 * CB);
  const int tid = threadIdx.x, lane = tid % 64, q = tid / 64;
  const sk_f32x4_t* in = reinterpret_cast<const sk_f32x4_t*>(ws) + (size_t)cg * per_slot + (size_t)blk * 256 + tid;
  sk_f32x4_t sum = in[0];
  for (int ks = 1; ks < KS; ks++) {
    const sk_f32x4_t v = in[(size_t)ks * groups * per_slot];
#pragma unroll
    for (int e = 0; e < 4; e++) sum[e] += v[e];
  }
#pragma unroll
  for (int e = 0; e < 4; e++) tile[lane & 31][q * 8 + (lane >> 5) * 4 + e] = sum[e];
  __syncthreads();
  const int row = tid / 8, j = tid % 8;
  const int m = ((wave >> 1) * 2 + r) * 32 + row;
  const int n = cg * cols_per_wg + ((wave & 1) + 2 * c) * 32 + 4 * j;
  const int n_end = min((cg + 1) * cols_per_wg, g.N);
  if (m >= g.M || n >= n_end) return;
  float v[4];
#pragma unroll
  for (int e = 0; e < 4; e++) v[e] = tile[row][4 * j + e];
  const size_t o = (size_t)m * (size_t)g.ldd + n, oc = (size_t)m * (size_t)g.ldc + n;
  const bool vec_ok = (g.ldd % 4 == 0) && (g.beta == 0 || g.ldc % 4 == 0) && ((reinterpret_cast<uintptr_t>(g.D) & 15u) == 0) &&
                      (g.beta == 0 || (reinterpret_cast<uintptr_t>(g.C) & 15u) == 0);
  if (vec_ok && n + 3 < n_end) {
    out_t cv[4] = {0, 0, 0, 0}, dv[4];
    if (g.beta != 0) __builtin_memcpy(cv, g.C + oc, sizeof(cv));
#pragma unroll
    for (int e = 0; e < 4; e++) dv[e] = epilogue<TYPES>(v[e], g.alpha, g.beta, &cv[e]);
    __builtin_memcpy(g.D + o, dv, sizeof(dv));
  } else {
#pragma unroll
    for (int e = 0; e < 4; e++)
      if (n + e < n_end) g.D[o + e] = epilogue<TYPES>(v[e], g.alpha, g.beta, g.C + oc + e);
  }
}

template <int TYPES> int launch_skinny(const GemmArgs<TYPES>& g, int variant, hipStream_t s) {
  if constexpr (!skinny_stream_types(TYPES)) {
    (void)g; (void)variant; (void)s;
    set_error("skinny rung is built for 8- and 16-bit elements with 32-bit accumulation only");
    return GZ_ERR_UNSUPPORTED;
  } else {
    if (variant > 1) {
      set_error("skinny rung has a single variant (got %d)", variant);
      return GZ_ERR_UNSUPPORTED;
    }
    if (!skinny_stream_supported(TYPES, g.M, g.N, g.K, g.layoutA, g.layoutB)) {
      set_error("skinny rung needs row-major A, column-major B, 1 <= M <= %d and whole 16-byte pieces of K (M=%d K=%d)",
                SKINNY_MAX_M, g.M, g.K);
      return GZ_ERR_UNSUPPORTED;
    }
    constexpr int ES = sizeof(typename Traits<TYPES>::in_t);
    if (((reinterpret_cast<uintptr_t>(g.A) | reinterpret_cast<uintptr_t>(g.B)) & 15u) || !skinny_lines_ok(ES, g.lda, g.ldb)) {
      set_error("skinny rung needs 16-byte aligned A and B and leading dimensions that are whole 16-byte pieces "
                "(lda=%lld ldb=%lld)", (long long)g.lda, (long long)g.ldb);
      return GZ_ERR_UNSUPPORTED;
    }
    const SkinnyCfg c = skinny_resolve(TYPES, g.M, g.N, g.K, device_compute_units(), (unsigned long long)workspace_limit(s));
    const dim3 grid((unsigned)c.grid_n), block((unsigned)c.threads);
    // (more than 64 KiB of dynamic LDS needs the opt-in; harmless below)
    auto one = [&](auto kern) {
      GZ_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     c.lds_bytes));
      hipLaunchKernelGGL(kern, grid, block, c.lds_bytes, s, g, c.cols_per_wg);
      GZ_HIP_TRY(hipGetLastError());
      return (int)GZ_OK;
    };
    if (c.kind == SKINNY_KIND_TILE) {
      if (c.mb == 32) return one(stream_tile_kernel<TYPES, 1, STREAM_TILE_STAGES_1>);
      if (c.mb == 64) return one(stream_tile_kernel<TYPES, 2, STREAM_TILE_STAGES_2>);
      return one(stream_tile_kernel<TYPES, 4, STREAM_TILE_STAGES_4>);
    }
    if (c.kind == SKINNY_KIND_DTL) {
      auto dtl = [&](auto ncp_c) {
        constexpr int NCP = decltype(ncp_c)::value;
        constexpr SkinnyDtlShape sh = skinny_dtl_shape(NCP);
        return (long long)g.K * ES % SKINNY_DTL_CHUNK_BYTES ? one(skinny_dtl_kernel<TYPES, NCP, sh.waves, sh.stages, true>)
                                                            : one(skinny_dtl_kernel<TYPES, NCP, sh.waves, sh.stages, false>);
      };
      switch (skinny_dtl_copies(c.cols_per_wg)) {
        case 1: return dtl(std::integral_constant<int, 1>{});
        case 2: return dtl(std::integral_constant<int, 2>{});
        case 4: return dtl(std::integral_constant<int, 4>{});
        default: return dtl(std::integral_constant<int, 8>{});
      }
    }
    if constexpr (skinny_rung_types(TYPES)) {   // wide column blocks, split K (skinny_resolve_wide)
      WorkspaceLease lease;
      const int st = lease.acquire((size_t)c.workspace_bytes, s);
      if (st != GZ_OK) return st;
      void* ws = lease.ptr;
      const int per_round = 8 / c.split_k;   // column groups per round of the eight XCDs
      const dim3 wgrid((unsigned)((c.grid_n + per_round - 1) / per_round * 8));
      auto k2 = stream_wide_kernel<TYPES, 2, STREAM_WIDE_STAGES_2>;
      auto k3 = stream_wide_kernel<TYPES, 3, STREAM_WIDE_STAGES_3>;
      auto k4 = stream_wide_kernel<TYPES, 4, STREAM_WIDE_STAGES_4>;
      auto kern = c.cb == 2 ? k2 : c.cb == 3 ? k3 : k4;
      GZ_HIP_TRY(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     c.lds_bytes));
      hipLaunchKernelGGL(kern, wgrid, block, c.lds_bytes, s, g, c.cols_per_wg, c.grid_n, c.split_k, static_cast<float*>(ws));
      GZ_HIP_TRY(hipGetLastError());
      hipLaunchKernelGGL((stream_wide_reduce_kernel<TYPES>), dim3((unsigned)(c.grid_n * 4 * 2 * c.cb)), dim3(256), 0, s, g,
                         c.cols_per_wg, c.grid_n, c.split_k, c.cb, static_cast<const float*>(ws));
      GZ_HIP_TRY(hipGetLastError());
      return GZ_OK;
    }
    set_error("skinny rung: no kernel for this plan");
    return GZ_ERR_UNSUPPORTED;
  }
}

template int launch_skinny<GZ_S8S8S32>(const GemmArgs<GZ_S8S8S32>&, int, hipStream_t);
template int launch_skinny<GZ_BF16BF16F32>(const GemmArgs<GZ_BF16BF16F32>&, int, hipStream_t);
template int launch_skinny<GZ_BF16BF16BF16>(const GemmArgs<GZ_BF16BF16BF16>&, int, hipStream_t);
template int launch_skinny<GZ_F16F16F16>(const GemmArgs<GZ_F16F16F16>&, int, hipStream_t);
template int launch_skinny<GZ_F32F32F32>(const GemmArgs<GZ_F32F32F32>&, int, hipStream_t);
template int launch_skinny<GZ_E4M3E4M3F16>(const GemmArgs<GZ_E4M3E4M3F16>&, int, hipStream_t);
template int launch_skinny<GZ_E5M2E5M2F16>(const GemmArgs<GZ_E5M2E5M2F16>&, int, hipStream_t);
template int launch_skinny<GZ_BF16BF16BF16_ACC16>(const GemmArgs<GZ_BF16BF16BF16_ACC16>&, int, hipStream_t);
template int launch_skinny<GZ_F16F16F16_ACC16>(const GemmArgs<GZ_F16F16F16_ACC16>&, int, hipStream_t);

}  // namespace gz
