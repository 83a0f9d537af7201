// NT GEMM kernel for gfx950 on bf16, int8 and fp8 (OCP e4m3fn) MFMA with a fused epilogue:
//
//   C[m][n] = epi( sum_k A[m][k] * B[n][k] )          A: [M, K] (lda), B: [N, K] (ldb), K contiguous
//   epi(acc) = act( round_opt( acc * alpha * a_scale[m] * b_scale[n] + bias[n] ) )   (+ C_old when accumulating)
//
// Matrix instructions: the 16x16 shapes (v_mfma_f32_16x16x32_bf16, v_mfma_i32_16x16x64_i8,
// v_mfma_f32_16x16x128_f8f6f4 without block scales). The part is limited by power, not by issue: on
// random operands held in registers (calib.hip) the 32x32 shapes run at 1750 / 3364 / 3903 T(FL)OP/s (bf16 / int8 /
// fp8) and the 16x16 shapes, walked so that successive MFMAs share one operand, at 2003 / 3975 / 4214. With the
// 32x32 shapes this GEMM's bf16 8192^3 kept the MFMA pipes busy 0.78 of the cycles at 1.48 GHz.
//
// Tiling: a workgroup of 8 wavefronts (two per SIMD, so that one wavefront's MFMAs issue while the other
// waits) computes a (32 MI) x 256 tile; wavefront w owns rows 16 MI (w / 4) .. +16 MI and columns
// 64 (w % 4) .. +64 as MI x 4 blocks of 16x16. The product is formed transposed (B rows are the
// instruction's rows), so a lane holds runs of columns of one row of C. MI is chosen by the
// launcher (gemm.hip).
//
// Stages of 128 K bytes per row (whole cache lines: half the L2 requests of 64-byte stages) go straight to
// LDS (global_load_lds) through a ring of slots per operand. A stage is KS k-steps (2 of 64 bytes for bf16 /
// int8, 1 of 128 bytes for fp8) of MI units; a unit is the 4 MFMAs of one A fragment. A fragments are read RA
// units ahead into a ring of R, the next k-step's B fragments during the units from MB on, so the barrier
// of stage s (all loads of stage s + 1 landed) sits before unit MB of its last k-step. At that point every
// wavefront has read all of B's stage s and all of A's stage s - 1: the loads of stage s + D + 1 go into
// those two slots, spread between the following MFMAs. 16-byte chunk c of a stage row is stored at gemm_slot,
// which makes the 16-row fragment reads conflict-free.
//
// What bounds it: power, then the tile loads. At 8192^3 in bf16 the kernel takes 788 us (877 with the 32x32
// shapes and 64-byte stages), 645 without its tile loads (timing only), 766 without its epilogue; the MFMA
// pipes are busy 0.77 of the cycles at 1.67 GHz. At 40,688 x 15,360 x 5,120, alternated with that kernel
// on one machine: int8 2422 us against 2812, fp8 2291 against 2664 (2642 and 2793 T(FL)OP/s). Bands that start their
// columns apart: 8192^3 bf16 775 -> 752 us, fp8 400 -> 380, int8 415 -> 393; 8,296 x 15,360 x 5,120 fp8 504 -> 487.
#pragma once
#include <type_traits>

#include "common.h"

namespace vdnh3 {

enum GemmKind { kBF16 = 0, kI8 = 1, kF8 = 2 };
enum OutType { kOutBF16 = 0, kOutF32 = 1, kOutI32 = 2 };

struct GemmEpi {
  const float *a_scale;  // [M] or null
  const float *b_scale;  // [N] or null (a single value when b_scale_n == 1)
  int b_scale_n;
  int a_scale_n;
  float alpha;
  const void *bias;  // [N] or null
  int bias_bf16;
  int act;            // 0 none, 1 sigmoid
  int act_cols;       // with the sigmoid: it applies to columns n < act_cols only (0: every column)
  int out_type;       // OutType
  int accumulate;     // C += epi(acc)
  int round_linear;   // bf16 output: round the linear result to bf16 before the activation
};

struct GemmArgs {
  const uint8_t *A, *B;
  int64_t lda_b, ldb_b;  // row strides in bytes
  void *C;
  int64_t ldc;
  int M, N;
  int nst;  // stages of kGemmSK bytes of K
  int tiles_m, tiles_n, per_xcd, total;
  GemmEpi epi;
};

constexpr int kGemmBN = 256;             // columns of a tile
constexpr int kGemmSK = 128;             // K bytes per row and stage
constexpr int kGemmThreads = 512;
constexpr int kGemmGroupRows = 1024;     // rows of C in a band of the tile order

// launches the kernel for tiles of 32 mi rows, mi one of 2, 4, 5, 6, 7, 8
template <int KIND>
void launch_gemm_tiles(int mi, const GemmArgs &args, hipStream_t stream);

#ifdef VDNH3_GEMM_KERNEL
namespace {

__device__ __forceinline__ float sigmoidf_(float x) { return 1.f / (1.f + __expf(-x)); }

// LDS slot of 16-byte chunk c of stage row r: a fragment read takes one chunk column of 16 consecutive rows
// per 16 lanes, and the slots put those in 16 different 16-byte bank groups (row % 2 x 8 slots)
__device__ __forceinline__ constexpr int gemm_slot(int r, int c) { return c ^ ((r >> 1) & 7); }

// Output stores, and the loads of the old values when accumulating, are non-temporal (the `nt`
// hint): the output streams through each XCD's L2 at 128 KB per tile, which would otherwise
// evict the A and B panels that the XCD's other workgroups are still reading.
// C is aligned to its elements only (any N and ldc; global accesses of any alignment are one instruction here), and
// the pointers say so: the types are no template arguments, which would lose their alignment.
typedef u32x4_t __attribute__((aligned(2))) u32x4_a2_t;
typedef u32x4_t __attribute__((aligned(4))) u32x4_a4_t;
typedef f32x4_t __attribute__((aligned(4))) f32x4_a4_t;
__device__ __forceinline__ void stream_store(u32x4_t v, uint16_t *p) {
  __builtin_nontemporal_store(v, reinterpret_cast<u32x4_a2_t *>(p));
}
__device__ __forceinline__ void stream_store(u32x4_t v, int32_t *p) {
  __builtin_nontemporal_store(v, reinterpret_cast<u32x4_a4_t *>(p));
}
__device__ __forceinline__ void stream_store(f32x4_t v, float *p) {
  __builtin_nontemporal_store(v, reinterpret_cast<f32x4_a4_t *>(p));
}
__device__ __forceinline__ u32x4_t stream_load(const uint16_t *p) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x4_a2_t *>(p));
}
__device__ __forceinline__ f32x4_t stream_load(const float *p) {
  return __builtin_nontemporal_load(reinterpret_cast<const f32x4_a4_t *>(p));
}

// Epilogue operands. Loaded at the start of the kernel, one column (its scale times alpha, its bias) and
// MI / 4 rows per lane, so that their latency hides behind the main loop at 2 + MI / 4 registers; the
// epilogue hands them round through a 1.5 KB LDS area of the wavefront.
template <int MI>
struct EpiOperands {
  static constexpr int kRows = (16 * MI + 63) / 64;
  float row[kRows], col, bias;
};
constexpr int kEpiWords = 256 + 64 + 64;  // row scales, column scales, biases

template <int MI>
__device__ __forceinline__ EpiOperands<MI> load_epi_operands(const GemmEpi &epi, int M, int N, int mb, int nb,
                                                             int lane) {
  EpiOperands<MI> o;
#pragma unroll
  for (int h = 0; h < EpiOperands<MI>::kRows; ++h) {
    const int m = min(mb + 64 * h + lane, M - 1);
    o.row[h] = epi.a_scale ? epi.a_scale[epi.a_scale_n == 1 ? 0 : m] : 1.f;
  }
  const int n = min(nb + lane, N - 1);
  o.col = epi.b_scale ? epi.alpha * epi.b_scale[epi.b_scale_n == 1 ? 0 : n] : epi.alpha;
  o.bias = !epi.bias ? 0.f
           : epi.bias_bf16 ? bf2f(static_cast<const uint16_t *>(epi.bias)[n])
                           : static_cast<const float *>(epi.bias)[n];
  return o;
}

// Lane (l16 = lane % 16, g = lane / 16) holds, of row 16 i + l16 of the wavefront's block, columns
// 32 jp + 8 g + 0 .. 7 in acc[i][2 jp] and acc[i][2 jp + 1]. bf16 output: lanes of an even and the next odd
// row swap halves (one DPP move per word), so that one store instruction writes eight whole 128-byte rows of
// the block; with 64-byte pieces of 16 rows instead the GEMM took 3-5% longer. A lane whose eight columns
// reach past N stores them one by one; nothing else depends on N or the alignment of C's rows.
template <int OUT, bool ACT, bool ACCUM, int MI, typename Acc>
__device__ __forceinline__ void store_block(const Acc (&acc)[MI][4], float *stage, const EpiOperands<MI> &eo,
                                            const GemmEpi &epi, void *C, int64_t ldc, int M, int N, int mb, int nb,
                                            int lane) {
  const int l16 = lane & 15, g = lane >> 4;
  float cs[16], bs[16];
  if constexpr (OUT != kOutI32) {
#pragma unroll
    for (int h = 0; h < EpiOperands<MI>::kRows; ++h) stage[64 * h + lane] = eo.row[h];
    stage[256 + lane] = eo.col;
    stage[320 + lane] = eo.bias;
    asm volatile("" ::: "memory");  // LDS operations of one wavefront complete in order
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      cs[k] = stage[256 + 32 * (k >> 3) + 8 * g + (k & 7)];
      bs[k] = stage[320 + 32 * (k >> 3) + 8 * g + (k & 7)];
    }
  }
  const int act_cols = epi.act_cols > 0 ? epi.act_cols : N;
  // the 8 values of block row i, column half jp
  auto values = [&](int i, int jp, float (&v)[8]) __device__ {
    const float rs = stage[16 * i + l16];
    const int n = nb + 32 * jp + 8 * g;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const auto e = acc[i][2 * jp + (k >> 2)][k & 3];
      float x = (float)e * rs;  // 1 without row scales
      x = x * cs[8 * jp + k] + bs[8 * jp + k];
      // bf16 output: rounding the linear value first only matters before the sigmoid (a
      // second rounding of a bf16 value, or the accumulation's own rounding, is exact)
      if constexpr (OUT == kOutBF16 && ACT) x = epi.round_linear ? round_bf(x) : x;
      if constexpr (ACT) x = n + k < act_cols ? sigmoidf_(x) : x;
      v[k] = x;
    }
  };
  if constexpr (OUT == kOutBF16) {
    const bool odd = lane & 1;
    const int n = nb + 8 * g + (odd ? 32 : 0);
    const int m0 = mb + (l16 & ~1);
    uint16_t *cp = static_cast<uint16_t *>(C) + (int64_t)m0 * ldc + n;
    // when accumulating, the old values of four block rows are loaded together, before their stores
    constexpr int kBatch = ACCUM ? 4 : 1;
#pragma unroll
    for (int i0 = 0; i0 < MI; i0 += kBatch) {
      u32x4_t old[kBatch][2];
      if constexpr (ACCUM) {
#pragma unroll
        for (int b = 0; b < kBatch; ++b)
#pragma unroll
          for (int r = 0; r < 2; ++r)
            if (i0 + b < MI && n + 8 <= N && m0 + 16 * (i0 + b) + r < M)
              old[b][r] = stream_load(cp + (int64_t)(16 * (i0 + b) + r) * ldc);
      }
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        const int i = i0 + b;
        if (i >= MI) break;
        u32x4_t w[2], o[2];
#pragma unroll
        for (int jp = 0; jp < 2; ++jp) {
          float v[8];
          values(i, jp, v);
#pragma unroll
          for (int h = 0; h < 4; ++h) w[jp][h] = pack_bf2(v[2 * h], v[2 * h + 1]);
        }
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          const uint32_t x = odd ? w[0][h] : w[1][h];
          const uint32_t y = (uint32_t)__builtin_amdgcn_mov_dpp((int)x, 0xB1, 0xf, 0xf, true);  // lane ^ 1
          o[0][h] = odd ? y : w[0][h];
          o[1][h] = odd ? w[1][h] : y;
        }
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          uint16_t *row = cp + (int64_t)(16 * i + r) * ldc;
          if (m0 + 16 * i + r >= M) continue;
          if (n + 8 <= N) {
            if constexpr (ACCUM) {
#pragma unroll
              for (int h = 0; h < 4; ++h)
                o[r][h] = pack_bf2(bf2f(old[b][r][h] & 0xffff) + bf2f(o[r][h] & 0xffff),
                                   bf2f(old[b][r][h] >> 16) + bf2f(o[r][h] >> 16));
            }
            stream_store(o[r], row);
          } else {
#pragma unroll
            for (int k = 0; k < 8; ++k) {
              const uint16_t e = (uint16_t)(o[r][k >> 1] >> (16 * (k & 1)));
              if (n + k < N) row[k] = ACCUM ? f2bf(bf2f(row[k]) + bf2f(e)) : e;
            }
          }
        }
      }
    }
  } else {
    // 32-bit output: the four lanes of a quad transpose their four rows' 16-byte pieces (swaps with the lane beside,
    // then two apart), so that one store instruction writes whole 256-byte runs of four rows: fp8 27,586 x 3,604 x
    // 1,408 204 us (485 with 16-byte pieces 32 bytes apart, 228 with 128-byte runs), int32 18,376 x 2,555 x 256 77
    // (109 with 128-byte runs).
    using elem = typename std::conditional<OUT == kOutI32, int32_t, float>::type;
    using vec = typename std::conditional<OUT == kOutI32, u32x4_t, f32x4_t>::type;
    const bool b0 = lane & 1, b1 = lane & 2;
    const int n = nb + 8 * g + (b0 ? 4 : 0) + (b1 ? 32 : 0), m0 = mb + (l16 & ~3);
    elem *cp = static_cast<elem *>(C) + (int64_t)m0 * ldc + n;
    auto swap = [](bool hi, u32x4_t &lo_v, u32x4_t &hi_v, auto ctrl) __device__ {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const uint32_t x = hi ? lo_v[k] : hi_v[k];
        const uint32_t y = (uint32_t)__builtin_amdgcn_mov_dpp((int)x, decltype(ctrl)::value, 0xf, 0xf, true);
        lo_v[k] = hi ? y : lo_v[k];
        hi_v[k] = hi ? hi_v[k] : y;
      }
    };
    // piece lane % 4 of rows 0 .. 3 of the quad in block row i
    auto transposed = [&](int i, u32x4_t (&o)[4]) __device__ {
#pragma unroll
      for (int jp = 0; jp < 2; ++jp) {
        u32x4_t &w0 = o[2 * jp], &w1 = o[2 * jp + 1];
        if constexpr (OUT == kOutI32) {
          w0 = __builtin_bit_cast(u32x4_t, acc[i][2 * jp]);
          w1 = __builtin_bit_cast(u32x4_t, acc[i][2 * jp + 1]);
        } else {
          float v[8];
          values(i, jp, v);
          w0 = __builtin_bit_cast(u32x4_t, f32x4_t{v[0], v[1], v[2], v[3]});
          w1 = __builtin_bit_cast(u32x4_t, f32x4_t{v[4], v[5], v[6], v[7]});
        }
        swap(b0, w0, w1, std::integral_constant<int, 0xB1>{});  // lane ^ 1
      }
      swap(b1, o[0], o[2], std::integral_constant<int, 0x4E>{});  // lane ^ 2
      swap(b1, o[1], o[3], std::integral_constant<int, 0x4E>{});
    };
    // as above, the old values of two block rows are loaded together, before their stores
    constexpr int kBatch = ACCUM ? 2 : 1;
#pragma unroll
    for (int i0 = 0; i0 < MI; i0 += kBatch) {
      vec old[kBatch][4];
      if constexpr (ACCUM) {
#pragma unroll
        for (int b = 0; b < kBatch; ++b)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            if (i0 + b >= MI || m0 + 16 * (i0 + b) + r >= M) continue;
            const elem *row = cp + (int64_t)(16 * (i0 + b) + r) * ldc;
            if (n + 4 <= N) {
              old[b][r] = stream_load(row);
            } else {
#pragma unroll
              for (int k = 0; k < 4; ++k) old[b][r][k] = n + k < N ? row[k] : 0;
            }
          }
      }
#pragma unroll
      for (int b = 0; b < kBatch; ++b) {
        const int i = i0 + b;
        if (i >= MI) break;
        u32x4_t o[4];
        transposed(i, o);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          if (m0 + 16 * i + r >= M) continue;
          elem *row = cp + (int64_t)(16 * i + r) * ldc;
          vec v = __builtin_bit_cast(vec, o[r]);
          if constexpr (ACCUM) v += old[b][r];
          if (n + 4 <= N) {
            stream_store(v, row);
          } else {
#pragma unroll
            for (int k = 0; k < 4; ++k)
              if (n + k < N) row[k] = (elem)v[k];
          }
        }
      }
    }
  }
}

// MFMA operands: 16 bytes per lane (bf16 / int8, 64 bytes of K) or 32 (fp8, 128 bytes of K)
template <int KIND>
struct Frag {
  using type = typename std::conditional<KIND == kF8, i32x8_t, u32x4_t>::type;
};

template <int KIND, int MI>
__global__ __launch_bounds__(kGemmThreads, 1) void gemm_nt_kernel(const GemmArgs args) {
  constexpr int BM = 32 * MI;
  constexpr int KS = KIND == kF8 ? 1 : 2;              // k-steps per stage
  constexpr int R = MI == 8 ? 4 : MI;                  // A fragment ring: divides the units of a stage
  constexpr int MB = MI / 2;                           // the barrier's unit in the last k-step
  constexpr int RA = MI - MB < 3 ? MI - MB : 3;        // units an A fragment is read ahead
  constexpr int U = KS * MI, UB = (KS - 1) * MI + MB;  // units per stage; the barrier's unit
  constexpr int A_STAGE = BM * kGemmSK, B_STAGE = kGemmBN * kGemmSK;
  constexpr int A_WL = BM / 8;  // an A stage in wavefront loads (8 rows, 1 KB each)
  constexpr int NA = (A_WL + 7) / 8, NB = kGemmBN / 64, NL = NA + NB;  // loads per wavefront and stage
  // Stages s + 1 .. s + D are in flight or landed while stage s is multiplied, through D + 2 slots for A and D + 1
  // for B: 160 KB for MI = 8, D = 1. A tile of at most 128 rows has its stage's MFMAs done before a load issued
  // one stage ahead returns, and LDS to spare.
  constexpr int D = MI <= 4 ? 2 : 1, SA = D + 2, SB = D + 1;
  // loads per unit from the barrier on; all go out at least half a stage before the barrier that waits for them
  constexpr int LPU = U == 2 ? 3 : KIND == kF8 || U < 2 * NL ? 2 : 1;
  static_assert(U % R == 0 && RA <= R && U * LPU >= NL, "fragment ring and load slots");
  __shared__ __attribute__((aligned(16))) uint8_t smem[SA * A_STAGE + SB * B_STAGE];
  static_assert(sizeof(smem) <= 160 * 1024 && (D == 1 || A_WL % 8 == 0), "LDS size; equal load counts per wavefront");
  static_assert(8 * kEpiWords * 4 <= (int)sizeof(smem), "epilogue operands must fit the stage slots");

  // XCD-aware tile order: workgroups are dealt round-robin over the 8 XCDs, so logical tile L of XCD x is
  // bid = 8 (L - x per_xcd) + x. Logical tiles walk bands of about kGemmGroupRows rows, column by column, so
  // the workgroups resident on one XCD share A rows and B columns in its L2.
  const int M = args.M, N = args.N, nst = args.nst;
  const int bid = blockIdx.x;
  const int L = (bid & 7) * args.per_xcd + (bid >> 3);
  if (L >= args.total) return;
  constexpr int kGroup = kGemmGroupRows / BM;
  const int band = L / (kGroup * args.tiles_n);
  const int band_m = min(kGroup, args.tiles_m - band * kGroup);
  const int in_band = L - band * kGroup * args.tiles_n;
  // A band starts its columns 5/8 of the way round from the last one's: the XCDs work on different bands, and
  // starting on the same columns they would all fetch the same B panels from the same memory channels at once
  const int column = (in_band / band_m + band * 5 * args.tiles_n / 8) % args.tiles_n;
  const int m0 = (band * kGroup + in_band % band_m) * BM, n0 = column * kGemmBN;

  const int tid = threadIdx.x, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = (wave >> 2) * (16 * MI), wn = (wave & 3) * 64;
  const EpiOperands<MI> eo = load_epi_operands<MI>(args.epi, M, N, m0 + wm, n0 + wn, lane);

  // Stage loads: load q of an operand covers stage rows 64 q .. +64 (8 per wavefront), lane tid % 8 of a row
  // fetching the chunk gemm_slot maps to slot tid % 8. Rows past M (N) read the last row; their results
  // are not stored. The source is a wave-uniform base plus a per-lane 32-bit offset that is the same
  // for every stage (the host checks that 256 rows of A and B span less than 4 GB). LDS row 64 w + 16 j + mm
  // of B holds column 64 w + 32 (j / 2) + 8 (mm / 4) + 4 (j % 2) + mm % 4 of the tile, so that the 16 rows
  // of each product fragment are consecutive and a lane's results are runs of 8 columns.
  const int lrow = tid >> 3;
  const int lchunk = gemm_slot(lrow, tid & 7);
  uint32_t a_off[NA], b_off[NB];
#pragma unroll
  for (int q = 0; q < NA; ++q)
    a_off[q] = (uint32_t)((min(m0 + 64 * q + lrow, M - 1) - m0) * args.lda_b + lchunk * 16);
  const int bcol = 32 * (lrow >> 5) + 8 * ((lrow >> 2) & 3) + 4 * ((lrow >> 4) & 1) + (lrow & 3);
#pragma unroll
  for (int q = 0; q < NB; ++q)
    b_off[q] = (uint32_t)((min(n0 + 64 * q + bcol, N - 1) - n0) * args.ldb_b + lchunk * 16);
  const uint8_t *a_tile = args.A + (int64_t)m0 * args.lda_b, *b_tile = args.B + (int64_t)n0 * args.ldb_b;
  const uint32_t lds0 = lds_address(&smem[0]) + wave * 1024;
  // load q of stage st: A for q < NA, then B, into the slots at bytes a_slot and b_slot
  auto load_part = [&](int st, uint32_t a_slot, uint32_t b_slot, int q) __device__ {
    const int64_t off = (int64_t)st * kGemmSK;
    if (q < NA) {
      if (A_WL % 8 == 0 || q + 1 < NA || wave < A_WL % 8)
        global_to_lds16_sbase(a_tile + off, a_off[q < NA ? q : 0], lds0 + a_slot + q * 8192);
    } else {
      global_to_lds16_sbase(b_tile + off, b_off[q >= NA ? q - NA : 0],
                            lds0 + SA * A_STAGE + b_slot + (q - NA) * 8192);
    }
  };

  // a lane's fragment: row l16, chunk 4 ks + g of the stage row (bf16 / int8), or chunks g and 4 + g (fp8);
  // A and B pair the same chunks, so the products pair the same k whatever order the instruction gives them
  uint32_t fo[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) fo[h] = l16 * kGemmSK + gemm_slot(l16, 4 * h + g) * 16;
  using frag_t = typename Frag<KIND>::type;
  using acc_t = typename std::conditional<KIND == kI8, i32x4_t, f32x4_t>::type;
  frag_t fa[R], fb[2][4];
  acc_t acc[MI][4];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = acc_t{};
  auto rd = [&](uint32_t base, int ks) __device__ {
    if constexpr (KIND == kF8) {
      const u32x4_t lo = ld16(smem + base + fo[0]), hi = ld16(smem + base + fo[1]);
      return frag_t{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
    } else {
      return frag_t(ld16(smem + base + fo[ks]));
    }
  };
  auto read_a = [&](uint32_t a_slot, int u) __device__ {  // the A fragment of unit u of a stage
    fa[u % R] = rd(a_slot + (uint32_t)wm * kGemmSK + (u % MI) * 16 * kGemmSK, u / MI);
  };
  auto read_b = [&](uint32_t b_slot, int ks, int buf, int j) __device__ {
    fb[buf][j] = rd(SA * A_STAGE + b_slot + (uint32_t)wn * kGemmSK + j * 16 * kGemmSK, ks);
  };
  auto next_a = [](uint32_t x) __device__ { return x == (SA - 1) * A_STAGE ? 0u : x + A_STAGE; };
  auto next_b = [](uint32_t x) __device__ { return x == (SB - 1) * B_STAGE ? 0u : x + B_STAGE; };

  // Stage s with its operands in slots sa and sb; P: the B fragment buffer of its first k-step. The last stage too waits at its
  // barrier and reads ahead (stale LDS bytes that nothing uses): a copy of the stage without them made the
  // register allocation spill.
  auto run_stage = [&](int s, uint32_t sa, uint32_t sb, auto parity) __device__ {
    constexpr int P = decltype(parity)::value;
    const uint32_t sa1 = next_a(sa), sb1 = next_b(sb);
    // slots of stage s + D (its loads that stage s - 1 left over go out before the barrier) and of stage
    // s + D + 1, whose A slot was that of stage s - 1 and whose B slot is this stage's
    const uint32_t la = D == 1 ? sa1 : next_a(sa1), lb = D == 1 ? sb1 : next_b(sb1);
    const uint32_t la1 = next_a(la), lb1 = sb;
    const bool load0 = s + D < nst, load1 = s + D + 1 < nst;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int ks = u / MI, i = u % MI, buf = (P + ks) & 1;
      if (u == UB) {
        // stage s + 1 has landed; the loads of a stage s + 2 may be in flight
        if (D == 1 || !load0) wait_vm<0>();
        else wait_vm<NL>();
        bare_barrier();
      }
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int j = (u & 1) ? 3 - x : x;  // successive MFMAs share an operand: less toggling, less power
        __builtin_amdgcn_sched_barrier(0);  // fixed issue order: each read and load sits between two MFMAs
        if constexpr (KIND == kF8)
          // scale operands 0 select the unscaled form
          acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb[buf][j], fa[u % R], acc[i][j], 0, 0, 0, 0, 0,
                                                                       0);
        else if constexpr (KIND == kBF16)
          acc[i][j] = mfma_bf16_16x16x32(as_bf16x8(fb[buf][j]), as_bf16x8(fa[u % R]), acc[i][j]);
        else
          acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4_t, fb[buf][j]),
                                                            __builtin_bit_cast(i32x4_t, fa[u % R]), acc[i][j], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
        if (x == 0) {
          if (u + RA < U) read_a(sa, u + RA);
          else read_a(sa1, u + RA - U);
        }
        if (x == 1 && i >= MB) {
          constexpr int per = (4 + MI - MB - 1) / (MI - MB);
#pragma unroll
          for (int t = 0; t < per; ++t) {
            const int jj = (i - MB) * per + t;
            if (jj < 4) {
              if (ks + 1 < KS) read_b(sb, ks + 1, buf ^ 1, jj);
              else read_b(sb1, 0, buf ^ 1, jj);
            }
          }
        }
#pragma unroll
        for (int t = 0; t < LPU; ++t) {
          const int q = (u >= UB ? u - UB : u + U - UB) * LPU + t;
          if (x == 2 + (t & 1) && q < NL) {
            if (u >= UB) { if (load1) load_part(s + D + 1, la1, lb1, q); }
            else if (load0) load_part(s + D, la, lb, q);
          }
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // prologue: stages 0 .. D - 1 whole, and of stage D what a stage issues after its barrier
  constexpr int kPost = (U - UB) * LPU < NL ? (U - UB) * LPU : NL;
#pragma unroll
  for (int st = 0; st <= D; ++st)
    if (st == 0 || st < nst) {
#pragma unroll
      for (int q = 0; q < (st < D ? NL : kPost); ++q) load_part(st, st * A_STAGE, st * B_STAGE, q);
    }
  if (nst > D && A_WL % 8 == 0) wait_vm<(D - 1) * NL + kPost>();
  else wait_vm<0>();
  bare_barrier();
#pragma unroll
  for (int j = 0; j < 4; ++j) read_b(0, 0, 0, j);
#pragma unroll
  for (int u = 0; u < RA; ++u) read_a(0, u);
  uint32_t sa = 0, sb = 0;
  auto step = [&](int s, auto parity) __device__ {
    run_stage(s, sa, sb, parity);
    sa = next_a(sa);
    sb = next_b(sb);
  };
  // A stage of a 64-row tile is short enough for instruction fetch to show: the padding keeps the loop's place against
  // 32-byte lines whatever code comes before (a longer epilogue had moved it: bf16 37.4 -> 39.0 us). 1,808 x 40 x 5,120
  // with 24 bytes of it: bf16 37.2 us against 39.1 / 38.5 / 37.6 with 0 / 8 / 16, int8 20.9 against 21.8 / 21.5 /
  // 21.0, fp8 20.0 against 20.6 / 20.3 / 20.3; at taller tiles it doesn't tell.
  if constexpr (MI == 2) asm volatile(".p2align 5\n.rept 6\ns_nop 0\n.endr");
  if constexpr (KS == 2) {
#pragma unroll 1
    for (int s = 0; s < nst; ++s) step(s, std::integral_constant<int, 0>{});
  } else {
    int s = 0;
#pragma unroll 1
    for (; s + 1 < nst; s += 2) {
      step(s, std::integral_constant<int, 0>{});
      step(s + 1, std::integral_constant<int, 1>{});
    }
    if (s < nst) step(s, std::integral_constant<int, 0>{});
  }

  // epilogue, specialised on the output type, activation and accumulation (one uniform branch here
  // instead of per-element tests); it reuses the LDS once every wavefront has read its last fragments
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  bare_barrier();
  float *stage = reinterpret_cast<float *>(smem) + wave * kEpiWords;
  const GemmEpi &epi = args.epi;
  void *C = args.C;
  const int mb = m0 + wm, nb = n0 + wn;
  if (epi.out_type == kOutI32) {
    if constexpr (KIND == kI8) store_block<kOutI32, false, false, MI>(acc, stage, eo, epi, C, args.ldc, M, N, mb, nb, lane);
  } else if (epi.out_type == kOutF32) {
    if (epi.act) store_block<kOutF32, true, false, MI>(acc, stage, eo, epi, C, args.ldc, M, N, mb, nb, lane);
    else if (epi.accumulate) store_block<kOutF32, false, true, MI>(acc, stage, eo, epi, C, args.ldc, M, N, mb, nb, lane);
    else store_block<kOutF32, false, false, MI>(acc, stage, eo, epi, C, args.ldc, M, N, mb, nb, lane);
  } else {
    if (epi.act) store_block<kOutBF16, true, false, MI>(acc, stage, eo, epi, C, args.ldc, M, N, mb, nb, lane);
    else if (epi.accumulate) store_block<kOutBF16, false, true, MI>(acc, stage, eo, epi, C, args.ldc, M, N, mb, nb, lane);
    else store_block<kOutBF16, false, false, MI>(acc, stage, eo, epi, C, args.ldc, M, N, mb, nb, lane);
  }
}

template <int KIND, int MI>
void launch_gemm_mi(const GemmArgs &args, hipStream_t stream) {
  hipLaunchKernelGGL((gemm_nt_kernel<KIND, MI>), dim3(args.per_xcd * 8), dim3(kGemmThreads), 0, stream, args);
}

}  // namespace

template <int KIND>
void launch_gemm_tiles(int mi, const GemmArgs &args, hipStream_t stream) {
  switch (mi) {
    case 2: return launch_gemm_mi<KIND, 2>(args, stream);
    case 4: return launch_gemm_mi<KIND, 4>(args, stream);
    case 5: return launch_gemm_mi<KIND, 5>(args, stream);
    case 6: return launch_gemm_mi<KIND, 6>(args, stream);
    case 7: return launch_gemm_mi<KIND, 7>(args, stream);
    default: return launch_gemm_mi<KIND, 8>(args, stream);
  }
}
#endif  // VDNH3_GEMM_KERNEL

}  // namespace vdnh3
