// Host side of the GEMM (gemm_kernel.h): argument checks, the choice of the tile height and the launch.
//
// It stands in for every projection of the hybrid block: F.linear in bf16 (gates, beta, the
// VDN to_out_linear, vdn_h3/projection.py:259-261), the fp8 `_scaled_mm(x_q, W_q^T, s_x, s_w)`
// (vdn_h3/fp8.py:254-262) and the W8A8 int8 projection with per-token x per-channel scales
// (the ComfyUI-native qkv_proj / out_proj of vdn_h3/hybrid.py:263, :535).
#include <initializer_list>

#include "gemm_kernel.h"

namespace vdnh3 {
namespace {

// Tile height (32 mi rows) for an M x N output: the one whose rounds of tiles over the 256 CUs, one workgroup
// each, take least. A round is taken to cost mi + 1.5 (the B tile's loads and reads, the prologue and the epilogue do
// not shrink with mi). Measured, one round for mi = 8 / 7 / 6 / 5 / 4 / 2: 185 / 170 / 151 / 130 / 114 / 74 us with
// 16,384 bytes of K in bf16, and for each type mi + 2 fits from 2,048 bytes on, mi + 3 512 bytes and mi + 4 one stage
// of 128 (bf16 10.0 / 8.9 / 7.8 / 6.8 / 6.5 / 4.9 us). Over 20,000 sizes drawn up to 40,688 x 15,360 the choice by
// mi + 2 differs for 0.6%, by at most 0.4% of the time, by mi + 4 for 1.1%, by at most 7%, so one line serves every
// type and K. Large outputs keep mi = 8; in between the height follows the last round (8,296 x 5,120: mi = 7, three
// full rounds, 346 us, against 348 with 8 and 2.6 rounds' worth of tiles; 1,808 x 5,120: mi = 5 79 us against 94;
// 40,688 x 208: mi = 5 123 us against 141), and few rows take low tiles, which leave fewer CUs idle (512 x
// 15,360 in int8: mi = 4 38.5 us against 50; 8,296 x 208: mi = 2 48 us against 101).
int gemm_mi(int M, int N) {
  const int64_t tiles_n = (N + kGemmBN - 1) / kGemmBN;
  int best = 8;
  int64_t best_cost = INT64_MAX;
  for (int mi : {8, 7, 6, 5, 4, 2}) {
    const int64_t tiles = tiles_n * ((M + 32 * mi - 1) / (32 * mi));
    const int64_t cost = (tiles + 255) / 256 * (2 * mi + 3);
    if (cost < best_cost) best = mi, best_cost = cost;
  }
  return best;
}

template <int KIND>
int launch_gemm(const void *A, int64_t lda, const void *B, int64_t ldb, void *C, int64_t ldc, int M, int N, int K,
                const GemmEpi &epi, hipStream_t stream) {
  const int eb = KIND == kBF16 ? 2 : 1;
  const int64_t kb = (int64_t)K * eb;
  VDNH3_HOST_CHECK(M > 0 && N > 0 && K > 0, VDNH3_ERR_INVALID, "gemm: M, N, K must be positive (%d, %d, %d)", M, N,
                   K);
  VDNH3_HOST_CHECK(kb % kGemmSK == 0, VDNH3_ERR_INVALID,
                   "gemm: K * element size must be a multiple of %d bytes (K=%d)", kGemmSK, K);
  VDNH3_HOST_CHECK((lda * eb) % 16 == 0 && (ldb * eb) % 16 == 0 && lda >= K && ldb >= K && ldc >= N,
                   VDNH3_ERR_INVALID, "gemm: leading dimensions must cover K/N and be 16-byte multiples");
  VDNH3_HOST_CHECK(reinterpret_cast<uintptr_t>(A) % 16 == 0 && reinterpret_cast<uintptr_t>(B) % 16 == 0,
                   VDNH3_ERR_INVALID, "gemm: A and B must be 16-byte aligned");
  VDNH3_HOST_CHECK((int64_t)256 * lda * eb < (int64_t(1) << 32) && (int64_t)256 * ldb * eb < (int64_t(1) << 32),
                   VDNH3_ERR_INVALID, "gemm: a 256-row panel of A or B must span less than 4 GB");
  const int mi = gemm_mi(M, N), bm = 32 * mi;
  GemmArgs args{static_cast<const uint8_t *>(A), static_cast<const uint8_t *>(B), lda * eb, ldb * eb, C, ldc, M, N,
                int(kb / kGemmSK)};
  args.tiles_m = (M + bm - 1) / bm;
  args.tiles_n = (N + kGemmBN - 1) / kGemmBN;
  args.total = args.tiles_m * args.tiles_n;
  args.per_xcd = (args.total + 7) / 8;
  args.epi = epi;
  launch_gemm_tiles<KIND>(mi, args, stream);
  return check_launch("gemm_nt");
}

}  // namespace
}  // namespace vdnh3

extern "C" int vdnh3_gemm_tile_rows(int M, int N) { return M > 0 && N > 0 ? 32 * vdnh3::gemm_mi(M, N) : 0; }

extern "C" int vdnh3_gemm(int kind, const void *A, int64_t lda, const void *B, int64_t ldb, void *C, int64_t ldc,
                          int M, int N, int K, const float *a_scale, int a_scale_n, const float *b_scale,
                          int b_scale_n, float alpha, const void *bias, int bias_bf16, int act, int out_type,
                          int accumulate, int round_linear, void *stream) {
  using namespace vdnh3;
  VDNH3_HOST_CHECK(A && B && C, VDNH3_ERR_INVALID, "gemm: null operand");
  VDNH3_HOST_CHECK(out_type >= kOutBF16 && out_type <= kOutI32, VDNH3_ERR_INVALID, "gemm: bad out_type %d", out_type);
  VDNH3_HOST_CHECK(out_type != kOutI32 || kind == kI8, VDNH3_ERR_INVALID, "gemm: int32 output needs int8 operands");
  VDNH3_HOST_CHECK(act == 0 || (act > 0 && (act & 1) && (act >> 1) <= N), VDNH3_ERR_INVALID,
                   "gemm: bad activation %d", act);
  VDNH3_HOST_CHECK(!(act && accumulate), VDNH3_ERR_INVALID, "gemm: a sigmoid epilogue cannot accumulate");
  VDNH3_HOST_CHECK(!a_scale || a_scale_n == 1 || a_scale_n == M, VDNH3_ERR_INVALID,
                   "gemm: a_scale must have 1 or M entries");
  VDNH3_HOST_CHECK(!b_scale || b_scale_n == 1 || b_scale_n == N, VDNH3_ERR_INVALID,
                   "gemm: b_scale must have 1 or N entries");
  GemmEpi epi{a_scale, b_scale, b_scale_n, a_scale_n, alpha, bias, bias_bf16, act & 1, act >> 1, out_type, accumulate,
              round_linear};
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (kind) {
    case kBF16:
      return launch_gemm<kBF16>(A, lda, B, ldb, C, ldc, M, N, K, epi, s);
    case kI8:
      return launch_gemm<kI8>(A, lda, B, ldb, C, ldc, M, N, K, epi, s);
    case kF8:
      return launch_gemm<kF8>(A, lda, B, ldb, C, ldc, M, N, K, epi, s);
    default:
      return set_error(VDNH3_ERR_INVALID, "gemm: unknown operand kind %d", kind);
  }
}
