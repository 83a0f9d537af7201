// Block-sparse local-window softmax attention for gfx950 (MI355X), bf16 MFMA.
//
// Computes O_i = softmax(scale * q_i K_A(i)^T) V_A(i) for the VDN-H3 window mask
// (vdn_h3/window.py:331-342) from a host-built tile plan (window_plan.cpp), with an
// optional fused per-head sigmoid gate (vdn_h3/hybrid.py:518-529).
//
// Work decomposition
//   one workgroup = 8 wavefronts = 256 query rows of one head x the key tiles of its run;
//   each wavefront owns 32 query rows and keeps its Q fragments in registers.
//   Scores are computed transposed, S^T = K Q^T, with v_mfma_f32_16x16x32_bf16: every lane
//   then owns one query of each 16-query block (lane % 16) and 24 of the 96 keys of a tile, so the row
//   maxima take three lane swaps and the probabilities P^T feed the next MFMA (O^T += V^T P^T)
//   straight from registers, without an LDS round trip. The 16x16 shape does the same work at 13% less
//   power than 32x32x16 (register-only rates 2003 against 1750 TFLOP/s on random operands), and this kernel
//   is power-bound: with the row sums below, 15.55 -> 15.02 ms at 40,688 x 40 x 128 and 2510 -> 2368 us at
//   16,007 x 56 x 128 (72 frames of 209 tokens), alternated on one machine. Where at most one workgroup a CU runs the
//   clock has room and the shape takes 2-4% longer (2,180 x 16 x 128 57.5 us against 55.9).
//   V^T is read from a copy made by a pre-pass (one extra 2*S*H*D-byte sweep): per head, one
//   contiguous image per 96-key tile, its 16-byte chunks already in the order and XOR swizzle of
//   the kernel's LDS tile, with keys interleaved in 16-key groups so that each lane's 8 MFMA
//   k-values are one 16-byte LDS read. K and V^T tiles go straight from HBM/L2 to LDS rings
//   (global_load_lds_dwordx4), each wavefront's load of a V^T tile one contiguous kilobyte; the
//   two halves of the workgroup alternate between the matrix cores and the VALU (see
//   window_attn_kernel).
//
// Scheduling
//   work items (query block, head) are ordered longest-first per head, and the flat
//   workgroup index is remapped so that each XCD (workgroups are dealt round-robin over
//   the 8 XCDs) runs a contiguous slice of that order: the resident workgroups of an
//   XCD work on the same head and neighbouring query blocks, so their K/V tiles are
//   shared in that XCD's L2.
#include "common.h"
#include "qk_norm.h"

namespace vdnh3 {
namespace {

constexpr int kBM = 256;  // query rows per workgroup (8 wavefronts x 32)
constexpr int kBN = 96;   // keys per tile: 102 MFMAs per wavefront and phase at D = 128
constexpr int kThreads = 512;
constexpr int kRing = 3;  // LDS slots per K and V^T ring (144 KB at D = 128): loads run kRing - 1 tiles ahead
// fragments a wavefront's LDS reads run ahead of its MFMAs: 8 / 6 / 5 / 4 measured 15.45 / 15.31 / 15.17 / 15.39 ms
// at the full shape, and with the row sums as MFMAs 6 / 5 / 4 15.04 / 15.09 / 15.02
constexpr int kAhead = 4;
constexpr float kLazy = 8.0f;  // log2 of the largest probability a stale running max allows
// The running max before the first score above it. Finite, so that a tile whose scores are all -inf (keys masked
// through a channel of q and k) adds zeros and not exp2(-inf + inf); and above every masked score of a type's
// lowest value, whose rounded product with the scale is no maximum to subtract: it is off by up to half its last place,
// and exp2 overflows at 128. A row with no score above it has no sum: 0 / 0, NaN, as of a row of -inf.
constexpr float kNoMax = -2147483648.0f;

// LDS position p (0..31) of V^T inside a 32-key group holds key offset kperm(p): the order in which lane
// group g = p / 8 holds its 8 keys of a k-step in two 16x16 blocks of S^T, whose rows are the K tile's LDS rows
// r, holding keys krow(r). The keys of lane groups 0 and 1 are those of the group's first half, so the PV product
// sums 16 keys before the next 16, bit for bit as 32x32x16 MFMAs do. Of the rounding only the row sums are
// then left apart from that shape's: 2e-5 of the output in 2-norm at 16,007 x 56 x 128 (with a lane group's keys 16
// apart 5e-5; a block's output 1.3e-5 to 2.5e-5 against 1.7e-4 to 2.4e-4). It costs nothing: the K tile loads
// fetch their rows in this order.
__host__ __device__ constexpr int kperm(int p) {
  return 16 * (p >> 4) + 8 * ((p & 7) >> 2) + 4 * ((p >> 3) & 1) + (p & 3);
}
__host__ __device__ constexpr int krow(int r) {
  return 32 * (r >> 5) + 16 * ((r >> 3) & 1) + 8 * ((r >> 4) & 1) + (r & 7);
}

// ---------------------------------------------------------------------------------
// LDS slots of the staged tiles. Each tile row is split into 16-byte chunks; chunk c of row r
// is stored at slot c ^ swizzle(r), so that the 16 lanes of one MFMA fragment read (16
// consecutive rows, one chunk column) hit 16 different 16-byte bank groups.
template <int D>
__device__ __forceinline__ int k_slot(int r, int c) {
  if constexpr (D == 128) return c ^ (r & 15);  // 16 chunks per 256-byte row
  else return c ^ ((r >> 1) & 7);               // 8 chunks per 128-byte row
}
__device__ __forceinline__ int v_slot(int d, int c) { return c ^ ((d >> 1) & 7); }  // 8 chunks per row
// the V^T tile's 32-key part (4 chunks per row): the 16 lanes of a fragment read (rows d..d+15)
// hit 16 different 16-byte bank groups
__device__ __forceinline__ int vb_slot(int d, int c) { return c ^ ((d >> 2) & 3); }

// Rows of the V^T copy and of the normalised q / k regions: seq rounded up to 192, a multiple of the
// pre-passes' 64-row blocks and of the attention's 96-key tiles, so a tile never reads past its head's
// region.
__host__ __device__ constexpr int pad_rows(int seq) { return (seq + 191) / 192 * 192; }

// ---------------------------------------------------------------------------------
// The V^T copy is a sequence of tile images, one per 96-key tile: the image of keys [ks, ks + 96)
// of head h starts at element (h * s_pad + ks) * D and holds the tile's 16-byte chunks in LDS
// order: position P < 8 D is (d = P / 8, slot P % 8) of the 64-key part, holding chunk
// v_slot(d, slot) of keys [ks, ks + 64) of V^T row d; position 8 D + 4 d + slot of the 32-key part
// holds chunk vb_slot(d, slot) of keys [ks + 64, ks + 96). Inside a chunk the 8 keys follow kperm
// within their 32-key group; keys past seq are zero. A tile load is then a contiguous copy.
// write_vt_image: the image chunks of the 64 keys [k0, k0 + 64) (k0 a multiple of 64) from their V rows
// staged in LDS (row r at rows + r * P), into the head's images at vt_head. A 64-key block holds whole
// 32-key groups, so every chunk it writes is complete; it covers one or two tiles.
template <int D, int P>
__device__ __forceinline__ void write_vt_image(const uint16_t *rows, int k0, uint16_t *__restrict__ vt_head,
                                               int tid) {
  for (int cc = tid; cc < D * 8; cc += kThreads) {
    const int d = cc >> 3, pc = cc & 7;  // V^T row; chunk pc holds key slots 8 pc .. 8 pc + 7 of the block
    const int key = k0 + 8 * pc, tile = key / kBN, sb = key - tile * kBN;
    const int pos = sb < 64 ? 8 * d + v_slot(d, sb >> 3) : 8 * D + 4 * d + vb_slot(d, (sb - 64) >> 3);
    uint16_t e[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int p = 8 * pc + j;
      e[j] = rows[((p & ~31) + kperm(p & 31)) * P + d];
    }
    uint4 o;
    o.x = uint32_t(e[0]) | (uint32_t(e[1]) << 16);
    o.y = uint32_t(e[2]) | (uint32_t(e[3]) << 16);
    o.z = uint32_t(e[4]) | (uint32_t(e[5]) << 16);
    o.w = uint32_t(e[6]) | (uint32_t(e[7]) << 16);
    *reinterpret_cast<uint4 *>(vt_head + (int64_t)tile * (kBN * D) + pos * 8) = o;
  }
}

// ---------------------------------------------------------------------------------
// Pre-pass: V [seq, heads, D] (strided view) -> the V^T tile images, 64 keys per workgroup.
// grid (s_pad / 64, heads), kThreads threads.
template <int D>
__global__ __launch_bounds__(kThreads) void vt_prepass_kernel(const uint16_t *__restrict__ v, int64_t v_row,
                                                              int64_t v_head, uint16_t *__restrict__ vt,
                                                              int seq, int s_pad) {
  constexpr int P = D + 8;
  __shared__ __attribute__((aligned(16))) uint16_t tile[64 * P];
  const int k0 = blockIdx.x * 64, head = blockIdx.y, tid = threadIdx.x;
  constexpr int CH = D / 8;  // 16-byte chunks per key row
  for (int c = tid; c < 64 * CH; c += kThreads) {
    int r = c / CH, col = c % CH, key = k0 + r;
    uint4 val = make_uint4(0, 0, 0, 0);
    if (key < seq) val = *reinterpret_cast<const uint4 *>(v + key * v_row + head * v_head + col * 8);
    *reinterpret_cast<uint4 *>(&tile[r * P + col * 8]) = val;
  }
  __syncthreads();
  write_vt_image<D, P>(tile, k0, vt + (int64_t)head * s_pad * D, tid);
}

// ---------------------------------------------------------------------------------
// The block's q_norm / k_norm (RMSNorm over the head dim, with ROPE the split-half rotation, one
// bf16 rounding: the arithmetic of qk_norm.h) of the BR rows [k0, k0 + BR) of one head at a
// time, written head-major (row r at dst + r * D), zero for rows at or past seq. Each row is
// normalised by an aligned group of D/8 lanes, one 8-channel chunk per lane (THREADS / (D/8) rows
// per pass; with D = 64 the last pass is partly idle). A lane loads the RoPE matrix rows its chunk
// uses once (the constructor) and reuses them for every head (run): row 0 (f00, f01) below half,
// row 1 (f10, f11) above.
template <int D, bool ROPE, int THREADS, int BR>
struct RowNorm {
  static constexpr int CH = D / 8, ROWS = THREADS / CH, ITER = (BR + ROWS - 1) / ROWS;
  // row r0 + it * ROWS lies in the block (a whole row group is in or out)
  __device__ __forceinline__ bool in_block(int it) const { return BR % ROWS == 0 || r0 + it * ROWS < BR; }
  int c, r0, half, k0, seq;
  bool first, rotated;
  float2 fm[ITER][ROPE ? 8 : 1];

  __device__ __forceinline__ RowNorm(const float *__restrict__ freqs, int64_t f_row, int rot, int k0_, int seq_,
                                     int tid)
      : c(tid % CH), r0(tid / CH), half(rot >> 1), k0(k0_), seq(seq_) {
    first = 8 * c < half;
    rotated = ROPE && 8 * c < rot;
    if constexpr (ROPE) {
#pragma unroll
      for (int it = 0; it < ITER; ++it) {
        const int key = k0 + r0 + it * ROWS;
        if (rotated && key < seq && in_block(it)) {
          const float *f = freqs + key * f_row + 4 * (first ? 8 * c : 8 * c - half) + (first ? 0 : 2);
#pragma unroll
          for (int j = 0; j < 8; ++j) fm[it][j] = *reinterpret_cast<const float2 *>(f + 4 * j);
        }
      }
    }
  }

  __device__ __forceinline__ void run(const uint16_t *__restrict__ x, int64_t x_row, int64_t x_head,
                                      const uint16_t *__restrict__ weight, float eps, uint16_t *__restrict__ dst,
                                      int head) const {
    float wf[8];
    {
      const u32x4_t w = ld16(weight + 8 * c);
#pragma unroll
      for (int j = 0; j < 8; ++j) wf[j] = __uint_as_float((j & 1) ? (w[j >> 1] & 0xffff0000u) : (w[j >> 1] << 16));
    }
    u32x4_t raw[ITER];
#pragma unroll
    for (int it = 0; it < ITER; ++it) {
      const int key = k0 + r0 + it * ROWS;
      raw[it] = key < seq && in_block(it) ? ld16(x + key * x_row + head * x_head + 8 * c) : u32x4_t{0, 0, 0, 0};
    }
#pragma unroll
    for (int it = 0; it < ITER; ++it) {
      if (!in_block(it)) continue;
      const int r = r0 + it * ROWS;
      const bool live = k0 + r < seq;
      float xf[8], y[8];
#pragma unroll
      for (int j = 0; j < 8; ++j)
        xf[j] = __uint_as_float((j & 1) ? (raw[it][j >> 1] & 0xffff0000u) : (raw[it][j >> 1] << 16));
      const float rr = rms_factor(group_tree_sum<CH>(chunk_sumsq(xf)), D, eps);
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = xf[j] * rr * wf[j];
      if constexpr (ROPE) {
        // the partner chunk (8c +- half) is lane c +- half / 8 of the same row group
        const int lane = __lane_id(), step = half >> 3;
        const int partner = rotated ? (first ? lane + step : lane - step) : lane;
        float o[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = __shfl(y[j], partner);
        if (rotated && live) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float2 m = fm[it][j];
            y[j] = rope_rotate(y[j], o[j], f32x4_t{m.x, m.y, m.x, m.y}, first);
          }
        }
      }
      if (!live) {
#pragma unroll
        for (int j = 0; j < 8; ++j) y[j] = 0.f;
      }
      st16(dst + r * D + 8 * c, u32x4_t{pack_bf2(y[0], y[1]), pack_bf2(y[2], y[3]), pack_bf2(y[4], y[5]),
                                        pack_bf2(y[6], y[7])});
    }
  }
};

// Heads per pre-pass workgroup. Without RoPE a workgroup has nothing to share between heads: one each
// (8,296 x 40 x 128: 70 us against 95 with ten, 40,688: 320 against 350, 1,808: 15 against 26). With RoPE the
// heads of a workgroup share its rows' matrices (about three heads' worth of work to load), against rounds
// of workgroups over the 512 places (two per CU); up to 256 workgroups have a CU each and run about a quarter
// faster. 40,688 rows so take 10 heads (519 us; 5: 522, 4: 538, 1: 680), 8,296 rows 6 (120 us; 10: 153, 5: 132,
// 1: 148) and 1,808 rows 3 (27 us; 10: 46, 4: 31, 1: 34).
int prepass_heads(int blocks, int heads, bool rope) {
  if (!rope) return 1;
  int best = 1;
  int64_t best_cost = INT64_MAX;
  for (int h = 1; h <= 10 && h <= heads; ++h) {
    const int64_t wgs = (int64_t)blocks * ((heads + h - 1) / h);
    const int64_t cost = (wgs <= 256 ? 3 : 4 * ((wgs + 511) / 512)) * (h + 3);
    if (cost < best_cost) best = h, best_cost = cost;
  }
  return best;
}

// Pre-pass of the normalising attention, for the 64 rows [k0, k0 + 64) of up to group_heads
// heads: the V^T image chunks of vt_prepass_kernel, the normalised keys kn[head][key][d] and, when q
// is given, the normalised queries qn[head][row][d] (RowNorm). V tiles alternate between two LDS
// buffers, so one barrier per head orders the tile's writes before its transposed reads, and the
// reads of a buffer before its next writes.
template <int D, bool ROPE>
__global__ __launch_bounds__(kThreads) void qkv_prepass_kernel(
    const uint16_t *__restrict__ q, int64_t q_row, int64_t q_head, const uint16_t *__restrict__ q_weight, float q_eps,
    const uint16_t *__restrict__ k, int64_t k_row, int64_t k_head, const uint16_t *__restrict__ k_weight, float k_eps,
    const uint16_t *__restrict__ v, int64_t v_row, int64_t v_head, const float *__restrict__ freqs, int64_t f_row,
    int rot, uint16_t *__restrict__ vt, uint16_t *__restrict__ kn, uint16_t *__restrict__ qn, int seq, int s_pad,
    int heads, int group_heads) {
  constexpr int P = D + 8;
  constexpr int CH = D / 8;  // 16-byte chunks per row
  __shared__ __attribute__((aligned(16))) uint16_t tile[2][64 * P];
  const int h0 = blockIdx.x * group_heads, h1 = min(heads, h0 + group_heads);
  const int k0 = blockIdx.y * 64, tid = threadIdx.x;
  const RowNorm<D, ROPE, kThreads, 64> norm(freqs, f_row, rot, k0, seq, tid);
  for (int head = h0; head < h1; ++head) {
    uint16_t *buf = tile[head & 1];
    for (int cc = tid; cc < 64 * CH; cc += kThreads) {
      int r = cc / CH, col = cc % CH, key = k0 + r;
      uint4 val = make_uint4(0, 0, 0, 0);
      if (key < seq) val = *reinterpret_cast<const uint4 *>(v + key * v_row + head * v_head + col * 8);
      *reinterpret_cast<uint4 *>(&buf[r * P + col * 8]) = val;
    }
    const int64_t off = ((int64_t)head * s_pad + k0) * D;
    norm.run(k, k_row, k_head, k_weight, k_eps, kn + off, head);
    if (q) norm.run(q, q_row, q_head, q_weight, q_eps, qn + off, head);
    __syncthreads();
    write_vt_image<D, P>(buf, k0, vt + (int64_t)head * s_pad * D, tid);
  }
}



// Reductions over the four 16-lane groups of a wavefront through v_permlane32_swap / v_permlane16_swap (gfx950).
// lanes < 32: max of a over lane groups (g, g + 2); lanes >= 32: the same of b
__device__ __forceinline__ float max_pair32(float a, float b) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
// a over the four lane groups, b over the four lane groups, each in every lane
__device__ __forceinline__ void group_max(float &a, float &b) {
  const uint32_t x = __float_as_uint(max_pair32(a, b));
  const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  const uint32_t y = __float_as_uint(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
  const auto q = __builtin_amdgcn_permlane32_swap(y, y, false, false);
  a = __uint_as_float(q[0]);
  b = __uint_as_float(q[1]);
}

constexpr int kNQ = 2;  // 16-query blocks per wavefront

// The Q^T fragments of a wavefront: lane (l16, g) holds channels 32 s + 8 g + j (j < 8) of query rows
// q0 + 16 n + l16, chunk 4 s + g (rows at or past q1 read row q1 - 1). QNORM: q is normalised as it is
// loaded (the block's q_norm with q_weight / q_eps, the arithmetic of qk_norm.h); otherwise q is used as given.
template <int D, bool QNORM>
__device__ __forceinline__ void load_q_frags(const uint16_t *__restrict__ q, int64_t q_row, int64_t q_head, int q0,
                                             int q1, int head, int l16, int g, const uint16_t *__restrict__ q_weight,
                                             float q_eps, bf16x8_t (&qf)[kNQ][D / 32]) {
  constexpr int NS = D / 32;
#pragma unroll
  for (int n = 0; n < kNQ; ++n) {
    const uint16_t *qp = q + (int64_t)min(q0 + 16 * n + l16, q1 - 1) * q_row + (int64_t)head * q_head + 8 * g;
    if constexpr (!QNORM) {
#pragma unroll
      for (int s = 0; s < NS; ++s) qf[n][s] = as_bf16x8(ld16(qp + 32 * s));
    } else {
      float y[NS][8], p[NS];
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const u32x4_t raw = ld16(qp + 32 * s);
#pragma unroll
        for (int j = 0; j < 8; ++j)
          y[s][j] = __uint_as_float((j & 1) ? (raw[j >> 1] & 0xffff0000u) : (raw[j >> 1] << 16));
        p[s] = chunk_sumsq(y[s]);
      }
      const float rr = rms_factor(quarters_tree_sum<NS>(p), D, q_eps);
#pragma unroll
      for (int s = 0; s < NS; ++s) {
        const u32x4_t w = ld16(q_weight + 32 * s + 8 * g);
#pragma unroll
        for (int j = 0; j < 8; ++j)
          y[s][j] = y[s][j] * rr * __uint_as_float((j & 1) ? (w[j >> 1] & 0xffff0000u) : (w[j >> 1] << 16));
        qf[n][s] = as_bf16x8(u32x4_t{pack_bf2(y[s][0], y[s][1]), pack_bf2(y[s][2], y[s][3]),
                                     pack_bf2(y[s][4], y[s][5]), pack_bf2(y[s][6], y[s][7])});
      }
    }
  }
}

// The output rows of a wavefront: O = O^T / l, rounded to bf16, times the row's gate when one is given
// (the gate fused into the attention epilogue). Every element of l[n] holds the row sum of the lane's query.
template <int D>
__device__ __forceinline__ void store_rows(const f32x4_t (&oacc)[D / 16][kNQ], const f32x4_t (&l)[kNQ], int q0,
                                           int q1, const uint16_t *__restrict__ gate, int64_t g_row, int head,
                                           uint16_t *__restrict__ out, int64_t o_row, int64_t o_head, int l16, int g) {
#pragma unroll
  for (int n = 0; n < kNQ; ++n) {
    const float inv = 1.f / l[n][0];
    const int qr = q0 + 16 * n + l16;
    if (qr >= q1) continue;
    const float gv = gate ? bf2f(gate[(int64_t)qr * g_row + head]) : 1.f;
    uint16_t *op = out + (int64_t)qr * o_row + (int64_t)head * o_head + 4 * g;
#pragma unroll
    for (int m = 0; m < D / 16; ++m) {
      float v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v[r] = round_bf(oacc[m][n][r] * inv);
        if (gate) v[r] *= gv;
      }
      *reinterpret_cast<uint2 *>(op + 16 * m) = make_uint2(pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]));
    }
  }
}

// The partial result of a wavefront's rows over one split of their key tiles: O^T unnormalised, the running
// max (base 2) and the row sum, [split][head][row][D] and [split][head][row][2] fp32.
struct Partial {
  float *o, *ml;  // null: the whole key set in one workgroup
};
template <int D>
__device__ __forceinline__ void store_partial(const f32x4_t (&oacc)[D / 16][kNQ], const f32x4_t (&l)[kNQ],
                                              const float (&m_run)[kNQ], int q0, int q1, const Partial &part,
                                              int64_t head_rows, int l16, int g) {
#pragma unroll
  for (int n = 0; n < kNQ; ++n) {
    const int qr = q0 + 16 * n + l16;
    if (qr >= q1) continue;
    float *op = part.o + (head_rows + qr) * D + 4 * g;
#pragma unroll
    for (int m = 0; m < D / 16; ++m) *reinterpret_cast<f32x4_t *>(op + 16 * m) = oacc[m][n];
    if (g == 0) *reinterpret_cast<float2 *>(part.ml + (head_rows + qr) * 2) = make_float2(m_run[n], l[n][0]);
  }
}

// Combines the splits of every row: O = sum_s 2^(m_s - m) O_s / sum_s 2^(m_s - m) l_s, m = max m_s; the
// rounding and the gate as store_rows. One thread per 8 channels of a (row, head).
template <int D>
__global__ __launch_bounds__(256) void combine_kernel(Partial part, int splits, int seq, int heads,
                                                      const uint16_t *__restrict__ gate, int64_t g_row,
                                                      uint16_t *__restrict__ out, int64_t o_row, int64_t o_head) {
  constexpr int CH = D / 8;
  const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int64_t rows = (int64_t)heads * seq;
  if (e >= rows * CH) return;
  const int64_t hr = e / CH;
  const int c = (int)(e - hr * CH), head = (int)(hr / seq), row = (int)(hr - (int64_t)head * seq);
  float m = -INFINITY;
  for (int s = 0; s < splits; ++s) m = fmaxf(m, part.ml[(s * rows + hr) * 2]);
  f32x4_t o[2] = {};
  float l = 0.f;
  for (int s = 0; s < splits; ++s) {
    const float2 ml = *reinterpret_cast<const float2 *>(part.ml + (s * rows + hr) * 2);
    const float w = __builtin_amdgcn_exp2f(ml.x - m);
    const f32x4_t *op = reinterpret_cast<const f32x4_t *>(part.o + (s * rows + hr) * D + 8 * c);
    o[0] += w * op[0];
    o[1] += w * op[1];
    l += w * ml.y;
  }
  const float inv = 1.f / l;
  const float gv = gate ? bf2f(gate[(int64_t)row * g_row + head]) : 1.f;
  float v[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    v[j] = round_bf(o[j >> 2][j & 3] * inv);
    if (gate) v[j] *= gv;
  }
  uint16_t *dst = out + (int64_t)row * o_row + (int64_t)head * o_head + 8 * c;  // 8-byte aligned
  *reinterpret_cast<uint2 *>(dst) = make_uint2(pack_bf2(v[0], v[1]), pack_bf2(v[2], v[3]));
  *reinterpret_cast<uint2 *>(dst + 4) = make_uint2(pack_bf2(v[4], v[5]), pack_bf2(v[6], v[7]));
}

// ---------------------------------------------------------------------------------
// Two-group ping-pong over the key tiles t = 0..T-1 of a work item (256 query rows of one head).
// Waves 0-3 (group A) and 4-7 (group B) each own 32 query rows; wave w and w + 4 share a SIMD.
// The item runs in barrier-separated phases p = 0 .. 2T+1; in each phase one group works on the
// matrix cores and the other on the VALU, so the two waves of every SIMD alternate:
//   MFMA phase of tile t :  O^T += V(t-1)^T P(t-1)^T, l += 1^T P(t-1)^T, S(t)^T = K(t) Q^T  (102 MFMAs)
//   VALU phase of tile t :  P(t) = exp2(scale S(t) - m), row max, O and l rescale   (softmax)
// Group A runs tile t's MFMA phase in phase 2t and its VALU phase in 2t+1; group B one phase
// later. K(t) and V(t-1) are read in phases 2t and 2t+1 only; tiles are loaded direct to LDS
// into three-slot rings, two tiles ahead: K tiles by group A and V^T tiles by group B, each at
// the start of the issuing group's VALU phase, so the MFMA stream carries no memory instruction
// and a tile that misses L2 has two tiles' time to land. A tile is 96 keys: every phase switch
// (a barrier, the first fragment reads of the MFMA phase) is shared by 96 16x16 MFMAs per wavefront, a
// third fewer switches than with 64-key tiles for the same work. The VALU phase is the longer one, so the row
// sums of P are six more MFMAs against a fragment of ones instead of 24 dot products in it (and come out
// summed over the lane groups): 15.30 -> 15.06 ms at 40,688 x 40 x 128, 2406 -> 2370 us at 16,007 x 56 x 128.
// QNORM: q is normalised as it is loaded (the block's q_norm with q_weight / q_eps, the arithmetic
// of qk_norm.h); otherwise q is used as given.
template <int D, bool QNORM>
__global__ __launch_bounds__(kThreads, 1) void window_attn_kernel(
    const uint16_t *__restrict__ q, int64_t q_row, int64_t q_head, const uint16_t *__restrict__ k, int64_t k_row,
    int64_t k_head, const uint16_t *__restrict__ vt, int s_pad, uint16_t *__restrict__ out, int64_t o_row,
    int64_t o_head, const uint16_t *__restrict__ gate, int64_t g_row, int seq, float scale_log2,
    const int4 *__restrict__ items, int n_items, const int2 *__restrict__ tiles, int per_xcd, int total,
    const uint16_t *__restrict__ q_weight, float q_eps, Partial part) {
  constexpr int KC = D / 8;    // 16-byte chunks per K row
  constexpr int NS = D / 32;   // k-steps of the QK^T contraction
  constexpr int NO = D / 16;   // 16-row blocks of O^T
  constexpr int NKB = kBN / 16;  // 16-key blocks of S^T
  constexpr int NT = kBN / 32;   // k-steps of the PV contraction
  constexpr int KT = kBN * D, VT = D * kBN;  // elements per tile
  // a V^T tile in LDS: keys 0..63 as [D][8 chunks] (v_slot), then keys 64..95 as [D][4 chunks] (vb_slot)
  constexpr int VA = D * 64;
  static_assert(kBN == 96, "the V^T tile layout is a 64-key part and a 32-key part");
  __shared__ __attribute__((aligned(16))) uint16_t Ks[kRing][KT];
  __shared__ __attribute__((aligned(16))) uint16_t Vs[kRing][VT];

  const int bid = blockIdx.x;
  const int L = (bid & 7) * per_xcd + (bid >> 3);
  if (L >= total) return;
  const int head = L / n_items;
  const int4 item = items[L - head * n_items];
  // grid.y splits of the item's key tiles
  const int t0 = item.w * (int)blockIdx.y / (int)gridDim.y, t1 = item.w * ((int)blockIdx.y + 1) / (int)gridDim.y;
  const int q0 = item.x, q1 = item.y, toff = item.z + t0, T = t1 - t0;

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  if (T == 0) {  // more splits than the item has tiles: this one adds nothing
    if (part.o) {
      const int64_t row = ((int64_t)blockIdx.y * (total / n_items) + head) * seq + q0;
      for (int e = tid; e < (q1 - q0) * D; e += kThreads) part.o[row * D + e] = 0.f;
      for (int r = tid; r < q1 - q0; r += kThreads)
        *reinterpret_cast<float2 *>(part.ml + (row + r) * 2) = make_float2(kNoMax, 0.f);
    }
    return;
  }
  const int l16 = lane & 15, g = lane >> 4;
  const int group = wave >> 2;
  // a wavefront whose 32 rows all lie past the item's end (the short last item of a run) skips
  // its fragment reads, MFMAs and softmax; it still issues its share of the tile loads and
  // joins every barrier
  const bool rows_live = q0 + wave * 32 < q1;

  bf16x8_t qf[kNQ][NS];
  load_q_frags<D, QNORM>(q, q_row, q_head, q0 + wave * 32, q1, head, l16, g, q_weight, q_eps, qf);

  const uint16_t *kbase = k + (int64_t)head * k_head;
  const uint16_t *vbase = vt + (int64_t)head * D * s_pad;
  // Tile loads, by one group of 256 threads: thread chunk i fills LDS position P = 256 i + gtid
  // (16-byte units) of the tile. In a K tile, P is (row P / KC, slot P % KC) and holds chunk
  // slot ^ swizzle(row) of key row krow(row); row kr0 + i * 256 / KC has the same swizzle for every i.
  // A V^T tile image is already in LDS order: P comes from position P of the image.
  // Rows past seq read row seq - 1 (their scores are masked).
  constexpr int KCG = kBN * KC / 256, VCG = D * (kBN / 8) / 256;  // 16-byte chunks per thread and tile
  static_assert(KCG >= 1 && VCG >= 1 && KCG == VCG, "both groups issue the same number of loads");
  const int gtid = tid & 255, gw = wave & 3;
  const int kr0 = gtid / KC;
  const int kslot = k_slot<D>(kr0, gtid % KC) * 8;
  // per-lane byte offsets of this group's chunks inside a tile's source rows (K rows for group
  // A, V^T rows for group B) and the tile's LDS base of this wavefront: an issue is a scalar
  // tile base, a scalar M0 and the load
  uint32_t doff[KCG];
#pragma unroll
  for (int i = 0; i < KCG; ++i) {
    const int P = 256 * i + gtid;
    doff[i] = 2u * (group == 0 ? (uint32_t)(krow(kr0 + i * (256 / KC)) * (int)k_row + kslot) : (uint32_t)(P * 8));
  }
  const uint32_t lds_dma = __builtin_amdgcn_readfirstlane(
      (group == 0 ? lds_address(&Ks[0][0]) : lds_address(&Vs[0][0])) + gw * 64 * 16);
  constexpr uint32_t kTileBytes = KT * 2;
  static_assert(KT == VT, "K and V^T tiles have the same size");
  // this group's loads of the tile whose first key is ks into ring slot `slot`; the last K tile
  // of the sequence reads rows past seq as row seq - 1 (their scores are masked)
  auto tile_dma = [&](int ks, int slot) __device__ {
    const uint16_t *base = group == 0 ? kbase + (int64_t)ks * k_row : vbase + (int64_t)ks * D;
    uint32_t off[KCG];
#pragma unroll
    for (int i = 0; i < KCG; ++i) off[i] = doff[i];
    if (group == 0 && ks + kBN > seq) {  // uniform: taken for the last tile of the sequence only
#pragma unroll
      for (int i = 0; i < KCG; ++i)
        off[i] = 2u * (uint32_t)((min(ks + krow(kr0 + i * (256 / KC)), seq - 1) - ks) * (int)k_row + kslot);
    }
#pragma unroll
    for (int i = 0; i < KCG; ++i)
      global_to_lds16_sbase(base, off[i], lds_dma + (uint32_t)slot * kTileBytes + (uint32_t)(i * 256 * 16));
  };

  // Fragment offsets inside a tile (elements). The swizzles depend on the row only through
  // l16 (r = 16 kb + l16, d = 16 m + l16), so the 16-row blocks differ by constant offsets.
  int kfo[NS], vfo[NT];
#pragma unroll
  for (int st = 0; st < NS; ++st) kfo[st] = (l16 * KC + k_slot<D>(l16, 4 * st + g)) * 8;
#pragma unroll
  for (int tt = 0; tt < NT; ++tt)
    vfo[tt] = tt < 2 ? (l16 * 8 + v_slot(l16, 4 * tt + g)) * 8 : VA + (l16 * 4 + vb_slot(l16, g)) * 8;

  f32x4_t oacc[NO][kNQ], sacc[NKB][kNQ];
  u32x4_t pb[NT][kNQ];  // P^T fragments: bf16 pairs
  f32x4_t l_run[kNQ];    // row sums of P: every element of a lane's vector is its query's sum
  const u32x4_t ones = {0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u};  // eight bf16 1.0
  float m_run[kNQ];
#pragma unroll
  for (int n = 0; n < kNQ; ++n) {
#pragma unroll
    for (int m = 0; m < NO; ++m) oacc[m][n] = f32x4_t{};
#pragma unroll
    for (int j = 0; j < NT; ++j) pb[j][n] = u32x4_t{};
    m_run[n] = kNoMax;
    l_run[n] = f32x4_t{};
  }

  // Rings: K(tau) and V(tau) live in slot tau % kRing. K(t) and V(t-1) are read in phases 2t
  // (group A) and 2t+1 (group B). Tile loads are issued by the group in its VALU phase, so the
  // MFMA stream carries no memory instruction: in its VALU phase of tile t, group A issues
  // K(t+kRing-1) (phase 2t+1) over K(t-1), last read in phase 2t-1, and group B issues
  // V(t+kRing-1) (phase 2t+2) over V(t-1), last read in phase 2t+1. In each phase the slot
  // being written differs from the K and V slots the MFMA group reads. Past the end the tile
  // index is clamped to T-1: such loads rewrite
  // slots that no real tile reads any more, and every VALU phase issues the same count, so each
  // group's vmcnt wait at the end of odd phases is exact.
  // prologue: K(0..kRing-2) by group A, V(0..kRing-3) by group B, all landed; V(-1), the V^T
  // slot read by the PV of tile 0 (with P(-1) = 0), is zeroed so that product is exactly zero.
  // Group B's first issue (phase 0) is V(kRing-2).
#pragma unroll
  for (int j = 0; j < kRing - 1; ++j)
    if (j < kRing - 2 || group == 0) tile_dma(tiles[toff + min(j, T - 1)].x, j);
  for (int i = tid; i < VT / 8; i += kThreads) st16(Vs[kRing - 1] + i * 8, u32x4_t{0, 0, 0, 0});
  wait_vm_lds<0>();
  bare_barrier();

  // Descriptors of the next VALU phase of this group (the key start of its tile load and the
  // mask bounds of its tile), scalar loads made at the end of the group's MFMA phase and
  // consumed after the barrier. Group B's first VALU phase (phase 0, tile -1) issues V(kRing-2).
  int dma_ks = group == 0 ? 0 : tiles[toff + min(kRing - 2, T - 1)].x;
  int mask = 0;

  const int phases = 2 * T + 2;
  for (int p = 0; p < phases; ++p) {
    // Group A (B) works on the matrix cores in even (odd) phases. Both tile indices depend on
    // p only, so tile descriptors are scalar loads.
    const int t_mfma = p >> 1;            // A: p = 2t; B: p = 2t + 1
    const int t_valu = (p - 1) >> 1;      // A: p = 2t + 1 (odd); B: p = 2t + 2 (even)
    if (group == (p & 1)) {
      if (!rows_live) {
        // descriptors of this group's next VALU phase (tile t_mfma)
        dma_ks = tiles[toff + min(t_mfma + kRing - 1, T - 1)].x;
      } else {
      // MFMA phase of tile t: O^T += V(t-1)^T P(t-1)^T, S(t)^T = K(t) Q^T (48 + 48 MFMAs at D = 128) and
      // l += 1^T P(t-1)^T (6).
      // t = 0 has no PV and t = T no QK: those phases run on a zero tile / discard the scores,
      // so the phase is one branch-free block. Fragment reads run kAhead fragments ahead.
      const int t = t_mfma;
      const uint16_t *vtile = Vs[(t + kRing - 1) % kRing];
      const uint16_t *ktile = Ks[t % kRing];
      // fragment i < NP: V^T block m = i % NO, k-step tt = i / NO; i >= NP: K block kb = (i - NP) % NKB,
      // k-step st = (i - NP) / NKB. Each feeds kNQ MFMAs (one per query block), the query blocks in
      // alternating order, so successive MFMAs share an operand (less toggling, less power) and none
      // waits for the result of the one before it.
      constexpr int NP = NO * NT, NF = NP + NKB * NS;
      auto frag = [&](int i) __device__ {
        if (i < NP) {
          const int m = i % NO, tt = i / NO;
          return ld16(vtile + (tt < 2 ? m * 16 * 64 : m * 16 * 32) + vfo[tt]);
        }
        return ld16(ktile + ((i - NP) % NKB) * 16 * D + kfo[(i - NP) / NKB]);
      };
      // the MFMA wave of each SIMD issues ahead of the VALU wave sharing it
      __builtin_amdgcn_s_setprio(1);
      u32x4_t fr[kAhead];
#pragma unroll
      for (int i = 0; i < kAhead; ++i) fr[i] = frag(i);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < NF; ++i) {
        const u32x4_t a = fr[i % kAhead];
#pragma unroll
        for (int x = 0; x < kNQ; ++x) {
          const int n = (i & 1) ? kNQ - 1 - x : x;
          if (i < NP) {
            oacc[i % NO][n] = mfma_bf16_16x16x32(as_bf16x8(a), as_bf16x8(pb[i / NO][n]), oacc[i % NO][n]);
            if (i % NO == NO - 1) l_run[n] = mfma_bf16_16x16x32(as_bf16x8(ones), as_bf16x8(pb[i / NO][n]), l_run[n]);
          } else {
            const int kb = (i - NP) % NKB, st = (i - NP) / NKB;
            if (st == 0) sacc[kb][n] = f32x4_t{};
            sacc[kb][n] = mfma_bf16_16x16x32(as_bf16x8(a), qf[n][st], sacc[kb][n]);
          }
        }
        if (i + kAhead < NF) fr[i % kAhead] = frag(i + kAhead);
        __builtin_amdgcn_sched_barrier(0);
      }
      __builtin_amdgcn_s_setprio(0);
      // descriptors of this group's next VALU phase (tile t): its DMA issue and its mask
      dma_ks = tiles[toff + min(t + kRing - 1, T - 1)].x;
      mask = t < T ? tiles[toff + t].y : 0;
      }
    } else {
      // VALU phase of tile t: first this group's tile loads (two tiles ahead), then the softmax
      // in base 2; a lane holds 24 of the 96 scores of each of its two queries. The running max m_run
      // moves only when this tile's max exceeds it by more than 2^kLazy: probabilities stay below
      // 2^kLazy (exact softmax either way, a common shift cancels in O / l) and most tiles skip the
      // rescale.
      tile_dma(dma_ks, (t_valu + kRing - 1) % kRing);
      const bool work = rows_live && p >= 1 + group && t_valu < T;
      if (work) {
        const int lo = mask & 0xffff, hi = mask >> 16;
        if (lo > 0 || hi < kBN) {
#pragma unroll
          for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int ko = krow(16 * kb) + krow(4 * g) + i;
              if (ko < lo || ko >= hi) {
#pragma unroll
                for (int n = 0; n < kNQ; ++n) sacc[kb][n][i] = -INFINITY;
              }
            }
        }
        // tile row max over the lane's 24 scores of a query as a tree of three-input maxima (8 + 3
        // v_max3), then over the four lane groups for both queries in three lane swaps
        static_assert(NKB == 6 && kNQ == 2, "the max tree is written for 2 x 24 scores per lane");
        float mt[kNQ];
#pragma unroll
        for (int n = 0; n < kNQ; ++n) {
          float m1[8];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            m1[i] = fmaxf(fmaxf(sacc[0][n][i], sacc[1][n][i]), sacc[2][n][i]);
            m1[4 + i] = fmaxf(fmaxf(sacc[3][n][i], sacc[4][n][i]), sacc[5][n][i]);
          }
          const float a = fmaxf(fmaxf(m1[0], m1[1]), m1[2]), b = fmaxf(fmaxf(m1[3], m1[4]), m1[5]);
          mt[n] = fmaxf(fmaxf(a, b), fmaxf(m1[6], m1[7]));
        }
        group_max(mt[0], mt[1]);
        bool grow = false;
#pragma unroll
        for (int n = 0; n < kNQ; ++n) {
          mt[n] *= scale_log2;
          grow = grow || mt[n] > m_run[n] + kLazy;
        }
        if (__any(grow)) {
#pragma unroll
          for (int n = 0; n < kNQ; ++n) {
            const float m_new = mt[n] > m_run[n] + kLazy ? mt[n] : m_run[n];
            const float corr = __builtin_amdgcn_exp2f(m_run[n] - m_new);
            m_run[n] = m_new;
            l_run[n] *= corr;
#pragma unroll
            for (int m = 0; m < NO; ++m) oacc[m][n] *= corr;
          }
        }
        // P in bf16 pairs (the values the PV product and the row sums use)
#pragma unroll
        for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
          for (int n = 0; n < kNQ; ++n)
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
              const float p0 = __builtin_amdgcn_exp2f(fmaf(sacc[kb][n][i], scale_log2, -m_run[n]));
              const float p1 = __builtin_amdgcn_exp2f(fmaf(sacc[kb][n][i + 1], scale_log2, -m_run[n]));
              pb[kb >> 1][n][2 * (kb & 1) + (i >> 1)] = pack_bf2(p0, p1);
            }
      }
    }
    // before an even phase 2(t+1): K(t+1) and V(t) (issued kRing - 1 issues ago by their group)
    // have landed; each group's two latest issues may still be in flight
    if (p & 1) wait_vm_lds<(kRing - 2) * KCG>();
    bare_barrier();
  }

  wait_vm_lds<0>();  // no tile load may land in LDS after the workgroup ends
  if (part.o)
    store_partial<D>(oacc, l_run, m_run, q0 + wave * 32, q1, part,
                     ((int64_t)blockIdx.y * (total / n_items) + head) * seq, l16, g);
  else
    store_rows<D>(oacc, l_run, q0 + wave * 32, q1, gate, g_row, head, out, o_row, o_head, l16, g);
}

template <int D>
int launch_prepass(const uint16_t *v, int64_t v_row, int64_t v_head, int seq, int heads, void *workspace,
                   hipStream_t stream) {
  const int s_pad = pad_rows(seq);
  hipLaunchKernelGGL(vt_prepass_kernel<D>, dim3(s_pad / 64, heads), dim3(kThreads), 0, stream, v, v_row, v_head,
                     static_cast<uint16_t *>(workspace), seq, s_pad);
  return check_launch("window vt_prepass");
}

// QNORM: q is normalised on load with q_weight / q_eps (see window_attn_kernel)
template <int D, bool QNORM>
int launch_attn(const uint16_t *q, int64_t q_row, int64_t q_head, const uint16_t *k, int64_t k_row, int64_t k_head,
                uint16_t *out, int64_t o_row, int64_t o_head, const uint16_t *gate, int64_t gate_row, int seq,
                int heads, float scale, const int32_t *items, int32_t n_items, const int32_t *tiles,
                const void *workspace, hipStream_t stream, const uint16_t *q_weight = nullptr, float q_eps = 0.f,
                int splits = 1, float *partial = nullptr) {
  const int s_pad = pad_rows(seq);
  const int total = n_items * heads;
  const int per_xcd = (total + 7) / 8;
  Partial part{nullptr, nullptr};
  if (splits > 1) part = Partial{partial, partial + (size_t)splits * heads * seq * D};
  hipLaunchKernelGGL((window_attn_kernel<D, QNORM>), dim3(per_xcd * 8, splits), dim3(kThreads), 0, stream, q, q_row, q_head, k,
                     k_row, k_head, static_cast<const uint16_t *>(workspace), s_pad, out, o_row, o_head, gate,
                     gate_row, seq, scale * 1.4426950408889634f, reinterpret_cast<const int4 *>(items), n_items,
                     reinterpret_cast<const int2 *>(tiles), per_xcd, total, q_weight, q_eps, part);
  int rc = check_launch("window_attn");
  if (rc || splits <= 1) return rc;
  const int64_t threads = (int64_t)heads * seq * (D / 8);
  hipLaunchKernelGGL(combine_kernel<D>, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream, part, splits, seq,
                     heads, gate, gate_row, out, o_row, o_head);
  return check_launch("window_attn combine");
}

template <int D>
int launch_qkv_prepass(const uint16_t *q, int64_t q_row, int64_t q_head, const uint16_t *q_weight, float q_eps,
                       const uint16_t *k, int64_t k_row, int64_t k_head, const uint16_t *k_weight, float k_eps,
                       const uint16_t *v, int64_t v_row, int64_t v_head, const float *freqs, int64_t f_row, int rot,
                       int seq, int heads, void *workspace, hipStream_t stream) {
  const int s_pad = pad_rows(seq);
  const size_t region = (size_t)heads * D * s_pad;
  uint16_t *vt = static_cast<uint16_t *>(workspace), *kn = vt + region, *qn = vt + 2 * region;
  const int gh = prepass_heads(s_pad / 64, heads, freqs != nullptr);
  const dim3 grid((heads + gh - 1) / gh, s_pad / 64);
  if (freqs)
    hipLaunchKernelGGL((qkv_prepass_kernel<D, true>), grid, dim3(kThreads), 0, stream, q, q_row, q_head, q_weight,
                       q_eps, k, k_row, k_head, k_weight, k_eps, v, v_row, v_head, freqs, f_row, rot, vt, kn, qn, seq,
                       s_pad, heads, gh);
  else
    hipLaunchKernelGGL((qkv_prepass_kernel<D, false>), grid, dim3(kThreads), 0, stream, q, q_row, q_head, q_weight,
                       q_eps, k, k_row, k_head, k_weight, k_eps, v, v_row, v_head, freqs, f_row, rot, vt, kn, qn, seq,
                       s_pad, heads, gh);
  return check_launch("window qkv_prepass");
}

int check_rope(const float *freqs, int64_t f_row, int rot, int head_dim) {
  if (!freqs) return VDNH3_OK;
  VDNH3_HOST_CHECK(rot > 0 && rot % 16 == 0 && rot <= head_dim, VDNH3_ERR_INVALID,
                   "rope: rot_dim must be a positive multiple of 16 and at most head_dim %d, got %d", head_dim, rot);
  VDNH3_HOST_CHECK(f_row >= 0 && f_row % 4 == 0 && reinterpret_cast<uintptr_t>(freqs) % 16 == 0, VDNH3_ERR_INVALID,
                   "rope: frequencies must be 16-byte aligned with a row stride multiple of 4");
  return VDNH3_OK;
}

int check_common(int seq, int heads, int head_dim, const void *workspace, size_t workspace_bytes) {
  VDNH3_HOST_CHECK(head_dim == 64 || head_dim == 128, VDNH3_ERR_INVALID,
                   "window attention supports head_dim 64 or 128, got %d", head_dim);
  VDNH3_HOST_CHECK(seq > 0 && heads > 0, VDNH3_ERR_INVALID, "seq and heads must be positive");
  VDNH3_HOST_CHECK(workspace != nullptr && reinterpret_cast<uintptr_t>(workspace) % 16 == 0, VDNH3_ERR_INVALID,
                   "workspace must be non-null and 16-byte aligned");
  VDNH3_HOST_CHECK(workspace_bytes >= vdnh3_window_workspace_bytes(seq, heads, head_dim), VDNH3_ERR_INVALID,
                   "workspace of %zu bytes is smaller than the %zu required", workspace_bytes,
                   vdnh3_window_workspace_bytes(seq, heads, head_dim));
  return VDNH3_OK;
}

int check_vec(const void *p, int64_t row, int64_t head, const char *name) {
  VDNH3_HOST_CHECK(p != nullptr, VDNH3_ERR_INVALID, "%s is null", name);
  VDNH3_HOST_CHECK(row % 8 == 0 && head % 8 == 0 && reinterpret_cast<uintptr_t>(p) % 16 == 0, VDNH3_ERR_INVALID,
                   "%s must be 16-byte aligned with row and head strides that are multiples of 8 elements", name);
  return VDNH3_OK;
}

}  // namespace
}  // namespace vdnh3

extern "C" int vdnh3_window_block_m(void) { return vdnh3::kBM; }
extern "C" int vdnh3_window_block_n(void) { return vdnh3::kBN; }

extern "C" size_t vdnh3_window_workspace_bytes(int seq, int heads, int head_dim) {
  if (seq <= 0 || heads <= 0 || head_dim <= 0) return 0;
  return size_t(heads) * size_t(head_dim) * size_t(vdnh3::pad_rows(seq)) * sizeof(uint16_t);
}

extern "C" int vdnh3_window_vt_prepass(const uint16_t *v, int64_t v_row, int64_t v_head, int seq, int heads,
                                       int head_dim, void *workspace, size_t workspace_bytes, void *stream) {
  int rc = vdnh3::check_common(seq, heads, head_dim, workspace, workspace_bytes);
  if (!rc) rc = vdnh3::check_vec(v, v_row, v_head, "v");
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  return head_dim == 128 ? vdnh3::launch_prepass<128>(v, v_row, v_head, seq, heads, workspace, s)
                         : vdnh3::launch_prepass<64>(v, v_row, v_head, seq, heads, workspace, s);
}

extern "C" size_t vdnh3_window_partial_bytes(int seq, int heads, int head_dim, int splits) {
  if (seq <= 0 || heads <= 0 || head_dim <= 0 || splits <= 1) return 0;
  return size_t(splits) * size_t(heads) * size_t(seq) * size_t(head_dim + 2) * sizeof(float);
}

namespace vdnh3 {
namespace {

int check_attn(const uint16_t *out, int64_t o_row, int64_t o_head, const int32_t *items, const int32_t *tiles,
               int32_t n_items) {
  VDNH3_HOST_CHECK(out != nullptr && o_row % 4 == 0 && o_head % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 8 == 0,
                   VDNH3_ERR_INVALID, "out must be 8-byte aligned with strides that are multiples of 4 elements");
  VDNH3_HOST_CHECK(items != nullptr && tiles != nullptr && n_items > 0, VDNH3_ERR_INVALID, "empty window plan");
  return VDNH3_OK;
}

int check_partial(int seq, int heads, int head_dim, int splits, const float *partial, size_t partial_bytes) {
  VDNH3_HOST_CHECK(splits >= 1 && splits <= 64, VDNH3_ERR_INVALID, "splits must be 1 to 64, got %d", splits);
  VDNH3_HOST_CHECK(splits == 1 || (partial && reinterpret_cast<uintptr_t>(partial) % 16 == 0 &&
                                   partial_bytes >= vdnh3_window_partial_bytes(seq, heads, head_dim, splits)),
                   VDNH3_ERR_INVALID, "the partial buffer must be 16-byte aligned and hold %zu bytes, got %zu",
                   vdnh3_window_partial_bytes(seq, heads, head_dim, splits), partial_bytes);
  return VDNH3_OK;
}

}  // namespace
}  // namespace vdnh3

extern "C" int vdnh3_window_attn_prepared_split(const uint16_t *q, int64_t q_row, int64_t q_head, const uint16_t *k,
                                                int64_t k_row, int64_t k_head, uint16_t *out, int64_t o_row,
                                                int64_t o_head, const uint16_t *gate, int64_t gate_row, int seq,
                                                int heads, int head_dim, float scale, const int32_t *items,
                                                int32_t n_items, const int32_t *tiles, const void *workspace,
                                                size_t workspace_bytes, int splits, float *partial,
                                                size_t partial_bytes, void *stream) {
  int rc = vdnh3::check_common(seq, heads, head_dim, workspace, workspace_bytes);
  if (!rc) rc = vdnh3::check_vec(q, q_row, q_head, "q");
  if (!rc) rc = vdnh3::check_vec(k, k_row, k_head, "k");
  if (!rc) rc = vdnh3::check_attn(out, o_row, o_head, items, tiles, n_items);
  if (!rc) rc = vdnh3::check_partial(seq, heads, head_dim, splits, partial, partial_bytes);
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (head_dim == 128)
    return vdnh3::launch_attn<128, false>(q, q_row, q_head, k, k_row, k_head, out, o_row, o_head, gate, gate_row, seq,
                                          heads, scale, items, n_items, tiles, workspace, s, nullptr, 0.f, splits,
                                          partial);
  return vdnh3::launch_attn<64, false>(q, q_row, q_head, k, k_row, k_head, out, o_row, o_head, gate, gate_row, seq,
                                       heads, scale, items, n_items, tiles, workspace, s, nullptr, 0.f, splits, partial);
}

extern "C" int vdnh3_window_attn_prepared(const uint16_t *q, int64_t q_row, int64_t q_head, const uint16_t *k,
                                          int64_t k_row, int64_t k_head, uint16_t *out, int64_t o_row,
                                          int64_t o_head, const uint16_t *gate, int64_t gate_row, int seq, int heads,
                                          int head_dim, float scale, const int32_t *items, int32_t n_items,
                                          const int32_t *tiles, const void *workspace, size_t workspace_bytes,
                                          void *stream) {
  return vdnh3_window_attn_prepared_split(q, q_row, q_head, k, k_row, k_head, out, o_row, o_head, gate, gate_row, seq,
                                          heads, head_dim, scale, items, n_items, tiles, workspace, workspace_bytes, 1,
                                          nullptr, 0, stream);
}

extern "C" int vdnh3_window_attn_fwd(const uint16_t *q, int64_t q_row, int64_t q_head, const uint16_t *k,
                                     int64_t k_row, int64_t k_head, const uint16_t *v, int64_t v_row, int64_t v_head,
                                     uint16_t *out, int64_t o_row, int64_t o_head, const uint16_t *gate,
                                     int64_t gate_row, int seq, int heads, int head_dim, float scale,
                                     const int32_t *items, int32_t n_items, const int32_t *tiles, void *workspace,
                                     size_t workspace_bytes, void *stream) {
  int rc = vdnh3_window_vt_prepass(v, v_row, v_head, seq, heads, head_dim, workspace, workspace_bytes, stream);
  if (rc) return rc;
  return vdnh3_window_attn_prepared(q, q_row, q_head, k, k_row, k_head, out, o_row, o_head, gate, gate_row, seq,
                                    heads, head_dim, scale, items, n_items, tiles, workspace, workspace_bytes, stream);
}

extern "C" size_t vdnh3_window_norm_workspace_bytes(int seq, int heads, int head_dim, int with_queries) {
  return (with_queries ? 3 : 2) * vdnh3_window_workspace_bytes(seq, heads, head_dim);
}

extern "C" int vdnh3_window_qkv_prepass(const uint16_t *q, int64_t q_row, int64_t q_head, const uint16_t *q_weight,
                                        float q_eps, const uint16_t *k, int64_t k_row, int64_t k_head,
                                        const uint16_t *k_weight, float k_eps, const uint16_t *v, int64_t v_row,
                                        int64_t v_head, const float *freqs, int64_t freqs_row, int rot_dim, int seq,
                                        int heads, int head_dim, void *workspace, size_t workspace_bytes,
                                        void *stream) {
  int rc = vdnh3::check_common(seq, heads, head_dim, workspace, workspace_bytes);
  if (!rc) rc = vdnh3::check_vec(k, k_row, k_head, "k");
  if (!rc) rc = vdnh3::check_vec(v, v_row, v_head, "v");
  if (!rc) rc = vdnh3::check_vec(k_weight, 0, 0, "k_weight");
  if (!rc && q) rc = vdnh3::check_vec(q, q_row, q_head, "q");
  if (!rc && q) rc = vdnh3::check_vec(q_weight, 0, 0, "q_weight");
  if (!rc) rc = vdnh3::check_rope(freqs, freqs_row, rot_dim, head_dim);
  if (rc) return rc;
  const size_t need = vdnh3_window_norm_workspace_bytes(seq, heads, head_dim, q != nullptr);
  VDNH3_HOST_CHECK(workspace_bytes >= need, VDNH3_ERR_INVALID,
                   "workspace of %zu bytes is smaller than the %zu the pre-pass writes", workspace_bytes, need);
  VDNH3_HOST_CHECK(vdnh3::pad_rows(seq) / 64 <= 65535, VDNH3_ERR_INVALID, "the pre-pass supports at most %d rows, got %d",
                   65535 * 64, seq);
  hipStream_t s = static_cast<hipStream_t>(stream);
  return head_dim == 128 ? vdnh3::launch_qkv_prepass<128>(q, q_row, q_head, q_weight, q_eps, k, k_row, k_head,
                                                          k_weight, k_eps, v, v_row, v_head, freqs, freqs_row, rot_dim,
                                                          seq, heads, workspace, s)
                         : vdnh3::launch_qkv_prepass<64>(q, q_row, q_head, q_weight, q_eps, k, k_row, k_head,
                                                         k_weight, k_eps, v, v_row, v_head, freqs, freqs_row, rot_dim,
                                                         seq, heads, workspace, s);
}

extern "C" int vdnh3_window_attn_qnorm_split(const uint16_t *q, int64_t q_row, int64_t q_head, const uint16_t *q_weight,
                                       float q_eps, uint16_t *out, int64_t o_row, int64_t o_head, const uint16_t *gate,
                                       int64_t gate_row, int seq, int heads, int head_dim, float scale,
                                       const int32_t *items, int32_t n_items, const int32_t *tiles,
                                       const void *workspace, size_t workspace_bytes, int splits, float *partial,
                                       size_t partial_bytes, void *stream) {
  int rc = vdnh3::check_common(seq, heads, head_dim, workspace, workspace_bytes);
  if (!rc) rc = vdnh3::check_vec(q, q_row, q_head, "q");
  if (!rc) rc = vdnh3::check_vec(q_weight, 0, 0, "q_weight");
  if (rc) return rc;
  VDNH3_HOST_CHECK(workspace_bytes >= vdnh3_window_norm_workspace_bytes(seq, heads, head_dim, 0), VDNH3_ERR_INVALID,
                   "workspace of %zu bytes is smaller than the %zu the normalising attention reads", workspace_bytes,
                   vdnh3_window_norm_workspace_bytes(seq, heads, head_dim, 0));
  rc = vdnh3::check_attn(out, o_row, o_head, items, tiles, n_items);
  if (!rc) rc = vdnh3::check_partial(seq, heads, head_dim, splits, partial, partial_bytes);
  if (rc) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const int s_pad = vdnh3::pad_rows(seq);
  // the normalised keys follow the V^T copy in the workspace: [heads][s_pad][head_dim]
  const uint16_t *kn = static_cast<const uint16_t *>(workspace) + (size_t)heads * head_dim * s_pad;
  const int64_t kn_row = head_dim, kn_head = (int64_t)s_pad * head_dim;
  if (head_dim == 128)
    return vdnh3::launch_attn<128, true>(q, q_row, q_head, kn, kn_row, kn_head, out, o_row, o_head, gate, gate_row,
                                         seq, heads, scale, items, n_items, tiles, workspace, s, q_weight, q_eps, splits,
                                         partial);
  return vdnh3::launch_attn<64, true>(q, q_row, q_head, kn, kn_row, kn_head, out, o_row, o_head, gate, gate_row, seq,
                                      heads, scale, items, n_items, tiles, workspace, s, q_weight, q_eps, splits,
                                         partial);
}

extern "C" int vdnh3_window_attn_qnorm(const uint16_t *q, int64_t q_row, int64_t q_head, const uint16_t *q_weight,
                                       float q_eps, uint16_t *out, int64_t o_row, int64_t o_head, const uint16_t *gate,
                                       int64_t gate_row, int seq, int heads, int head_dim, float scale,
                                       const int32_t *items, int32_t n_items, const int32_t *tiles,
                                       const void *workspace, size_t workspace_bytes, void *stream) {
  return vdnh3_window_attn_qnorm_split(q, q_row, q_head, q_weight, q_eps, out, o_row, o_head, gate, gate_row, seq, heads,
                                       head_dim, scale, items, n_items, tiles, workspace, workspace_bytes, 1, nullptr,
                                       0, stream);
}
