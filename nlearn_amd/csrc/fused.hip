// fused.hip — the elementwise tail of the training step around the GEMMs:
// LayerNorm (forward with the residual add folded in, backward with the
// residual gradient folded in), column sums for bias gradients, and the token
// + learned-position embedding (forward and backward).
//
// Math (nlearn/model.py:216-241 normalisation params and call, model.py:315-324
// pre-norm residual blocks, model.py:75-86 embedding lookup; the LayerNorm with
// gamma/beta and the learned position table are the layout the benchmark
// configuration trains):
//   LN:   y = (x - mean) * rstd * gamma + beta,  rstd = 1/sqrt(var + eps)
//   dLN:  dx = rstd * (g - mean(g) - xh * mean(g * xh)),  g = dy * gamma, xh = (x - mean) * rstd
//         dgamma = sum_rows dy * xh,  dbeta = sum_rows dy
//
// MI355X design: one 64-lane wave per row (a 512-wide bf16 row is one 16-byte
// vector per lane), wave sums by DPP adds and row swaps for the row statistics,
// no LDS in the forward. Parameter-gradient sums are per-workgroup partial rows combined
// in a fixed order by a second kernel (deterministic, no atomics).
#include <type_traits>

#include "common.h"

namespace nl {
namespace {

constexpr int kRowsPerBlock = 4;   // LayerNorm: one wave per row, 4 waves per workgroup
constexpr int kMaxD = 4096;        // LayerNorm width limit (8 vectors of 8 per lane)
constexpr int kLnBwdBlocks = 1024; // LayerNorm backward: most workgroups, and the partial rows of dgamma / dbeta the workspace holds
constexpr int kColsumRows = 64;    // column sums: rows per partial

// Lane `lane` holds columns (i*64 + lane)*8 .. +7 of the row in vector i.
template <int VPL>
__device__ __forceinline__ void load_row(u32x4 (&v)[VPL], const uint16_t* p, int D, int lane) {
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int c = (i * 64 + lane) * 8;
    v[i] = (c < D) ? *reinterpret_cast<const u32x4*>(p + c) : u32x4{0u, 0u, 0u, 0u};
  }
}

__device__ __forceinline__ void unpack8(const u32x4& v, float f[8]) {
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    f[2 * q] = bf16_lo(v[q]);
    f[2 * q + 1] = bf16_hi(v[q]);
  }
}
__device__ __forceinline__ u32x4 pack8(const float f[8]) {
  u32x4 v;
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = pack_bf16x2(f[2 * q], f[2 * q + 1]);
  return v;
}
__device__ __forceinline__ void load8f(const float* p, float f[8]) {
  const f32x4 a = *reinterpret_cast<const f32x4*>(p), b = *reinterpret_cast<const f32x4*>(p + 4);
  f[0] = a[0], f[1] = a[1], f[2] = a[2], f[3] = a[3], f[4] = b[0], f[5] = b[1], f[6] = b[2], f[7] = b[3];
}

// y = LN(s), s = x (+ r). With r, s is rounded to bf16 and stored to s_out (the
// residual stream the next block reads) before it is normalised.
// One row per wave, every load (x, r, gamma, beta) issued before the first use.
// Bound by HBM from about 8000 rows of 512 (16384: 67 MB in 15 us); below, by
// the chain load -> sum -> squares -> store, which is why a wave takes one row
// and sums without LDS permutes. Four rows per wave one after the other, with
// permutes: 200 x 512 5.0 us against 2.4, 4096 x 512 7.3 against 5.4, 32768 x 512
// 28.4 against 25.5.
template <int VPL>
__global__ __launch_bounds__(64 * kRowsPerBlock) void ln_fwd_kernel(int rows, int D, const uint16_t* __restrict__ x,
                                                                    const uint16_t* __restrict__ r,
                                                                    uint16_t* __restrict__ s_out,
                                                                    const float* __restrict__ gamma,
                                                                    const float* __restrict__ beta,
                                                                    uint16_t* __restrict__ y, float* __restrict__ mean_out,
                                                                    float* __restrict__ rstd_out, float eps) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * kRowsPerBlock + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int64_t off = (int64_t)row * D;
  u32x4 xv[VPL], rv[VPL];
  load_row<VPL>(xv, x + off, D, lane);
  if (r) load_row<VPL>(rv, r + off, D, lane);
  float gg[VPL][8], bb[VPL][8];
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int c = (i * 64 + lane) * 8;
    if (c < D) {
      load8f(gamma + c, gg[i]);
      load8f(beta + c, bb[i]);
    }
  }
  float f[VPL][8];
#pragma unroll
  for (int i = 0; i < VPL; ++i) unpack8(xv[i], f[i]);
  if (r) {
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      float g[8];
      unpack8(rv[i], g);
#pragma unroll
      for (int j = 0; j < 8; ++j) f[i][j] = bf16_to_f32(f32_to_bf16(f[i][j] + g[j]));
      const int c = (i * 64 + lane) * 8;
      if (c < D) *reinterpret_cast<u32x4*>(s_out + off + c) = pack8(f[i]);
    }
  }
  // columns beyond D hold zeros, so they add nothing to the sum
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < VPL; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) s += f[i][j];
  const float mean = wave_sum(s) / (float)D;
  float v = 0.f;
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const bool in = (i * 64 + lane) * 8 < D;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float d = in ? f[i][j] - mean : 0.f;
      v += d * d;
    }
  }
  const float rstd = rsqrtf(wave_sum(v) / (float)D + eps);
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int c = (i * 64 + lane) * 8;
    if (c >= D) continue;
    float o[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = (f[i][j] - mean) * rstd * gg[i][j] + bb[i][j];
    *reinterpret_cast<u32x4*>(y + off + c) = pack8(o);
  }
  if (lane == 0) {
    mean_out[row] = mean;
    rstd_out[row] = rstd;
  }
}

// out[c] (+)= sum_{p<P} part[p][c] for one or two (part, out) pairs
// (blockIdx.y picks the pair), summed in a fixed order. A workgroup owns 16
// columns: thread (ph, q), ph < 64, q < 4, sums rows p = ph, ph+64, ... of
// columns [4q, 4q+4) of its strip; the 64 phase sums are then added in groups
// of 4 (phases 4g..4g+3) and the 16 group sums in g order. The strips are
// narrow so that a 512-column sum still spreads over 32 workgroups per pair
// with every row load in flight at once (LayerNorm's P <= 1024: 16 loads a thread).
__device__ __forceinline__ void sum_partials_strip(int bx, int pair, int P, int D, const float* __restrict__ part0,
                                                   float* __restrict__ out0, const float* __restrict__ part1,
                                                   float* __restrict__ out1, int accumulate) {
  __shared__ float s[64][17];
  __shared__ float s2[16][17];
  const float* __restrict__ part = pair ? part1 : part0;
  float* __restrict__ out = pair ? out1 : out0;
  const int q = threadIdx.x & 3, ph = threadIdx.x >> 2;
  const int c = bx * 16 + q * 4;
  float a[4] = {0.f, 0.f, 0.f, 0.f};
  if ((D & 3) == 0) {
    if (c < D) {
#pragma unroll 16
      for (int p = ph; p < P; p += 64) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(part + (int64_t)p * D + c);
#pragma unroll
        for (int j = 0; j < 4; ++j) a[j] += v[j];
      }
    }
  } else {
#pragma unroll 4
    for (int p = ph; p < P; p += 64) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (c + j < D) a[j] += part[(int64_t)p * D + c + j];
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) s[ph][q * 4 + j] = a[j];
  __syncthreads();
  {
    const int col = threadIdx.x & 15, g = threadIdx.x >> 4;
    s2[g][col] = ((s[4 * g][col] + s[4 * g + 1][col]) + s[4 * g + 2][col]) + s[4 * g + 3][col];
  }
  __syncthreads();
  if (threadIdx.x < 16) {
    const int cc = bx * 16 + threadIdx.x;
    if (cc < D) {
      float t = 0.f;
#pragma unroll
      for (int g = 0; g < 16; ++g) t += s2[g][threadIdx.x];
      out[cc] = accumulate ? out[cc] + t : t;
    }
  }
}

// A reduction of partial rows that rides along in another kernel's launch.
struct PartialSums {
  int P, D, strips;  // strips: (D + 15) / 16 workgroups per pair; 0 = none
  const float* part_g;
  float* dgamma;
  const float* part_b;
  float* dbeta;
  int accumulate;
};

// dx = dLN(dy) (+ dres). Each of the first nblk workgroups also writes one
// partial row of dgamma and one of dbeta (its 4 waves combined in wave order).
// Workgroups past nblk reduce `prev`, the partial rows of an earlier call.
template <int VPL>
__global__ __launch_bounds__(64 * kRowsPerBlock) void ln_bwd_kernel(
    int rows, int D, const uint16_t* __restrict__ dy, const uint16_t* __restrict__ x, const float* __restrict__ mean_in,
    const float* __restrict__ rstd_in, const float* __restrict__ gamma, const uint16_t* __restrict__ dres,
    uint16_t* __restrict__ dx, float* __restrict__ part_g, float* __restrict__ part_b, int nblk, PartialSums prev) {
  if ((int)blockIdx.x >= nblk) {
    const int j = blockIdx.x - nblk;
    sum_partials_strip(j % prev.strips, j / prev.strips, prev.P, prev.D, prev.part_g, prev.dgamma, prev.part_b,
                       prev.dbeta, prev.accumulate);
    return;
  }
  // [wave][j][lane]: the sums of column (i*64 + lane)*8 + j; the 72-float pitch
  // keeps both the per-wave writes and the per-column reads off shared banks
  __shared__ float sg[kRowsPerBlock][8 * 72];
  __shared__ float sb[kRowsPerBlock][8 * 72];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  float ag[VPL][8], ab[VPL][8], gam[VPL][8];
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    const int c = (i * 64 + lane) * 8;
#pragma unroll
    for (int j = 0; j < 8; ++j) ag[i][j] = ab[i][j] = gam[i][j] = 0.f;
    if (c < D) load8f(gamma + c, gam[i]);
  }
  // Rows are software-pipelined: the next row's dy, x, dres, mean and rstd are
  // in flight while this row is computed and stored.
  const int stride = nblk * kRowsPerBlock;
  int row = blockIdx.x * kRowsPerBlock + wave;
  u32x4 dv[VPL], xv[VPL], rv[VPL];
  float mu = 0.f, rs = 0.f;
  auto fetch = [&](int rw, u32x4 (&d)[VPL], u32x4 (&xx)[VPL], u32x4 (&rr)[VPL], float& m, float& q) {
    const int64_t o = (int64_t)rw * D;
    load_row<VPL>(d, dy + o, D, lane);
    load_row<VPL>(xx, x + o, D, lane);
    if (dres) load_row<VPL>(rr, dres + o, D, lane);
    m = mean_in[rw];
    q = rstd_in[rw];
  };
  if (row < rows) fetch(row, dv, xv, rv, mu, rs);
  while (row < rows) {
    const int64_t off = (int64_t)row * D;
    const int nxt = row + stride;
    u32x4 dn[VPL], xn[VPL], rn[VPL];
    float mun = 0.f, rsn = 0.f;
    if (nxt < rows) fetch(nxt, dn, xn, rn, mun, rsn);
    float g[VPL][8], xh[VPL][8];
    float s1 = 0.f, s2 = 0.f;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      float dyf[8], xf[8];
      unpack8(dv[i], dyf);
      unpack8(xv[i], xf);
      const bool in = (i * 64 + lane) * 8 < D;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        xh[i][j] = in ? (xf[j] - mu) * rs : 0.f;
        g[i][j] = dyf[j] * gam[i][j];
        s1 += g[i][j];
        s2 += g[i][j] * xh[i][j];
        ag[i][j] += dyf[j] * xh[i][j];
        ab[i][j] += dyf[j];
      }
    }
    const float m1 = wave_sum(s1) / (float)D, m2 = wave_sum(s2) / (float)D;
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      const int c = (i * 64 + lane) * 8;
      if (c >= D) continue;
      float o[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = rs * (g[i][j] - m1 - xh[i][j] * m2);
      if (dres) {
        float rf[8];
        unpack8(rv[i], rf);
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] += rf[j];
      }
      *reinterpret_cast<u32x4*>(dx + off + c) = pack8(o);
    }
#pragma unroll
    for (int i = 0; i < VPL; ++i) {
      dv[i] = dn[i];
      xv[i] = xn[i];
      rv[i] = rn[i];
    }
    mu = mun;
    rs = rsn;
    row = nxt;
  }
  // combine the 4 waves in wave order (deterministic), one partial row per workgroup
#pragma unroll
  for (int i = 0; i < VPL; ++i) {
    if (i > 0) __syncthreads();
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      sg[wave][j * 72 + lane] = ag[i][j];
      sb[wave][j * 72 + lane] = ab[i][j];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < 512; e += blockDim.x) {
      const int c = i * 512 + e;
      if (c >= D) break;
      const int o = (e & 7) * 72 + (e >> 3);
      part_g[(int64_t)blockIdx.x * D + c] = ((sg[0][o] + sg[1][o]) + sg[2][o]) + sg[3][o];
      part_b[(int64_t)blockIdx.x * D + c] = ((sb[0][o] + sb[1][o]) + sb[2][o]) + sb[3][o];
    }
  }
}

__global__ __launch_bounds__(256) void sum_partials_kernel(int P, int D, const float* __restrict__ part0,
                                                           float* __restrict__ out0, const float* __restrict__ part1,
                                                           float* __restrict__ out1, int accumulate) {
  sum_partials_strip(blockIdx.x, blockIdx.y, P, D, part0, out0, part1, out1, accumulate);
}

// Partial column sums of a bf16 [rows][cols] matrix (row stride ld, ld % 8 == 0):
// workgroup (bx, by) sums rows [by*kColsumRows, +kColsumRows) of columns
// [bx*512, +512). 64 lanes x 8 columns, 4 row phases combined in order.
__global__ __launch_bounds__(256) void colsum_partial_kernel(int rows, int cols, const uint16_t* __restrict__ x,
                                                             int64_t ld, float* __restrict__ part) {
  __shared__ float s[4][512];
  const int lane = threadIdx.x & 63, ph = threadIdx.x >> 6;
  const int c = blockIdx.x * 512 + lane * 8;
  const int r0 = blockIdx.y * kColsumRows;
  const int r1 = min(rows, r0 + kColsumRows);
  float a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (c < cols) {
    if (c + 8 <= cols) {
#pragma unroll 4
      for (int r = r0 + ph; r < r1; r += 4) {
        float f[8];
        unpack8(*reinterpret_cast<const u32x4*>(x + (int64_t)r * ld + c), f);
#pragma unroll
        for (int j = 0; j < 8; ++j) a[j] += f[j];
      }
    } else {
      for (int r = r0 + ph; r < r1; r += 4)
        for (int j = 0; j < cols - c; ++j) a[j] += bf16_to_f32(x[(int64_t)r * ld + c + j]);
    }
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) s[ph][lane * 8 + j] = a[j];
  __syncthreads();
  for (int k = threadIdx.x; k < 512; k += 256) {
    const int cc = blockIdx.x * 512 + k;
    if (cc < cols) part[(int64_t)blockIdx.y * cols + cc] = ((s[0][k] + s[1][k]) + s[2][k]) + s[3][k];
  }
}

// out[t, :] = bf16(tok[ids[t]] + pos[t % S])  (fp32 tables, D % 4 == 0).
// An id outside [0, vocab) yields a NaN row.
__global__ __launch_bounds__(128) void embed_fwd_kernel(int S, int D, const int32_t* __restrict__ ids,
                                                        const float* __restrict__ tok, const float* __restrict__ pos,
                                                        uint16_t* __restrict__ out, int vocab) {
  const int t = blockIdx.x;
  const int s = t % S;
  const int id = ids[t];
  const bool ok = id >= 0 && id < vocab;
  for (int c = threadIdx.x * 4; c < D; c += 128 * 4) {
    const f32x4 a = ok ? *reinterpret_cast<const f32x4*>(tok + (int64_t)id * D + c) : f32x4{NAN, NAN, NAN, NAN};
    const f32x4 p = *reinterpret_cast<const f32x4*>(pos + (int64_t)s * D + c);
    *reinterpret_cast<u32x2*>(out + (int64_t)t * D + c) =
        u32x2{pack_bf16x2(a[0] + p[0], a[1] + p[1]), pack_bf16x2(a[2] + p[2], a[3] + p[3])};
  }
}

// The embedding backward, deterministic (no floating-point atomics), in three
// launches over a workspace of exactly one 8-byte entry per token:
//
// embed_count_kernel: workgroup k counts, for each bucket b of W vocabulary
// rows [b W, b W + W), the positions of the k-th of P equal token ranges whose
// id falls in it: counts[b][k] (integer counts; the order of the LDS
// increments does not change them). Ids outside [0, vocab) go nowhere.
//
// embed_bucket_kernel: workgroup (b, k) appends, in increasing t, the (t,
// ids[t]) of its range whose id falls in bucket b to its segment of the list,
// which starts at the number of entries of every (b', k') before (b, k) in
// (bucket, range) order, and records that start in offsets[b][k]. The segments
// of a bucket are then contiguous and in increasing t, and the lists hold
// exactly the valid tokens.
//
// embed_bwd_kernel:
// * workgroups [0, S) form dpos[s] (+)= sum_b dx[b, s] in batch order;
// * workgroup S + g owns R token-table rows of one bucket (their sums in LDS)
//   and walks the bucket's list 512 entries at a time: its waves sort the
//   entries of the owned rows by row (ballots keep the tokens of a row in
//   increasing t), then every thread adds its CW columns of dx[t] along the
//   sorted entries, holding the current row's sum in registers: each (row,
//   column) is summed by one thread in increasing t (np.add.at's order). Every
//   owned row is then written, zero when no token has its id, so dtok needs no
//   zeroing first.
//   What bounds it: ids as spread as a uniform draw leave mostly the write of
//   dtok (103 MB at 50257 x 512), hence few registers and many workgroups per
//   CU. Ids with the 1/rank frequencies of text put a fifth of all tokens on
//   the first 8 rows, one serial chain by contract: what counts there is how
//   many dx rows are in flight and how few instructions an entry takes. The
//   whole backward at 50257 x 512, against one wave per 8 rows that loads and
//   adds one token at a time: 8 x 512 tokens of such ids 545 -> 72 us, 32 x 512
//   2150 -> 245 us; of uniform ids 27 -> 30 and 38 -> 39 us.
constexpr int kEmbTokLds = 16384;  // a bucket is a whole number of 16384 / (4 D)-row groups
constexpr int kEmbBuckets = 256;   // target number of buckets
constexpr int kEmbParts = 4;       // token ranges per bucket (one scanning workgroup each)
constexpr int kEmbMaxBuckets = 256;  // W = ceil(vocab / 256) rounded up to a whole group: at most 256 buckets
constexpr int kEmbChunk = 512;     // list entries sorted into per-row lists at a time

struct EmbPlan {
  int W;        // rows per bucket
  int buckets;  // ceil(vocab / W)
};
EmbPlan emb_plan(int D, int vocab) {
  EmbPlan p;
  const int unit = std::max(1, kEmbTokLds / (D * 4));
  const int want = (vocab + kEmbBuckets - 1) / kEmbBuckets;
  p.W = (want + unit - 1) / unit * unit;
  p.buckets = (vocab + p.W - 1) / p.W;
  return p;
}

__global__ __launch_bounds__(256) void embed_count_kernel(int T, int vocab, int W, int buckets,
                                                          const int32_t* __restrict__ ids, int* __restrict__ counts) {
  __shared__ int hist[kEmbMaxBuckets];
  const int tid = threadIdx.x, k_part = blockIdx.x;
  for (int b = tid; b < buckets; b += 256) hist[b] = 0;
  __syncthreads();
  const int span = (T + kEmbParts - 1) / kEmbParts;
  const int t0 = k_part * span, t1 = min(T, t0 + span);
  // eight ids per thread loaded before any is counted: a load per increment
  // made each thread a chain of dependent global loads
  for (int c = t0 + tid; c < t1; c += 256 * 8) {
    int v[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = c + e * 256 < t1 ? ids[c + e * 256] : -1;
#pragma unroll
    for (int e = 0; e < 8; ++e)
      if ((uint32_t)v[e] < (uint32_t)vocab) atomicAdd(&hist[v[e] / W], 1);
  }
  __syncthreads();
  for (int b = tid; b < buckets; b += 256) counts[b * kEmbParts + k_part] = hist[b];
}

__global__ __launch_bounds__(256) void embed_bucket_kernel(int T, int vocab, int W, const int32_t* __restrict__ ids,
                                                           const int* __restrict__ counts, int* __restrict__ offsets,
                                                           int2* __restrict__ lists) {
  __shared__ int wave_tot[4];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int b = blockIdx.x / kEmbParts, k_part = blockIdx.x % kEmbParts;
  const int v0 = b * W;
  const int nrows = min(W, vocab - v0);
  const int span = (T + kEmbParts - 1) / kEmbParts;
  const int t0 = k_part * span, t1 = min(T, t0 + span);
  // start of this segment: the entries of every (bucket, range) before it
  int before = 0;
  for (int i = tid; i < (int)blockIdx.x; i += 256) before += counts[i];
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) before += __shfl_xor(before, d, 64);
  if (lane == 0) wave_tot[wave] = before;
  __syncthreads();
  const int seg0 = wave_tot[0] + wave_tot[1] + wave_tot[2] + wave_tot[3];
  if (tid == 0) offsets[blockIdx.x] = seg0;
  __syncthreads();  // wave_tot is reused below
  int2* list = lists + seg0;
  int cursor = 0;
  // thread tid holds positions c0 + 4 tid + e: in t order thread by thread, e
  // within; the next chunk's ids are loaded before this chunk is placed
  int cur[4], nxt[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) cur[e] = t0 + 4 * tid + e < t1 ? ids[t0 + 4 * tid + e] : -1;
  for (int c0 = t0; c0 < t1; c0 += 1024) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int t = c0 + 1024 + 4 * tid + e;
      nxt[e] = t < t1 ? ids[t] : -1;
    }
    bool hit[4];
    int k = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      hit[e] = (uint32_t)(cur[e] - v0) < (uint32_t)nrows;
      k += hit[e];
    }
    // exclusive prefix of k over the workgroup (wave scan, then wave totals)
    int incl = k;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int y = __shfl_up(incl, d, 64);
      if (lane >= d) incl += y;
    }
    if (lane == 63) wave_tot[wave] = incl;
    __syncthreads();
    int base = cursor, total = 0;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      if (w < wave) base += wave_tot[w];
      total += wave_tot[w];
    }
    int pos = base + incl - k;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (hit[e]) list[pos++] = int2{c0 + 4 * tid + e, cur[e]};
    cursor += total;
    __syncthreads();  // wave_tot is rewritten by the next chunk
#pragma unroll
    for (int e = 0; e < 4; ++e) cur[e] = nxt[e];
  }
}

// CW bf16 columns of a dx row (CW / 2 dwords; rows are 8-byte aligned)
template <int CW>
struct EmbCols {
  uint32_t d[CW / 2];
};

// accumulators per row: a column for every lane of the waves that cover D
template <int CW>
__host__ __device__ constexpr int emb_pitch(int D) { return (D + 64 * CW - 1) / (64 * CW) * (64 * CW); }

template <int CW, int R>
__global__ __launch_bounds__(256, CW == 2 ? 7 : 6) void embed_bwd_kernel(int B, int S, int D, const uint16_t* __restrict__ dx,
                                                        float* __restrict__ dtok, int vocab, int W, int groups,
                                                        const int* __restrict__ counts,
                                                        const int* __restrict__ offsets,
                                                        const int2* __restrict__ lists, float* __restrict__ dpos,
                                                        int accumulate) {
  const int tid = threadIdx.x, nt = blockDim.x;
  if ((int)blockIdx.x < S) {
    const int s = blockIdx.x;
    for (int c = tid; c < D; c += nt) {
      float a = 0.f;
#pragma unroll 8
      for (int b = 0; b < B; ++b) a += bf16_to_f32(dx[((int64_t)b * S + s) * D + c]);
      float* o = dpos + (int64_t)s * D + c;
      *o = accumulate ? *o + a : a;
    }
    return;
  }
  typedef __attribute__((__vector_size__(CW * sizeof(float)))) float facc;
  __shared__ int2 sorted[kEmbChunk];              // (t, row) of the chunk's owned entries, by row, then t
  extern __shared__ __attribute__((aligned(16))) float acc[];  // [R][pitch]; a thread touches its own columns only
  const int lane = tid & 63, nw = nt >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = (int)blockIdx.x - S;
  const int b = g / groups;
  const int64_t v0 = (int64_t)b * W + (int64_t)(g - b * groups) * R;
  const int64_t vend = min((int64_t)vocab, (int64_t)(b + 1) * W);
  if (v0 >= vend) return;
  const int nrows = (int)min((int64_t)R, vend - v0);

  // the segments of a bucket are contiguous: one list of n entries
  int n = 0;
  const int2* list = lists;
  if (B > 0 && S > 0) {
#pragma unroll
    for (int k = 0; k < kEmbParts; ++k) n += counts[b * kEmbParts + k];
    list += offsets[b * kEmbParts];
  }
  constexpr int PER = kEmbChunk / 64;
  int et[PER], er[PER];  // the chunk's entries: token, row - v0 (negative or >= R: another workgroup's)
  auto fetch = [&](int c0) {
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int2 e = c0 + i * 64 + lane < n ? list[c0 + i * 64 + lane] : int2{0, -1};
      et[i] = e.x;
      er[i] = e.y - (int)v0;
    }
  };
  const int pitch = emb_pitch<CW>(D);
  uint32_t seen = 0;  // rows with an accumulator
  if (n > 0) fetch(0);
  for (int c0 = 0; c0 < n; c0 += kEmbChunk) {
    // every wave counts the chunk's entries of each owned row; wave r % nw then
    // writes row r's, in order, behind those of the rows before it
    uint32_t has = 0;
#pragma unroll
    for (int i = 0; i < PER; ++i)
      if (__ballot((uint32_t)er[i] < (uint32_t)R)) has |= 1u << i;
    int m = 0;
    uint32_t now = 0;  // rows with tokens in this chunk
    if (has) {
#pragma unroll
      for (int r = 0; r < R; ++r) {
        int cur = m;
#pragma unroll
        for (int i = 0; i < PER; ++i)
          if (has >> i & 1) {
            const bool hit = er[i] == r;
            const uint64_t k = __ballot(hit);
            if (hit && r % nw == wave)
              sorted[cur + __builtin_amdgcn_mbcnt_hi((uint32_t)(k >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)k, 0))] =
                  int2{et[i], r};
            cur += __popcll(k);
          }
        if (cur > m) now |= 1u << r;
        m = cur;
      }
    }
    if (c0 + kEmbChunk < n) fetch(c0 + kEmbChunk);
    if (m == 0) continue;  // the same in every wave
    __syncthreads();
    constexpr int DEPTH = CW == 2 ? 32 : 16, REST = 8;
    // a wave's lanes past column D read the row's last columns and sum them into
    // accumulators of their own, which nobody stores: no lane masks in the loop
    for (int w0 = wave * 64 * CW; w0 < D; w0 += nt * CW) {
      const int c = w0 + lane * CW;
      const int co = min(c, D - CW);
      float* ac = acc + c;
#pragma unroll
      for (int r = 0; r < R; ++r)
        if ((now & ~seen) >> r & 1) *reinterpret_cast<facc*>(ac + r * pitch) = facc{};
      int row = __builtin_amdgcn_readfirstlane(sorted[0].y);  // the row whose sum is in `cur`
      facc cur = *reinterpret_cast<const facc*>(ac + row * pitch);
      auto add = [&](const EmbCols<CW>& x) __attribute__((always_inline)) {
#pragma unroll
        for (int e = 0; e < CW / 2; ++e) {
          cur[2 * e] += bf16_lo(x.d[e]);
          cur[2 * e + 1] += bf16_hi(x.d[e]);
        }
      };
      // entries i .. i + N - 1 (those past m repeat the last and are not added):
      // every lane forms one entry's row address, so a load costs two lane reads
      auto batch = [&](auto nn, int i) __attribute__((always_inline)) {
        constexpr int N = decltype(nn)::value;
        const int k = min(i + (lane & (N - 1)), m - 1);
        const int2 e = sorted[k];
        const uint64_t ad = (uint64_t)(dx + (int64_t)e.x * D);
        const bool end = i + (lane & (N - 1)) >= m;
        const uint32_t stop = (uint32_t)__ballot(end || (k > 0 && sorted[k - 1].y != e.y));  // not simply "add to cur"
        EmbCols<CW> x[N];
#pragma unroll
        for (int j = 0; j < N; ++j) {
          const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)ad, j);
          const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)(ad >> 32), j);
          const uint16_t* q = reinterpret_cast<const uint16_t*>(((uint64_t)hi << 32) | lo) + (uint32_t)co;
          if constexpr (CW == 2) x[j].d[0] = *reinterpret_cast<const uint32_t*>(q);
          else {
            const u32x2 v = *reinterpret_cast<const u32x2*>(q);
            x[j].d[0] = v[0];
            x[j].d[1] = v[1];
          }
        }
#pragma unroll
        for (int j0 = 0; j0 < N; j0 += 4) {
          if ((stop >> j0 & 15u) == 0) {
#pragma unroll
            for (int j = j0; j < j0 + 4; ++j) add(x[j]);
          } else {
#pragma unroll
            for (int j = j0; j < j0 + 4; ++j) {
              if (i + j >= m) continue;
              const int r = __builtin_amdgcn_readlane(e.y, j);
              if (r != row) {
                *reinterpret_cast<facc*>(ac + row * pitch) = cur;
                cur = *reinterpret_cast<const facc*>(ac + r * pitch);
                row = r;
              }
              add(x[j]);
            }
          }
        }
      };
      for (int i = 0; i < m;) {
        if (m - i > REST) {
          batch(std::integral_constant<int, DEPTH>{}, i);
          i += DEPTH;
        } else {
          batch(std::integral_constant<int, REST>{}, i);
          i += REST;
        }
      }
      *reinterpret_cast<facc*>(ac + row * pitch) = cur;
    }
    seen |= now;
    __syncthreads();  // the sorted entries are rewritten by the next chunk
  }
  // the owned rows are contiguous in dtok: 16 bytes per lane (the last barrier
  // made every column's sum visible)
  const int d4 = D / 4, n4 = nrows * d4;
  f32x4* out = reinterpret_cast<f32x4*>(dtok + v0 * D);
  if (seen == 0) {
    for (int i = tid; i < n4; i += nt) out[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    return;
  }
  for (int i = tid; i < n4; i += nt) {
    const int r = i / d4;
    out[i] = seen >> r & 1 ? *reinterpret_cast<const f32x4*>(acc + r * pitch + (i - r * d4) * 4) : f32x4{0.f, 0.f, 0.f, 0.f};
  }
}

// rows per row workgroup: at most 16 KB of accumulators
int emb_rows(int D) { return D <= 512 ? 8 : D <= 1024 ? 4 : D <= 2048 ? 2 : 1; }

template <int CW, int R>
void launch_embed_bwd(hipStream_t st, int64_t grid, int batch, int seq, int D, const uint16_t* dx, float* dtok,
                      int vocab, int W, const int* counts, const int* offsets, const int2* lists, float* dpos,
                      int accumulate) {
  const int nt = std::min(256, (D / CW + 63) / 64 * 64);
  hipLaunchKernelGGL((embed_bwd_kernel<CW, R>), dim3((unsigned)grid), dim3(nt), R * emb_pitch<CW>(D) * sizeof(float), st, batch, seq,
                     D, dx, dtok, vocab, W, (W + R - 1) / R, counts, offsets, lists, dpos, accumulate);
}

int vectors_per_lane(int D) {
  const int v = (D + 511) / 512;
  return v <= 1 ? 1 : v <= 2 ? 2 : v <= 4 ? 4 : 8;
}

// Workgroups of the LayerNorm backward, each leaving one partial row of dgamma
// and dbeta: few, because the partials cost as much traffic per workgroup as
// 8 rows of data and their sum is a launch that waits for all of them; enough
// to keep the loads in flight. Measured with the sum (us, 1024 / 512 / 256):
//   4096 x 512   15.1 / 11.6 / 10.3     16384 x 512   24.0 / 21.3 / 26.1
//   8192 x 512   18.4 / 14.7 / 16.0     32768 x 512   35.9 / 32.2 / 43.0
//   8191 x 1024  25.2 / 19.4 / 19.6     8191 x 2048   47.0 / 36.5 / 31.5
// A row of up to 256 columns leaves half of a wave's lanes or more without a
// load, so the same bytes need more waves, most of all where the sum is left to
// the next call (us of nl_layernorm_bwd_deferred, 1024 / 768 / 512 / 256):
//   4096 x 256    5.1 /  4.8 /  4.4 /  5.1    32768 x 256  17.3 / 17.4 / 18.8 / 27.7
//   8191 x 256    6.3 /  5.7 /  6.0 /  7.6    65536 x 256  28.1 / 28.9 / 32.2 / 51.1
int ln_bwd_blocks(int rows, int D) {
  const int most = D > 256 ? (rows >= 8192 ? 512 : 256)
                           : (rows >= 49152 ? kLnBwdBlocks : rows >= 20000 ? 768 : rows >= 5000 ? 512 : 256);
  return std::min(most, (rows + kRowsPerBlock - 1) / kRowsPerBlock);
}

}  // namespace
}  // namespace nl

using namespace nl;

extern "C" int nl_layernorm_fwd(void* stream, int rows, int D, const nl_bf16* x, const nl_bf16* residual,
                                nl_bf16* sum_out, const float* gamma, const float* beta, float eps, nl_bf16* y,
                                float* mean, float* rstd) {
  if (rows < 0 || D <= 0 || (D % 8) != 0 || D > kMaxD)
    return nl_set_error(NL_EINVAL, "layernorm: need 0 < D <= 4096 and D % 8 == 0");
  if (rows == 0) return NL_OK;
  if (!x || !gamma || !beta || !y || !mean || !rstd || (residual && !sum_out))
    return nl_set_error(NL_EINVAL, "layernorm: null pointer");
  if ((((uintptr_t)x | (uintptr_t)y | (uintptr_t)gamma | (uintptr_t)beta | (uintptr_t)residual | (uintptr_t)sum_out) &
       15) != 0)
    return nl_set_error(NL_EALIGN, "layernorm: buffers must be 16-byte aligned");
  const dim3 block(64 * kRowsPerBlock);
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((rows + kRowsPerBlock - 1) / kRowsPerBlock);
  switch (vectors_per_lane(D)) {
#define NL_LNF(N)                                                                                                    \
  case N:                                                                                                            \
    hipLaunchKernelGGL(ln_fwd_kernel<N>, grid, block, 0, st, rows, D, x, residual, sum_out, gamma, beta, y, mean,    \
                       rstd, eps);                                                                                   \
    break;
    NL_LNF(1)
    NL_LNF(2)
    NL_LNF(4)
    NL_LNF(8)
#undef NL_LNF
  }
  return nl_check_launch("nl_layernorm_fwd");
}

extern "C" size_t nl_layernorm_bwd_ws_bytes(int rows, int D) {
  if (rows <= 0 || D <= 0) return 0;
  return (size_t)2 * std::min(kLnBwdBlocks, (rows + kRowsPerBlock - 1) / kRowsPerBlock) * D * sizeof(float);
}

#define NL_TRY(x)        \
  do {                   \
    int rc_ = (x);       \
    if (rc_) return rc_; \
  } while (0)

namespace nl {
namespace {
PartialSums no_partial_sums() {
  PartialSums r{};
  return r;
}

// Checks the arguments of one LayerNorm backward and launches ln_bwd_kernel,
// its parameter sums left as partial rows in ws, plus the workgroups of prev.
int ln_bwd_launch(void* stream, int rows, int D, const nl_bf16* dy, const nl_bf16* x, const float* mean,
                  const float* rstd, const float* gamma, const nl_bf16* dres, nl_bf16* dx, void* ws, size_t ws_bytes,
                  const PartialSums& prev, const char* who) {
  if (rows < 0 || D <= 0 || (D % 8) != 0 || D > kMaxD)
    return nl_set_error(NL_EINVAL, std::string(who) + ": need 0 < D <= 4096 and D % 8 == 0");
  const int nblk = rows > 0 ? ln_bwd_blocks(rows, D) : 0;
  if (rows > 0) {
    if (!dy || !x || !mean || !rstd || !gamma || !dx || !ws)
      return nl_set_error(NL_EINVAL, std::string(who) + ": null pointer");
    if ((((uintptr_t)dy | (uintptr_t)x | (uintptr_t)dx | (uintptr_t)dres | (uintptr_t)gamma | (uintptr_t)ws) & 15) != 0)
      return nl_set_error(NL_EALIGN, std::string(who) + ": buffers must be 16-byte aligned");
    if (ws_bytes < nl_layernorm_bwd_ws_bytes(rows, D))
      return nl_set_error(NL_EINVAL, std::string(who) + ": workspace smaller than nl_layernorm_bwd_ws_bytes()");
  }
  const int grid = nblk + 2 * prev.strips;
  if (grid == 0) return NL_OK;
  float* pg = static_cast<float*>(ws);
  float* pb = rows > 0 ? pg + (size_t)nblk * D : nullptr;
  hipStream_t st = (hipStream_t)stream;
  switch (vectors_per_lane(D)) {
#define NL_LNB(N)                                                                                                 \
  case N:                                                                                                         \
    hipLaunchKernelGGL(ln_bwd_kernel<N>, dim3(grid), dim3(64 * kRowsPerBlock), 0, st, rows, D, dy, x, mean, rstd, \
                       gamma, dres, dx, pg, pb, nblk, prev);                                                      \
    break;
    NL_LNB(1)
    NL_LNB(2)
    NL_LNB(4)
    NL_LNB(8)
#undef NL_LNB
  }
  return NL_OK;
}

// The reduction of the partial rows a deferred call left in ws.
int partial_sums_of(int rows, int D, const void* ws, float* dgamma, float* dbeta, int accumulate, PartialSums& out,
                    const char* who) {
  out = no_partial_sums();
  if (rows <= 0 || !ws) return NL_OK;
  if (D <= 0 || (D % 8) != 0 || D > kMaxD)
    return nl_set_error(NL_EINVAL, std::string(who) + ": partial sums need 0 < D <= 4096 and D % 8 == 0");
  if (!dgamma || !dbeta) return nl_set_error(NL_EINVAL, std::string(who) + ": null dgamma or dbeta");
  if (((uintptr_t)ws & 15) != 0) return nl_set_error(NL_EALIGN, std::string(who) + ": partials must be 16-byte aligned");
  out.P = ln_bwd_blocks(rows, D);
  out.D = D;
  out.strips = (D + 15) / 16;
  out.part_g = static_cast<const float*>(ws);
  out.part_b = out.part_g + (size_t)out.P * D;
  out.dgamma = dgamma;
  out.dbeta = dbeta;
  out.accumulate = accumulate;
  return NL_OK;
}
}  // namespace
}  // namespace nl

extern "C" int nl_layernorm_bwd(void* stream, int rows, int D, const nl_bf16* dy, const nl_bf16* x, const float* mean,
                                const float* rstd, const float* gamma, const nl_bf16* dres, nl_bf16* dx, float* dgamma,
                                float* dbeta, int accumulate, void* ws, size_t ws_bytes) {
  if (rows < 0 || D <= 0 || (D % 8) != 0 || D > kMaxD)
    return nl_set_error(NL_EINVAL, "layernorm: need 0 < D <= 4096 and D % 8 == 0");
  if (rows == 0) return NL_OK;
  if (!dgamma || !dbeta) return nl_set_error(NL_EINVAL, "layernorm_bwd: null pointer");
  NL_TRY(ln_bwd_launch(stream, rows, D, dy, x, mean, rstd, gamma, dres, dx, ws, ws_bytes, no_partial_sums(),
                       "layernorm_bwd"));
  const int blocks = ln_bwd_blocks(rows, D);
  const float* pg = static_cast<const float*>(ws);
  hipLaunchKernelGGL(sum_partials_kernel, dim3((D + 15) / 16, 2), dim3(256), 0, (hipStream_t)stream, blocks, D, pg,
                     dgamma, pg + (size_t)blocks * D, dbeta, accumulate);
  return nl_check_launch("nl_layernorm_bwd");
}

extern "C" int nl_layernorm_bwd_deferred(void* stream, int rows, int D, const nl_bf16* dy, const nl_bf16* x,
                                         const float* mean, const float* rstd, const float* gamma,
                                         const nl_bf16* dres, nl_bf16* dx, void* ws, size_t ws_bytes, int prev_rows,
                                         int prev_D, const void* prev_ws, float* prev_dgamma, float* prev_dbeta,
                                         int prev_accumulate) {
  PartialSums prev;
  NL_TRY(partial_sums_of(prev_rows, prev_D, prev_ws, prev_dgamma, prev_dbeta, prev_accumulate, prev,
                         "layernorm_bwd_deferred"));
  NL_TRY(ln_bwd_launch(stream, rows, D, dy, x, mean, rstd, gamma, dres, dx, ws, ws_bytes, prev,
                       "layernorm_bwd_deferred"));
  return nl_check_launch("nl_layernorm_bwd_deferred");
}

extern "C" int nl_layernorm_param_sums(void* stream, int rows, int D, const void* ws, float* dgamma, float* dbeta,
                                       int accumulate) {
  if (rows < 0) return nl_set_error(NL_EINVAL, "layernorm_param_sums: rows < 0");
  PartialSums ps;
  NL_TRY(partial_sums_of(rows, D, ws, dgamma, dbeta, accumulate, ps, "layernorm_param_sums"));
  if (ps.strips == 0) return NL_OK;
  hipLaunchKernelGGL(sum_partials_kernel, dim3(ps.strips, 2), dim3(256), 0, (hipStream_t)stream, ps.P, ps.D,
                     ps.part_g, ps.dgamma, ps.part_b, ps.dbeta, accumulate);
  return nl_check_launch("nl_layernorm_param_sums");
}

extern "C" size_t nl_colsum_ws_bytes(int rows, int cols) {
  if (rows <= 0 || cols <= 0) return 0;
  return (size_t)((rows + kColsumRows - 1) / kColsumRows) * cols * sizeof(float);
}

extern "C" int nl_colsum_bf16(void* stream, int rows, int cols, const nl_bf16* x, int64_t ld, float* out,
                              int accumulate, void* ws, size_t ws_bytes) {
  if (rows <= 0 || cols <= 0) return nl_set_error(NL_EINVAL, "colsum: need rows > 0 and cols > 0");
  if (ld < cols) return nl_set_error(NL_EINVAL, "colsum: ld < cols");
  if (!x || !out || !ws) return nl_set_error(NL_EINVAL, "colsum: null pointer");
  if ((((uintptr_t)x | (uintptr_t)ws) & 15) != 0 || (ld & 7) != 0)
    return nl_set_error(NL_EALIGN, "colsum: x and ws must be 16-byte aligned and ld % 8 == 0");
  if (ws_bytes < nl_colsum_ws_bytes(rows, cols))
    return nl_set_error(NL_EINVAL, "colsum: workspace smaller than nl_colsum_ws_bytes()");
  const int P = (rows + kColsumRows - 1) / kColsumRows;
  if (P > 65535) return nl_set_error(NL_EINVAL, "colsum: too many rows");
  float* part = static_cast<float*>(ws);
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(colsum_partial_kernel, dim3((cols + 511) / 512, P), dim3(256), 0, st, rows, cols, x, ld, part);
  hipLaunchKernelGGL(sum_partials_kernel, dim3((cols + 15) / 16, 1), dim3(256), 0, st, P, cols, (const float*)part, out,
                     (const float*)nullptr, (float*)nullptr, accumulate);
  return nl_check_launch("nl_colsum_bf16");
}

extern "C" int nl_embedding_fwd(void* stream, int batch, int seq, int D, int vocab, const int32_t* ids,
                                const float* tok, const float* pos, nl_bf16* out) {
  if (batch < 0 || seq < 0 || D <= 0 || (D % 4) != 0 || vocab <= 0)
    return nl_set_error(NL_EINVAL, "embedding: need D % 4 == 0 and vocab > 0");
  if (batch == 0 || seq == 0) return NL_OK;
  if (!ids || !tok || !pos || !out) return nl_set_error(NL_EINVAL, "embedding: null pointer");
  if ((((uintptr_t)tok | (uintptr_t)pos) & 15) != 0 || ((uintptr_t)out & 7) != 0)
    return nl_set_error(NL_EALIGN, "embedding: tables must be 16-byte and out 8-byte aligned");
  if ((int64_t)batch * seq > 0x7fffffff) return nl_set_error(NL_EINVAL, "embedding: too many tokens");
  hipLaunchKernelGGL(embed_fwd_kernel, dim3(batch * seq), dim3(128), 0, (hipStream_t)stream, seq, D, ids, tok, pos,
                     out, vocab);
  return nl_check_launch("nl_embedding_fwd");
}

// counts and segment offsets ([buckets][parts] ints each), then one 8-byte
// (t, id) entry per token from a 16-byte boundary
static size_t emb_head_bytes(const EmbPlan& p) { return ((size_t)p.buckets * kEmbParts * 2 * sizeof(int) + 15) / 16 * 16; }

extern "C" size_t nl_embedding_bwd_ws_bytes(int batch, int seq, int D, int vocab) {
  if (batch <= 0 || seq <= 0 || D <= 0 || vocab <= 0) return 0;
  const EmbPlan p = emb_plan(D, vocab);
  return emb_head_bytes(p) + (size_t)batch * seq * sizeof(int2);
}

extern "C" int nl_embedding_bwd(void* stream, int batch, int seq, int D, int vocab, const int32_t* ids,
                                const nl_bf16* dx, float* dtok, float* dpos, int accumulate_pos, void* ws,
                                size_t ws_bytes) {
  if (batch < 0 || seq < 0 || D <= 0 || (D % 4) != 0 || vocab <= 0)
    return nl_set_error(NL_EINVAL, "embedding_bwd: need D % 4 == 0 and vocab > 0");
  if (D * 4 > kEmbTokLds) return nl_set_error(NL_EINVAL, "embedding_bwd: D above 4096");
  const int64_t T64 = (int64_t)batch * seq;
  if (!dtok || (seq > 0 && !dpos) || (T64 > 0 && (!ids || !dx)))
    return nl_set_error(NL_EINVAL, "embedding_bwd: null pointer");
  if ((((uintptr_t)dtok) & 15) != 0 || (((uintptr_t)dx) & 7) != 0)
    return nl_set_error(NL_EALIGN, "embedding_bwd: dtok must be 16-byte and dx 8-byte aligned");
  if (T64 > 0x7fffffff - 1024) return nl_set_error(NL_EINVAL, "embedding_bwd: too many tokens");
  const EmbPlan p = emb_plan(D, vocab);
  const int64_t grid = seq + (int64_t)p.buckets * ((p.W + emb_rows(D) - 1) / emb_rows(D));
  if (grid > 0x7fffffff) return nl_set_error(NL_EINVAL, "embedding_bwd: vocabulary too large");
  const int T = (int)T64;
  hipStream_t st = (hipStream_t)stream;
  int* counts = nullptr;
  int* offsets = nullptr;
  int2* lists = nullptr;
  if (T > 0) {
    if (!ws || ws_bytes < nl_embedding_bwd_ws_bytes(batch, seq, D, vocab) || ((uintptr_t)ws & 15) != 0)
      return nl_set_error(NL_EINVAL, "embedding_bwd: workspace below nl_embedding_bwd_ws_bytes()");
    if (p.buckets > kEmbMaxBuckets) return nl_set_error(NL_EUNSUPPORTED, "embedding_bwd: too many buckets");
    counts = reinterpret_cast<int*>(ws);
    offsets = counts + (size_t)p.buckets * kEmbParts;
    lists = reinterpret_cast<int2*>(reinterpret_cast<char*>(ws) + emb_head_bytes(p));
    hipLaunchKernelGGL(embed_count_kernel, dim3(kEmbParts), dim3(256), 0, st, T, vocab, p.W, p.buckets, ids, counts);
    hipLaunchKernelGGL(embed_bucket_kernel, dim3(p.buckets * kEmbParts), dim3(256), 0, st, T, vocab, p.W, ids, counts,
                       offsets, lists);
  }
  // with no tokens every row of dtok is still written (zero): counts is not read then
  auto go = [&](auto f) {
    f(st, grid, batch, seq, D, dx, dtok, vocab, p.W, counts, offsets, lists, dpos, accumulate_pos);
  };
  switch (emb_rows(D)) {
    case 8: go(launch_embed_bwd<2, 8>); break;
    case 4: go(launch_embed_bwd<4, 4>); break;
    case 2: go(launch_embed_bwd<4, 2>); break;
    default: go(launch_embed_bwd<4, 1>); break;
  }
  return nl_check_launch("nl_embedding_bwd");
}
