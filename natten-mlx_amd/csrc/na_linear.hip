// na_linear.hip — pieces of the attention layer around the fused op: the packed
// projection [token, 3, H D] taken apart into q, k and v and their gradients put
// back together (k_pack3), and the weight and bias gradient of the projections:
// dW[n, k] = sum over tokens of G[m, n] X[m, k], db[n] = the
// column sums of G, for bf16 / fp16 rows.
//
// The sum runs over tens of thousands of tokens into a matrix of a few tiles,
// so the tokens are split over the chip.  A workgroup of four waves takes a
// 128 x 128 tile of dW over one run of tokens: 64 rows of G and X are staged in
// one of two LDS buffers while the rows before them are multiplied, both
// operands come out of LDS through the transposing read (the tokens are the
// contraction), and each wave holds a 64 x 64 block in 16 accumulators of
// 16x16x32 MFMAs.  Partial sums stay float32; a second pass adds them in token
// order and rounds once, so the result does not depend on the run.  db is one
// more column of the product (a ones operand) in the workgroups of the first
// column of tiles.
//
// What bounds it: each workgroup's chain of stages (load 64 rows, wait, store,
// barrier, 32 MFMAs per wave), with two workgroups on a CU to overlap.  By
// counters (bf16, 25088 rows, 768 x 256) k_wgrad reads 51.5 MB, G and X once, and
// writes 31.6 MB of partial sums in 27 us, 3.0 TB/s against 4.8 of a copy; its waves
// spend 34% of their time waiting for loads and barriers, 25% for an issue slot,
// and the matrix cores are busy 15% of it.  k_wgrad_sum reads the partial sums
// back in 6.6 us at the copy's rate.  The library's kernels for these shapes give
// a tile the whole sum and leave most of the chip idle (25088 rows, with
// db: 768 x 256 163 -> 33 us, 256 x 256 121 -> 21, 1536 x 512 198 -> 82; 41472 rows,
// 768 x 256: 234 -> 43).
#include "na_launch.h"
#include "na_lean.h"

namespace na {
namespace {

constexpr int kWgTile = 128;  // rows and columns of dW per workgroup
constexpr int kWgRows = 64;   // tokens per stage
constexpr int kWgRS = kWgTile + 8;  // LDS row stride in elements

struct WgProb {
  int32_t N, K;        // columns of G and of X
  int64_t M;           // tokens
  int32_t mper, S;     // tokens per split, splits
  int32_t tn, tk;      // tiles over N and K
  int32_t n_launch;
  FastDiv ftiles, ftk;
};

template <typename T>
__global__ void __launch_bounds__(256)
    k_wgrad(WgProb P, const T *__restrict__ g, const T *__restrict__ x, float *__restrict__ part,
            int has_bias) {
  typedef L16<T> M;
  typedef typename M::v8 v8;
  typedef typename M::v4 v4;
  typedef typename M::e E;
  extern __shared__ __align__(16) char smem[];
  E *const buf = reinterpret_cast<E *>(smem);  // [2][G rows, X rows]
  constexpr int BUF = kWgRows * kWgRS;

  const int id = xcd_tile(blockIdx.x, P.n_launch);  // a split's tiles share an XCD's L2
  const int split = (int)fdiv((uint32_t)id, P.ftiles);
  if (split >= P.S) return;
  const int tile = id - split * (int)P.ftiles.d;
  const int ti = (int)fdiv((uint32_t)tile, P.ftk), tj = tile - ti * P.tk;
  const int n0 = ti * kWgTile, k0 = tj * kWgTile;
  const int64_t m0 = (int64_t)split * P.mper;
  const int rows = (int)min((int64_t)P.mper, P.M - m0);

  const int tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
  const int n = lane & 15, gq = lane >> 4;
  // staging: the thread's 16-byte column unit and rows r0 + 16 i
  const int cu = 8 * (tid & 15), r0 = tid >> 4;
  const bool gok = n0 + cu < P.N, xok = k0 + cu < P.K;
  const T *gp = g + (m0 + r0) * P.N + n0 + cu;
  const T *xp = x + (m0 + r0) * P.K + k0 + cu;
  v8 gr[4], xr[4];
  auto load = [&](int s) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = s + 16 * i;  // relative to r0
      const bool in = r0 + r < rows;
      v8 z;
#pragma unroll
      for (int e = 0; e < 8; ++e) z[e] = (E)0.f;
      gr[i] = in && gok ? *reinterpret_cast<const v8 *>(gp + (int64_t)r * P.N) : z;
      xr[i] = in && xok ? *reinterpret_cast<const v8 *>(xp + (int64_t)r * P.K) : z;
    }
  };
  auto store = [&](int b) {
    E *d = buf + b * 2 * BUF + r0 * kWgRS + cu;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      *reinterpret_cast<v8 *>(d + 16 * i * kWgRS) = gr[i];
      *reinterpret_cast<v8 *>(d + BUF + 16 * i * kWgRS) = xr[i];
    }
  };

  f32x4 acc[4][4], accb[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    accb[i] = zero4();
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = zero4();
  }
  const int wn = 64 * (w >> 1), wk = 64 * (w & 1);
  const bool bias = has_bias != 0 && tj == 0 && wk == 0;  // wave-uniform
  v8 ones;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = (E)1.f;
  const int tr = (4 * gq + (n >> 2)) * kWgRS + 4 * (n & 3);
  load(0);
  store(0);
  __syncthreads();
  const int steps = (rows + kWgRows - 1) / kWgRows;
  for (int s = 0; s < steps; ++s) {
    const bool more = s + 1 < steps;
    if (more) load((s + 1) * kWgRows);
    const E *gs = buf + (s & 1) * 2 * BUF + tr + wn, *xs = buf + (s & 1) * 2 * BUF + BUF + tr + wk;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      v8 a[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const v4 a0 = M::tr(gs + 32 * h * kWgRS + 16 * i), a1 = M::tr(gs + (32 * h + 16) * kWgRS + 16 * i);
        a[i] = __builtin_shufflevector(a0, a1, 0, 1, 2, 3, 4, 5, 6, 7);
        const v4 b0 = M::tr(xs + 32 * h * kWgRS + 16 * i), b1 = M::tr(xs + (32 * h + 16) * kWgRS + 16 * i);
        b[i] = __builtin_shufflevector(b0, b1, 0, 1, 2, 3, 4, 5, 6, 7);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = M::mma(a[i], b[j], acc[i][j]);
      if (bias)
#pragma unroll
        for (int i = 0; i < 4; ++i) accb[i] = M::mma(a[i], ones, accb[i]);
    }
    if (more) store((s + 1) & 1);
    __syncthreads();
  }
  // lane: rows 4 gq + r of block i, column n of block j
  float *pd = part + (int64_t)split * (P.N * (int64_t)P.K + P.N);  // dW, then db
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = n0 + wn + 16 * i + 4 * gq + r;
      if (row >= P.N) continue;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int col = k0 + wk + 16 * j + n;
        if (col < P.K) pd[(int64_t)row * P.K + col] = acc[i][j][r];
      }
      if (bias && n == 0) pd[(int64_t)P.N * P.K + row] = accb[i][r];
    }
}

// dW and db from the splits' sums: a workgroup takes 32 columns of four values,
// eight threads share a column (thread row j the splits j, j + 8, ...) and their
// sums meet in LDS, always in the same order.  (One thread per column, 98 splits
// of a 256 x 256 gradient over 25088 rows: 47 us with the product, this way 21.)
template <typename T>
__global__ void __launch_bounds__(256)
    k_wgrad_sum(const float *__restrict__ part, T *__restrict__ dw, T *__restrict__ db, int64_t nw,
                int64_t count, int S) {
  __shared__ float4 sums[8][32];
  const int c = threadIdx.x & 31, j = threadIdx.x >> 5;
  const int64_t i = ((int64_t)blockIdx.x * 32 + c) * 4;
  const bool live = i < (db != nullptr ? count : nw);
  float4 s = make_float4(0.f, 0.f, 0.f, 0.f);
  if (live) {
#pragma unroll 4
    for (int k = j; k < S; k += 8) {
      const float4 v = *reinterpret_cast<const float4 *>(part + k * count + i);
      s.x += v.x;
      s.y += v.y;
      s.z += v.z;
      s.w += v.w;
    }
  }
  sums[j][c] = s;
  __syncthreads();
  if (j != 0 || !live) return;
  float r[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float4 v = sums[k][c];
    r[0] += v.x;
    r[1] += v.y;
    r[2] += v.z;
    r[3] += v.w;
  }
  VecIO<T, 4>::store(i < nw ? dw + i : db + (i - nw), r);
}

// [tokens, 3, U] <-> [3, tokens, U] in 16-byte units: one launch and one pass in
// place of three strided copies each way (bf16 [8, 56, 56, 3, 8, 32]: 3 x 7 us -> 12 us, 6.4 TB/s).
template <bool SPLIT>
__global__ void __launch_bounds__(256)
    k_pack3(const uint4 *__restrict__ src, uint4 *__restrict__ dst, int64_t n, FastDiv fU,
            int64_t tokens) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;  // unit of [tokens, 3, U]
  if (i >= n) return;
  const uint32_t row = fdiv((uint32_t)i, fU);  // 3 token + part
  const uint32_t u = (uint32_t)i - row * fU.d;
  const uint32_t tok = row / 3u, s = row - 3u * tok;
  const int64_t j = ((int64_t)s * tokens + tok) * fU.d + u;
  if (SPLIT)
    dst[j] = src[i];
  else
    dst[i] = src[j];
}

WgProb make_wgprob(int64_t M, int N, int K) {
  WgProb P{};
  P.M = M;
  P.N = N;
  P.K = K;
  P.tn = (N + kWgTile - 1) / kWgTile;
  P.tk = (K + kWgTile - 1) / kWgTile;
  const int tiles = P.tn * P.tk;
  // about two workgroups per CU, runs of at least 256 tokens
  const int64_t want = std::max(1, 2 * kLeanCUs / tiles), most = std::max<int64_t>(1, M / 256);
  const int64_t S = std::min(want, most);
  P.mper = (int32_t)(((M + S - 1) / S + kWgRows - 1) / kWgRows * kWgRows);
  P.S = (int32_t)((M + P.mper - 1) / P.mper);
  P.n_launch = (tiles * P.S + 7) & ~7;
  P.ftiles = make_fastdiv((uint32_t)tiles);
  P.ftk = make_fastdiv((uint32_t)P.tk);
  return P;
}

}  // namespace

bool pack3_ok(int64_t tokens, int64_t row_bytes) {
  return tokens > 0 && row_bytes > 0 && row_bytes % 16 == 0 &&
         3 * tokens * (row_bytes / 16) < ((int64_t)1 << 31);
}

void pack3(bool split, int64_t tokens, int64_t row_bytes, const void *src, void *dst, hipStream_t st) {
  const int64_t n = 3 * tokens * (row_bytes / 16);
  const FastDiv fU = make_fastdiv((uint32_t)(row_bytes / 16));
  const dim3 grid((unsigned)((n + 255) / 256)), block(256);
  if (split)
    hipLaunchKernelGGL((k_pack3<true>), grid, block, 0, st, (const uint4 *)src, (uint4 *)dst, n, fU, tokens);
  else
    hipLaunchKernelGGL((k_pack3<false>), grid, block, 0, st, (const uint4 *)src, (uint4 *)dst, n, fU, tokens);
}

bool linear_wgrad_ok(int dtype, int64_t M, int64_t N, int64_t K) {
  return (dtype == NA_BF16 || dtype == NA_F16) && N > 0 && K > 0 && N % 8 == 0 && K % 8 == 0 &&
         N <= 16384 && K <= 16384 && M > 0 && M < ((int64_t)1 << 31);
}

size_t linear_wgrad_workspace(int64_t M, int64_t N, int64_t K) {
  const WgProb P = make_wgprob(M, (int)N, (int)K);
  return sizeof(float) * (size_t)P.S * (size_t)(N * K + N);
}

void linear_wgrad(int dtype, int64_t M, int64_t N, int64_t K, const void *g, const void *x,
                  void *dw, void *db, void *workspace, hipStream_t st) {
  const WgProb P = make_wgprob(M, (int)N, (int)K);
  float *part = static_cast<float *>(workspace);
  const size_t lds = sizeof(uint16_t) * 4 * kWgRows * kWgRS;
  auto run = [&](auto tag) {
    using T = decltype(tag);
    hipLaunchKernelGGL((k_wgrad<T>), dim3(P.n_launch), dim3(256), lds, st, P, (const T *)g,
                       (const T *)x, part, db != nullptr ? 1 : 0);
    const int64_t nw = N * K, count = nw + N;
    hipLaunchKernelGGL((k_wgrad_sum<T>), dim3((unsigned)((count / 4 + 31) / 32)), dim3(256), 0, st,
                       part, (T *)dw, (T *)db, nw, count, P.S);
  };
  if (dtype == NA_BF16) run(bf16_t{});
  else run(f16_t{});
}

}  // namespace na
