// na_wave.h — pieces of the wave kernels (one wave, one 16-row tile, float32
// matrix cores): the fused op (na_wave.hip) and the split and
// position-bias ops (na_wsplit.hip).  Problem and tile description, the box of
// rows a tile's windows cover and its points, packed window tests, the score
// and accumulate products, and the host-side choice of tiles.
#pragma once

#include <algorithm>
#include <cmath>

#include "na_common.h"
#include "na_launch.h"

namespace na {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

// A lane's 16-byte fragment of each 64-byte piece of a row, the 16x16 score
// product over one piece, and the fragment as float32 (EPF elements from
// element EPF * gq of the piece).
template <typename T>
struct Wv;
template <>
struct Wv<float> {
  typedef f32x4 frag;
  static constexpr int EPF = 4;
  static __device__ __forceinline__ f32x4 mma(frag a, frag b, f32x4 c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a[i], b[i], c, 0, 0, 0);
    return c;
  }
};
template <>
struct Wv<bf16_t> {
  typedef __bf16 frag __attribute__((ext_vector_type(8)));
  static constexpr int EPF = 8;
  static __device__ __forceinline__ f32x4 mma(frag a, frag b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
  }
};
template <>
struct Wv<f16_t> {
  typedef _Float16 frag __attribute__((ext_vector_type(8)));
  static constexpr int EPF = 8;
  static __device__ __forceinline__ f32x4 mma(frag a, frag b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
  }
};

// Tiling of the query grid (forward, dQ) or the key grid (dK / dV).
struct WvGrid {
  int32_t T[3], lgT[3], nt[3];  // tile extents (powers of two), tiles per phase
  FastDiv fG[3], fnt[3];        // d * nt, nt
  FastDiv fGrid;                // tiles per (sample, head)
  int32_t n_tiles, n_wg;        // waves, workgroups launched (a multiple of 8)
};

struct WvAx {
  int32_t K, nh, d, s, causal, O;
  int32_t Lq, Lrem;    // phase r of the keys holds Lq + (r < Lrem) points
  int32_t tok, otok;   // token strides of one position: input and output grid
};

struct WvProb {
  WvAx ax[3];
  int32_t B, H, Hkv, rep;
  int64_t Ltot, Otot;  // tokens per sample: input and output grid
  FastDiv fH, fHkv, fRep;
  float scale, sl2;    // sl2 = scale * log2(e)
  WvGrid gq, gk;       // query tiles, key tiles
};

// Box coordinates packed into one word, a guard bit above each field.
template <int R>
struct Pk {
  static constexpr int W = R == 1 ? 32 : R == 2 ? 16 : 10;  // field width
  static constexpr uint32_t kMax = (1u << (W - 1)) - 1;     // largest coordinate
  static constexpr uint32_t kGuard =
      R == 1 ? 0x80000000u : R == 2 ? 0x80008000u : (1u << 9) | (1u << 19) | (1u << 29);
  static constexpr uint32_t kAll =
      R == 1 ? kMax : R == 2 ? kMax * 0x10001u : kMax * 0x100401u;
  static __device__ __forceinline__ constexpr int shift(int a) { return (2 - a) * (R == 1 ? 0 : W); }
};

struct WvTile {
  int b, h;
  int r[3], i0[3], nv[3], Lr[3], Qr[3];
};

__device__ __forceinline__ int wv_start(const WvAx &x, int ip, int Lr) {
  return x.causal ? max(ip - x.K + 1, 0) : min(max(ip - x.nh, 0), Lr - x.K);
}
__device__ __forceinline__ int wv_end(const WvAx &x, int ip, int Lr) {
  return x.causal ? ip + 1 : min(max(ip - x.nh, 0), Lr - x.K) + x.K;
}
// Query indices [first, last) whose windows hold key j: the positions are
// [j <= K-1 ? 0 : j - K/2, j >= Lr-K ? Lr : j + K/2 + 1) (causal [j, j + K)),
// of which every s-th carries a query.
__device__ __forceinline__ int wv_istart(const WvAx &x, int j) {
  const int p = x.causal ? j : (j <= x.K - 1 ? 0 : j - x.nh);
  return x.s == 1 ? p : (p + x.s - 1) / x.s;
}
__device__ __forceinline__ int wv_iend(const WvAx &x, int j, int Lr, int Qr) {
  const int p = x.causal ? min(j + x.K, Lr) : (j >= Lr - x.K ? Lr : j + x.nh + 1);
  return x.s == 1 ? p : min((p + x.s - 1) / x.s, Qr);
}

template <int R>
__device__ __forceinline__ bool wv_decode(const WvProb &P, const WvGrid &G, const FastDiv &fHn,
                                          uint32_t tile, bool keys, WvTile &t) {
  const uint32_t rest = fdiv(tile, G.fGrid);
  uint32_t sp = tile - rest * G.fGrid.d;
  const uint32_t bq = fdiv(rest, fHn);
  t.h = (int)(rest - bq * fHn.d);
  t.b = (int)bq;
  bool any = t.b < P.B;
#pragma unroll
  for (int a = 2; a >= 3 - R; --a) {
    const WvAx &x = P.ax[a];
    uint32_t g = sp;
    if (a > 3 - R) {
      const uint32_t qd = fdiv(sp, G.fG[a]);
      g = sp - qd * G.fG[a].d;
      sp = qd;
    }
    const int rr = (int)fdiv(g, G.fnt[a]);
    t.r[a] = rr;
    t.i0[a] = ((int)g - rr * G.nt[a]) << G.lgT[a];
    t.Lr[a] = x.Lq + (rr < x.Lrem ? 1 : 0);
    t.Qr[a] = x.s == 1 ? t.Lr[a] : x.O;
    t.nv[a] = min((keys ? t.Lr[a] : t.Qr[a]) - t.i0[a], G.T[a]);
    any = any && t.nv[a] > 0;
  }
  return any;
}

// Index of the lane's row (position n of the tile, the last one past its end)
// on axis a.
__device__ __forceinline__ int wv_row(const WvGrid &G, const WvTile &t, int a, int n, bool &valid) {
  int sh = 0;
  for (int c = 2; c > a; --c) sh += G.lgT[c];
  const int u = (n >> sh) & (G.T[a] - 1);
  valid = valid && u < t.nv[a];
  return t.i0[a] + min(u, t.nv[a] - 1);
}

// A box of rows numbered row-major: extents, byte strides of its points in
// one tensor (and a second one), and the decoding of a point's number.
template <int R, bool TWO>
struct WvBox {
  int lo[3], E[3], npts;
  uint32_t SK[3], SO[3];
  float r2, r1;
  __device__ __forceinline__ void finish() {
    npts = 1;
#pragma unroll
    for (int a = 3 - R; a < 3; ++a) npts *= max(E[a], 0);
    r2 = __builtin_amdgcn_rcpf((float)E[2]);
    r1 = R == 3 ? __builtin_amdgcn_rcpf((float)E[1]) : 0.f;
  }
  // Packed coordinates and byte offsets of point x.  The quotients come
  // from a product with the reciprocal: (x + 1/2) / E is at least 1/(2 E)
  // from an integer and the product is off by less than x 2^-22 / E, so they
  // are exact for x < 2^20.
  __device__ __forceinline__ uint32_t coords(int x, int (&e)[3]) const {
    const int xc = min(x, npts - 1);
    e[0] = e[1] = 0;
    e[2] = xc;
    if (R >= 2) {
      e[1] = (int)(((float)xc + 0.5f) * r2);
      e[2] = xc - e[1] * E[2];
    }
    if (R == 3) {
      e[0] = (int)(((float)e[1] + 0.5f) * r1);
      e[1] -= e[0] * E[1];
    }
    uint32_t c = (uint32_t)e[2];
    if (R >= 2) c |= (uint32_t)e[1] << Pk<R>::shift(1);
    if (R == 3) c |= (uint32_t)e[0] << Pk<R>::shift(0);
    return x < npts ? c : Pk<R>::kAll;  // past the box: in no window
  }
  static __device__ __forceinline__ uint32_t offset(const int (&e)[3], const uint32_t (&S)[3]) {
    uint32_t off = (uint32_t)e[2] * S[2];
    if (R >= 2) off += (uint32_t)e[1] * S[1];
    if (R == 3) off += (uint32_t)e[0] * S[0];
    return off;
  }
  __device__ __forceinline__ uint32_t point(int x, uint32_t &off, uint32_t &off2) const {
    int e[3];
    const uint32_t c = coords(x, e);
    off = offset(e, SK);
    off2 = TWO ? offset(e, SO) : off;
    return c;
  }
};

// A lane's window in box coordinates, packed: wl its first point, wh its last.
template <int R>
struct WvWin {
  uint32_t wl = 0, wh = 0;
  bool none = false;
  __device__ __forceinline__ void axis(int a, int first, int last) {
    none = none || last < first;
    wl |= (uint32_t)first << Pk<R>::shift(a);
    wh |= (uint32_t)last << Pk<R>::shift(a);
  }
  __device__ __forceinline__ void finish() {
    if (none) {
      wl = Pk<R>::kAll;
      wh = 0;
    }
  }
  // every field of (c - wl) and (wh - c) is non-negative
  __device__ __forceinline__ bool holds(uint32_t c) const {
    constexpr uint32_t g = Pk<R>::kGuard;
    return (((c | g) - wl) & ((wh | g) - c) & g) == g;
  }
};

template <typename T, int NF>
__device__ __forceinline__ void ld_row(const char *base, uint32_t off, typename Wv<T>::frag (&f)[NF]) {
#pragma unroll
  for (int i = 0; i < NF; ++i)
    f[i] = *reinterpret_cast<const typename Wv<T>::frag *>(base + (size_t)(off + 64u * i));
}

// Four consecutive elements as float32, and their store.
template <typename T>
__device__ __forceinline__ f32x4 ld4(const char *p) {
  f32x4 v;
  if constexpr (sizeof(T) == 4) {
    v = *reinterpret_cast<const f32x4 *>(p);
  } else {
    float x[4];
    VecIO<T, 4>::load(reinterpret_cast<const T *>(p), x);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = x[r];
  }
  return v;
}
template <typename T>
__device__ __forceinline__ void st4(char *p, f32x4 v) {
  const float x[4] = {v[0], v[1], v[2], v[3]};
  VecIO<T, 4>::store(reinterpret_cast<T *>(p), x);
}

template <typename T>
__device__ __forceinline__ float wv_dot(typename Wv<T>::frag a, typename Wv<T>::frag b, float c) {
#pragma unroll
  for (int e = 0; e < Wv<T>::EPF; ++e) c = fmaf((float)a[e], (float)b[e], c);
  return c;
}

// The lane's fragments of its row n into LDS row `row` as float32.
template <typename T, int NF>
__device__ __forceinline__ void wv_lds(float *row, int gq, const typename Wv<T>::frag (&f)[NF]) {
  constexpr int N = Wv<T>::EPF;
#pragma unroll
  for (int i = 0; i < NF; ++i)
#pragma unroll
    for (int e = 0; e < N; e += 4) {
      const f32x4 v = {(float)f[i][e], (float)f[i][e + 1], (float)f[i][e + 2], (float)f[i][e + 3]};
      *reinterpret_cast<f32x4 *>(row + 4 * N * i + N * gq + e) = v;
    }
}

// The 16x16 products of rows a[0..NF) with rows b: up to four sums of their
// own, added pairwise (a single chain over head_dim lost 1.2e-7 of a forward's
// output where the lane-group sums of na_valu.hip lose 1.0e-7), which also
// keeps several products in flight.
template <typename T, int NF>
__device__ __forceinline__ f32x4 wv_scores(const typename Wv<T>::frag (&a)[NF],
                                           const typename Wv<T>::frag (&b)[NF]) {
  constexpr int N = NF < 4 ? NF : 4;
  f32x4 s[N];
#pragma unroll
  for (int i = 0; i < N; ++i) s[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NF; ++i) s[i % N] = Wv<T>::mma(a[i], b[i], s[i % N]);
  if constexpr (N == 4) return (s[0] + s[1]) + (s[2] + s[3]);
  if constexpr (N == 2) return s[0] + s[1];
  return s[0];
}

// acc^T += X^T W: X the 16 LDS rows, the lane's w[r] the weight of row
// 4 gq + r in its column.
template <int NDB, int RS>
__device__ __forceinline__ void wv_acc(const float *xt, const float (&w)[4], f32x4 (&acc)[NDB]) {
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int db = 0; db < NDB; ++db)
      acc[db] = __builtin_amdgcn_mfma_f32_16x16x4f32(xt[r * RS + 16 * db], w[r], acc[db], 0, 0, 0);
}

__device__ __forceinline__ float wv_quad_max(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float wv_quad_sum(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// This wave's LDS operations so far are complete.
__device__ __forceinline__ void wv_lds_sync() {
  __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  __builtin_amdgcn_wave_barrier();
  asm volatile("" ::: "memory");
}

template <int NDB>
__device__ __forceinline__ bool wv_nan(const f32x4 (&a)[NDB], float t) {
#pragma unroll
  for (int db = 0; db < NDB; ++db)
#pragma unroll
    for (int r = 0; r < 4; ++r) t += a[db][r];
  return __builtin_amdgcn_ballot_w64(!(t == t)) != 0;  // inf - inf too: no harm
}

// Workgroups reach the 8 XCDs in turn; each XCD gets a contiguous run of them.
__device__ __forceinline__ int wv_wg(int bid, int n_wg) { return (bid & 7) * (n_wg >> 3) + (bid >> 3); }

// Waves per workgroup (they are independent; at head_dim 128 the backward's
// LDS rows of four would pass 64 KB).
template <int D>
constexpr int wv_waves() {
  return D == 128 ? 2 : 4;
}
// LDS row stride in floats: 4 mod 64 banks apart (36, 68, ...; 20 for 16), so
// the 16 rows' 16-byte writes and the transposed reads of 4 row groups x 16
// columns are free of conflicts.
template <int D>
constexpr int wv_rs() {
  return D + 4;
}

// ---------------------------------------------------------------------------
// Host side.

int phase_max(const Axis &x) { return (int)(((int64_t)x.L + x.d - 1) / x.d); }

// Tile extents (product 16) with the fewest chunks over the grid.
void wv_tile(const Prob &P, bool keys, int T[3]) {
  const int lead = 3 - P.rank;
  double best = 1e300;
  for (int l0 = 0; l0 <= 4; ++l0)
    for (int l1 = 0; l0 + l1 <= 4; ++l1) {
      const int Tt[3] = {1 << l0, 1 << l1, 1 << (4 - l0 - l1)};
      bool ok = true;
      for (int a = 0; a < lead; ++a) ok = ok && Tt[a] == 1;
      if (!ok) continue;
      double tiles = 1.0, pts = 1.0;
      for (int a = lead; a < 3; ++a) {
        const Axis &x = P.ax[a];
        const int Lr = phase_max(x), Qr = x.s == 1 ? Lr : x.O;
        const int len = keys ? Lr : Qr;
        tiles *= (double)x.d * ((len + Tt[a] - 1) / Tt[a]);
        pts *= keys ? std::min(Qr, (Tt[a] + x.K - 2) / x.s + 1)
                    : std::min(Lr, (Tt[a] - 1) * x.s + x.K);
      }
      const double cost = tiles * std::ceil(pts / 16.0);
      if (cost < best) {
        best = cost;
        for (int a = 0; a < 3; ++a) T[a] = Tt[a];
      }
    }
}

WvGrid wv_grid(const Prob &P, bool keys, int waves) {
  WvGrid G{};
  int T[3] = {1, 1, 16};
  wv_tile(P, keys, T);
  int64_t grid = 1;
  for (int a = 0; a < 3; ++a) {
    const Axis &x = P.ax[a];
    const int Lr = phase_max(x), len = keys || x.s == 1 ? Lr : x.O;
    G.T[a] = T[a];
    while ((1 << G.lgT[a]) < T[a]) ++G.lgT[a];
    G.nt[a] = (len + T[a] - 1) / T[a];
    G.fG[a] = make_fastdiv((uint32_t)(x.d * G.nt[a]));
    G.fnt[a] = make_fastdiv((uint32_t)G.nt[a]);
    grid *= (int64_t)x.d * G.nt[a];
  }
  G.fGrid = make_fastdiv((uint32_t)grid);
  G.n_tiles = (int32_t)(P.B * (keys ? P.Hkv : P.H) * grid);
  G.n_wg = ((G.n_tiles + waves - 1) / waves + 7) & ~7;
  return G;
}

WvProb make_wvprob(const Prob &P, bool backward, int waves) {
  WvProb W{};
  W.B = P.B;
  W.H = P.H;
  W.Hkv = P.Hkv;
  W.rep = P.rep;
  int32_t tok = 1, otok = 1;
  for (int a = 2; a >= 0; --a) {
    const Axis &x = P.ax[a];
    WvAx &y = W.ax[a];
    y.K = x.K;
    y.nh = x.K / 2;
    y.d = x.d;
    y.s = x.s;
    y.causal = x.causal;
    y.O = x.O;
    y.Lq = x.L / x.d;
    y.Lrem = x.L % x.d;
    y.tok = tok;
    y.otok = otok;
    tok *= x.L;
    otok *= x.O;
  }
  W.Ltot = tok;
  W.Otot = otok;
  W.fH = make_fastdiv((uint32_t)P.H);
  W.fHkv = make_fastdiv((uint32_t)P.Hkv);
  W.fRep = make_fastdiv((uint32_t)P.rep);
  W.scale = P.scale;
  W.sl2 = P.scale * kLog2e;
  W.gq = wv_grid(P, false, waves);
  if (backward) W.gk = wv_grid(P, true, waves);
  return W;
}

// The launch of both grids (a backward's two passes) holds fewer than 2^32
// threads: ragged phases (three points of 16 rows each, or d > L on a causal axis)
// take up to a wave per point.
bool wv_launch_ok(const Prob &P) {
  constexpr int64_t most = ((int64_t)1 << 32) / 64 - 64;  // waves, the last workgroups' apart
  auto points = [&](int a) { return (int64_t)P.ax[a].d * phase_max(P.ax[a]); };
  if (points(0) >= most || points(1) >= most || points(2) >= most) return false;
  // every tile holds a point: far below the limit without the tiles
  const double all = (double)P.B * P.H * points(0) * points(1) * points(2);
  if (2.0 * all < (double)most) return true;
  double waves = 0.0;
  for (int keys = 0; keys < 2; ++keys) {
    int T[3] = {1, 1, 16};
    wv_tile(P, keys != 0, T);
    double n = (double)P.B * (keys ? P.Hkv : P.H);
    for (int a = 0; a < 3; ++a) {
      const Axis &x = P.ax[a];
      const int len = keys || x.s == 1 ? phase_max(x) : x.O;
      n *= (double)x.d * ((len + T[a] - 1) / T[a]);
    }
    waves += n;
  }
  return waves < (double)most;
}

// Window rules, box sizes and index arithmetic of the wave kernels, for rows
// of `es`-byte elements.
bool wv_geometry_ok(const Prob &P, int64_t es) {
  // box extents within the packed coordinate fields, box points within the
  // range of the reciprocal division (an inverse box spans at most
  // T + 2 (K - 1) points, a forward one (T - 1) s + K, s <= K: T <= 16)
  const int64_t field = P.rank == 1 ? (int64_t)1 << 18 : P.rank == 2 ? 32767 : 511;
  int64_t pts = 1;
  for (int a = 3 - P.rank; a < 3; ++a) {
    const Axis &x = P.ax[a];
    if (x.s != 1 && (x.d != 1 || x.s > x.K)) return false;
    if (!x.causal && ((x.K % 2) == 0 || (int64_t)x.d * x.K > x.L)) return false;
    const int64_t e = std::min<int64_t>(phase_max(x), 16 + std::max<int64_t>(2 * x.K, 16 * x.s + x.K));
    if (e > field) return false;
    pts *= e;
  }
  if (pts > ((int64_t)1 << 18)) return false;
  // 32-bit byte offsets inside a sample, 32-bit tile numbers
  const int64_t tokens = (int64_t)P.ax[0].L * P.ax[1].L * P.ax[2].L;
  if (tokens * std::max(P.H, P.Hkv) * P.D * es >= ((int64_t)1 << 31)) return false;
  return (int64_t)P.B * P.H * tokens < ((int64_t)1 << 30) && wv_launch_ok(P);
}

}  // namespace
}  // namespace na
