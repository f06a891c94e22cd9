// na_wsplit.hip — float32 split ops (QK logits, AV, and their backward) and
// the DiNAT QK + relative-position-bias / AV ops on float32 matrix cores, on
// the wave tiles of na_wave.h: one wave per 16 queries (or 16 keys), no
// barrier, rows and compact rows of its own in LDS.
//
// Compact rows [query, K0 K1 K2] hold one value per window slot, row-major over
// the axes.  The slot of the key at box coordinates e in a query's window that
// starts at wl is sum (e_a - wl_a) st_a, so a key's part (its linear slot
// index, computed once per row and handed over through LDS) minus a constant
// of the query's lane; the bias cell is the same with the table's strides.
//   ws_qk   compact = mult <x, y_key> (+ bias), `fill` outside the window:
//           logits, and dattn from (dout, v).  Scores go to their slots in
//           LDS, then the 16 rows leave as whole runs.
//   ws_av   out = mult sum_slot a y_key: AV, and dq from (dlogits, k).  The
//           compact rows come into LDS as whole runs; a lane gathers the four
//           weights of its query by slot, zero outside the window.
//   ws_inv  z_key = mult sum a[q, slot(q, key)] x_q over the queries whose
//           windows hold the key: dk and dv.  The weights are gathered from
//           memory one chunk ahead; every one is read by exactly one key.
// A backward call's two passes share one launch, the key-side one first (its
// chains are the longer ones).
//
// What bounds it: at these sizes the chain of the few waves a SIMD has (load,
// LDS, product) rather than the matrix cores: by counters, over float32
// [4, 56, 56, 2, 32] K = 7 with position bias, one to three waves per SIMD that wait
// for memory or LDS 42 to 58% of their time and for an issue slot 14 to 32%, matrix
// cores 7 to 13% busy; 12 to 24 MB of traffic per launch, 1.0 to 1.4 times its own
// tensors, take 3 to 5 us at a copy's rate.  Against the vector-ALU kernels,
// which read every neighbour row per query and divide per candidate in the
// inverse pass: float32 [4, 56, 56, 2, 32] K = 7 with position bias, logits
// 32.1 -> 13.5 us, AV 27.9 -> 10.4, QK backward 137 -> 21.6 (with the bias
// gradient), AV backward 117 -> 14.7; split ops on [4, 80, 80, 8,
// 32] K = 5: 75 -> 33, 56 -> 32, 188 -> 52, 196 -> 51.
//
// As in na_wave.hip a result with a NaN is computed again key by key, so a
// value that is not finite reaches only the rows whose windows hold it.
#include "na_wave.h"

namespace na {
namespace {

struct WsLay {
  int32_t KK, KP;          // slots per compact row, LDS stride of a row (odd)
  int32_t st[3], rs[3];    // slot and bias-cell strides per axis
  int32_t cells;           // bias cells per head
  int32_t q_rt, q_rh;      // rows per position and per head, query-side rows
  int32_t k_rt, k_rh;      // the same of the key-side rows
  int32_t prefill;         // a slot may lie outside the window (causal axes)
  int32_t lw;              // LDS floats per wave
};

// Rows in the wave's LDS: X rows [16][RS], compact rows [16][KP], then per
// chunk row: packed coordinates, linear slot | cell << 16, gather base.
template <int D>
constexpr int ws_x() {
  return 16 * wv_rs<D>();
}

// What a lane knows of its query: row, window (packed and as slot and cell
// constants), and the tile's key box.
template <int R>
struct WsQuery {
  WvBox<R, false> box;
  WvWin<R> win;
  bool valid = true;
  int row = 0;         // query-side row inside the sample
  int slot0 = 0, cell0 = 0;
  uint32_t pb = 0;     // bias row of slot 0 per axis (axis 1 << 16 | axis 2)
  int64_t krow = 0;    // key-side row of box point 0 (head 0)
  template <int D>
  __device__ __forceinline__ void init(const WvProb &P, const WsLay &S, const WvTile &t, int n) {
#pragma unroll
    for (int a = 3 - R; a < 3; ++a) {
      const WvAx &x = P.ax[a];
      box.lo[a] = wv_start(x, t.i0[a], t.Lr[a]);
      box.E[a] = wv_end(x, t.i0[a] + t.nv[a] - 1, t.Lr[a]) - box.lo[a];
      box.SK[a] = (uint32_t)(x.d * x.tok) * (uint32_t)(S.k_rt * D * 4);
      krow += (int64_t)(t.r[a] + x.d * box.lo[a]) * x.tok * S.k_rt;
      const int i = wv_row(P.gq, t, a, n, valid);
      row += (t.r[a] + x.d * i) * x.tok * S.q_rt;
      // a causal window's slot 0 may lie before the sample: raw start
      const int raw = x.causal ? i - x.K + 1 : wv_start(x, i, t.Lr[a]);
      win.axis(a, wv_start(x, i, t.Lr[a]) - box.lo[a], wv_end(x, i, t.Lr[a]) - 1 - box.lo[a]);
      slot0 += (box.lo[a] - raw) * S.st[a];
      cell0 += (box.lo[a] - i + x.K - 1) * S.rs[a];
      if (a > 0) pb |= (uint32_t)((raw - i + x.K - 1) & 0xffff) << (a == 1 ? 16 : 0);
    }
    row += t.h * S.q_rh;
    box.finish();
    win.finish();
  }
};

// A box point's slot and cell parts in one word.
__device__ __forceinline__ uint32_t ws_lin(const WsLay &S, const int (&e)[3]) {
  const uint32_t s = e[0] * S.st[0] + e[1] * S.st[1] + e[2] * S.st[2];
  const uint32_t c = e[0] * S.rs[0] + e[1] * S.rs[1] + e[2] * S.rs[2];
  return s | (c << 16);
}

// Copy the tile's 16 compact rows between memory and LDS, one row at a time
// (a row is one contiguous run; its place is the lane's of that row).
template <bool LOAD>
__device__ __forceinline__ void ws_rows(const WsLay &S, float *sm, float *g, const float *gl, int row,
                                        bool valid, int lane) {
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const uint32_t r = (uint32_t)__builtin_amdgcn_readlane(row, i);
    if (!LOAD && __builtin_amdgcn_readlane((int)valid, i) == 0) continue;
    for (int c = lane; c < S.KK; c += 64) {
      if constexpr (LOAD)
        sm[i * S.KP + c] = gl[(uint64_t)r * S.KK + c];
      else
        g[(uint64_t)r * S.KK + c] = sm[i * S.KP + c];
    }
  }
}

template <int D, int R>
__device__ __forceinline__ void ws_qk(const WvProb &P, const WsLay &S, uint32_t tile, float *sm, int lane,
                                      const float *x, const float *y, const float *bias, float *out,
                                      float pre, float mult, float fill) {
  typedef Wv<float>::frag frag;
  constexpr int NF = D / 16;
  const int n = lane & 15, gq = lane >> 4;
  WvTile t;
  if (!wv_decode<R>(P, P.gq, P.fH, tile, false, t)) return;
  const int hk = (int)fdiv((uint32_t)t.h, P.fRep);
  WsQuery<R> Q;
  Q.template init<D>(P, S, t, n);
  const char *yb = reinterpret_cast<const char *>(y) +
                   (t.b * P.Ltot * P.Hkv + Q.krow + (int64_t)hk * S.k_rh) * (D * 4);
  const float *xb = x + t.b * P.Ltot * P.H * D;
  frag qf[NF], kf[NF];
  ld_row<float>(reinterpret_cast<const char *>(xb), (uint32_t)Q.row * (D * 4u) + 16u * gq, qf);
  uint32_t cd, lin;
  auto load = [&](int c) {
    int e[3];
    cd = Q.box.coords(16 * c + n, e);
    lin = ws_lin(S, e);
    ld_row<float>(yb, Q.box.offset(e, Q.box.SK) + 16u * gq, kf);
  };
  load(0);
  float *cr = sm + ws_x<D>();
  uint32_t *crow = reinterpret_cast<uint32_t *>(cr + 16 * S.KP), *lrow = crow + 16;
  if (S.prefill)
    for (int c = lane; c < 16 * S.KP; c += 64) cr[c] = fill;
#pragma unroll
  for (int i = 0; i < NF; ++i) qf[i] *= pre;
  const float *bh = bias != nullptr ? bias + t.h * S.cells : nullptr;
  const int nch = (Q.box.npts + 15) >> 4;
  for (int c = 0; c < nch; ++c) {
    const f32x4 s = wv_scores<float>(kf, qf);
    if (gq == 0) {
      crow[n] = cd;
      lrow[n] = lin;
    }
    load(c + 1);
    wv_lds_sync();
    const uint4 cc = *reinterpret_cast<const uint4 *>(crow + 4 * gq);
    const uint4 ll = *reinterpret_cast<const uint4 *>(lrow + 4 * gq);
    const uint32_t c4[4] = {cc.x, cc.y, cc.z, cc.w}, l4[4] = {ll.x, ll.y, ll.z, ll.w};
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const bool ok = Q.win.holds(c4[r]);
      const int slot = ok ? (int)(l4[r] & 0xffffu) + Q.slot0 : S.KK;  // KK: a spare column
      float v = s[r] * mult;
      if (bh != nullptr) v += bh[ok ? (int)(l4[r] >> 16) + Q.cell0 : 0];
      cr[n * S.KP + slot] = v;
    }
  }
  wv_lds_sync();
  ws_rows<false>(S, cr, out + t.b * P.Ltot * P.H * S.KK, nullptr, Q.row, Q.valid, lane);
}

// The tile's part of the bias gradient (rank 2), in float64: for each cell of
// the table the sum over the tile's queries of the compact value whose slot has
// that cell, to bpart[(head, cell)][tile of the head].  Where no window of the
// tile is clamped slot 0's cell is K/2 on both axes: the K0 K1 cells from there
// hold one sum each, the others are zero.  A tile past the end of a short phase
// has no query and writes zeros (`any` false): every partial is written.
// The rows are in LDS for dq already; read again by a pass of its own they
// made QK backward 31.7 us at [4, 56, 56, 2, 32] K = 7 (21.6 so), 137 at
// [6, 80, 80, 8, 32] K = 5 (89), 115 at [2, 56, 56, 4, 32] K = 13 (53).  At
// rank 1 a table has too few cells for 64 lanes (82.0 -> 83.4 at [6, 6000, 12,
// 32] K = 7 d = 2): it keeps the pass.
__device__ __forceinline__ void ws_bias(const WvProb &P, const WsLay &S, const WvTile &t, uint32_t tile,
                                        const WsQuery<2> &Q, const float *cr, int lane, bool any,
                                        double *bpart) {
  const WvAx &x1 = P.ax[1], &x2 = P.ax[2];
  const int grid = (int)P.gq.fGrid.d, per_head = P.B * grid;
  const int sp = (int)tile - (t.b * P.H + t.h) * grid;
  double *dst = bpart + (int64_t)t.h * S.cells * per_head + t.b * grid + sp;
  if (!any) {
    for (int c = lane; c < S.cells; c += 64) dst[(int64_t)c * per_head] = 0.0;
    return;
  }
  const uint32_t mid = (uint32_t)x1.nh << 16 | (uint32_t)x2.nh;
  const uint32_t live = (uint32_t)__builtin_amdgcn_ballot_w64(Q.valid) & 0xffffu;
  const bool inner = __builtin_amdgcn_ballot_w64(Q.pb != mid) == 0;
  const int R2 = 2 * x2.K - 1;
  const float rr = __builtin_amdgcn_rcpf((float)R2);
  for (int c = lane; c < S.cells; c += 64) {
    const int c1 = (int)(((float)c + 0.5f) * rr), c2 = c - c1 * R2;
    double s = 0.0;
    if (inner) {
      const int k1 = c1 - x1.nh, k2 = c2 - x2.nh;
      const bool ok = (unsigned)k1 < (unsigned)x1.K && (unsigned)k2 < (unsigned)x2.K;
      const float *p = cr + (ok ? k1 * x2.K + k2 : 0);
#pragma unroll
      for (int i = 0; i < 16; ++i)
        if (live >> i & 1u) s += (double)p[i * S.KP];
      s = ok ? s : 0.0;
    } else {
#pragma unroll 4
      for (int i = 0; i < 16; ++i) {
        const uint32_t pb = (uint32_t)__builtin_amdgcn_readlane((int)Q.pb, i);
        const int k1 = c1 - (int)(pb >> 16), k2 = c2 - (int)(pb & 0xffffu);
        const bool ok = (live >> i & 1u) && (unsigned)k1 < (unsigned)x1.K &&
                        (unsigned)k2 < (unsigned)x2.K;
        const float v = cr[i * S.KP + (ok ? k1 * x2.K + k2 : 0)];
        s += ok ? (double)v : 0.0;
      }
    }
    dst[(int64_t)c * per_head] = s;
  }
}

template <int D, int R>
__device__ __forceinline__ void ws_av(const WvProb &P, const WsLay &S, uint32_t tile, float *sm, int lane,
                                      const float *a, const float *y, float *out, float mult,
                                      double *bpart) {
  typedef Wv<float>::frag frag;
  constexpr int NF = D / 16, NDB = D / 16, RS = wv_rs<D>();
  const int n = lane & 15, gq = lane >> 4;
  WvTile t;
  WsQuery<R> Q;
  if (!wv_decode<R>(P, P.gq, P.fH, tile, false, t)) {
    if constexpr (R == 2)
      if (bpart != nullptr && t.b < P.B) ws_bias(P, S, t, tile, Q, sm, lane, false, bpart);
    return;
  }
  const int hk = (int)fdiv((uint32_t)t.h, P.fRep);
  Q.template init<D>(P, S, t, n);
  const char *yb = reinterpret_cast<const char *>(y) +
                   (t.b * P.Ltot * P.Hkv + Q.krow + (int64_t)hk * S.k_rh) * (D * 4);
  frag kf[NF];
  uint32_t cd, lin;
  auto load = [&](int c) {
    int e[3];
    cd = Q.box.coords(16 * c + n, e);
    lin = ws_lin(S, e);
    ld_row<float>(yb, Q.box.offset(e, Q.box.SK) + 16u * gq, kf);
  };
  load(0);
  float *cr = sm + ws_x<D>();
  uint32_t *crow = reinterpret_cast<uint32_t *>(cr + 16 * S.KP), *lrow = crow + 16;
  ws_rows<true>(S, cr, nullptr, a + t.b * P.Ltot * P.H * S.KK, Q.row, true, lane);
  const float *xt = sm + 4 * gq * RS + n;
  f32x4 acc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) acc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int nch = (Q.box.npts + 15) >> 4;
  for (int c = 0; c < nch; ++c) {
    wv_lds<float>(sm + n * RS, gq, kf);
    if (gq == 0) {
      crow[n] = cd;
      lrow[n] = lin;
    }
    load(c + 1);
    wv_lds_sync();
    const uint4 cc = *reinterpret_cast<const uint4 *>(crow + 4 * gq);
    const uint4 ll = *reinterpret_cast<const uint4 *>(lrow + 4 * gq);
    const uint32_t c4[4] = {cc.x, cc.y, cc.z, cc.w}, l4[4] = {ll.x, ll.y, ll.z, ll.w};
    float w[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const bool ok = Q.win.holds(c4[r]);
      const float v = cr[n * S.KP + (ok ? (int)(l4[r] & 0xffffu) + Q.slot0 : 0)];
      w[r] = ok ? v : 0.f;
    }
    wv_acc<NDB, RS>(xt, w, acc);
  }
  if (wv_nan(acc, 0.f)) {  // again, key by key
#pragma unroll
    for (int db = 0; db < NDB; ++db) acc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int p = 0; p < Q.box.npts; ++p) {
      int e[3];
      cd = Q.box.coords(p, e);
      if (!Q.win.holds(cd)) continue;
      const float w = cr[n * S.KP + (int)(ws_lin(S, e) & 0xffffu) + Q.slot0];
      const char *yr = yb + Q.box.offset(e, Q.box.SK) + 16 * gq;
#pragma unroll
      for (int db = 0; db < NDB; ++db) acc[db] += w * ld4<float>(yr + 64 * db);
    }
  }
  if constexpr (R == 2)
    if (bpart != nullptr) ws_bias(P, S, t, tile, Q, cr, lane, true, bpart);
  if (!Q.valid) return;
  char *ob = reinterpret_cast<char *>(out + t.b * P.Ltot * P.H * D) + (uint64_t)(uint32_t)Q.row * (D * 4);
#pragma unroll
  for (int db = 0; db < NDB; ++db) st4<float>(ob + (16 * db + 4 * gq) * 4, acc[db] * mult);
}

template <int D, int R>
__device__ __forceinline__ void ws_inv(const WvProb &P, const WsLay &S, uint32_t tile, float *sm, int lane,
                                       const float *a, const float *x, float *z, float mult) {
  typedef Wv<float>::frag frag;
  constexpr int NF = D / 16, NDB = D / 16, RS = wv_rs<D>();
  const int n = lane & 15, gq = lane >> 4;
  WvTile t;
  if (!wv_decode<R>(P, P.gk, P.fHkv, tile, true, t)) return;
  WvBox<R, false> box;  // the queries whose windows hold the tile's keys
  WvWin<R> win;
  bool kv = true;
  int krow = 0, jl = 0;  // key row inside the sample; its linear slot part
  int64_t qrow = 0;      // query-side row of box point 0
  int brow[3];           // rows per box step
#pragma unroll
  for (int a_ = 3 - R; a_ < 3; ++a_) {
    const WvAx &ax = P.ax[a_];
    box.lo[a_] = wv_istart(ax, t.i0[a_]);
    box.E[a_] = wv_iend(ax, t.i0[a_] + t.nv[a_] - 1, t.Lr[a_], t.Qr[a_]) - box.lo[a_];
    brow[a_] = ax.d * ax.tok * S.q_rt;
    box.SK[a_] = (uint32_t)brow[a_];
    qrow += (int64_t)(t.r[a_] + ax.d * box.lo[a_]) * ax.tok * S.q_rt;
    const int j = wv_row(P.gk, t, a_, n, kv);
    krow += (t.r[a_] + ax.d * j) * ax.tok * S.k_rt;
    jl += j * S.st[a_];
    win.axis(a_, wv_istart(ax, j) - box.lo[a_],
             wv_iend(ax, j, t.Lr[a_], t.Qr[a_]) - 1 - box.lo[a_]);
  }
  krow += t.h * S.k_rh;
  box.finish();
  win.finish();
  uint32_t *crow = reinterpret_cast<uint32_t *>(sm + ws_x<D>());
  const float *xt = sm + 4 * gq * RS + n;
  f32x4 acc[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) acc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int nch = (box.npts + 15) >> 4;
  // a box point's compact row minus its window's start, in floats: the weight
  // of the key with linear part jl is at that plus jl
  auto gather0 = [&](const int (&e)[3], uint32_t row) {
    int s0 = 0;
#pragma unroll
    for (int a_ = 3 - R; a_ < 3; ++a_) {
      const WvAx &ax = P.ax[a_];
      const int i = box.lo[a_] + e[a_];
      s0 += (ax.causal ? i - ax.K + 1 : wv_start(ax, i, t.Lr[a_])) * S.st[a_];
    }
    return (int)(row * (uint32_t)S.KK) - s0;
  };
  for (int hr = 0; hr < P.rep && nch > 0; ++hr) {
    const int64_t base = t.b * P.Ltot * P.H + qrow + (int64_t)(t.h * P.rep + hr) * S.q_rh;
    const char *xb = reinterpret_cast<const char *>(x + base * D);
    const float *ab = a + base * S.KK;
    frag xf[NF];
    float wn[4];
    // chunk c: its rows on their way to registers, and its weights
    auto load = [&](int c) {
      int e[3];
      const uint32_t cd = box.coords(16 * c + n, e);
      const uint32_t row = box.offset(e, box.SK);
      ld_row<float>(xb, row * (D * 4u) + 16u * gq, xf);
      uint32_t *cb = crow + 32 * (c & 1);
      if (gq == 0) {
        cb[n] = cd;
        cb[16 + n] = (uint32_t)gather0(e, row);
      }
      wv_lds_sync();
      const uint4 cc = *reinterpret_cast<const uint4 *>(cb + 4 * gq);
      const uint4 gg = *reinterpret_cast<const uint4 *>(cb + 16 + 4 * gq);
      const uint32_t c4[4] = {cc.x, cc.y, cc.z, cc.w}, g4[4] = {gg.x, gg.y, gg.z, gg.w};
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool ok = win.holds(c4[r]);
        const float v = ab[ok ? (int)g4[r] + jl : 0];
        wn[r] = ok ? v : 0.f;
      }
    };
    load(0);
    for (int c = 0; c < nch; ++c) {
      wv_lds<float>(sm + n * RS, gq, xf);
      const float w[4] = {wn[0], wn[1], wn[2], wn[3]};
      load(c + 1);
      wv_acc<NDB, RS>(xt, w, acc);
    }
  }
  if (wv_nan(acc, 0.f)) {  // again, query by query
#pragma unroll
    for (int db = 0; db < NDB; ++db) acc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int hr = 0; hr < P.rep; ++hr) {
      const int64_t base = t.b * P.Ltot * P.H + qrow + (int64_t)(t.h * P.rep + hr) * S.q_rh;
      for (int p = 0; p < box.npts; ++p) {
        int e[3];
        if (!win.holds(box.coords(p, e))) continue;
        const uint32_t row = box.offset(e, box.SK);
        const float w = a[base * S.KK + gather0(e, row) + jl];
        const char *xr = reinterpret_cast<const char *>(x + base * D) + (uint64_t)row * (D * 4) + 16 * gq;
#pragma unroll
        for (int db = 0; db < NDB; ++db) acc[db] += w * ld4<float>(xr + 64 * db);
      }
    }
  }
  if (!kv) return;
  char *zb = reinterpret_cast<char *>(z + t.b * P.Ltot * P.Hkv * D) + (uint64_t)(uint32_t)krow * (D * 4);
#pragma unroll
  for (int db = 0; db < NDB; ++db) st4<float>(zb + (16 * db + 4 * gq) * 4, acc[db] * mult);
}

// One kernel, its passes by block range: [0, n_inv) the key-side pass (when
// there is one), the rest the query-side one (QK: ws_qk, else ws_av).
template <int D, int R, bool QK>
__global__ void __launch_bounds__(256)
    k_wsplit(WvProb P, WsLay S, int n_inv, const float *__restrict__ x, const float *__restrict__ y,
             const float *__restrict__ bias, const float *__restrict__ a, float *__restrict__ out,
             float pre, float mult, float fill, const float *__restrict__ ia,
             const float *__restrict__ ix, float *__restrict__ iz, float imult,
             double *__restrict__ bpart) {
  extern __shared__ __align__(16) float ws_smem[];
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int nw = blockDim.x >> 6;
  float *sm = ws_smem + w * S.lw;
  if ((int)blockIdx.x < n_inv) {
    ws_inv<D, R>(P, S, (uint32_t)(wv_wg(blockIdx.x, P.gk.n_wg) * nw + w), sm, lane, ia, ix, iz, imult);
    return;
  }
  const uint32_t tile = (uint32_t)(wv_wg((int)blockIdx.x - n_inv, P.gq.n_wg) * nw + w);
  if constexpr (QK)
    ws_qk<D, R>(P, S, tile, sm, lane, x, y, bias, out, pre, mult, fill);
  else
    ws_av<D, R>(P, S, tile, sm, lane, a, y, out, mult, bpart);
}

// ---------------------------------------------------------------------------
// Host side.

constexpr int kMaxSlots = 512;

bool ws_ok(const Prob &P) {
  if (P.dense || P.sample_extent != nullptr || P.n_extra > 0) return false;
  if (P.D != 16 && P.D != 32 && P.D != 64 && P.D != 128) return false;
  int64_t kk = 1, cells = 1;
  for (int a = 0; a < 3; ++a) {
    if (P.ax[a].s != 1) return false;
    kk *= P.ax[a].K;
    cells *= 2 * P.ax[a].K - 1;
  }
  // slot and cell parts share a word, with room for a box's extent past the
  // window (its 15 points or so more per axis)
  int64_t sl = 0, ce = 0;
  {
    int64_t st = 1, rs = 1;
    for (int a = 2; a >= 0; --a) {
      const Axis &x = P.ax[a];
      const int64_t e = std::min<int64_t>(phase_max(x), x.K + 16);
      sl += e * st;
      ce += e * rs;
      st *= x.K;
      rs *= 2 * x.K - 1;
    }
  }
  if (kk > kMaxSlots || sl >= 65536 || ce >= 65536) return false;
  const int64_t tokens = (int64_t)P.ax[0].L * P.ax[1].L * P.ax[2].L;
  if (tokens * P.H * kk >= ((int64_t)1 << 29)) return false;  // 32-bit float offsets
  return wv_geometry_ok(P, 4);
}

struct WsPass {  // the query-side pass
  bool qk;
  const float *x, *y, *bias, *a;
  float *out, pre, mult, fill;
};
struct WsInv {   // the key-side pass (z null: none)
  const float *a, *x;
  float *z, mult;
};

void ws_launch(const Prob &P, bool heads_first, const WsPass &p, const WsInv &v, hipStream_t st,
               double *bpart = nullptr) {
  if (P.B == 0) return;
  WsLay S{};
  S.KK = P.kprod;
  S.KP = (P.kprod + 1) | 1;
  int32_t ss = 1, rs = 1;
  for (int a = 2; a >= 0; --a) {
    S.st[a] = ss;
    S.rs[a] = rs;
    ss *= P.ax[a].K;
    rs *= 2 * P.ax[a].K - 1;
    S.prefill |= P.ax[a].causal;
  }
  S.cells = rs;
  const int tokens = P.ax[0].L * P.ax[1].L * P.ax[2].L;
  S.q_rt = heads_first ? 1 : P.H;
  S.q_rh = heads_first ? tokens : 1;
  S.k_rt = heads_first ? 1 : P.Hkv;
  S.k_rh = heads_first ? tokens : 1;
  S.lw = 16 * (P.D + 4) + ((16 * S.KP + 3) & ~3) + 64;
  // four independent waves per workgroup within 64 KB of LDS, else two or one
  const int nw = S.lw * 16 <= 65536 ? 4 : S.lw * 8 <= 65536 ? 2 : 1;
  const WvProb W = make_wvprob(P, v.z != nullptr, nw);
  const int n_inv = v.z != nullptr ? W.gk.n_wg : 0;
  const dim3 grid(n_inv + (p.out != nullptr ? W.gq.n_wg : 0)), block(64 * nw);
  if (grid.x == 0) return;
#define WS_L(DD, RR, QQ)                                                                        \
  hipLaunchKernelGGL((k_wsplit<DD, RR, QQ>), grid, block, (size_t)S.lw * 4 * nw, st, W, S, n_inv, \
                     p.x, p.y, p.bias, p.a, p.out, p.pre, p.mult, p.fill, v.a, v.x, v.z, v.mult, bpart)
#define WS_Q(DD, RR)                                     \
  do {                                                   \
    if (p.qk) WS_L(DD, RR, true); else WS_L(DD, RR, false); \
  } while (0)
#define WS_R(DD)                       \
  do {                                 \
    if (P.rank == 1) WS_Q(DD, 1);      \
    else if (P.rank == 2) WS_Q(DD, 2); \
    else WS_Q(DD, 3);                  \
  } while (0)
  if (P.D == 16) WS_R(16);
  else if (P.D == 32) WS_R(32);
  else if (P.D == 64) WS_R(64);
  else WS_R(128);
#undef WS_R
#undef WS_Q
#undef WS_L
}

Prob rpb_prob(const RpbProb &A) {
  Prob P{};
  P.B = A.B;
  P.H = P.Hkv = A.H;
  P.rep = 1;
  P.D = A.D;
  P.rank = A.rank;
  P.kprod = A.KK;
  const int32_t L[2] = {A.L0, A.L1}, K[2] = {A.K0, A.K1}, d[2] = {A.d0, A.d1};
  for (int a = 0; a < 3; ++a) {
    const int i = a - (3 - A.rank);
    P.ax[a] = i < 0 ? Axis{1, 1, 1, 1, 0, 1} : Axis{L[i], K[i], d[i], 1, 0, L[i]};
  }
  return P;
}

}  // namespace

// Where a window has few slots, a tile's 16-point chunks are mostly points of
// no window and the vector ALU's one pass over the window is shorter; and a
// small launch is one chain of chunks (load, LDS, product), the longer the wider
// the head.  Times here over there, float32, by slots, head_dim and rows (queries
// times heads):
//   QK   3 slots, D 128: 1.34 to 1.50 up to 4.4e3 rows, 0.7 to 0.8 from 3e4; 5 slots,
//        D 64 / 128: 1.07 to 1.25, 0.5 to 0.8; 7 and 9 slots: D 32 0.81 to 1.01, D 64
//        0.42 to 0.97, D 128 up to 1.08 below 1e3 rows, 0.35 to 0.98 above; D 16 up to
//        9 slots 1.2; from 13 slots on 0.12 to 0.91
//   AV   13 to 27 slots, D 64 / 128: 1.04 to 1.54 up to 5e3 rows, 0.25 to 0.79 from
//        1.6e4; 31 to 49 slots, D 128: 0.95 to 1.07, 0.2 to 0.5; 25 slots, D 16 / 32: 0.58
//        to 1.02; otherwise 0.15 to 0.99.  9 slots lose (D 32 / 64: 26.2 -> 29.1 us, 4.6
//        -> 7.5 on a small one)
// A backward call's two passes gain from 3 slots on at every size (0.1 to 0.7).
constexpr int64_t kFilled = 1 << 14;  // rows that fill the chip: four waves per CU

bool wsplit_eligible(const Prob &P, int dtype, WsplitPass pass) {
  const int kk = P.kprod;
  const int64_t rows = (int64_t)P.B * P.H * P.ax[0].L * P.ax[1].L * P.ax[2].L;
  bool gains = kk >= 3;
  if (pass == kWsQk)
    gains = kk >= 13 || (kk >= 7 ? P.D >= 32 && (P.D < 128 || rows >= kFilled / 4)
                                 : kk * P.D >= 224 && rows >= kFilled);
  if (pass == kWsAv)
    gains = P.D < 64 ? kk >= 25 : kk >= (rows >= kFilled ? 13 : P.D == 64 ? 31 : 49);
  return dtype == NA_F32 && gains && ws_ok(P);
}

void wsplit_qk(const Prob &P, const void *q, const void *k, void *logits, hipStream_t st) {
  ws_launch(P, false,
            {true, (const float *)q, (const float *)k, nullptr, nullptr, (float *)logits, 1.f, P.scale,
             -INFINITY},
            {}, st);
}

void wsplit_av(const Prob &P, const void *attn, const void *v, void *out, hipStream_t st) {
  ws_launch(P, false, {false, nullptr, (const float *)v, nullptr, (const float *)attn, (float *)out, 1.f,
                       1.f, 0.f},
            {}, st);
}

void wsplit_qk_bwd(const Prob &P, const void *q, const void *k, const void *dl, void *dq, void *dk,
                   hipStream_t st) {
  ws_launch(P, false,
            {false, nullptr, (const float *)k, nullptr, (const float *)dl, (float *)dq, 1.f, P.scale, 0.f},
            {(const float *)dl, (const float *)q, (float *)dk, P.scale}, st);
}

void wsplit_av_bwd(const Prob &P, const void *attn, const void *v, const void *dout, void *dattn,
                   void *dv, hipStream_t st) {
  ws_launch(P, false,
            {true, (const float *)dout, (const float *)v, nullptr, nullptr, (float *)dattn, 1.f, 1.f, 0.f},
            {(const float *)attn, (const float *)dout, (float *)dv, 1.f}, st);
}

// Rank 1 up to head_dim 16 has kernels of its own (na_rpb.hip) that stage
// whole blocks of rows.  Times here over there (the generic kernels), by slots,
// head_dim and rows:
//   logits, dattn alone   rank 1: 3 and 5 slots, D 64 / 128 0.95 to 1.5; 7 slots 0.65 to
//        1.4; 9 slots, D 32 / 128 0.57 to 1.0, D 64 0.6 to 1.11; rank 2, 9 slots, D 32
//        0.80 to 0.86, but 1.08 at 4e4 rows, D 64 / 128 0.79 to 0.98
//   AV, dq alone          7 slots 0.7 to 1.54; 9 slots 0.89 to 1.26 up to 5e4 rows (D 16
//        1.18 at 3e5), 0.57 to 0.81 from 2.4e5 with D 32 and more
// and from 13 slots on 0.08 to 0.92 for every pass, but at rank 1 with up to four
// heads, whose rows lie closer together for the generic kernels, 1.04 to 1.4 at 9 to
// 25 slots from 3e4 rows on (AV of head_dim 128 at any), 0.3 to 0.6 at 31.  A
// backward call's two passes together gain from 7 slots on at every size (0.1 to
// 0.84).
bool wsplit_rpb_eligible(const RpbProb &A, WsplitPass pass) {
  const int64_t rows = (int64_t)A.n_rows;
  bool gains = A.KK >= 7;
  if (pass == kWsQk)
    gains = A.KK >= 13 || (A.KK >= 9 && (A.rank == 1 ? A.D != 64
                                                     : A.D >= 64 || (A.D == 32 && (rows < kFilled ||
                                                                                   rows >= 8 * kFilled))));
  if (pass == kWsAv) gains = A.KK >= 13 || (A.KK >= 9 && A.D >= 32 && rows >= 8 * kFilled);
  if (pass != kWsBwd && A.rank == 1 && A.H <= 4) gains = A.KK >= 31;
  return gains && (A.rank == 2 || A.D > 16) && A.n_rows > 0 && ws_ok(rpb_prob(A));
}

void wsplit_rpb_dot(const RpbProb &A, const float *x, const float *y, const float *rpb, float *out,
                    int scale_x, float fill, hipStream_t st) {
  ws_launch(rpb_prob(A), A.heads_first != 0,
            {true, x, y, rpb, nullptr, out, scale_x ? A.scale : 1.f, 1.f, fill}, {}, st);
}

void wsplit_rpb_gather(const RpbProb &A, const float *w, const float *y, float *out, float post,
                       hipStream_t st) {
  ws_launch(rpb_prob(A), A.heads_first != 0, {false, nullptr, y, nullptr, w, out, 1.f, post, 0.f}, {}, st);
}

void wsplit_rpb_inverse(const RpbProb &A, const float *w, const float *x, float *out, float post,
                        hipStream_t st) {
  ws_launch(rpb_prob(A), A.heads_first != 0, {}, {w, x, out, post}, st);
}

// One partial per tile of a head, for each cell of the bias table (rank 2).
int32_t wsplit_rpb_bias_tiles(const RpbProb &A) {
  if (A.rank != 2 || !wsplit_rpb_eligible(A, kWsBwd)) return 0;
  const WvGrid G = wv_grid(rpb_prob(A), false, 4);
  return (int32_t)(A.B * (int64_t)G.fGrid.d);
}

void wsplit_rpb_qk_bwd(const RpbProb &A, const float *dl, const float *q, const float *key, float *dq,
                       float *dk, double *bias_part, hipStream_t st) {
  const float post = A.has_scale ? A.scale : 1.f;
  ws_launch(rpb_prob(A), A.heads_first != 0, {false, nullptr, key, nullptr, dl, dq, 1.f, post, 0.f},
            {dl, q, dk, post}, st, bias_part);
}

void wsplit_rpb_av_bwd(const RpbProb &A, const float *attn, const float *v, const float *dout,
                       float *dattn, float *dv, hipStream_t st) {
  ws_launch(rpb_prob(A), A.heads_first != 0, {true, dout, v, nullptr, nullptr, dattn, 1.f, 1.f, 0.f},
            {attn, dout, dv, 1.f}, st);
}

}  // namespace na
