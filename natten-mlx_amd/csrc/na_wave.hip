// na_wave.hip — fused neighborhood attention on matrix cores in 32-bit
// arithmetic: float32 tensors, and bf16 / fp16 tensors with strided queries.
//
// Problem class (wave_eligible): float32 with head_dim 16/32/64/128, or
// bf16/fp16 with head_dim 32/64/128 where some axis is strided; on every axis
// stride 1 or dilation 1, and a causal axis or an odd K with d*K <= L; no
// per-sample extents, additional tokens or dense mode.  Everything else of
// those types stays with the vector-ALU kernels (na_valu.hip), whose results
// these match to rounding: probabilities, score gradients and sums stay
// float32 for every storage type.
//
// One wave owns 16 queries of one dilation phase (a T0 x T1 x T2 box) and
// needs no other wave: no barrier, 16 rows of its own in LDS.  The keys its
// queries' windows cover form a box [lo, lo + E) per axis; its points are
// numbered row-major and taken 16 at a time, so a chunk is always full
// (K = 7, tile 4 x 4: 100 points = 7 chunks; one chunk per box row would be
// 10).  Lane l = 16 gq + n loads row n of the chunk (16 bytes of every 64):
// the A operand of S^T = K Q^T as it lies in memory.  V goes through the
// wave's LDS rows, as float32, to be read transposed for O^T += V^T P^T on
// v_mfma_f32_16x16x4_f32: the lane's scores of step r are that step's B
// operand as they come out of the score MFMA.  The rows' box coordinates,
// packed into one word with a guard bit per axis, go through LDS too; one
// subtraction each way tests a key against all axes of a query's window.
// The next chunk's loads are issued once its operands are free, so they fly
// during the softmax and the second product.
//
// What bounds it: the f32 matrix cores run 64 FLOP per cycle and SIMD (157
// TFLOP/s on the chip), and a 16-query tile multiplies the whole box, about
// twice its windows' keys; then the chain load -> scores -> softmax -> product
// of the few waves a small problem has.  By counters, float32 [2, 61, 45, 8, 32]
// K = 7: the forward (2944 waves) reads its inputs once (17.0 MB), its waves wait
// for memory or LDS 56% of their time and for an issue slot 26%, matrix cores 23%
// busy; the backward's (5888) 29% and 58%, matrix cores 33% busy.  So the forward
// is its loads' latency, the backward its dependent products and their issue.
// Against the vector-ALU kernels, which
// read every key row once per query from L2: float32 [2, 61, 45, 8, 32] K = 7
// forward 52 -> 17 us, backward 279 -> 41 us; bf16 [4, 57, 75, 4, 64] K = 7
// stride 2 forward 40 -> 18 us, backward 188 -> 34 us; float32 [4, 128, 128,
// 8, 64] K = 3, the least work per key, 249 -> 137 and 985 -> 425 us.
//
// A value that is not finite must reach only the queries whose windows hold
// it, but 0 * inf in a product over the box is NaN.  So a wave whose result
// holds a NaN computes its rows again key by key (the `again` blocks).
#include "na_wave.h"

namespace na {
namespace {

template <typename T, int D, int R>
__global__ void __launch_bounds__(64 * wv_waves<D>())
    k_wvfwd(WvProb P, const T *__restrict__ q, const T *__restrict__ k, const T *__restrict__ v,
            T *__restrict__ out, float *__restrict__ lse) {
  typedef typename Wv<T>::frag frag;
  constexpr int ES = sizeof(T), NF = D * ES / 64, NDB = D / 16, RS = wv_rs<D>(), NW = wv_waves<D>();
  __shared__ __align__(16) float smem[NW * (16 * RS + 16)];

  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, n = lane & 15, gq = lane >> 4;
  const uint32_t tile = (uint32_t)(wv_wg(blockIdx.x, P.gq.n_wg) * NW + w);
  WvTile t;
  if (!wv_decode<R>(P, P.gq, P.fH, tile, false, t)) return;
  const int hk = (int)fdiv((uint32_t)t.h, P.fRep);

  // the tile's key box, the lane's query and its window
  WvBox<R, false> box;
  WvWin<R> win;
  bool qv = true;
  int64_t ktok = 0;
  int qtok = 0, otok = 0;
#pragma unroll
  for (int a = 3 - R; a < 3; ++a) {
    const WvAx &x = P.ax[a];
    box.lo[a] = wv_start(x, t.i0[a] * x.s, t.Lr[a]);
    box.E[a] = wv_end(x, (t.i0[a] + t.nv[a] - 1) * x.s, t.Lr[a]) - box.lo[a];
    box.SK[a] = (uint32_t)(x.d * x.tok) * (uint32_t)(P.Hkv * D * ES);
    ktok += (int64_t)(t.r[a] + x.d * box.lo[a]) * x.tok;
    const int i = wv_row(P.gq, t, a, n, qv);
    qtok += (t.r[a] + x.d * x.s * i) * x.tok;
    otok += (t.r[a] + x.d * i) * x.otok;
    win.axis(a, wv_start(x, i * x.s, t.Lr[a]) - box.lo[a],
             wv_end(x, i * x.s, t.Lr[a]) - 1 - box.lo[a]);
  }
  box.finish();
  win.finish();
  const int64_t kofs = ((t.b * P.Ltot + ktok) * P.Hkv + hk) * (D * ES);
  const char *kb = reinterpret_cast<const char *>(k) + kofs;
  const char *vb = reinterpret_cast<const char *>(v) + kofs;
  const char *qb = reinterpret_cast<const char *>(q) + (t.b * P.Ltot * P.H + t.h) * (D * ES);

  frag qf[NF], kf[NF], vf[NF];
  ld_row<T>(qb, (uint32_t)qtok * (uint32_t)(P.H * D * ES) + 16u * gq, qf);
  uint32_t cd, ko, unused;
  auto load = [&](int c) {
    cd = box.point(16 * c + n, ko, unused);
    ld_row<T>(kb, ko + 16u * gq, kf);
    ld_row<T>(vb, ko + 16u * gq, vf);
  };
  load(0);

  float *vrow = smem + w * (16 * RS + 16);
  uint32_t *crow = reinterpret_cast<uint32_t *>(vrow + 16 * RS);
  const float *vt = vrow + 4 * gq * RS + n;
  f32x4 o[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) o[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY, l = 0.f;
  const int nch = (box.npts + 15) >> 4;
  for (int c = 0; c < nch; ++c) {
    f32x4 s = wv_scores<T>(kf, qf);
    wv_lds<T>(vrow + n * RS, gq, vf);
    if (gq == 0) crow[n] = cd;
    load(c + 1);  // past the last chunk: its last point again
    wv_lds_sync();
    const uint4 cc = *reinterpret_cast<const uint4 *>(crow + 4 * gq);
    const uint32_t c4[4] = {cc.x, cc.y, cc.z, cc.w};
    float mx = -INFINITY;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      s[r] = win.holds(c4[r]) ? s[r] : -INFINITY;
      mx = fmaxf(mx, s[r]);
    }
    mx = wv_quad_max(mx) * P.sl2;
    // the reference point may trail the running maximum by up to 8 (a
    // factor 2^8 in P, exact after the division by l)
    if (__builtin_amdgcn_ballot_w64(mx > m + 8.f) != 0) {
      const float mn = fmaxf(m, mx);
      const float alpha = __builtin_amdgcn_exp2f(m - (mn == -INFINITY ? 0.f : mn));
      l *= alpha;
#pragma unroll
      for (int db = 0; db < NDB; ++db) o[db] *= alpha;
      m = mn;
    }
    const float mu = m == -INFINITY ? 0.f : m;
    float p[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      p[r] = __builtin_amdgcn_exp2f(fmaf(s[r], P.sl2, -mu));
      l += p[r];
    }
    wv_acc<NDB, RS>(vt, p, o);
  }
  l = wv_quad_sum(l);
  if (wv_nan(o, l)) {  // again, key by key
    m = -INFINITY;
    l = 0.f;
#pragma unroll
    for (int db = 0; db < NDB; ++db) o[db] = f32x4{0.f, 0.f, 0.f, 0.f};
    for (int x = 0; x < box.npts; ++x) {
      cd = box.point(x, ko, unused);
      ld_row<T>(kb, ko + 16u * gq, kf);
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < NF; ++i) s = wv_dot<T>(qf[i], kf[i], s);
      s = wv_quad_sum(s) * P.sl2;
      if (win.holds(cd)) {
        const float mn = fmaxf(m, s);
        const float mu = mn == -INFINITY ? 0.f : mn;
        const float alpha = exp2f(m - mu), pr = exp2f(s - mu);
        l = fmaf(l, alpha, pr);
        m = mn;
#pragma unroll
        for (int db = 0; db < NDB; ++db)
          o[db] = o[db] * alpha + pr * ld4<T>(vb + ko + (16 * db + 4 * gq) * ES);
      }
    }
  }
  if (!qv) return;
  const float inv = 1.f / l;
  const int64_t orow = (t.b * P.Otot + otok) * P.H + t.h;
  char *ob = reinterpret_cast<char *>(out) + orow * (D * ES);
#pragma unroll
  for (int db = 0; db < NDB; ++db) st4<T>(ob + (16 * db + 4 * gq) * ES, o[db] * inv);
  if (lse != nullptr && gq == 0) lse[orow] = (m + __log2f(l)) * kLn2;
}

// Backward.  Workgroups [0, gk.n_wg) own key tiles (dK, dV; the longer role,
// dispatched first), the rest query tiles (dQ); delta = rowsum(dO * O) - dlse
// is formed from the rows each role reads anyway plus O.
template <typename T, int D, int R, bool STR>
__global__ void __launch_bounds__(64 * wv_waves<D>())
    k_wvbwd(WvProb P, const T *__restrict__ q, const T *__restrict__ k, const T *__restrict__ v,
            const T *__restrict__ out, const float *__restrict__ lse, const T *__restrict__ dout,
            const float *__restrict__ dlse, T *__restrict__ dq, T *__restrict__ dk,
            T *__restrict__ dv) {
  typedef typename Wv<T>::frag frag;
  constexpr int ES = sizeof(T), NF = D * ES / 64, NDB = D / 16, RS = wv_rs<D>(), NW = wv_waves<D>();
  constexpr int LW = 2 * 16 * RS + 48;  // floats per wave
  __shared__ __align__(16) float smem[NW * LW];

  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, n = lane & 15, gq = lane >> 4;
  float *xrow = smem + w * LW;
  uint32_t *crow = reinterpret_cast<uint32_t *>(xrow + 2 * 16 * RS);
  const float *xt = xrow + 4 * gq * RS + n;
  const char *qc = reinterpret_cast<const char *>(q), *kc = reinterpret_cast<const char *>(k);
  const char *vc = reinterpret_cast<const char *>(v), *oc = reinterpret_cast<const char *>(out);
  const char *gc = reinterpret_cast<const char *>(dout);
  const uint32_t HB = (uint32_t)(P.H * D * ES);  // bytes per token of q, out, dout
  WvTile t;
  WvWin<R> win;

  if ((int)blockIdx.x >= P.gk.n_wg) {
    // =============================== dQ ===============================
    const uint32_t tile =
        (uint32_t)(wv_wg((int)blockIdx.x - P.gk.n_wg, P.gq.n_wg) * NW + w);
    if (!wv_decode<R>(P, P.gq, P.fH, tile, false, t)) return;
    const int hk = (int)fdiv((uint32_t)t.h, P.fRep);
    WvBox<R, false> box;
    bool qv = true;
    int64_t ktok = 0;
    int qtok = 0, otok = 0;
#pragma unroll
    for (int a = 3 - R; a < 3; ++a) {
      const WvAx &x = P.ax[a];
      box.lo[a] = wv_start(x, t.i0[a] * x.s, t.Lr[a]);
      box.E[a] = wv_end(x, (t.i0[a] + t.nv[a] - 1) * x.s, t.Lr[a]) - box.lo[a];
      box.SK[a] = (uint32_t)(x.d * x.tok) * (uint32_t)(P.Hkv * D * ES);
      ktok += (int64_t)(t.r[a] + x.d * box.lo[a]) * x.tok;
      const int i = wv_row(P.gq, t, a, n, qv);
      qtok += (t.r[a] + x.d * x.s * i) * x.tok;
      otok += (t.r[a] + x.d * i) * x.otok;
      win.axis(a, wv_start(x, i * x.s, t.Lr[a]) - box.lo[a],
               wv_end(x, i * x.s, t.Lr[a]) - 1 - box.lo[a]);
    }
    box.finish();
    win.finish();
    const int64_t kofs = ((t.b * P.Ltot + ktok) * P.Hkv + hk) * (D * ES);
    const char *kb = kc + kofs, *vb = vc + kofs;
    const int64_t qofs = (t.b * P.Ltot * P.H + t.h) * (D * ES);
    const int64_t orow0 = t.b * P.Otot * P.H + t.h;
    const uint32_t qo = (uint32_t)qtok * HB, oo = (uint32_t)otok * HB;

    frag qf[NF], df[NF], kf[NF], vf[NF];
    ld_row<T>(qc + qofs, qo + 16u * gq, qf);
    ld_row<T>(gc + orow0 * (D * ES), oo + 16u * gq, df);
    float delta = 0.f;
    {
      frag of[NF];
      ld_row<T>(oc + orow0 * (D * ES), oo + 16u * gq, of);
#pragma unroll
      for (int i = 0; i < NF; ++i) delta = wv_dot<T>(df[i], of[i], delta);
    }
    uint32_t cd, ko, unused;
    auto load = [&](int c) {
      cd = box.point(16 * c + n, ko, unused);
      ld_row<T>(kb, ko + 16u * gq, kf);
      ld_row<T>(vb, ko + 16u * gq, vf);
    };
    load(0);
    const int64_t orow = orow0 + (int64_t)otok * P.H;
    const float lse2 = lse[orow] * kLog2e;
    delta = wv_quad_sum(delta) - (dlse != nullptr ? dlse[orow] : 0.f);
    f32x4 acc[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db) acc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int nch = (box.npts + 15) >> 4;
    for (int c = 0; c < nch; ++c) {
      const f32x4 s = wv_scores<T>(kf, qf), dp = wv_scores<T>(vf, df);
      wv_lds<T>(xrow + n * RS, gq, kf);
      if (gq == 0) crow[n] = cd;
      load(c + 1);
      wv_lds_sync();
      const uint4 cc = *reinterpret_cast<const uint4 *>(crow + 4 * gq);
      const uint32_t c4[4] = {cc.x, cc.y, cc.z, cc.w};
      float ds[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float p = __builtin_amdgcn_exp2f(fmaf(s[r], P.sl2, -lse2));
        ds[r] = win.holds(c4[r]) ? p * (dp[r] - delta) : 0.f;
      }
      wv_acc<NDB, RS>(xt, ds, acc);
    }
    if (wv_nan(acc, 0.f)) {  // again, key by key
#pragma unroll
      for (int db = 0; db < NDB; ++db) acc[db] = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int x = 0; x < box.npts; ++x) {
        cd = box.point(x, ko, unused);
        ld_row<T>(kb, ko + 16u * gq, kf);
        ld_row<T>(vb, ko + 16u * gq, vf);
        float s = 0.f, dp = 0.f;
#pragma unroll
        for (int i = 0; i < NF; ++i) {
          s = wv_dot<T>(qf[i], kf[i], s);
          dp = wv_dot<T>(df[i], vf[i], dp);
        }
        s = wv_quad_sum(s);
        dp = wv_quad_sum(dp);
        if (win.holds(cd)) {
          const float ds = exp2f(fmaf(s, P.sl2, -lse2)) * (dp - delta);
#pragma unroll
          for (int db = 0; db < NDB; ++db)
            acc[db] += ds * ld4<T>(kb + ko + (16 * db + 4 * gq) * ES);
        }
      }
    }
    if (!qv) return;
    char *db_ = reinterpret_cast<char *>(dq) + qofs + qo;
#pragma unroll
    for (int db = 0; db < NDB; ++db) st4<T>(db_ + (16 * db + 4 * gq) * ES, acc[db] * P.scale);
    return;
  }

  // ============================== dK / dV ==============================
  const uint32_t tile = (uint32_t)(wv_wg(blockIdx.x, P.gk.n_wg) * NW + w);
  if (!wv_decode<R>(P, P.gk, P.fHkv, tile, true, t)) return;
  // the box of queries whose windows hold the tile's keys
  WvBox<R, STR> box;
  bool kv = true, on = true;  // on: the key's position carries a query
  int64_t qtok = 0, otok = 0;
  int ktok = 0;
#pragma unroll
  for (int a = 3 - R; a < 3; ++a) {
    const WvAx &x = P.ax[a];
    box.lo[a] = wv_istart(x, t.i0[a]);
    box.E[a] = wv_iend(x, t.i0[a] + t.nv[a] - 1, t.Lr[a], t.Qr[a]) - box.lo[a];
    box.SK[a] = (uint32_t)(x.d * x.s * x.tok) * HB;
    box.SO[a] = (uint32_t)(x.d * x.otok) * HB;
    qtok += (int64_t)(t.r[a] + x.d * x.s * box.lo[a]) * x.tok;
    otok += (int64_t)(t.r[a] + x.d * box.lo[a]) * x.otok;
    const int j = wv_row(P.gk, t, a, n, kv);
    ktok += (t.r[a] + x.d * j) * x.tok;
    on = on && (!STR || j % x.s == 0);
    win.axis(a, wv_istart(x, j) - box.lo[a], wv_iend(x, j, t.Lr[a], t.Qr[a]) - 1 - box.lo[a]);
  }
  box.finish();
  win.finish();
  const int64_t kofs = (t.b * P.Ltot * P.Hkv + t.h) * (D * ES);
  const uint32_t ko = (uint32_t)ktok * (uint32_t)(P.Hkv * D * ES);
  frag kf[NF], vf[NF];
  ld_row<T>(kc + kofs, ko + 16u * gq, kf);
  ld_row<T>(vc + kofs, ko + 16u * gq, vf);
  f32x4 adk[NDB], adv[NDB];
#pragma unroll
  for (int db = 0; db < NDB; ++db) {
    adk[db] = f32x4{0.f, 0.f, 0.f, 0.f};
    adv[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  float *const grow = xrow + 16 * RS;                              // dO rows
  float *const lrow = reinterpret_cast<float *>(crow) + 16;        // lse * log2(e)
  float *const drow = lrow + 16;                                   // delta
  const float *const gt = xt + 16 * RS;
  const int nch = (box.npts + 15) >> 4;
  // (row of the output grid, head h) at byte offset oo of that head's rows
  const uint32_t rowsh = (uint32_t)(D * ES);
  for (int hr = 0; hr < P.rep && nch > 0; ++hr) {
    const int h = t.h * P.rep + hr;
    const char *qb = qc + ((t.b * P.Ltot + qtok) * P.H + h) * (D * ES);
    const int64_t orow0 = (t.b * P.Otot + otok) * P.H + h;
    const char *gb = gc + orow0 * (D * ES), *ob = oc + orow0 * (D * ES);
    const float *lb = lse + orow0, *dlb = dlse != nullptr ? dlse + orow0 : nullptr;
    frag qf[NF], gf[NF], of[NF];
    uint32_t cd, qo, oo;
    float ls, dl;
    auto load = [&](int c) {
      cd = box.point(16 * c + n, qo, oo);
      ld_row<T>(qb, qo + 16u * gq, qf);
      ld_row<T>(gb, oo + 16u * gq, gf);
      ld_row<T>(ob, oo + 16u * gq, of);
      ls = lb[oo / rowsh];
      dl = dlb != nullptr ? dlb[oo / rowsh] : 0.f;
    };
    load(0);
    for (int c = 0; c < nch; ++c) {
      const f32x4 s = wv_scores<T>(qf, kf), dp = wv_scores<T>(gf, vf);
      float delta = 0.f;
#pragma unroll
      for (int i = 0; i < NF; ++i) delta = wv_dot<T>(gf[i], of[i], delta);
      delta = wv_quad_sum(delta) - dl;
      wv_lds<T>(xrow + n * RS, gq, qf);
      wv_lds<T>(grow + n * RS, gq, gf);
      if (gq == 0) {
        crow[n] = cd;
        lrow[n] = ls * kLog2e;
        drow[n] = delta;
      }
      load(c + 1);
      wv_lds_sync();
      const uint4 cc = *reinterpret_cast<const uint4 *>(crow + 4 * gq);
      const uint32_t c4[4] = {cc.x, cc.y, cc.z, cc.w};
      const f32x4 l4 = *reinterpret_cast<const f32x4 *>(lrow + 4 * gq);
      const f32x4 d4 = *reinterpret_cast<const f32x4 *>(drow + 4 * gq);
      float p[4], ds[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float e = __builtin_amdgcn_exp2f(fmaf(s[r], P.sl2, -l4[r]));
        p[r] = win.holds(c4[r]) ? e : 0.f;
        ds[r] = win.holds(c4[r]) ? e * (dp[r] - d4[r]) : 0.f;
      }
      wv_acc<NDB, RS>(gt, p, adv);
      wv_acc<NDB, RS>(xt, ds, adk);
    }
  }
  if (wv_nan(adk, 0.f) || wv_nan(adv, 0.f)) {  // again, query by query
#pragma unroll
    for (int db = 0; db < NDB; ++db) {
      adk[db] = f32x4{0.f, 0.f, 0.f, 0.f};
      adv[db] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    for (int hr = 0; hr < P.rep; ++hr) {
      const int h = t.h * P.rep + hr;
      const char *qb = qc + ((t.b * P.Ltot + qtok) * P.H + h) * (D * ES);
      const int64_t orow0 = (t.b * P.Otot + otok) * P.H + h;
      for (int x = 0; x < box.npts; ++x) {
        frag qf[NF], gf[NF], of[NF];
        uint32_t qo, oo;
        const uint32_t cd = box.point(x, qo, oo);
        const char *gb = gc + orow0 * (D * ES), *ob = oc + orow0 * (D * ES);
        ld_row<T>(qb, qo + 16u * gq, qf);
        ld_row<T>(gb, oo + 16u * gq, gf);
        ld_row<T>(ob, oo + 16u * gq, of);
        float s = 0.f, dp = 0.f, delta = 0.f;
#pragma unroll
        for (int i = 0; i < NF; ++i) {
          s = wv_dot<T>(kf[i], qf[i], s);
          dp = wv_dot<T>(vf[i], gf[i], dp);
          delta = wv_dot<T>(gf[i], of[i], delta);
        }
        s = wv_quad_sum(s);
        dp = wv_quad_sum(dp);
        delta = wv_quad_sum(delta);
        const int64_t orow = orow0 + oo / rowsh;
        if (dlse != nullptr) delta -= dlse[orow];
        if (win.holds(cd)) {
          const float pr = exp2f(fmaf(s, P.sl2, -lse[orow] * kLog2e));
          const float ds = pr * (dp - delta);
#pragma unroll
          for (int db = 0; db < NDB; ++db) {
            adv[db] += pr * ld4<T>(gb + oo + (16 * db + 4 * gq) * ES);
            adk[db] += ds * ld4<T>(qb + qo + (16 * db + 4 * gq) * ES);
          }
        }
      }
    }
  }
  if (!kv) return;
  char *dkb = reinterpret_cast<char *>(dk) + kofs + ko;
  char *dvb = reinterpret_cast<char *>(dv) + kofs + ko;
#pragma unroll
  for (int db = 0; db < NDB; ++db) {
    st4<T>(dkb + (16 * db + 4 * gq) * ES, adk[db] * P.scale);
    st4<T>(dvb + (16 * db + 4 * gq) * ES, adv[db]);
  }
  if (STR && !on) {  // no query here: its rows of dq are zero
    for (int hr = 0; hr < P.rep; ++hr) {
      char *zb = reinterpret_cast<char *>(dq) +
                 ((t.b * P.Ltot + ktok) * P.H + t.h * P.rep + hr) * (D * ES);
#pragma unroll
      for (int db = 0; db < NDB; ++db)
        st4<T>(zb + (16 * db + 4 * gq) * ES, f32x4{0.f, 0.f, 0.f, 0.f});
    }
  }
}

// ---------------------------------------------------------------------------
// Host side.

bool strided(const Prob &P) { return P.ax[0].s != 1 || P.ax[1].s != 1 || P.ax[2].s != 1; }

}  // namespace

bool wave_eligible(const Prob &P, int dtype) {
  if (P.dense || P.sample_extent != nullptr || P.n_extra > 0) return false;
  if (dtype == NA_F32 ? (P.D != 16 && P.D != 32 && P.D != 64 && P.D != 128)
                      : ((P.D != 32 && P.D != 64 && P.D != 128) || !strided(P)))
    return false;
  // the running maximum is taken over unscaled scores
  if (!(P.scale > 0.f) || !std::isfinite(P.scale)) return false;
  return wv_geometry_ok(P, dtype == NA_F32 ? 4 : 2);
}

// The forward where a tile's box holds many times a window's keys (few slots,
// strided queries): the product over the box costs more than the window alone on
// the vector ALU, the sooner the wider the head and the smaller the launch (one
// chain of chunks per wave).  Times here over there by box over window (K = 3
// stride 1 on one axis 6, stride 2 11, stride 3 16, 3 x 3 stride 2 9, 5 x 5 stride 3
// 7.8) and output rows (positions times heads):
//   float32  D 128: 5 to 8 1.03 to 1.2 up to 4e3 rows, 0.58 to 0.83 from 2.4e4 (1.01 at
//            7e3); 9 1.0 to 1.12.  D 64: 7 to 8 at most 1.0; 9 to 11 0.96 to 1.16, 0.83 to
//            0.87 from 8e4; 16 1.03 to 1.34.  D 16 / 32: up to 11 at most 1.0, 16 0.7 to
//            1.15
//   16 bits  D 128: 8 to 11 0.78 to 1.12 up to 7e3, 0.72 to 0.92 from 1.7e4; 16 1.0 to
//            1.25.  D 32 / 64: up to 11 at most 1.0, 16 0.68 to 1.18
// The backward gains at every ratio.
bool wave_fwd_eligible(const Prob &P, int dtype) {
  if (!wave_eligible(P, dtype)) return false;
  if (P.any_size != 0) return true;
  int T[3] = {1, 1, 16};
  wv_tile(P, false, T);
  int64_t pts = 1, rows = (int64_t)P.B * P.H;
  for (int a = 3 - P.rank; a < 3; ++a) {
    const Axis &x = P.ax[a];
    pts *= std::min(phase_max(x), (T[a] - 1) * x.s + x.K);
    rows *= x.O;
  }
  int most = 12;
  if (P.D == 128) most = rows < 1 << 14 ? (dtype == NA_F32 ? 5 : 7) : (dtype == NA_F32 ? 8 : 12);
  if (P.D == 64 && dtype == NA_F32) most = rows < 1 << 16 ? 8 : 12;
  return pts <= (int64_t)P.kprod * most;
}

#define WV_R(KERNEL, TT, DD)                       \
  do {                                             \
    if (P.rank == 1) KERNEL(TT, DD, 1);            \
    else if (P.rank == 2) KERNEL(TT, DD, 2);       \
    else KERNEL(TT, DD, 3);                        \
  } while (0)
#define WV_D(KERNEL, TT)                           \
  do {                                             \
    if (P.D == 32) WV_R(KERNEL, TT, 32);           \
    else if (P.D == 64) WV_R(KERNEL, TT, 64);      \
    else WV_R(KERNEL, TT, 128);                    \
  } while (0)
#define WV_ALL(KERNEL)                                    \
  do {                                                    \
    if (dtype == NA_F32) {                                \
      if (P.D == 16) WV_R(KERNEL, float, 16);             \
      else WV_D(KERNEL, float);                           \
    } else if (dtype == NA_BF16) {                        \
      WV_D(KERNEL, bf16_t);                               \
    } else {                                              \
      WV_D(KERNEL, f16_t);                                \
    }                                                     \
  } while (0)

void wave_fwd(const Prob &P, int dtype, const void *q, const void *k, const void *v, void *out,
              float *lse, hipStream_t st) {
  const WvProb W = make_wvprob(P, false, P.D == 128 ? wv_waves<128>() : wv_waves<64>());
  if (W.gq.n_tiles == 0) return;
#define WV_F(TT, DD, RR)                                                                        \
  hipLaunchKernelGGL((k_wvfwd<TT, DD, RR>), dim3(W.gq.n_wg), dim3(64 * wv_waves<DD>()), 0, st, W, \
                     (const TT *)q, (const TT *)k, (const TT *)v, (TT *)out, lse)
  WV_ALL(WV_F);
#undef WV_F
}

void wave_bwd(const Prob &P, int dtype, const void *q, const void *k, const void *v,
              const void *out, const float *lse, const void *dout, const float *dlse, void *dq,
              void *dk, void *dv, hipStream_t st) {
  const WvProb W = make_wvprob(P, true, P.D == 128 ? wv_waves<128>() : wv_waves<64>());
  if (W.gq.n_tiles == 0) return;
  const bool str = strided(P);
#define WV_BL(TT, DD, RR, SS)                                                               \
  hipLaunchKernelGGL((k_wvbwd<TT, DD, RR, SS>), dim3(W.gk.n_wg + W.gq.n_wg),                \
                     dim3(64 * wv_waves<DD>()), 0, st, W, (const TT *)q, (const TT *)k,     \
                     (const TT *)v, (const TT *)out, lse, (const TT *)dout, dlse, (TT *)dq, \
                     (TT *)dk, (TT *)dv)
  // 16-bit problems come here only with a stride
#define WV_B(TT, DD, RR)                                                       \
  do {                                                                         \
    if (sizeof(TT) == 2 || str) WV_BL(TT, DD, RR, true);                       \
    else WV_BL(TT, DD, RR, (sizeof(TT) == 2));                                 \
  } while (0)
  WV_ALL(WV_B);
#undef WV_B
#undef WV_BL
}

#undef WV_ALL
#undef WV_D
#undef WV_R

}  // namespace na
