// The differentiable ops as torch custom operators with their autograd nodes
// in C++ over the C ABI of libnatten_amd.so: the fused op (natten_amd::na_fused),
// the split ops (na_split_qk, na_split_av), the DiNAT ops (na_rpb_qk, na_rpb_av)
// and a layer's projections (na_linear).
//
// The reference's autograd layer (autograd/na1d.py:34-53, na2d.py:34-64,
// na3d.py) wraps the fused forward / backward in an mx.custom_function; the
// Python twins here are autograd/fused.py's _FusedNA, autograd/split.py's and
// autograd/allin1.py's Functions.  These nodes do the same work without
// Python in the backward and without ctypes marshalling in either direction:
// an eager training step is host-bound (the config-2 kernels take ~21 us per
// step, the host path several times that), so the per-call host cost is what a
// caller who does not capture graphs sees.  A split or DiNAT step has two nodes
// each way: eager, against the Python Functions over ctypes, split
// [4, 56, 56, 4, 32] K = 7 186 -> 107 us, DiNAT [8, 2048, 12, 12] K = 7
// 188 -> 116 us (66 and 57 us of them on the GPU).
//
// Built with the host compiler against torch's headers only (no HIP
// headers): the caller passes torch's current stream handle, and the
// backward launches on the forward's stream (torch runs a node's backward
// on the stream of its forward).

#include <ATen/ATen.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/library.h>

#include <cstdint>
#include <cstring>
#include <vector>

#include "natten_amd.h"

namespace {

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

void check_rc(int rc, const char *what) {
  TORCH_CHECK(rc == NA_OK, "natten_amd ", what, " failed (", rc, "): ", na_last_error());
}

void check_device(const at::Tensor &t) {
  if (!t.defined()) return;
  TORCH_CHECK(t.is_cuda(),
              "natten_amd's hip backend runs on MI355X (HIP) tensors only; got a tensor on ",
              t.device(), ". There is no CPU implementation.");
}

// `t` is on `q`'s device (checked after the shapes: a mismatched call raises
// the same wherever its tensors are).
void check_devices(const at::Tensor &q, std::initializer_list<const at::Tensor *> others) {
  check_device(q);
  for (const at::Tensor *t : others)
    if (t->defined())
      TORCH_CHECK(t->device() == q.device(), "tensors are on different devices: ", q.device(),
                  " and ", t->device());
}

int32_t dtype_code(at::ScalarType s) {
  switch (s) {
    case at::kFloat:
      return NA_F32;
    case at::kHalf:
      return NA_F16;
    case at::kBFloat16:
      return NA_BF16;
    default:
      TORCH_CHECK(false, "natten_amd supports float32/float16/bfloat16 tensors, got ", s);
  }
  return -1;
}

const void *cptr(const at::Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }
void *mptr(const at::Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }

// q [B, X..., H, D], k [B, X..., H_kv, D]; per-axis fields hold the rank's
// axes first and 1 (0 for causal) after them, as na_params documents.
na_params make_params(const at::Tensor &q, const at::Tensor &k, at::IntArrayRef kernel,
                      at::IntArrayRef stride, at::IntArrayRef dilation,
                      at::IntArrayRef causal, double scale, int64_t n_extra, int64_t flags,
                      const at::Tensor &sample_extent) {
  const int64_t rank = q.dim() - 3;
  TORCH_CHECK(rank >= 1 && rank <= 3, "natten_amd: q must be [B, *spatial, heads, dim]");
  TORCH_CHECK((int64_t)kernel.size() == rank && (int64_t)stride.size() == rank &&
                  (int64_t)dilation.size() == rank && (int64_t)causal.size() == rank,
              "natten_amd: per-axis parameters must have one entry per spatial axis");
  for (int64_t a = 0; a < rank; ++a)
    TORCH_CHECK(kernel[a] > 0 && stride[a] > 0 && dilation[a] > 0,
                "natten_amd: kernel, stride and dilation must be positive");
  na_params p{};
  p.rank = (int32_t)rank;
  p.batch = (int32_t)q.size(0);
  p.heads = (int32_t)q.size(-2);
  p.kv_heads = (int32_t)k.size(-2);
  p.head_dim = (int32_t)q.size(-1);
  p.dtype = dtype_code(q.scalar_type());
  for (int a = 0; a < 3; ++a) {
    p.extent[a] = 1;
    p.kernel[a] = 1;
    p.dilation[a] = 1;
    p.stride[a] = 1;
    p.causal[a] = 0;
  }
  for (int64_t a = 0; a < rank; ++a) {
    p.extent[a] = (int32_t)q.size(1 + a);
    p.kernel[a] = (int32_t)kernel[a];
    p.dilation[a] = (int32_t)dilation[a];
    p.stride[a] = (int32_t)stride[a];
    p.causal[a] = causal[a] != 0 ? 1 : 0;
  }
  p.scale = (float)scale;
  p.n_extra = (int32_t)n_extra;
  p.flags = (int32_t)flags;
  p.sample_extent =
      sample_extent.defined() ? static_cast<const int32_t *>(sample_extent.data_ptr()) : nullptr;
  return p;
}

// A node's parameters as one saved value: the parameter block's bytes in
// 64-bit words, then `more`.  No device pointer is kept in it.
template <typename P>
std::vector<int64_t> pack(const P &p, std::initializer_list<int64_t> more) {
  std::vector<int64_t> v((sizeof(P) + 7) / 8);
  std::memcpy(v.data(), &p, sizeof(P));
  v.insert(v.end(), more);
  return v;
}
template <typename P>
P unpack(const std::vector<int64_t> &v, const int64_t **more) {
  P p;
  std::memcpy(&p, v.data(), sizeof(P));
  *more = v.data() + (sizeof(P) + 7) / 8;
  return p;
}

void *as_stream(int64_t s) { return reinterpret_cast<void *>(s); }

at::Tensor contig(const at::Tensor &t) { return t.defined() ? t.contiguous() : t; }

struct FusedNA : public torch::autograd::Function<FusedNA> {
  // The optional inputs come as std::optional so that an absent one is not
  // taken for an (undefined) variable input of the node.
  static variable_list forward(AutogradContext *ctx, at::Tensor q, at::Tensor k, at::Tensor v,
                               std::optional<at::Tensor> extra_k_opt,
                               std::optional<at::Tensor> extra_v_opt,
                               std::optional<at::Tensor> sample_extent_opt,
                               std::vector<int64_t> kernel, std::vector<int64_t> stride,
                               std::vector<int64_t> dilation, std::vector<int64_t> causal,
                               double scale, int64_t flags, int64_t stream) {
    at::Tensor extra_k = extra_k_opt.value_or(at::Tensor());
    at::Tensor extra_v = extra_v_opt.value_or(at::Tensor());
    const at::Tensor sample_extent = sample_extent_opt.value_or(at::Tensor());
    for (const at::Tensor *t : std::initializer_list<const at::Tensor *>{
             &q, &k, &v, &extra_k, &extra_v, &sample_extent})
      check_device(*t);
    // the shape rules the functional layer has already applied, restated for
    // direct callers of the operator
    TORCH_CHECK(q.dim() == k.dim() && q.dim() == v.dim() && q.size(0) == k.size(0) &&
                    q.size(0) == v.size(0) && k.sizes() == v.sizes() && q.size(-1) == k.size(-1),
                "natten_amd na_fused: q [B, *spatial, H, D], k / v [B, *spatial, H_kv, D]");
    for (int64_t a = 1; a + 2 < q.dim(); ++a)
      TORCH_CHECK(q.size(a) == k.size(a), "natten_amd na_fused: spatial extents differ");
    TORCH_CHECK(k.size(-2) > 0 && q.size(-2) % k.size(-2) == 0,
                "natten_amd na_fused: heads_q must be divisible by heads_kv");
    TORCH_CHECK(k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type(),
                "natten_amd na_fused: q, k and v must share a dtype");
    TORCH_CHECK(extra_k.defined() == extra_v.defined(),
                "natten_amd na_fused: extra_k and extra_v come together");
    if (extra_k.defined())
      TORCH_CHECK(extra_k.dim() == 4 && extra_k.sizes() == extra_v.sizes() &&
                      extra_k.size(0) == q.size(0) && extra_k.size(2) == k.size(-2) &&
                      extra_k.size(3) == q.size(-1) && extra_k.scalar_type() == q.scalar_type() &&
                      extra_v.scalar_type() == q.scalar_type(),
                  "natten_amd na_fused: extra_k / extra_v [B, N_extra, H_kv, D] in q's dtype");
    if (sample_extent.defined())
      TORCH_CHECK(sample_extent.scalar_type() == at::kInt && sample_extent.is_contiguous() &&
                      sample_extent.numel() == q.size(0) * (q.dim() - 3),
                  "natten_amd na_fused: sample_extent is a contiguous int32 [B, rank] tensor");
    q = q.contiguous();
    k = contig(k);
    v = contig(v);
    extra_k = contig(extra_k);
    extra_v = contig(extra_v);
    const int64_t n_extra = extra_k.defined() ? extra_k.size(1) : 0;
    const na_params p = make_params(q, k, kernel, stride, dilation, causal, scale, n_extra, flags,
                                    sample_extent);
    std::vector<int64_t> osz(q.sizes().begin(), q.sizes().end());
    for (size_t a = 0; a < kernel.size(); ++a)
      osz[1 + a] = (osz[1 + a] + stride[a] - 1) / stride[a];
    at::Tensor out = at::empty(osz, q.options());
    osz.pop_back();
    at::Tensor lse = at::empty(osz, q.options().dtype(at::kFloat));
    check_rc(na_fwd(&p, q.data_ptr(), k.data_ptr(), v.data_ptr(), cptr(extra_k), cptr(extra_v),
                    out.data_ptr(), static_cast<float *>(lse.data_ptr()),
                    reinterpret_cast<void *>(stream)),
             "na_fwd");
    ctx->save_for_backward({q, k, v, extra_k, extra_v, out, lse, sample_extent});
    na_params saved = p;
    saved.sample_extent = nullptr;  // read from the saved tensor again
    ctx->saved_data["p"] = pack(saved, {stream});
    // lse is differentiable too: its gradient enters the backward as
    // delta - dlse
    ctx->set_materialize_grads(false);
    return {out, lse};
  }

  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const at::Tensor &q = s[0], &k = s[1], &v = s[2], &extra_k = s[3], &extra_v = s[4],
                     &out = s[5], &lse = s[6], &sample_extent = s[7];
    at::Tensor gout = grads[0], glse = grads.size() > 1 ? grads[1] : at::Tensor();
    if (!gout.defined()) gout = at::zeros_like(out);
    gout = gout.contiguous();
    if (gout.scalar_type() != q.scalar_type()) gout = gout.to(q.scalar_type());
    if (glse.defined()) {
      glse = glse.contiguous();
      if (glse.scalar_type() != at::kFloat) glse = glse.to(at::kFloat);
    }
    const std::vector<int64_t> packed = ctx->saved_data["p"].toIntVector();
    const int64_t *more;
    na_params p = unpack<na_params>(packed, &more);
    p.sample_extent = static_cast<const int32_t *>(cptr(sample_extent));
    void *stream = as_stream(more[0]);
    const int64_t n_extra = p.n_extra;
    const size_t ws_bytes = na_bwd_workspace_bytes(&p);
    at::Tensor dq = at::empty_like(q), dk = at::empty_like(k), dv = at::empty_like(v);
    at::Tensor dek = n_extra ? at::empty_like(extra_k) : at::Tensor();
    at::Tensor dev = n_extra ? at::empty_like(extra_v) : at::Tensor();
    at::Tensor ws = ws_bytes ? at::empty({(int64_t)ws_bytes}, q.options().dtype(at::kByte))
                             : at::Tensor();
    const float *dlse = glse.defined() ? static_cast<const float *>(glse.data_ptr()) : nullptr;
    check_rc(na_bwd(&p, q.data_ptr(), k.data_ptr(), v.data_ptr(), cptr(extra_k), cptr(extra_v),
                    out.data_ptr(), static_cast<const float *>(lse.data_ptr()), gout.data_ptr(),
                    dlse, dq.data_ptr(),
                    dk.data_ptr(), dv.data_ptr(), mptr(dek), mptr(dev), mptr(ws), ws_bytes,
                    stream),
             "na_bwd");
    // one entry per forward input: q, k, v, extra_k, extra_v, then the
    // non-differentiable sample extents and parameters
    return {dq, dk, dv, dek, dev, at::Tensor(), at::Tensor(), at::Tensor(),
            at::Tensor(), at::Tensor(), at::Tensor(), at::Tensor(), at::Tensor()};
  }
};

std::tuple<at::Tensor, at::Tensor> na_fused(const at::Tensor &q, const at::Tensor &k,
                                            const at::Tensor &v,
                                            const std::optional<at::Tensor> &extra_k,
                                            const std::optional<at::Tensor> &extra_v,
                                            const std::optional<at::Tensor> &sample_extent,
                                            at::IntArrayRef kernel, at::IntArrayRef stride,
                                            at::IntArrayRef dilation, at::IntArrayRef causal,
                                            double scale, int64_t flags, int64_t stream) {
  auto r = FusedNA::apply(q, k, v, extra_k, extra_v, sample_extent, kernel.vec(), stride.vec(),
                          dilation.vec(), causal.vec(), scale, flags, stream);
  return {r[0], r[1]};
}

// The fused op on a layer's packed projection qkv [B, X..., 3, H, D] (nn.py): the
// three tensors come out of it in one pass and their gradients go back into one
// packed gradient.
struct FusedQKV : public torch::autograd::Function<FusedQKV> {
  static variable_list forward(AutogradContext *ctx, at::Tensor qkv, at::IntArrayRef kernel,
                               at::IntArrayRef stride, at::IntArrayRef dilation,
                               at::IntArrayRef causal, double scale, int64_t flags,
                               int64_t stream) {
    TORCH_CHECK(qkv.dim() >= 5 && qkv.dim() <= 7 && qkv.size(-3) == 3,
                "natten_amd na_fused_qkv: qkv is [B, *spatial, 3, H, D], got ", qkv.sizes());
    qkv = qkv.contiguous();
    std::vector<int64_t> sz(qkv.sizes().begin(), qkv.sizes().end());
    const int64_t row = qkv.size(-1) * qkv.size(-2) * (int64_t)qkv.element_size();
    sz.erase(sz.end() - 3);
    std::vector<int64_t> all(sz);
    all.insert(all.begin(), 3);
    const int64_t tokens = row > 0 ? (int64_t)(qkv.numel() * qkv.element_size() / (3 * row)) : 0;
    at::Tensor parts = at::empty(all, qkv.options());
    const at::Tensor q = parts.select(0, 0), k = parts.select(0, 1), v = parts.select(0, 2);
    const na_params p =
        make_params(q, k, kernel, stride, dilation, causal, scale, 0, flags, at::Tensor());
    check_device(qkv);
    check_rc(na_pack3(1, tokens, row, qkv.data_ptr(), parts.data_ptr(), as_stream(stream)),
             "na_pack3");
    for (size_t a = 0; a < kernel.size(); ++a) sz[1 + a] = (sz[1 + a] + stride[a] - 1) / stride[a];
    at::Tensor out = at::empty(sz, qkv.options());
    sz.pop_back();
    at::Tensor lse = at::empty(sz, qkv.options().dtype(at::kFloat));
    check_rc(na_fwd(&p, q.data_ptr(), k.data_ptr(), v.data_ptr(), nullptr, nullptr, out.data_ptr(),
                    static_cast<float *>(lse.data_ptr()), as_stream(stream)),
             "na_fwd");
    ctx->save_for_backward({parts, out, lse});
    ctx->saved_data["p"] = pack(p, {stream, tokens, row});
    return {out};
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const at::Tensor &parts = s[0], &out = s[1], &lse = s[2];
    const std::vector<int64_t> packed = ctx->saved_data["p"].toIntVector();
    const int64_t *more;
    const na_params p = unpack<na_params>(packed, &more);
    void *stream = as_stream(more[0]);
    const at::Tensor g = (grads[0].scalar_type() == parts.scalar_type()
                              ? grads[0] : grads[0].to(parts.scalar_type())).contiguous();
    const size_t ws_bytes = na_bwd_workspace_bytes(&p);
    at::Tensor d = at::empty_like(parts);
    at::Tensor ws = ws_bytes ? at::empty({(int64_t)ws_bytes}, parts.options().dtype(at::kByte))
                             : at::Tensor();
    auto part = [](const at::Tensor &t, int i) {
      return static_cast<void *>(static_cast<char *>(t.data_ptr()) +
                                 i * (t.numel() / 3) * (int64_t)t.element_size());
    };
    check_rc(na_bwd(&p, part(parts, 0), part(parts, 1), part(parts, 2), nullptr, nullptr,
                    out.data_ptr(), static_cast<const float *>(lse.data_ptr()), g.data_ptr(),
                    nullptr, part(d, 0), part(d, 1), part(d, 2), nullptr, nullptr, mptr(ws),
                    ws_bytes, stream),
             "na_bwd");
    std::vector<int64_t> sz(parts.sizes().begin() + 1, parts.sizes().end());
    sz.insert(sz.end() - 2, 3);
    at::Tensor dqkv = at::empty(sz, parts.options());
    check_rc(na_pack3(0, more[1], more[2], d.data_ptr(), dqkv.data_ptr(), stream), "na_pack3");
    const at::Tensor none;
    return {dqkv, none, none, none, none, none, none, none};
  }
};

at::Tensor na_fused_qkv(const at::Tensor &qkv, at::IntArrayRef kernel, at::IntArrayRef stride,
                        at::IntArrayRef dilation, at::IntArrayRef causal, double scale,
                        int64_t flags, int64_t stream) {
  return FusedQKV::apply(qkv, kernel, stride, dilation, causal, scale, flags, stream)[0];
}

// ---- split ops (autograd/split.py) ----------------------------------------
// The functional layer has validated the call; its shape rules are restated for
// direct callers of the operators, whose kernels index by these sizes.

std::vector<int64_t> split_sizes(const at::Tensor &x, at::IntArrayRef stride, int64_t last) {
  std::vector<int64_t> sz(x.sizes().begin(), x.sizes().end());
  for (size_t a = 0; a < stride.size(); ++a) sz[1 + a] = (sz[1 + a] + stride[a] - 1) / stride[a];
  sz.back() = last;
  return sz;
}

int64_t product(at::IntArrayRef v) {
  int64_t n = 1;
  for (const int64_t x : v) n *= x;
  return n;
}

at::Tensor to_type(const at::Tensor &t, at::ScalarType s) {
  return t.scalar_type() == s ? t : t.to(s);
}

struct SplitQK : public torch::autograd::Function<SplitQK> {
  static at::Tensor forward(AutogradContext *ctx, at::Tensor q, at::Tensor k,
                            at::IntArrayRef kernel, at::IntArrayRef stride,
                            at::IntArrayRef dilation, at::IntArrayRef causal, double scale,
                            int64_t flags, int64_t stream) {
    TORCH_CHECK(q.dim() == k.dim() && q.dim() >= 4 && q.dim() <= 6 &&
                    q.sizes().slice(0, q.dim() - 2) == k.sizes().slice(0, q.dim() - 2) &&
                    q.size(-1) == k.size(-1) && k.size(-2) > 0 && q.size(-2) % k.size(-2) == 0,
                "natten_amd na_split_qk: q [B, *spatial, H, D], k [B, *spatial, H_kv, D], got ",
                q.sizes(), " and ", k.sizes());
    const na_params p =
        make_params(q, k, kernel, stride, dilation, causal, scale, 0, flags, at::Tensor());
    check_devices(q, {&k});
    const auto kd = k.scalar_type();
    q = q.contiguous();
    k = to_type(k, q.scalar_type()).contiguous();
    at::Tensor logits = at::empty(split_sizes(q, stride, product(kernel)), q.options());
    check_rc(na_qk_fwd(&p, q.data_ptr(), k.data_ptr(), logits.data_ptr(), as_stream(stream)),
             "na_qk_fwd");
    ctx->save_for_backward({q, k});
    ctx->saved_data["p"] = pack(p, {stream, (int64_t)kd});
    return logits;
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const at::Tensor &q = s[0], &k = s[1];
    const std::vector<int64_t> packed = ctx->saved_data["p"].toIntVector();
    const int64_t *more;
    const na_params p = unpack<na_params>(packed, &more);
    const at::Tensor g = to_type(grads[0], q.scalar_type()).contiguous();
    at::Tensor dq = at::empty_like(q), dk = at::empty_like(k);
    check_rc(na_qk_bwd(&p, q.data_ptr(), k.data_ptr(), g.data_ptr(), dq.data_ptr(),
                       dk.data_ptr(), as_stream(more[0])),
             "na_qk_bwd");
    const at::Tensor none;
    return {dq, to_type(dk, (at::ScalarType)more[1]), none, none, none, none, none, none, none};
  }
};

struct SplitAV : public torch::autograd::Function<SplitAV> {
  static at::Tensor forward(AutogradContext *ctx, at::Tensor attn, at::Tensor v,
                            at::IntArrayRef kernel, at::IntArrayRef stride,
                            at::IntArrayRef dilation, at::IntArrayRef causal, int64_t stream) {
    const auto ad = attn.scalar_type(), vd = v.scalar_type();
    const auto dt = at::promote_types(ad, vd);
    na_params p = make_params(v, v, kernel, stride, dilation, causal, 1.0, 0, 0, at::Tensor());
    p.dtype = dtype_code(dt);
    std::vector<int64_t> want = split_sizes(v, stride, product(kernel));
    if (attn.dim() == v.dim()) want[want.size() - 2] = attn.size(-2);
    TORCH_CHECK(attn.sizes() == at::IntArrayRef(want) && v.size(-2) > 0 &&
                    attn.size(-2) % v.size(-2) == 0,
                "natten_amd na_split_av: attn is [B, *ceil(spatial / stride), H, slots] for v "
                "[B, *spatial, H_kv, D], got ", attn.sizes(), " and ", v.sizes());
    check_devices(attn, {&v});
    attn = to_type(attn, dt).contiguous();
    v = to_type(v, dt).contiguous();
    p.heads = (int32_t)attn.size(-2);
    std::vector<int64_t> osz(attn.sizes().begin(), attn.sizes().end());
    osz.back() = v.size(-1);
    at::Tensor out = at::empty(osz, v.options());
    check_rc(na_av_fwd(&p, attn.data_ptr(), v.data_ptr(), out.data_ptr(), as_stream(stream)),
             "na_av_fwd");
    ctx->save_for_backward({attn, v});
    ctx->saved_data["p"] = pack(p, {stream, (int64_t)ad, (int64_t)vd});
    return out;
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const at::Tensor &attn = s[0], &v = s[1];
    const std::vector<int64_t> packed = ctx->saved_data["p"].toIntVector();
    const int64_t *more;
    const na_params p = unpack<na_params>(packed, &more);
    const at::Tensor g = to_type(grads[0], v.scalar_type()).contiguous();
    at::Tensor dattn = at::empty_like(attn), dv = at::empty_like(v);
    check_rc(na_av_bwd(&p, attn.data_ptr(), v.data_ptr(), g.data_ptr(), dattn.data_ptr(),
                       dv.data_ptr(), as_stream(more[0])),
             "na_av_bwd");
    const at::Tensor none;
    return {to_type(dattn, (at::ScalarType)more[1]), to_type(dv, (at::ScalarType)more[2]),
            none, none, none, none, none};
  }
};

// ---- DiNAT ops (autograd/allin1.py) ----------------------------------------

na_rpb_params make_rpb(const at::Tensor &x, at::IntArrayRef kernel, at::IntArrayRef dilation,
                       double scale, bool has_scale, bool heads_first) {
  const int64_t rank = x.dim() - 3;
  TORCH_CHECK((rank == 1 || rank == 2) && (int64_t)kernel.size() == rank &&
                  (int64_t)dilation.size() == rank,
              "natten_amd: a rank-1 or rank-2 tensor with one kernel and dilation per axis");
  for (int64_t a = 0; a < rank; ++a)
    TORCH_CHECK(kernel[a] > 0 && dilation[a] > 0, "natten_amd: kernel and dilation must be positive");
  na_rpb_params p{};
  p.rank = (int32_t)rank;
  p.batch = (int32_t)x.size(0);
  p.heads = (int32_t)x.size(heads_first ? 1 : -2);
  p.head_dim = (int32_t)x.size(-1);
  for (int a = 0; a < 2; ++a) {
    p.extent[a] = a < rank ? (int32_t)x.size((heads_first ? 2 : 1) + a) : 1;
    p.kernel[a] = a < rank ? (int32_t)kernel[a] : 1;
    p.dilation[a] = a < rank ? (int32_t)dilation[a] : 1;
  }
  p.heads_first = heads_first ? 1 : 0;
  p.dtype = dtype_code(x.scalar_type());
  p.scale = has_scale ? (float)scale : 1.f;
  p.has_scale = has_scale ? 1 : 0;
  return p;
}

at::Tensor f32(const at::Tensor &t) { return to_type(t, at::kFloat).contiguous(); }

struct RpbQK : public torch::autograd::Function<RpbQK> {
  // rpb: float [H, 2K-1] (rank 2: [H, 2K0-1, 2K1-1]) or absent
  static at::Tensor forward(AutogradContext *ctx, at::Tensor q, at::Tensor k,
                            std::optional<at::Tensor> rpb_opt, at::IntArrayRef kernel,
                            at::IntArrayRef dilation, double scale, bool has_scale,
                            bool heads_first, int64_t stream) {
    const at::Tensor rpb = rpb_opt.value_or(at::Tensor());
    const na_rpb_params p = make_rpb(q, kernel, dilation, scale, has_scale, heads_first);
    TORCH_CHECK(q.sizes() == k.sizes(), "natten_amd na_rpb_qk: q and k must have identical shapes, "
                "got ", q.sizes(), " and ", k.sizes());
    if (rpb.defined()) {
      std::vector<int64_t> want{p.heads};
      for (const int64_t x : kernel) want.push_back(2 * x - 1);
      TORCH_CHECK(rpb.is_floating_point() && rpb.sizes() == at::IntArrayRef(want),
                  "natten_amd na_rpb_qk: rpb must have shape ", at::IntArrayRef(want), ", got ",
                  rpb.sizes());
    }
    check_devices(q, {&k, &rpb});
    const auto kd = k.scalar_type();
    q = q.contiguous();
    k = to_type(k, q.scalar_type()).contiguous();
    const at::Tensor bias = rpb.defined() ? f32(rpb) : rpb;
    std::vector<int64_t> osz(q.sizes().begin(), q.sizes().end());
    osz.back() = product(kernel);
    at::Tensor out = at::empty(osz, q.options().dtype(at::kFloat));
    check_rc(na_rpb_qk_fwd(&p, q.data_ptr(), k.data_ptr(), static_cast<const float *>(cptr(bias)),
                           static_cast<float *>(out.data_ptr()), as_stream(stream)),
             "na_rpb_qk_fwd");
    ctx->save_for_backward({q, k});
    ctx->saved_data["p"] = pack(
        p, {stream, (int64_t)kd, rpb.defined() ? (int64_t)rpb.scalar_type() : (int64_t)-1});
    return out;
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const at::Tensor &q = s[0], &k = s[1];
    const std::vector<int64_t> packed = ctx->saved_data["p"].toIntVector();
    const int64_t *more;
    const na_rpb_params p = unpack<na_rpb_params>(packed, &more);
    const bool has_rpb = more[2] >= 0;
    const at::Tensor g = f32(grads[0]);
    at::Tensor dq, dk, drpb, ws;
    if (ctx->needs_input_grad(0)) dq = at::empty_like(q);
    if (ctx->needs_input_grad(1)) dk = at::empty_like(k);
    size_t ws_bytes = 0;
    if (has_rpb && ctx->needs_input_grad(2)) {
      std::vector<int64_t> bsz{p.heads};
      for (int a = 0; a < p.rank; ++a) bsz.push_back(2 * p.kernel[a] - 1);
      drpb = at::empty(bsz, q.options().dtype(at::kFloat));
      ws_bytes = na_rpb_bwd_workspace_bytes(&p);
      ws = at::empty({(int64_t)std::max<size_t>(ws_bytes, 1)}, q.options().dtype(at::kByte));
    }
    check_rc(na_rpb_qk_bwd(&p, q.data_ptr(), k.data_ptr(), static_cast<const float *>(g.data_ptr()),
                           mptr(dq), mptr(dk), static_cast<float *>(mptr(drpb)), mptr(ws),
                           ws_bytes, as_stream(more[0])),
             "na_rpb_qk_bwd");
    if (dk.defined()) dk = to_type(dk, (at::ScalarType)more[1]);
    if (drpb.defined()) drpb = to_type(drpb, (at::ScalarType)more[2]);
    const at::Tensor none;
    return {dq, dk, drpb, none, none, none, none, none, none};
  }
};

struct RpbAV : public torch::autograd::Function<RpbAV> {
  // out_f32: the output (and its gradient) is float32, else v's dtype
  static at::Tensor forward(AutogradContext *ctx, at::Tensor attn, at::Tensor v,
                            at::IntArrayRef kernel, at::IntArrayRef dilation, bool heads_first,
                            bool out_f32, int64_t stream) {
    const na_rpb_params p = make_rpb(v, kernel, dilation, 1.0, false, heads_first);
    std::vector<int64_t> want(v.sizes().begin(), v.sizes().end());
    want.back() = product(kernel);
    TORCH_CHECK(attn.sizes() == at::IntArrayRef(want), "natten_amd na_rpb_av: attn must have shape ",
                at::IntArrayRef(want), ", got ", attn.sizes());
    check_devices(v, {&attn});
    const auto ad = attn.scalar_type();
    v = v.contiguous();
    attn = f32(attn);
    at::Tensor out =
        at::empty(v.sizes(), out_f32 ? v.options().dtype(at::kFloat) : v.options());
    check_rc(na_rpb_av_fwd(&p, static_cast<const float *>(attn.data_ptr()), v.data_ptr(),
                           out.data_ptr(), dtype_code(out.scalar_type()), as_stream(stream)),
             "na_rpb_av_fwd");
    ctx->save_for_backward({attn, v});
    ctx->saved_data["p"] = pack(p, {stream, (int64_t)ad});
    return out;
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const at::Tensor &attn = s[0], &v = s[1];
    const std::vector<int64_t> packed = ctx->saved_data["p"].toIntVector();
    const int64_t *more;
    const na_rpb_params p = unpack<na_rpb_params>(packed, &more);
    at::Tensor g = grads[0];
    if (g.scalar_type() != at::kFloat && g.scalar_type() != v.scalar_type()) g = g.to(at::kFloat);
    g = g.contiguous();
    at::Tensor dattn, dv;
    if (ctx->needs_input_grad(0)) dattn = at::empty_like(attn);
    if (ctx->needs_input_grad(1)) dv = at::empty_like(v);
    check_rc(na_rpb_av_bwd(&p, static_cast<const float *>(attn.data_ptr()), v.data_ptr(),
                           g.data_ptr(), dtype_code(g.scalar_type()),
                           static_cast<float *>(mptr(dattn)), mptr(dv), as_stream(more[0])),
             "na_rpb_av_bwd");
    if (dattn.defined()) dattn = to_type(dattn, (at::ScalarType)more[1]);
    const at::Tensor none;
    return {dattn, dv, none, none, none, none, none};
  }
};

// ---- a layer's projection (nn.py) -------------------------------------------
// torch's linear, with the weight and bias gradient from na_linear_wgrad: the
// caller passes contiguous-last-dim bf16 / fp16 tensors it takes.  A backward
// that records a graph goes through torch's own ops.
struct Linear : public torch::autograd::Function<Linear> {
  static at::Tensor forward(AutogradContext *ctx, at::Tensor x, at::Tensor w,
                            std::optional<at::Tensor> b, int64_t stream) {
    TORCH_CHECK(x.dim() >= 1 && w.dim() == 2 && x.size(-1) == w.size(1) &&
                    (!b.has_value() || (b->dim() == 1 && b->size(0) == w.size(0))),
                "natten_amd na_linear: x [..., k], weight [n, k], bias [n], got ", x.sizes(),
                " and ", w.sizes());
    dtype_code(x.scalar_type());  // one the backward knows
    const at::Tensor bias = b.value_or(at::Tensor());
    check_devices(x, {&w, &bias});
    ctx->save_for_backward({x, w});
    ctx->saved_data["p"] = std::vector<int64_t>{stream, b.has_value() ? 1 : 0};
    return at::linear(x, w, b);
  }
  static variable_list backward(AutogradContext *ctx, variable_list grads) {
    const variable_list s = ctx->get_saved_variables();
    const at::Tensor &x = s[0], &w = s[1];
    const std::vector<int64_t> p = ctx->saved_data["p"].toIntVector();
    const int64_t n = w.size(0), k = w.size(1);
    const at::Tensor g = grads[0].reshape({-1, n}), x2 = x.reshape({-1, k});
    at::Tensor dx, dw, db;
    if (ctx->needs_input_grad(0)) dx = g.mm(w).view_as(x);
    const bool want_w = ctx->needs_input_grad(1);
    const bool want_b = p[1] != 0 && ctx->needs_input_grad(2);
    const int32_t dt = dtype_code(x.scalar_type());
    const size_t bytes = na_linear_wgrad_workspace_bytes(dt, g.size(0), n, k);
    // beyond 1M weights the library's kernels fill the chip (3072 x 1024 over
    // 25088 rows: 278 us there, 314 here; 1536 x 512: 197 and 82)
    if (want_w && bytes > 0 && n * k <= (1 << 20) && !at::GradMode::is_enabled() &&
        g.scalar_type() == x.scalar_type()) {
      const at::Tensor gc = g.contiguous(), xc = x2.contiguous();
      dw = at::empty_like(w, at::MemoryFormat::Contiguous);
      if (want_b) db = at::empty({n}, w.options());
      at::Tensor ws = at::empty({(int64_t)bytes}, w.options().dtype(at::kByte));
      check_rc(na_linear_wgrad(dt, g.size(0), n, k, gc.data_ptr(), xc.data_ptr(), dw.data_ptr(),
                               mptr(db), ws.data_ptr(), bytes, as_stream(p[0])),
               "na_linear_wgrad");
    } else {
      if (want_w) dw = g.t().mm(x2);
      if (want_b) db = g.sum(0);
    }
    return {dx, dw, db, at::Tensor()};
  }
};

at::Tensor na_linear(const at::Tensor &x, const at::Tensor &w, const std::optional<at::Tensor> &b,
                     int64_t stream) {
  return Linear::apply(x, w, b, stream);
}

at::Tensor na_split_qk(const at::Tensor &q, const at::Tensor &k, at::IntArrayRef kernel,
                       at::IntArrayRef stride, at::IntArrayRef dilation, at::IntArrayRef causal,
                       double scale, int64_t flags, int64_t stream) {
  return SplitQK::apply(q, k, kernel, stride, dilation, causal, scale, flags, stream);
}
at::Tensor na_split_av(const at::Tensor &attn, const at::Tensor &v, at::IntArrayRef kernel,
                       at::IntArrayRef stride, at::IntArrayRef dilation, at::IntArrayRef causal,
                       int64_t stream) {
  return SplitAV::apply(attn, v, kernel, stride, dilation, causal, stream);
}
at::Tensor na_rpb_qk(const at::Tensor &q, const at::Tensor &k, const std::optional<at::Tensor> &rpb,
                     at::IntArrayRef kernel, at::IntArrayRef dilation, double scale,
                     bool has_scale, bool heads_first, int64_t stream) {
  return RpbQK::apply(q, k, rpb, kernel, dilation, scale, has_scale, heads_first, stream);
}
at::Tensor na_rpb_av(const at::Tensor &attn, const at::Tensor &v, at::IntArrayRef kernel,
                     at::IntArrayRef dilation, bool heads_first, bool out_f32, int64_t stream) {
  return RpbAV::apply(attn, v, kernel, dilation, heads_first, out_f32, stream);
}

}  // namespace

TORCH_LIBRARY(natten_amd, m) {
  m.def(
      "na_fused(Tensor q, Tensor k, Tensor v, Tensor? extra_k, Tensor? extra_v, "
      "Tensor? sample_extent, int[] kernel, int[] stride, int[] dilation, int[] causal, "
      "float scale, int flags, int stream) -> (Tensor, Tensor)");
  m.def(
      "na_split_qk(Tensor q, Tensor k, int[] kernel, int[] stride, int[] dilation, "
      "int[] causal, float scale, int flags, int stream) -> Tensor");
  m.def(
      "na_split_av(Tensor attn, Tensor v, int[] kernel, int[] stride, int[] dilation, "
      "int[] causal, int stream) -> Tensor");
  m.def(
      "na_rpb_qk(Tensor q, Tensor k, Tensor? rpb, int[] kernel, int[] dilation, float scale, "
      "bool has_scale, bool heads_first, int stream) -> Tensor");
  m.def(
      "na_rpb_av(Tensor attn, Tensor v, int[] kernel, int[] dilation, bool heads_first, "
      "bool out_f32, int stream) -> Tensor");
  m.def(
      "na_fused_qkv(Tensor qkv, int[] kernel, int[] stride, int[] dilation, int[] causal, "
      "float scale, int flags, int stream) -> Tensor");
  m.def("na_linear(Tensor x, Tensor weight, Tensor? bias, int stream) -> Tensor");
}

TORCH_LIBRARY_IMPL(natten_amd, CompositeImplicitAutograd, m) {
  m.impl("na_fused", na_fused);
  m.impl("na_split_qk", na_split_qk);
  m.impl("na_split_av", na_split_av);
  m.impl("na_rpb_qk", na_rpb_qk);
  m.impl("na_rpb_av", na_rpb_av);
  m.impl("na_linear", na_linear);
  m.impl("na_fused_qkv", na_fused_qkv);
}
