// Host path of the block's forward, decode step and training backward in native code: one call
// from Python checks, allocates (PyTorch's caching allocator) and launches everything that
// HdcMamba9v3Block's Python composition does, in the same order and on the same kernels and
// library products.  A block forward is 7-9 launches; issued one by one through ctypes they cost
// about 190 us of Python per block, more than the kernels take below ~8192 rows.  Nothing is kept
// between calls: workspaces that outlive a call are passed in.
#include <torch/extension.h>

#include <optional>
#include <tuple>
#include <vector>

#include "../../include/hdcm.h"

namespace {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

// A library status other than 0; surfaces in Python as hdcmamba_amd._ops.HdcmError.
struct StatusError : std::exception {
  const char* op;
  int code;
  StatusError(const char* o, int c) : op(o), code(c) {}
  const char* what() const noexcept override { return op; }
};
void check(const char* op, int code) {
  if (code != HDCM_OK) throw StatusError(op, code);
}

int dtype_of(const Tensor& t) {
  if (t.scalar_type() == at::kBFloat16) return HDCM_BF16;
  TORCH_CHECK_TYPE(t.scalar_type() == at::kFloat, "unsupported dtype ", t.scalar_type(), "; expected float32 or bfloat16");
  return HDCM_F32;
}

// Held by every entry point: no autograd, and no autocast, which would give a product another dtype than
// the kernels around it are told (a backward may be called inside a region that its forward was not in).
struct Entry {
  at::NoGradGuard no_grad;
  c10::impl::ExcludeDispatchKeyGuard no_autocast{c10::autocast_dispatch_keyset};
};

void on_gpu(const Tensor& t) {
  TORCH_CHECK(t.is_cuda(), "hdcmamba_amd kernels need ROCm GPU tensors; got a tensor on ", t.device(),
              " (there is no CPU path)");
}

// t in ref's dtype, contiguous, on ref's device
Tensor same(const Tensor& t, const Tensor& ref, const char* name) {
  TORCH_CHECK(t.device() == ref.device(), name, " is on ", t.device(), ", expected ", ref.device());
  return (t.scalar_type() == ref.scalar_type() ? t : t.to(ref.scalar_type())).contiguous();
}

// Stride of the rows of [B, L, W], which must be uniform
int64_t row_stride(const Tensor& t, const char* name) {
  if (t.numel() == 0) return t.size(2);
  TORCH_CHECK(t.stride(2) == 1, name, ": last dimension must be contiguous");
  const int64_t B = t.size(0), L = t.size(1);
  const int64_t rs = L > 1 ? t.stride(1) : B > 1 ? t.stride(0) : t.size(2);
  TORCH_CHECK(B <= 1 || t.stride(0) == rs * L, name, ": leading dimensions must collapse to uniformly strided rows");
  return rs;
}

// Batch stride of [B, L, W] rows for a kernel: a batch of one may come with any, which is not used.
int64_t batch_stride(const Tensor& t) { return t.size(0) > 1 ? t.stride(0) : t.size(1) * t.size(2); }

bool aligned(const Tensor& t, size_t n) { return (uintptr_t)t.const_data_ptr() % n == 0; }

Tensor bytes(size_t n, const Tensor& like) {
  return at::empty({(int64_t)std::max<size_t>(n, 256)}, like.options().dtype(at::kByte));
}
Tensor fp32(at::IntArrayRef shape, const Tensor& like) { return at::empty(shape, like.options().dtype(at::kFloat)); }

// Where the SSM scan runs relative to the slot kernels (HdcMamba9v3Block.ssm_overlap): on the main
// stream, or on the side stream joined before, between or after them.
enum Overlap { kMain = 0, kNone = 1, kState = 2, kGate = 3, kAfterState = 4 };

struct Streams {
  void *main, *side;
  int overlap;
  Tensor ssm_ws;
};
using StreamArgs = std::tuple<int64_t, int64_t, int, Tensor>;
Streams streams_of(const StreamArgs& a) {
  return {(void*)std::get<0>(a), (void*)std::get<1>(a), std::get<2>(a), std::get<3>(a)};
}

struct Dims {
  int64_t ds, H, C;
};
using DimArgs = std::tuple<int64_t, int64_t, int64_t>;
Dims dims_of(const DimArgs& a) { return {std::get<0>(a), std::get<1>(a), std::get<2>(a)}; }

// A block's parameters in the activation dtype, as passed: norm w, b; conv w, b; in_proj w, b; A_log;
// gamma; GroupNorm w, b; out_proj w.
struct Params {
  Tensor nw, nb, cw, cb, w_in, b_in, A_log, gamma, gnw, gnb, w_out;
  double eps;
};
Params params_of(const std::vector<Tensor>& p, const Tensor& x, const Dims& d, double eps) {
  TORCH_CHECK(p.size() == 11, "a block has 11 parameters");
  const int64_t dm = x.size(-1), K = d.ds + dm;
  static const char* names[] = {"norm.weight", "norm.bias", "conv1d.weight", "conv1d.bias", "in_proj.weight",
                                "in_proj.bias", "A_log", "gamma_buf", "group_norm.weight", "group_norm.bias",
                                "out_proj.weight"};
  std::vector<Tensor> q;
  q.reserve(11);
  for (size_t i = 0; i < 11; ++i) q.push_back(same(p[i], x, names[i]));
  // the kernels get pointers: the projections' shapes as a product would check them, the vectors' lengths
  const Tensor &w_in = q[4], &w_out = q[10];
  TORCH_CHECK(w_in.dim() == 2 && w_in.size(1) == dm && w_in.size(0) >= 3 * d.ds + 4 * dm && q[5].numel() == w_in.size(0),
              "in_proj ", w_in.sizes(), " + ", q[5].sizes(), " does not take x of width ", dm);
  TORCH_CHECK(w_out.dim() == 2 && w_out.size(1) == K && w_out.size(0) == dm, "out_proj ", w_out.sizes(), " should be [", dm, ", ",
              K, "]");
  const int64_t least[] = {dm, dm, 4 * dm, dm, 0, 0, d.ds, d.H, dm, dm};
  for (size_t i = 0; i < 10; ++i)
    TORCH_CHECK(q[i].numel() >= least[i], names[i], " has ", q[i].numel(), " values, expected ", least[i]);
  return {q[0], q[1], q[2].view({dm, 4}), q[3], q[4], q[5], q[6], q[7], q[8], q[9], q[10], eps};
}

// ------------------------------------------------------------------------ single operations
Tensor norm_conv(const Tensor& x, const Tensor& nw, const Tensor& nb, const Tensor& cw, const Tensor& cb, double eps,
                 void* s) {
  const int64_t B = x.size(0), L = x.size(1), D = x.size(2);
  Tensor out = at::empty({B, L, D}, x.options());
  check("hdcm_norm_conv_fwd", hdcm_norm_conv_fwd(x.const_data_ptr(), batch_stride(x), x.stride(1), nw.const_data_ptr(),
                                                 nb.const_data_ptr(), cw.const_data_ptr(), cb.const_data_ptr(),
                                                 out.mutable_data_ptr(), out.stride(0), out.stride(1), B, L, D,
                                                 (float)eps, dtype_of(x), s));
  return out;
}

// dx (x's dtype; with res [B, L, D] contiguous, plus res) and, as one fp32 buffer [7 D], d norm w, d norm b,
// d conv w [D, 4], d conv b
std::pair<Tensor, Tensor> norm_conv_bwd(const Tensor& go, const Tensor& x, const Tensor& nw, const Tensor& nb, const Tensor& cw,
                                  const Tensor* res, double eps, void* s) {
  const int64_t B = x.size(0), L = x.size(1), D = x.size(2);
  Tensor dx = at::empty({B, L, D}, x.options());
  Tensor dw = fp32({7 * D}, x);
  float* p = dw.mutable_data_ptr<float>();
  const size_t n = hdcm_norm_conv_bwd_workspace_bytes(B, L, D);
  Tensor ws = bytes(n, x);
  check("hdcm_norm_conv_bwd_add",
        hdcm_norm_conv_bwd_add(go.const_data_ptr(), batch_stride(go), go.stride(1), x.const_data_ptr(), batch_stride(x), x.stride(1),
                           nw.const_data_ptr(), nb.const_data_ptr(), cw.const_data_ptr(), res ? res->const_data_ptr() : nullptr,
                           L * D, D, dx.mutable_data_ptr(),
                           dx.stride(0), dx.stride(1), p, p + D, p + 2 * D, p + 6 * D, ws.mutable_data_ptr(), n, B, L, D,
                           (float)eps, dtype_of(x), s));
  return {dx, dw};
}

// x w^T (+ bias) (+ res) into out, fp32 rows [M, K] and [M, N]
void gemm_f32(const Tensor& x, const Tensor& w, const float* bias, const float* res, Tensor& out, int64_t M, void* s) {
  const int64_t K = w.size(1), N = w.size(0);
  check("hdcm_gemm_f32_fwd", hdcm_gemm_f32_fwd(x.const_data_ptr<float>(), K, w.const_data_ptr<float>(), K, bias, res, N,
                                               out.mutable_data_ptr<float>(), N, M, N, K, s));
}

Tensor in_proj(const Tensor& x, const Tensor& w, const Tensor& b, bool library, void* s) {
  const int64_t K = x.size(-1), M = K ? x.numel() / K : 0, N = w.size(0);
  const bool f32 = dtype_of(x) == HDCM_F32;
  if (library || !(f32 ? hdcm_gemm_f32_preferred(M, N, K) : hdcm_gemm_preferred(M, N, K, HDCM_BF16)) ||
      !aligned(x, 16) || !aligned(w, 16) || !aligned(b, f32 ? 16 : 8))
    return at::linear(x, w, b);
  Tensor out = at::empty({x.size(0), x.size(1), N}, x.options());
  if (f32) {
    gemm_f32(x, w, b.const_data_ptr<float>(), nullptr, out, M, s);
    return out;
  }
  check("hdcm_gemm_fwd", hdcm_gemm_fwd(x.const_data_ptr(), K, w.const_data_ptr(), K, b.const_data_ptr(),
                                       out.mutable_data_ptr(), N, M, N, K, HDCM_BF16, s));
  return out;
}

void ssm(const Tensor& projs, const Tensor& A_log, int64_t ds, Tensor& combined, float* h_final, float* stats,
         const Tensor& ws, void* s) {
  const int64_t B = projs.size(0), L = projs.size(1);
  check("hdcm_ssm_fwd", hdcm_ssm_fwd(projs.const_data_ptr(), row_stride(projs, "projs"), A_log.const_data_ptr(), nullptr,
                                     combined.mutable_data_ptr(), combined.size(2), h_final, stats, stats ? B * L : 0,
                                     ws.mutable_data_ptr(), ws.numel(), B, L, ds, dtype_of(projs), s));
}

struct Mixed {
  Tensor combined, x_conv, projs, slot_ws;
};
// SSM and slot memory + gate from projs into one row buffer [y_ssm | gated slot output]; with
// stats, the partial row statistics [P, B L, 2] of its rows.
void mixer(Mixed& m, const Params& p, const Dims& d, const Streams& st, int device, float* stats, float* h_final,
           float* S_final) {
  const Tensor& projs = m.projs;
  const int64_t B = projs.size(0), L = projs.size(1), dm = p.w_out.size(0), ds = d.ds;
  const int dt = dtype_of(projs);
  m.combined = at::empty({B, L, ds + dm}, projs.options());
  const size_t n = hdcm_slot_workspace_bytes(B, L, dm, d.H, d.C, dt);
  if (n == 0 && B * L > 0) throw StatusError("hdcm_slot_workspace_bytes", HDCM_EUNSUPPORTED);
  m.slot_ws = bytes(n, projs);
  const int64_t q = 3 * ds, prs = row_stride(projs, "projs");
  const auto after = [&](void* a, void* b) { check("hdcm_stream_after", hdcm_stream_after(a, b, device)); };
  const auto scan = [&] {
    if (st.overlap == kMain) return ssm(projs, p.A_log, ds, m.combined, h_final, stats, st.ssm_ws, st.main);
    after(st.side, st.main);
    ssm(projs, p.A_log, ds, m.combined, h_final, stats, st.ssm_ws, st.side);
    if (st.overlap == kNone) after(st.main, st.side);
  };
  if (st.overlap != kAfterState) scan();
  check("hdcm_slot_state_fwd",
        hdcm_slot_state_fwd(projs.const_data_ptr(), prs, q, p.gamma.const_data_ptr(), nullptr,
                            m.slot_ws.mutable_data_ptr(), m.slot_ws.numel(), B, L, dm, d.H, d.C, dt, st.main));
  if (st.overlap == kAfterState) scan();
  if (st.overlap == kState) after(st.main, st.side);
  const int64_t parts = (ds + 31) / 32;
  check("hdcm_slot_gate_fwd",
        hdcm_slot_gate_fwd(projs.const_data_ptr(), prs, q, p.gamma.const_data_ptr(), p.gnw.const_data_ptr(),
                           p.gnb.const_data_ptr(), 1e-5f, m.slot_ws.mutable_data_ptr(), m.slot_ws.numel(),
                           m.combined.mutable_data_ptr(), ds + dm, ds, S_final,
                           stats ? stats + 2 * parts * B * L : nullptr, stats ? B * L : 0, B, L, dm, d.H, d.C, dt, st.main));
  if (st.overlap == kGate || st.overlap == kAfterState) after(st.main, st.side);
}

// Row LayerNorm without affine into out (which may be x)
void row_norm(const Tensor& x, Tensor& out, void* s) {
  const int64_t W = x.size(-1);
  check("hdcm_rowln_fwd", hdcm_rowln_fwd(x.const_data_ptr(), W, out.mutable_data_ptr(), W, nullptr, nullptr,
                                         W ? x.numel() / W : 0, W, 1e-5f, dtype_of(x), s));
}

// ------------------------------------------------------------------------ block forward
struct ForwardOut {
  Tensor y;
  Mixed m;
};
// One block on chunk-aligned contiguous x [B, L, dm]; y into `out` (which may be x) when given.
ForwardOut forward(const Tensor& x, const Params& p, const Dims& d, const Streams& st, const OptTensor& out_, bool fused,
                   const OptTensor& w_sums, bool library, float* h_final, float* S_final) {
  const int64_t B = x.size(0), L = x.size(1), dm = x.size(2), M = B * L, ds = d.ds, K = ds + dm;
  Mixed m;
  m.x_conv = norm_conv(x, p.nw, p.nb, p.cw, p.cb, p.eps, st.main);
  m.projs = in_proj(m.x_conv, p.w_in, p.b_in, library, st.main);
  Tensor out = out_ ? *out_ : at::empty_like(x);
  const int device = x.get_device();
  if (fused && w_sums) {  // the GEMM takes the row statistics from the scan and the gate pass
    const int64_t parts = (ds + 31) / 32 + d.H;
    Tensor stats = fp32({parts, M, 2}, x);
    mixer(m, p, d, st, device, stats.mutable_data_ptr<float>(), h_final, S_final);
    check("hdcm_rowln_gemm_stats_fwd",
          hdcm_rowln_gemm_stats_fwd(m.combined.const_data_ptr(), K, p.w_out.const_data_ptr(), K,
                                    w_sums->const_data_ptr<float>(), stats.const_data_ptr<float>(), parts, M,
                                    x.const_data_ptr(), dm, out.mutable_data_ptr(), dm, M, dm, K, 1e-5f, dtype_of(x),
                                    st.main));
    return {out, m};
  }
  mixer(m, p, d, st, device, nullptr, h_final, S_final);
  if (fused) {
    check("hdcm_rowln_gemm_fwd",
          hdcm_rowln_gemm_fwd(m.combined.const_data_ptr(), K, p.w_out.const_data_ptr(), K, x.const_data_ptr(), dm,
                              out.mutable_data_ptr(), dm, M, dm, K, 1e-5f, dtype_of(x), st.main));
  } else {
    row_norm(m.combined, m.combined, st.main);
    Tensor o2 = out.view({M, dm});
    if (dtype_of(x) == HDCM_F32 && !library && hdcm_gemm_f32_preferred(M, dm, K) && aligned(m.combined, 16) &&
        aligned(p.w_out, 16) && aligned(x, 16) && aligned(out, 16))
      gemm_f32(m.combined, p.w_out, nullptr, x.const_data_ptr<float>(), o2, M, st.main);
    else if (out.const_data_ptr() == x.const_data_ptr()) o2.addmm_(m.combined.view({M, K}), p.w_out.t());
    else at::addmm_out(o2, x.view({M, dm}), m.combined.view({M, K}), p.w_out.t());
  }
  return {out, m};
}

void on_device_of(const Tensor& t, const Tensor& ref, const char* name) {
  TORCH_CHECK(t.device() == ref.device(), name, " is on ", t.device(), ", expected ", ref.device());
}

// A state the kernels write through its pointer: fp32, contiguous, on x's device.
float* opt_ptr(const OptTensor& t, at::IntArrayRef shape, const Tensor& x, const char* name) {
  if (!t) return nullptr;
  on_device_of(*t, x, name);
  TORCH_CHECK(t->scalar_type() == at::kFloat && t->is_contiguous() && t->sizes() == shape, name,
              " must be a contiguous fp32 tensor of shape ", shape);
  return t->mutable_data_ptr<float>();
}

Tensor block_forward(const Tensor& x, const std::vector<Tensor>& params, double eps, const DimArgs& dims,
                     const StreamArgs& streams, const OptTensor& out, bool fused, const OptTensor& w_sums, bool library,
                     const OptTensor& h_final, const OptTensor& S_final) {
  Entry entry;
  on_gpu(x);
  const Dims d = dims_of(dims);
  const int64_t B = x.size(0), dm = x.size(2), hd = dm / d.H;
  return forward(x, params_of(params, x, d, eps), d, streams_of(streams), out, fused, w_sums, library,
                 opt_ptr(h_final, {B, d.ds}, x, "h"), opt_ptr(S_final, {B, d.H, hd, hd}, x, "S_prev"))
      .y;
}

// [B, pad + L, dm] with pad zero rows in front of every sequence's rows
Tensor pad_rows(const Tensor& x_, int64_t pad, int64_t stream) {
  Entry entry;
  on_gpu(x_);
  const int dt = dtype_of(x_);
  const int64_t E = dt == HDCM_BF16 ? 8 : 4;
  Tensor x = x_;
  const int64_t B = x.size(0), L = x.size(1), D = x.size(2);
  const auto fits = [&] {
    return x.stride(2) == 1 && (B <= 1 || x.stride(0) % E == 0) && (L <= 1 || (x.stride(1) % E == 0 && x.stride(1) >= D)) &&
           aligned(x, 16);
  };
  if (!fits()) x = x.contiguous();
  if (D % E || !fits()) return at::constant_pad_nd(x, {0, 0, pad, 0});
  Tensor out = at::empty({B, L + pad, D}, x.options());
  check("hdcm_pad_rows_fwd", hdcm_pad_rows_fwd(x.const_data_ptr(), batch_stride(x), L > 1 ? x.stride(1) : D, out.mutable_data_ptr(), B, L,
                                               pad, D, dt, (void*)stream));
  return out;
}

void refresh_gamma(const Tensor& decay_log, const Tensor& gamma, int64_t stream) {
  on_gpu(gamma);
  TORCH_CHECK(decay_log.scalar_type() == gamma.scalar_type() && decay_log.is_contiguous() && gamma.is_contiguous() &&
                  decay_log.numel() == gamma.numel() && decay_log.device() == gamma.device(),
              "decay_log and gamma_buf must match");
  check("hdcm_gamma_fwd", hdcm_gamma_fwd(decay_log.const_data_ptr(), gamma.mutable_data_ptr(), gamma.numel(),
                                         dtype_of(gamma), (void*)stream));
  gamma.unsafeGetTensorImpl()->bump_version();
}

// ------------------------------------------------------------------------ decode step
// One token per row of x [B, dm]; the states advance in place.
Tensor block_step(const Tensor& x_, const std::vector<Tensor>& params, double eps, const DimArgs& dims, const Tensor& conv,
                  const Tensor& h, const Tensor& S_prev, const Tensor& S_intra, int64_t pos, const OptTensor& pos_dev,
                  bool fused_front, bool fused_out, const OptTensor& step_ws, int64_t stream) {
  Entry entry;
  on_gpu(x_);
  const Dims d = dims_of(dims);
  TORCH_CHECK(x_.dim() == 2, "step expects x of shape [B, d_model]");
  const bool fits =
      x_.stride(1) == 1 && (x_.size(0) <= 1 || x_.stride(0) % (16 / x_.element_size()) == 0) && aligned(x_, 16);
  const Tensor x = fits ? x_ : x_.clone(at::MemoryFormat::Contiguous);
  const int64_t B = x.size(0), dm = x.size(1), ds = d.ds, hd = dm / d.H, K = ds + dm, xs = B > 1 ? x.stride(0) : dm;
  const Params p = params_of(params, x, d, eps);
  const int64_t N = p.w_in.size(0);
  const int dt = dtype_of(x);
  void* s = (void*)stream;
  TORCH_CHECK(conv.scalar_type() == x.scalar_type() && conv.is_contiguous() && conv.sizes() == at::IntArrayRef({B, 3, dm}),
              "step: conv must be a contiguous [B,3,D] tensor of x's dtype");
  on_device_of(conv, x, "conv");
  if (pos_dev) on_device_of(*pos_dev, x, "pos_dev");
  float* hp = opt_ptr(h, {B, ds}, x, "h");
  float* sp = opt_ptr(S_prev, {B, d.H, hd, hd}, x, "S_prev");
  float* si = opt_ptr(S_intra, {B, d.H, hd, hd}, x, "S_intra");
  Tensor projs = at::empty({B, N}, x.options()), u = at::empty({B, dm}, x.options());
  const bool bf = dt == HDCM_BF16, rows16 = bf && B >= 1 && B <= 16;
  if (fused_front && rows16 && dm % 32 == 0 && dm <= 2048 && N >= 2048) {
    TORCH_CHECK(step_ws, "step: the fused front needs its workspace");
    check("hdcm_norm_conv_in_proj_step_fwd",
          hdcm_norm_conv_in_proj_step_fwd(x.const_data_ptr(), xs, p.nw.const_data_ptr(), p.nb.const_data_ptr(),
                                          p.cw.const_data_ptr(), p.cb.const_data_ptr(), conv.mutable_data_ptr(), (float)eps,
                                          u.mutable_data_ptr(), dm, p.w_in.const_data_ptr(), dm, p.b_in.const_data_ptr(),
                                          projs.mutable_data_ptr(), N, B, dm, N, step_ws->mutable_data_ptr(),
                                          step_ws->numel(), dt, s));
  } else {
    check("hdcm_norm_conv_step_fwd",
          hdcm_norm_conv_step_fwd(x.const_data_ptr(), xs, p.nw.const_data_ptr(), p.nb.const_data_ptr(),
                                  p.cw.const_data_ptr(), p.cb.const_data_ptr(), conv.mutable_data_ptr(),
                                  u.mutable_data_ptr(), dm, B, dm, (float)eps, dt, s));
    if (bf && B <= 16 && dm % 32 == 0 && dm <= 3072) {
      check("hdcm_skinny_gemm_fwd",
            hdcm_skinny_gemm_fwd(u.const_data_ptr(), dm, p.w_in.const_data_ptr(), dm, p.b_in.const_data_ptr(), nullptr, 0,
                                 projs.mutable_data_ptr(), N, B, N, dm, dt, s));
    } else {
      projs = at::linear(u, p.w_in, p.b_in);
    }
  }
  Tensor c = at::empty({B, K}, x.options());
  check("hdcm_mixer_step_fwd",
        hdcm_mixer_step_fwd(projs.const_data_ptr(), N, 3 * ds, p.A_log.const_data_ptr(), hp, p.gamma.const_data_ptr(), sp,
                            si, pos, pos_dev ? pos_dev->const_data_ptr<int>() : nullptr, d.C, p.gnw.const_data_ptr(),
                            p.gnb.const_data_ptr(), 1e-5f, c.mutable_data_ptr(), K, 0, ds, B, dm, ds, d.H, dt, s));
  if (fused_out) {
    Tensor y = at::empty({B, dm}, x.options());
    check("hdcm_rowln_gemm_fwd",
          hdcm_rowln_gemm_fwd(c.const_data_ptr(), K, p.w_out.const_data_ptr(), K, x.const_data_ptr(), xs,
                              y.mutable_data_ptr(), dm, B, dm, K, 1e-5f, dt, s));
    return y;
  }
  row_norm(c, c, s);
  if (bf && B <= 16 && K % 32 == 0 && K <= 3072) {
    Tensor y = at::empty({B, dm}, x.options());
    check("hdcm_skinny_gemm_fwd",
          hdcm_skinny_gemm_fwd(c.const_data_ptr(), K, p.w_out.const_data_ptr(), K, nullptr, x.const_data_ptr(),
                               xs, y.mutable_data_ptr(), dm, B, dm, K, dt, s));
    return y;
  }
  return at::addmm(x, c, p.w_out.t());
}

// ------------------------------------------------------------------------ training
// Gradients of the mixer from dcomb [B, L, ds + dm] (contiguous, projs' dtype): dprojs and, as one
// fp32 buffer [2 dm + ds], d GroupNorm w, d GroupNorm b, d A_log.
std::pair<Tensor, Tensor> mixer_grads(const Tensor& projs, const Tensor& A_log, const Tensor& gamma, const Tensor& gnw,
                                const Tensor& gnb, const Tensor& combined, const Tensor& slot_ws, const Tensor& dcomb,
                                const Dims& d, void* s) {
  const int64_t B = projs.size(0), L = projs.size(1), ds = d.ds, dm = gnw.numel(), W = ds + dm, P = row_stride(projs, "projs"), DP = projs.size(2);
  const int dt = dtype_of(projs);
  const int64_t esz = dt == HDCM_BF16 ? 2 : 4;
  Tensor dprojs = at::empty(projs.sizes(), projs.options());
  Tensor g = fp32({2 * dm + ds}, projs);
  float* gp = g.mutable_data_ptr<float>();
  {
    const size_t n = hdcm_slot_grad_workspace_bytes(B, L, dm, d.H, d.C, dt);
    Tensor ws = bytes(n, projs);
    check("hdcm_slot_grad",
          hdcm_slot_grad(projs.const_data_ptr(), P, 3 * ds, gamma.const_data_ptr(), gnw.const_data_ptr(),
                         gnb.const_data_ptr(), 1e-5f, slot_ws.const_data_ptr(), slot_ws.numel(),
                         (const char*)dcomb.const_data_ptr() + ds * esz, W, dprojs.mutable_data_ptr(), DP, gp,
                         gp + dm, ws.mutable_data_ptr(), ws.numel(), B, L, dm, d.H, d.C, dt, s));
  }
  const size_t n = hdcm_ssm_bwd_workspace_bytes(B, L, ds, dt);
  Tensor ws = bytes(n, projs);
  check("hdcm_ssm_bwd",
        hdcm_ssm_bwd(projs.const_data_ptr(), P, A_log.const_data_ptr(), combined.const_data_ptr(), W,
                     dcomb.const_data_ptr(), W, dprojs.mutable_data_ptr(), DP, gp + 2 * dm,
                     ws.mutable_data_ptr(), ws.numel(), B, L, ds, dt, s));
  return {dprojs, g};
}

// SlotSsmMixerFunction: (combined, slot workspace) from projs [B, L, P]
std::vector<Tensor> mixer_forward(const Tensor& projs, const Tensor& A_log, const Tensor& gamma, const Tensor& gnw,
                                  const Tensor& gnb, const DimArgs& dims, const StreamArgs& streams) {
  Entry entry;
  on_gpu(projs);
  Params p;
  p.A_log = same(A_log, projs, "A_log");
  p.gamma = same(gamma, projs, "gamma");
  p.gnw = same(gnw, projs, "gn_w");
  p.gnb = same(gnb, projs, "gn_b");
  p.w_out = p.gnw;  // (its row count is d_model)
  Mixed m;
  m.projs = projs;
  mixer(m, p, dims_of(dims), streams_of(streams), projs.get_device(), nullptr, nullptr, nullptr);
  return {m.combined, m.slot_ws};
}

std::vector<Tensor> mixer_backward(const Tensor& dcomb_, const Tensor& projs, const Tensor& A_log, const Tensor& gamma,
                                   const Tensor& gnw, const Tensor& gnb, const Tensor& combined, const Tensor& slot_ws,
                                   const DimArgs& dims, int64_t stream) {
  Entry entry;
  on_gpu(dcomb_);
  Tensor dcomb = same(dcomb_, projs, "grad");
  if (!aligned(dcomb, 16)) dcomb = dcomb.clone();
  const Dims d = dims_of(dims);
  auto g = mixer_grads(projs, same(A_log, projs, "A_log"), same(gamma, projs, "gamma"), same(gnw, projs, "gn_w"),
                       same(gnb, projs, "gn_b"), combined, slot_ws, dcomb, d, (void*)stream);
  const int64_t dm = gnw.numel();
  const Tensor w = g.second.to(gnw.scalar_type());
  return {g.first, g.second.narrow(0, 2 * dm, d.ds).to(A_log.scalar_type()), w.narrow(0, 0, dm),
          gnb.scalar_type() == gnw.scalar_type() ? w.narrow(0, dm, dm) : g.second.narrow(0, dm, dm).to(gnb.scalar_type())};
}

// FusedNormConv1dFunction
Tensor norm_conv_forward(const Tensor& x_, const Tensor& nw, const Tensor& nb, const Tensor& cw, const Tensor& cb,
                         double eps, int64_t stream) {
  Entry entry;
  on_gpu(x_);
  TORCH_CHECK(x_.dim() == 3, "norm_conv expects x of shape [B, L, D]");
  const Tensor x = x_.stride(2) == 1 ? x_ : x_.contiguous();
  const int64_t D = x.size(2);
  return norm_conv(x, same(nw, x, "ln_w"), same(nb, x, "ln_b"), same(cw.reshape({D, 4}), x, "conv_w"), same(cb, x, "conv_b"),
                   eps, (void*)stream);
}

std::vector<Tensor> norm_conv_backward(const Tensor& go_, const Tensor& x_, const Tensor& nw, const Tensor& nb,
                                       const Tensor& cw, double eps, int64_t stream) {
  Entry entry;
  on_gpu(go_);
  const Tensor x = x_.stride(2) == 1 ? x_ : x_.contiguous();
  const int64_t D = x.size(2);
  auto g = norm_conv_bwd(same(go_, x, "grad_out"), x, same(nw, x, "ln_w"), same(nb, x, "ln_b"),
                         same(cw.reshape({D, 4}), x, "conv_w"), nullptr, eps, (void*)stream);
  const Tensor w = g.second.to(x.scalar_type());
  return {g.first, w.narrow(0, 0, D), w.narrow(0, D, D), w.narrow(0, 2 * D, 4 * D).view(cw.sizes()), w.narrow(0, 6 * D, D)};
}

// Weight gradient y^T x of row-major y [M, N], x [M, K] and, with sums, y's column sums.  By the rule on sizes
// also where recorded library solutions are in use: those are of the forward's products.
std::pair<Tensor, Tensor> weight_grad(const Tensor& y, const Tensor& x, bool sums, void* s) {
  const int64_t M = y.size(0), N = y.size(1), K = x.size(1);
  if (!hdcm_gemm_tn_preferred(M, N, K, sums, dtype_of(y)) || !aligned(y, 16) || !aligned(x, 16))
    return {at::mm(y.t(), x), sums ? y.sum(0) : Tensor()};
  Tensor w = at::empty({N, K}, y.options()), c = sums ? at::empty({N}, y.options()) : Tensor();
  const size_t n = hdcm_gemm_tn_workspace_bytes(M, N, K);
  Tensor ws = bytes(n, y);
  check("hdcm_gemm_tn", hdcm_gemm_tn(y.const_data_ptr(), N, x.const_data_ptr(), K, w.mutable_data_ptr(), K,
                                     sums ? c.mutable_data_ptr() : nullptr, ws.mutable_data_ptr(), ws.numel(), M, N, K,
                                     HDCM_BF16, s));
  return {w, c};
}

// Recompute and backward of one block in training from x and dy [B, L, dm] (chunk-aligned,
// contiguous): gradients of x and of the parameters in params_of's order (undefined where there is
// none), in the parameters' dtypes.  mixer_grad: the differentiable mixer; otherwise the SSM and slot
// kernels are constants and only x and out_proj receive gradients.  need[0]: x; need[1..11]: the
// parameters.
std::vector<OptTensor> block_backward(const Tensor& x, const Tensor& dy, const std::vector<Tensor>& params, double eps,
                                      const DimArgs& dims, const StreamArgs& streams, bool mixer_grad, bool library,
                                      const std::vector<bool>& need) {
  Entry entry;
  on_gpu(x);
  const Dims d = dims_of(dims);
  const Streams st = streams_of(streams);
  const Params p = params_of(params, x, d, eps);
  const int64_t B = x.size(0), L = x.size(1), dm = x.size(2), M = B * L, K = d.ds + dm, N = p.w_in.size(0);
  std::vector<OptTensor> out(12);
  const auto give = [&](int i, const Tensor& g) {  // i: params_of's index
    if (need[i + 1]) out[i + 1] = g.scalar_type() == params[i].scalar_type() ? g : g.to(params[i].scalar_type());
  };
  // Parts [start, start + n) of fp32 sums, rounded once, to the type of each parameter (one conversion for
  // a run of parameters of one type).
  struct Part {
    int i;
    int64_t start, n;
  };
  const auto give_sums = [&](const Tensor& sums, std::initializer_list<Part> parts) {
    Tensor w = sums;
    for (const Part& q : parts) {
      if (!need[q.i + 1]) continue;
      if (w.scalar_type() != params[q.i].scalar_type()) w = sums.to(params[q.i].scalar_type());
      give(q.i, w.narrow(0, q.start, q.n).view(params[q.i].sizes()));
    }
  };
  if (!mixer_grad && !need[11]) {
    if (need[0]) out[0] = dy;
    return out;
  }
  Mixed m;
  m.x_conv = norm_conv(x, p.nw, p.nb, p.cw, p.cb, p.eps, st.main);
  m.projs = in_proj(m.x_conv, p.w_in, p.b_in, library, st.main);
  mixer(m, p, d, st, x.get_device(), nullptr, nullptr, nullptr);
  const Tensor dy2 = dy.view({M, dm});
  if (need[11]) {
    Tensor c = at::empty_like(m.combined);
    row_norm(m.combined, c, st.main);
    give(10, weight_grad(dy2, c.view({M, K}), false, st.main).first);
  }
  if (!mixer_grad) {
    if (need[0]) out[0] = dy;
    return out;
  }
  Tensor dcomb = at::empty_like(m.combined);
  {
    const Tensor dc = at::mm(dy2, p.w_out);  // d LN(combined)
    check("hdcm_rowln_bwd", hdcm_rowln_bwd(dc.const_data_ptr(), K, m.combined.const_data_ptr(), K, nullptr,
                                           dcomb.mutable_data_ptr(), K, nullptr, nullptr, nullptr, 0, M, K, 1e-5f,
                                           dtype_of(x), st.main));
  }
  auto g = mixer_grads(m.projs, p.A_log, p.gamma, p.gnw, p.gnb, m.combined, m.slot_ws, dcomb, d, st.main);
  m.projs.reset();
  m.combined.reset();
  dcomb.reset();
  give_sums(g.second, {{8, 0, dm}, {9, dm, dm}, {6, 2 * dm, d.ds}});
  const Tensor dproj2 = g.first.view({M, N});
  if (need[5]) {
    const auto wg = weight_grad(dproj2, m.x_conv.view({M, dm}), need[6], st.main);
    give(4, wg.first);
    if (need[6]) give(5, wg.second);
  } else if (need[6]) {
    give(5, dproj2.sum(0));
  }
  if (need[0] || need[1] || need[2] || need[3] || need[4]) {
    Tensor dxc = at::mm(dproj2, p.w_in).view({B, L, dm});
    const bool add = aligned(dy, 16);
    auto n = norm_conv_bwd(dxc, x, p.nw, p.nb, p.cw, add ? &dy : nullptr, p.eps, st.main);
    if (need[0]) out[0] = add ? n.first : n.first.add_(dy);
    give_sums(n.second, {{0, 0, dm}, {1, dm, dm}, {2, 2 * dm, 4 * dm}, {3, 6 * dm, dm}});
  }
  return out;
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  pybind11::register_exception_translator([](std::exception_ptr p) {
    try {
      if (p) std::rethrow_exception(p);
    } catch (const StatusError& e) {
      const auto cls = pybind11::module_::import("hdcmamba_amd._ops").attr("HdcmError");
      PyErr_SetObject(cls.ptr(), cls(e.op, e.code).ptr());
    }
  });
  m.attr("MAIN") = (int)kMain;
  m.attr("OVERLAP") = pybind11::dict(pybind11::arg("none") = (int)kNone, pybind11::arg("state") = (int)kState,
                                     pybind11::arg("gate") = (int)kGate, pybind11::arg("after_state") = (int)kAfterState);
  m.def("block_forward", &block_forward);
  m.def("block_step", &block_step);
  m.def("block_backward", &block_backward);
  m.def("pad_rows", &pad_rows);
  m.def("refresh_gamma", &refresh_gamma);
  m.def("mixer_forward", &mixer_forward);
  m.def("mixer_backward", &mixer_backward);
  m.def("norm_conv_forward", &norm_conv_forward);
  m.def("norm_conv_backward", &norm_conv_backward);
}
