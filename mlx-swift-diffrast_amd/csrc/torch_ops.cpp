// The differentiable ops as torch::autograd::Function nodes: argument
// checks, allocation of outputs and gradients, and the calls of the C ABI
// (include/diffrast_mi355x.h), whose library the Python layer names.
//
// Small calls are bound by the host: one triangle at 256^2, rasterize ->
// interpolate -> MSE and back, is nine launches of a few microseconds each,
// and the same nodes as Python autograd functions over ctypes calls took
// 112 to 173 us a pass, depending on the host (these: 70 to 98; one view of
// the textured chain at 512^2: 235 to 355, now 144 to 208).  Each op's
// semantics (checks, messages, reuse rules) are those of diffrast/ops.py's
// documentation.
#include <dlfcn.h>

#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/extension.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <string>
#include <tuple>
#include <vector>

#include "diffrast_mi355x.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::Variable;
using torch::autograd::variable_list;
using OptTensor = std::optional<Tensor>;

// ---- the C ABI ---------------------------------------------------------------

struct Api {
#define DR_FN(name) decltype(&::name) name = nullptr
  DR_FN(dr_get_last_error);
  DR_FN(dr_rasterize_fwd_ex);
  DR_FN(dr_rasterize_fwd_again);
  DR_FN(dr_rasterize_bwd);
  DR_FN(dr_interpolate_fwd);
  DR_FN(dr_interpolate_bwd);
  DR_FN(dr_interpolate_fwd_idx);
  DR_FN(dr_interpolate_bwd_idx);
  DR_FN(dr_texture_mip_levels);
  DR_FN(dr_texture_mip_size);
  DR_FN(dr_texture_build_mip);
  DR_FN(dr_texture_fwd);
  DR_FN(dr_texture_bwd);
  DR_FN(dr_antialias_topology);
  DR_FN(dr_antialias_fwd);
  DR_FN(dr_antialias_bwd);
  DR_FN(dr_antialias_saved_bytes);
  DR_FN(dr_antialias_fwd_save);
  DR_FN(dr_antialias_bwd_saved);
  DR_FN(dr_mse_loss);
#undef DR_FN
};
Api api;

void load_api(const std::string& path) {
  void* h = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
  TORCH_CHECK(h != nullptr, "diffrast: ", dlerror());
  Api a;
#define DR_FN(name)                                               \
  a.name = reinterpret_cast<decltype(a.name)>(dlsym(h, #name));   \
  TORCH_CHECK(a.name != nullptr, "diffrast: ", path, " has no " #name)
  DR_FN(dr_get_last_error);
  DR_FN(dr_rasterize_fwd_ex);
  DR_FN(dr_rasterize_fwd_again);
  DR_FN(dr_rasterize_bwd);
  DR_FN(dr_interpolate_fwd);
  DR_FN(dr_interpolate_bwd);
  DR_FN(dr_interpolate_fwd_idx);
  DR_FN(dr_interpolate_bwd_idx);
  DR_FN(dr_texture_mip_levels);
  DR_FN(dr_texture_mip_size);
  DR_FN(dr_texture_build_mip);
  DR_FN(dr_texture_fwd);
  DR_FN(dr_texture_bwd);
  DR_FN(dr_antialias_topology);
  DR_FN(dr_antialias_fwd);
  DR_FN(dr_antialias_bwd);
  DR_FN(dr_antialias_saved_bytes);
  DR_FN(dr_antialias_fwd_save);
  DR_FN(dr_antialias_bwd_saved);
  DR_FN(dr_mse_loss);
#undef DR_FN
  api = a;
}

void check(int rc) {
  if (rc == DR_OK) return;
  const std::string msg = api.dr_get_last_error();
  TORCH_CHECK_VALUE(rc != DR_ERR_ARGUMENT, msg);
  TORCH_CHECK(false, "diffrast error ", rc, ": ", msg);
}

// ---- helpers -------------------------------------------------------------------

dr_stream_t stream() { return (dr_stream_t)c10::hip::getCurrentHIPStream().stream(); }

const float* f(const Tensor& t) { return t.defined() ? (const float*)t.const_data_ptr() : nullptr; }
float* fm(const Tensor& t) { return t.defined() ? (float*)t.data_ptr() : nullptr; }
const int32_t* i32(const Tensor& t) { return t.defined() ? (const int32_t*)t.const_data_ptr() : nullptr; }

// Optional tensors: a node's optional inputs are given to apply() as
// std::optional (it takes every plain Tensor for a defined one).
Tensor opt(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }
OptTensor some(const Tensor& t) { return t.defined() ? OptTensor(t) : OptTensor(); }

// Differentiable conversion to contiguous float32 (the tensor itself when it
// is that already).
Tensor f32(const Tensor& t) { return t.to(at::kFloat).contiguous(); }

Tensor tri_of(const Tensor& t, at::Device dev) {
  return t.detach().to(dev, at::kInt).contiguous();
}

Tensor empty(at::IntArrayRef sizes, const Tensor& like) {
  return at::empty(sizes, like.options().dtype(at::kFloat).requires_grad(false).memory_format(
                              at::MemoryFormat::Contiguous));
}
Tensor zeros(at::IntArrayRef sizes, const Tensor& like) {
  return at::zeros(sizes, like.options().dtype(at::kFloat).requires_grad(false));
}
// A float32 buffer of t's shape with the standard contiguous strides, for a
// gradient returned to autograd: a size-1 dimension of the input may carry
// any stride, and autograd copies a returned gradient whose strides differ
// from the standard ones instead of keeping it as the leaf's .grad.
Tensor grad_buf(const Tensor& t) { return empty(t.sizes(), t); }

// An incoming cotangent, zeros where nothing reached the output.
Tensor cotangent(const Tensor& g, at::IntArrayRef sizes, const Tensor& like) {
  return g.defined() ? f32(g) : zeros(sizes, like);
}

// A side input is read by the kernels that run on the main input's device.
void check_device(const char* what, const Tensor& t, const Tensor& main) {
  TORCH_CHECK_VALUE(t.is_cuda() && t.device() == main.device(), what, " must be on the device of ",
                    "the other tensors (got ", t.device(), " and ", main.device(), ")");
}

void check_tri(const char* op, const Tensor& tri) {
  TORCH_CHECK_VALUE(tri.dim() == 2 && tri.size(1) == 3, op, ": tri must be [T, 3] (got ",
                    tri.sizes(), ")");
}

// ---- rasterize (Rasterize.swift:44-157) ------------------------------------------

using Where = std::pair<int, void*>;  // device, stream

Where place_of(const Tensor& t) {
  const auto d = t.device().index();
  return {(int)d, (void*)c10::hip::getCurrentHIPStream(d).stream()};
}

// The last rasterize call per (device, stream): the caller's pos and tri
// (weak references), read in place (no conversion copy), and their autograd
// versions.  A peel layer given the same tensors, unchanged since (same
// versions), reuses that call's triangle setup and tile lists
// (dr_rasterize_fwd_again, which also checks every pointer and size itself).
struct LastRaster {
  c10::weak_intrusive_ptr<c10::TensorImpl> pos, tri;
  int64_t pos_version, tri_version;
  std::vector<int64_t> pos_sizes, tri_sizes;
  int64_t N, H, W, max_per_tile;
  bool range;
  std::vector<int32_t> ranges;
};
// The last rasterize forward per (device, stream): its pos and tri buffers
// (storage, address, shape, strides) and pos's version.  A backward whose pos
// and tri are those buffers, pos at that version, differentiates a forward
// over the same data (autograd has checked that its saved pos is unchanged
// since its own forward; a later in-place change would have bumped the
// version), so it may reuse the per-triangle values the last forward stored
// (DR_RASTERIZE_BWD_REUSE; the peel layers of one pos all qualify).  The
// storages are weak references: an address alone may by then be that of
// another tensor (a hook on saved tensors brings pos back in new memory).
using WeakStorage = c10::weak_intrusive_ptr<c10::StorageImpl>;
struct FwdKey {
  WeakStorage pos_storage, tri_storage;
  const void *pos, *tri;
  int64_t version;
  std::vector<int64_t> pos_sizes, pos_strides, tri_sizes;
  bool operator==(const FwdKey& o) const {
    return pos_storage._unsafe_get_target() == o.pos_storage._unsafe_get_target() &&
           tri_storage._unsafe_get_target() == o.tri_storage._unsafe_get_target() &&
           pos == o.pos && tri == o.tri && version == o.version && pos_sizes == o.pos_sizes &&
           pos_strides == o.pos_strides && tri_sizes == o.tri_sizes;
  }
};
std::mutex g_mu;
std::map<Where, LastRaster> g_last_raster;
std::map<Where, FwdKey> g_last_fwd;

FwdKey fwd_key(const Tensor& pos, const Tensor& tri) {
  return {pos.storage().getWeakStorageImpl(), tri.storage().getWeakStorageImpl(),
          pos.const_data_ptr(), tri.const_data_ptr(), (int64_t)pos._version(), pos.sizes().vec(),
          pos.strides().vec(), tri.sizes().vec()};
}

struct RasterizeFn : torch::autograd::Function<RasterizeFn> {
  static variable_list forward(AutogradContext* ctx, const Variable& pos, const Tensor& tri,
                               const OptTensor& ranges_, const OptTensor& peel_, int64_t H,
                               int64_t W, bool grad_db, int64_t max_per_tile, bool again) {
    const Tensor ranges = opt(ranges_), peel = opt(peel_);
    const bool range = ranges.defined();
    const int64_t N = range ? ranges.size(0) : pos.size(0);
    const int64_t V = range ? pos.size(0) : pos.size(1), T = tri.size(0);
    Tensor rast = empty({N, H, W, 4}, pos);
    Tensor rast_db = empty({N, H, W, grad_db ? 4 : 0}, pos);
    auto fwd = again ? api.dr_rasterize_fwd_again : api.dr_rasterize_fwd_ex;
    check(fwd(f(pos), range ? 0 : V * 4, i32(tri), i32(ranges), f(peel), (int)N, (int)V, (int)T,
              (int)H, (int)W, fm(rast), grad_db ? fm(rast_db) : nullptr, (int)max_per_tile,
              stream()));
    {
      FwdKey key = fwd_key(pos, tri);
      std::lock_guard<std::mutex> lk(g_mu);
      g_last_fwd.insert_or_assign(place_of(pos), std::move(key));
    }
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({pos, tri, rast});
    ctx->saved_data["m"] = std::vector<int64_t>{range, N, V, H, W};
    return {rast, rast_db};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &pos = saved[0], &tri = saved[1], &rast = saved[2];
    const auto m = ctx->saved_data["m"].toIntVector();
    const Tensor d_rast = cotangent(g[0], rast.sizes(), rast);
    const Tensor db = g[1].defined() && g[1].size(3) == 4 ? f32(g[1]) : Tensor();
    Tensor d_pos = grad_buf(pos);
    unsigned flags = 0;
    {
      const FwdKey key = fwd_key(pos, tri);
      std::lock_guard<std::mutex> lk(g_mu);
      const auto it = g_last_fwd.find(place_of(pos));
      if (it != g_last_fwd.end() && it->second == key) flags = DR_RASTERIZE_BWD_REUSE;
    }
    check(api.dr_rasterize_bwd(f(pos), m[0] ? 0 : m[2] * 4, i32(tri), f(rast), f(d_rast), f(db),
                               (int)m[1], (int)m[2], (int)tri.size(0), (int)m[3], (int)m[4],
                               fm(d_pos), flags, stream()));
    return {d_pos, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

std::tuple<Tensor, Tensor> rasterize_op(const Tensor& pos, const Tensor& tri, int64_t H, int64_t W,
                                        bool grad_db, const OptTensor& ranges_cpu,
                                        const OptTensor& peel_layer, int64_t max_per_tile) {
  Tensor posf;
  if (pos.requires_grad()) {
    posf = pos.to(at::kFloat);
    TORCH_CHECK_VALUE(posf.is_cuda(), "rasterize: pos must be on a ROCm device");
  } else {
    TORCH_CHECK_VALUE(pos.is_cuda(), "rasterize: pos must be a tensor on a ROCm device");
    posf = pos.to(at::kFloat);
  }
  const Tensor tri32 = tri_of(tri, posf.device());
  check_tri("rasterize", tri32);
  const Tensor ranges = opt(ranges_cpu);
  int64_t N;
  if (ranges.defined()) {
    TORCH_CHECK_VALUE(posf.dim() == 2 && posf.size(1) == 4,
                      "rasterize: with `ranges`, pos must be [V, 4] (got ", posf.sizes(), ")");
    TORCH_CHECK_VALUE(ranges.dim() == 2 && ranges.size(1) == 2,
                      "rasterize: ranges must be [N, 2] (got ", ranges.sizes(), ")");
    TORCH_CHECK(ranges.device().is_cpu() && ranges.scalar_type() == at::kInt &&
                ranges.is_contiguous(), "rasterize: ranges must be contiguous int32 on the host");
    N = ranges.size(0);
  } else {
    TORCH_CHECK_VALUE(posf.dim() == 3 && posf.size(2) == 4, "rasterize: pos must be [N, V, 4] (got ",
                      posf.sizes(), ")");
    N = posf.size(0);
  }
  Tensor peel;
  if (peel_layer.has_value()) {
    TORCH_CHECK_VALUE(peel_layer->is_cuda(), "peelLayer must be a tensor on a ROCm device");
    peel = f32(peel_layer->detach());
    TORCH_CHECK_VALUE(peel.sizes() == at::IntArrayRef({N, H, W, 4}),
                      "rasterize: peelLayer must match rast shape [N, H, W, 4] (got ", peel.sizes(),
                      ")");
  }
  TORCH_CHECK_VALUE(0 <= max_per_tile && max_per_tile <= 1024,
                    "rasterize: maxPerTile must be in [0, 1024] (0: no limit)");
  const Tensor posc = posf.contiguous();
  // Reuse (peel layers only): the same pos and tri tensors as the previous
  // call on this stream, read in place and unchanged since.  (A transform's
  // wrapper has no storage: apply() refuses it by name.)
  const bool in_place = pos.has_storage() && tri32.has_storage() && tri.is_cuda() &&
                        posc.const_data_ptr() == pos.const_data_ptr() &&
                        tri32.const_data_ptr() == tri.const_data_ptr();
  const Where at_ = place_of(posc);
  bool again = false;
  int64_t pv = 0, tv = 0;
  const int32_t* rp = i32(ranges);
  const int64_t nr = ranges.defined() ? 2 * N : 0;
  if (in_place) {
    pv = (int64_t)pos._version();
    tv = (int64_t)tri._version();
    if (peel.defined()) {
      std::lock_guard<std::mutex> lk(g_mu);
      const auto it = g_last_raster.find(at_);
      if (it != g_last_raster.end()) {
        const LastRaster& L = it->second;
        // (a weak reference keeps the address from being given to another)
        again = L.pos._unsafe_get_target() == pos.unsafeGetTensorImpl() &&
                L.tri._unsafe_get_target() == tri.unsafeGetTensorImpl() && L.pos_version == pv &&
                L.tri_version == tv && at::IntArrayRef(L.pos_sizes) == pos.sizes() &&
                at::IntArrayRef(L.tri_sizes) == tri.sizes() && L.N == N && L.H == H && L.W == W &&
                L.max_per_tile == max_per_tile && L.range == ranges.defined() &&
                (int64_t)L.ranges.size() == nr && std::equal(L.ranges.begin(), L.ranges.end(), rp);
      }
    }
  }
  auto out = RasterizeFn::apply(posc, tri32, some(ranges), some(peel), H, W, grad_db, max_per_tile, again);
  {
    std::lock_guard<std::mutex> lk(g_mu);
    g_last_raster.erase(at_);
    if (in_place)
      g_last_raster.emplace(
          at_, LastRaster{c10::weak_intrusive_ptr<c10::TensorImpl>(pos.getIntrusivePtr()),
                          c10::weak_intrusive_ptr<c10::TensorImpl>(tri.getIntrusivePtr()), pv, tv,
                          pos.sizes().vec(), tri.sizes().vec(), N, H, W, max_per_tile,
                          ranges.defined(), std::vector<int32_t>(rp, rp + nr)});
  }
  return {out[0], out[1]};
}

// ---- interpolate (Interpolate.swift:43-132) ----------------------------------------

// diff: the attribute indices (empty: all of them when K = A); passed with
// the launch up to DR_INTERPOLATE_HOST_IDX, else read from diff_dev.
struct InterpolateFn : torch::autograd::Function<InterpolateFn> {
  static variable_list forward(AutogradContext* ctx, const Variable& attr, const Variable& rast,
                               const OptTensor& rast_db_, const Tensor& tri,
                               const std::vector<int64_t>& diff, const OptTensor& diff_dev_,
                               int64_t K, bool shared) {
    const Tensor rast_db = opt(rast_db_), diff_dev = opt(diff_dev_);
    const int64_t N = rast.size(0), H = rast.size(1), W = rast.size(2);
    const int64_t V = attr.size(-2), A = attr.size(-1), stride = shared ? 0 : V * A;
    Tensor out = empty({N, H, W, A}, rast), out_da = empty({N, H, W, 2 * K}, rast);
    const std::vector<int32_t> idx(diff.begin(), diff.end());
    const bool host = !idx.empty() && !diff_dev.defined();
    check((host ? api.dr_interpolate_fwd_idx : api.dr_interpolate_fwd)(
        f(attr), stride, f(rast), f(rast_db), i32(tri), host ? idx.data() : i32(diff_dev), (int)K,
        (int)N, (int)H, (int)W, (int)V, (int)tri.size(0), (int)A, fm(out), K ? fm(out_da) : nullptr,
        stream()));
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({attr, rast, rast_db, tri, diff_dev});
    ctx->saved_data["k"] = K;
    ctx->saved_data["s"] = shared;
    if (host) ctx->saved_data["d"] = diff;
    return {out, out_da};
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &attr = saved[0], &rast = saved[1], &rast_db = saved[2], &tri = saved[3],
                 &diff_dev = saved[4];
    const int64_t K = ctx->saved_data["k"].toInt();
    const bool shared = ctx->saved_data["s"].toBool();
    std::vector<int32_t> idx;
    const auto d = ctx->saved_data.find("d");
    if (d != ctx->saved_data.end())
      for (const int64_t i : d->second.toIntVector()) idx.push_back((int32_t)i);
    const int64_t N = rast.size(0), H = rast.size(1), W = rast.size(2);
    const int64_t V = attr.size(-2), A = attr.size(-1), stride = shared ? 0 : V * A;
    const Tensor d_out = cotangent(g[0], {N, H, W, A}, rast);
    const Tensor d_out_da = K ? cotangent(g[1], {N, H, W, 2 * K}, rast) : Tensor();
    Tensor d_attr = grad_buf(attr), d_rast = grad_buf(rast);
    Tensor d_rast_db = K ? grad_buf(rast) : Tensor();
    check((!idx.empty() ? api.dr_interpolate_bwd_idx : api.dr_interpolate_bwd)(
        f(attr), stride, f(rast), f(rast_db), i32(tri), !idx.empty() ? idx.data() : i32(diff_dev),
        (int)K, f(d_out), f(d_out_da), (int)N, (int)H, (int)W, (int)V, (int)tri.size(0), (int)A,
        fm(d_attr), stride, fm(d_rast), fm(d_rast_db), 0, stream()));
    return {d_attr, d_rast, d_rast_db, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// mode 0: no derivatives; 1: of all attributes; 2: of those in `diff`.
std::tuple<Tensor, Tensor> interpolate_op(const Tensor& attr, const Tensor& rast,
                                          const Tensor& tri, const OptTensor& rast_db, int mode,
                                          const std::vector<int64_t>& diff) {
  TORCH_CHECK_VALUE(rast.dim() == 4 && rast.size(3) == 4,
                    "interpolate: rast must be [N, H, W, 4] (got ", rast.sizes(), ")");
  TORCH_CHECK_VALUE(attr.dim() == 2 || attr.dim() == 3,
                    "interpolate: attr must be [V, A] or [N, V, A] (got ", attr.sizes(), ")");
  const int64_t N = rast.size(0), A = attr.size(-1);
  const Tensor tri32 = tri_of(tri, rast.device());
  check_tri("interpolate", tri32);
  TORCH_CHECK_VALUE(attr.dim() == 2 || attr.size(0) == 1 || attr.size(0) == N,
                    "interpolate: attr batch dim ", attr.size(0), " incompatible with rast batch ",
                    N);
  const bool shared = attr.dim() == 2 || (attr.size(0) == 1 && N != 1);
  TORCH_CHECK_VALUE(rast.is_cuda() && attr.is_cuda(), "interpolate: tensors must be on a ROCm device");
  const Tensor rastf = f32(rast), attrf = f32(attr);
  if (mode == 0) {
    auto out = InterpolateFn::apply(attrf, rastf, OptTensor(), tri32, std::vector<int64_t>(),
                                    OptTensor(), (int64_t)0, shared);
    return {out[0], empty({N, rast.size(1), rast.size(2), 0}, rastf)};
  }
  TORCH_CHECK_VALUE(rast_db.has_value(), "interpolate: rastDB is required when diffAttrs is set");
  TORCH_CHECK_VALUE(rast_db->sizes() == rast.sizes(), "interpolate: rastDB must match rast shape (got ",
                    rast_db->sizes(), " vs ", rast.sizes(), ")");
  check_device("interpolate: rastDB", *rast_db, rast);
  Tensor diff_dev;
  if (mode == 2) {
    TORCH_CHECK_VALUE(!diff.empty(), "interpolate: diffAttrs.indices must be non-empty");
    for (const int64_t i : diff)
      TORCH_CHECK_VALUE(0 <= i && i < A, "interpolate: diffAttrs.indices values must be in [0, A) (A=",
                        A, ")");
    if (diff.size() > DR_INTERPOLATE_HOST_IDX)
      diff_dev = at::tensor(diff, at::TensorOptions().dtype(at::kInt)).to(rast.device());
  }
  auto out = InterpolateFn::apply(attrf, rastf, OptTensor(f32(*rast_db)), tri32, diff, some(diff_dev),
                                  mode == 1 ? A : (int64_t)diff.size(), shared);
  return {out[0], out[1]};
}

// ---- texture (Texture.swift:62-327) ---------------------------------------------------

struct TextureFn : torch::autograd::Function<TextureFn> {
  static Tensor forward(AutogradContext* ctx, const Variable& tex, const Variable& uv,
                        const OptTensor& uv_da_, const OptTensor& bias_map_, int64_t filt,
                        int64_t boundary, double bias, int64_t levels, const OptTensor& pyramid_,
                        bool dir_grad) {
    const Tensor uv_da = opt(uv_da_), bias_map = opt(bias_map_), pyramid = opt(pyramid_);
    const bool cube = boundary == DR_BOUNDARY_CUBE;
    const int64_t N = uv.size(0), Hi = uv.size(1), Wi = uv.size(2), Nt = tex.size(0);
    const int64_t Ht = tex.size(cube ? 2 : 1), Wt = tex.size(cube ? 3 : 2), C = tex.size(cube ? 4 : 3);
    int64_t L = 1;
    Tensor pyr;
    if (filt >= DR_FILTER_LINEAR_MIPMAP_NEAREST && pyramid.defined()) {
      L = levels;
      pyr = pyramid;
    } else if (filt >= DR_FILTER_LINEAR_MIPMAP_NEAREST) {
      const int64_t faces = cube ? Nt * 6 : Nt;  // a cube map's pyramid: every face's
      L = api.dr_texture_mip_levels((int)Ht, (int)Wt, -1, nullptr, nullptr);
      const int64_t size = api.dr_texture_mip_size((int)faces, (int)Ht, (int)Wt, (int)C, (int)L);
      pyr = empty({std::max<int64_t>(size, 1)}, tex);
      check(api.dr_texture_build_mip(f(tex), (int)faces, (int)Ht, (int)Wt, (int)C, (int)L, fm(pyr),
                                     stream()));
    }
    Tensor out = empty({N, Hi, Wi, C}, uv);
    check(api.dr_texture_fwd(f(tex), f(pyr), (int)Nt, (int)Ht, (int)Wt, (int)C, (int)L, f(uv),
                             f(uv_da), f(bias_map), (float)bias, (int)filt, (int)boundary, (int)N,
                             (int)Hi, (int)Wi, fm(out), stream()));
    const bool want[3] = {uv.requires_grad(), uv_da.defined() && uv_da.requires_grad(),
                          bias_map.defined() && bias_map.requires_grad()};
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({tex, uv, uv_da, bias_map, pyr});
    ctx->saved_data["m"] = std::vector<int64_t>{filt, boundary, L, Nt, Ht, Wt, C, dir_grad, want[0],
                                                want[1], want[2]};
    ctx->saved_data["b"] = bias;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &tex = saved[0], &uv = saved[1], &uv_da = saved[2], &bias_map = saved[3],
                 &pyr = saved[4];
    const auto m = ctx->saved_data["m"].toIntVector();
    const int64_t N = uv.size(0), Hi = uv.size(1), Wi = uv.size(2);
    const Tensor d_out = cotangent(g[0], {N, Hi, Wi, m[6]}, uv);
    Tensor d_tex = grad_buf(tex);
    Tensor d_uv = m[8] ? grad_buf(uv) : Tensor();
    Tensor d_uv_da = m[9] ? grad_buf(uv_da) : Tensor();
    Tensor d_bias = m[10] ? grad_buf(bias_map) : Tensor();
    check(api.dr_texture_bwd(f(tex), f(pyr), (int)m[3], (int)m[4], (int)m[5], (int)m[6], (int)m[2],
                             f(uv), f(uv_da), f(bias_map), (float)ctx->saved_data["b"].toDouble(),
                             (int)m[0], (int)m[1], (int)N, (int)Hi, (int)Wi, f(d_out), fm(d_tex),
                             fm(d_uv), fm(d_uv_da), fm(d_bias), m[7] ? DR_CUBE_DIR_GRAD : 0u,
                             stream()));
    return {d_tex,    d_uv,     d_uv_da,  d_bias,   Tensor(),
            Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// Texture.swift:104-108: [N, H_img, W_img] or [N, H_img, W_img, 1].
Tensor bias_map_of(const OptTensor& m, const Tensor& uv) {
  if (!m.has_value()) return Tensor();
  TORCH_CHECK_VALUE((m->dim() == 3 || (m->dim() == 4 && m->size(3) == 1)) &&
                        m->sizes().slice(0, 3) == uv.sizes().slice(0, 3),
                    "texture: mipLevelBiasMap must be [N, H_img, W_img] or [N, H_img, W_img, 1] (got ",
                    m->sizes(), ")");
  check_device("texture: mipLevelBiasMap", *m, uv);
  return f32(*m);
}

// levels / pyramid: a prebuilt pyramid (2D mip filters), else undefined.
Tensor texture_op(const Tensor& tex, const Tensor& uv, const OptTensor& uv_da, int64_t filt,
                  int64_t boundary, double bias, const OptTensor& bias_map, int64_t levels,
                  const OptTensor& pyramid, bool dir_grad) {
  const Tensor texf = f32(tex), uvf = f32(uv);
  TORCH_CHECK_VALUE(texf.is_cuda() && uvf.is_cuda(), "texture: tensors must be on a ROCm device");
  const bool mip = filt >= DR_FILTER_LINEAR_MIPMAP_NEAREST;
  const bool da_fits = uv_da.has_value() && uv_da->dim() == 4 && uvf.dim() == 4 &&
                       uv_da->sizes().slice(0, 3) == uvf.sizes().slice(0, 3);
  if (boundary == DR_BOUNDARY_CUBE) {
    TORCH_CHECK_VALUE(filt != DR_FILTER_NEAREST,
                      "texture: cube textures support the linear and mipmap filterModes");
    TORCH_CHECK_VALUE(texf.dim() == 5 && texf.size(1) == 6,
                      "texture: cube tex must be [N, 6, H, W, C] (got ", texf.sizes(), ")");
    TORCH_CHECK_VALUE(uvf.dim() == 4 && uvf.size(3) == 3,
                      "texture: cube uv must be [N, H_img, W_img, 3] direction vector (got ",
                      uvf.sizes(), ")");
    TORCH_CHECK_VALUE(texf.size(0) == 1 || texf.size(0) == uvf.size(0),
                      "texture: tex batch dim incompatible with uv batch");
    TORCH_CHECK_VALUE(!pyramid.has_value(), "texture: a prebuilt `mip` is for 2D textures");
    if (!mip)
      return TextureFn::apply(texf, uvf, OptTensor(), OptTensor(), filt, boundary, 0.0, (int64_t)0,
                              OptTensor(), dir_grad);
    TORCH_CHECK_VALUE(da_fits && uv_da->size(3) == 6,
                      "texture: cube mipmap filterModes require uvDA [N, H_img, W_img, 6] "
                      "(direction derivatives)");
    check_device("texture: uvDA", *uv_da, uvf);
    return TextureFn::apply(texf, uvf, OptTensor(f32(*uv_da)), some(bias_map_of(bias_map, uvf)),
                            filt, boundary, bias, (int64_t)0, OptTensor(), dir_grad);
  }
  TORCH_CHECK_VALUE(texf.dim() == 4, "texture: tex must be [N, H_tex, W_tex, C] (got ", texf.sizes(),
                    ")");
  TORCH_CHECK_VALUE(uvf.dim() == 4 && uvf.size(3) == 2,
                    "texture: uv must be [N, H_img, W_img, 2] (got ", uvf.sizes(), ")");
  TORCH_CHECK_VALUE(texf.size(0) == 1 || texf.size(0) == uvf.size(0), "texture: tex batch dim ",
                    texf.size(0), " incompatible with uv batch ", uvf.size(0));
  if (!mip)
    return TextureFn::apply(texf, uvf, OptTensor(), OptTensor(), filt, boundary, 0.0, (int64_t)0,
                            OptTensor(), false);
  TORCH_CHECK_VALUE(uv_da.has_value(), "texture: mipmap filterModes require uvDA");
  TORCH_CHECK_VALUE(da_fits && uv_da->size(3) == 4,
                    "texture: uvDA must be [N, H_img, W_img, 4] (got ", uv_da->sizes(), ")");
  check_device("texture: uvDA", *uv_da, uvf);
  return TextureFn::apply(texf, uvf, OptTensor(f32(*uv_da)), some(bias_map_of(bias_map, uvf)), filt,
                          boundary, bias, levels, pyramid, false);
}

// ---- antialias (Antialias.swift:90-131) -------------------------------------------------

struct AntialiasFn : torch::autograd::Function<AntialiasFn> {
  static Tensor forward(AutogradContext* ctx, const Variable& color, const Variable& pos,
                        const Tensor& rast, const Tensor& tri, const Tensor& topo) {
    const int64_t N = color.size(0), H = color.size(1), W = color.size(2), C = color.size(3);
    const int64_t V = pos.size(1), T = tri.size(0);
    Tensor out = empty(color.sizes(), color), saved;
    const bool want[2] = {color.requires_grad(), pos.requires_grad()};
    if (want[0] || want[1]) {
      // the saved state (blend mask, edge records) spares the backward the
      // pixels without blends and the per-triangle setup
      saved = at::empty({api.dr_antialias_saved_bytes((int)N, (int)H, (int)W, (int)T)},
                        color.options().dtype(at::kByte).requires_grad(false));
      check(api.dr_antialias_fwd_save(f(color), f(rast), f(pos), i32(tri), i32(topo), (int)N, (int)H,
                                      (int)W, (int)C, (int)V, (int)T, fm(out), saved.data_ptr(),
                                      stream()));
    } else {
      check(api.dr_antialias_fwd(f(color), f(rast), f(pos), i32(tri), i32(topo), (int)N, (int)H,
                                 (int)W, (int)C, (int)V, (int)T, fm(out), stream()));
    }
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({color, pos, rast, tri, topo, saved});
    ctx->saved_data["m"] = std::vector<int64_t>{want[0], want[1]};
    return out;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const auto s = ctx->get_saved_variables();
    const Tensor &color = s[0], &pos = s[1], &rast = s[2], &tri = s[3], &topo = s[4], &saved = s[5];
    const auto m = ctx->saved_data["m"].toIntVector();
    const int64_t N = color.size(0), H = color.size(1), W = color.size(2), C = color.size(3);
    const int64_t V = pos.size(1), T = tri.size(0);
    const Tensor d_out = cotangent(g[0], color.sizes(), color);
    Tensor d_color = m[0] ? grad_buf(color) : Tensor(), d_pos = m[1] ? grad_buf(pos) : Tensor();
    if (saved.defined())
      check(api.dr_antialias_bwd_saved(f(color), f(rast), f(pos), i32(tri), i32(topo), f(d_out),
                                       saved.const_data_ptr(), (int)N, (int)H, (int)W, (int)C, (int)V,
                                       (int)T, fm(d_color), fm(d_pos), 0, stream()));
    else
      check(api.dr_antialias_bwd(f(color), f(rast), f(pos), i32(tri), i32(topo), f(d_out), (int)N,
                                 (int)H, (int)W, (int)C, (int)V, (int)T, fm(d_color), fm(d_pos), 0,
                                 stream()));
    return {d_color, d_pos, Tensor(), Tensor(), Tensor()};
  }
};

// topo undefined: built here.
Tensor antialias_op(const Tensor& color, const Tensor& rast, const Tensor& pos, const Tensor& tri,
                    const OptTensor& topology) {
  TORCH_CHECK_VALUE(color.dim() == 4, "antialias: color must be [N, H, W, C] (got ", color.sizes(),
                    ")");
  TORCH_CHECK_VALUE(rast.dim() == 4 && rast.size(3) == 4 &&
                        rast.sizes().slice(0, 3) == color.sizes().slice(0, 3),
                    "antialias: rast must match color in [N, H, W] and have 4 channels");
  TORCH_CHECK_VALUE(pos.dim() == 3 && pos.size(2) == 4, "antialias: pos must be [N, V, 4] (got ",
                    pos.sizes(), ")");
  TORCH_CHECK_VALUE(color.is_cuda() && rast.is_cuda() && pos.is_cuda(),
                    "antialias: tensors must be on a ROCm device");
  // (read per image and per triangle)
  TORCH_CHECK_VALUE(pos.size(0) >= color.size(0), "antialias: pos must have color's batch (got ",
                    pos.sizes(), " for ", color.size(0), " images)");
  const Tensor tri32 = tri_of(tri, color.device());
  check_tri("antialias", tri32);
  Tensor topo;
  if (topology.has_value()) {
    topo = tri_of(*topology, color.device());
    TORCH_CHECK_VALUE(topo.numel() >= tri32.numel(), "antialias: topologyHash must be [T, 3] (got ",
                      topo.sizes(), " for ", tri32.size(0), " triangles)");
  } else {
    topo = at::empty_like(tri32);
    check(api.dr_antialias_topology(i32(tri32), (int)tri32.size(0), (int32_t*)topo.data_ptr(),
                                    stream()));
  }
  return AntialiasFn::apply(f32(color), f32(pos), f32(rast.detach()), tri32, topo);
}

// ---- MSE loss (ColorFitExample/main.swift:62-66) -----------------------------------------

struct MseFn : torch::autograd::Function<MseFn> {
  static Tensor forward(AutogradContext* ctx, const Variable& out, const Tensor& target) {
    Tensor loss = empty({}, out);
    Tensor d_out = out.requires_grad() ? grad_buf(out) : Tensor();
    check(api.dr_mse_loss(f(out), f(target), out.numel(), fm(loss), fm(d_out), stream()));
    ctx->set_materialize_grads(false);
    ctx->save_for_backward({d_out});
    return loss;
  }
  static variable_list backward(AutogradContext* ctx, const variable_list& g) {
    const auto s = ctx->get_saved_variables();
    return {g[0].defined() ? s[0] * g[0] : Tensor(), Tensor()};
  }
};

Tensor mse_loss_op(const Tensor& out, const Tensor& target) {
  TORCH_CHECK_VALUE(out.sizes() == target.sizes(), "mse_loss: shapes differ (", out.sizes(), " vs ",
                    target.sizes(), ")");
  TORCH_CHECK_VALUE(out.is_cuda() && target.is_cuda(), "mse_loss: tensors must be on a ROCm device");
  TORCH_CHECK_VALUE(out.numel() != 0, "mse_loss: empty tensors");
  return MseFn::apply(f32(out), f32(target.detach()));
}

}  // namespace

PYBIND11_MODULE(_torch_ops, m) {
  m.def("load", torch::wrap_pybind_function_no_gil(load_api));
  m.def("rasterize", torch::wrap_pybind_function_no_gil(rasterize_op));
  m.def("interpolate", torch::wrap_pybind_function_no_gil(interpolate_op));
  m.def("texture", torch::wrap_pybind_function_no_gil(texture_op));
  m.def("antialias", torch::wrap_pybind_function_no_gil(antialias_op));
  m.def("mse_loss", torch::wrap_pybind_function_no_gil(mse_loss_op));
}
