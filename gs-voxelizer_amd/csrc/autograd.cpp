// autograd.cpp — the projection's and the voxelization's autograd nodes, native.
//
// The same steps as the Python classes of optim_to_render.py and voxelize.py
// (allocate the outputs, enqueue the library's entry points on the current
// stream, save what the backward reads), without the interpreter: a Python
// autograd.Function costs ~24 us a forward and takes the interpreter from the
// engine's thread in the backward, and the step at 128^3 / 50k, whose kernels
// take 130 us, spent 380 us on the host.  Only plain calls come here; the Python
// modules keep everything else (first calls, graph capture, transforms, odd
// inputs and every error message).  Nothing is kept between calls.
//
// libgsvox.so is loaded by _lib.py; its entry points are handed over once by
// address (bind), so this file links against torch alone.
#include <torch/extension.h>

#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include <atomic>
#include <map>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/gsvox.h"
#include "gsv_numerics.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// The library's entry points (gsvox.h), set by bind().
#define GSV_ENTRIES(X)                                                                            \
    X(gsv_status_string) X(gsv_last_hip_error) X(gsv_project_fwd) X(gsv_project_bwd)               \
    X(gsv_cumsum_bin_workspace_bytes) X(gsv_cumsum_bin_and_sort_device_count) X(gsv_voxelize_fwd)  \
    X(gsv_voxelize_fwd_l1_workspace_bytes) X(gsv_voxelize_fwd_l1)                                  \
    X(gsv_voxelize_bwd_workspace_bytes) X(gsv_voxelize_bwd) X(gsv_voxelize_bwd_l1)
struct Library {
#define GSV_FIELD(name) decltype(&::name) name = nullptr;
    GSV_ENTRIES(GSV_FIELD)
#undef GSV_FIELD
} lib;

void bind(const std::map<std::string, uintptr_t> &addresses) {
#define GSV_BIND(name) lib.name = reinterpret_cast<decltype(&::name)>(addresses.at(#name));
    GSV_ENTRIES(GSV_BIND)
#undef GSV_BIND
}

void check(int status, const char *name) {
    if (status == GSV_OK) return;
    std::string text = lib.gsv_status_string(status);
    if (status == GSV_ERR_HIP)
        text += " (hipError_t " + std::to_string(lib.gsv_last_hip_error()) + ")";
    TORCH_CHECK(false, "gs_voxelizer.", name, ": ", text);
}

template <class T>
T *ptr(const Tensor &t) {
    return t.defined() && t.numel() > 0 ? static_cast<T *>(t.data_ptr()) : nullptr;
}

void *stream_of(const Tensor &t) {
    return reinterpret_cast<void *>(c10::hip::getCurrentHIPStream(t.get_device()).stream());
}

Tensor empty(at::IntArrayRef size, const Tensor &like, at::ScalarType type) {
    return at::empty(size, at::TensorOptions().device(like.device()).dtype(type));
}

Tensor workspace(size_t bytes, const Tensor &like) {
    return empty({(int64_t)std::max<size_t>(bytes, 1)}, like, at::kByte);
}

struct Volume {
    int D, H, W;
    int64_t tiles() const {
        return (int64_t)gsv_tiles_along(D) * gsv_tiles_along(H) * gsv_tiles_along(W);
    }
};

struct World {
    float wz, wy, wx, cz, cy, cx;
};

// A contiguous tensor of this type, row width and count on `dev`.
bool is_rows(const Tensor &t, at::ScalarType type, const at::Device &dev, int64_t n, int64_t width) {
    return t.defined() && t.layout() == at::kStrided && t.scalar_type() == type &&
           t.device() == dev && t.dim() == 2 && t.size(0) == n && t.size(1) == width &&
           t.is_contiguous();
}

bool is_vector(const Tensor &t, at::ScalarType type, const at::Device &dev, int64_t n) {
    return t.defined() && t.layout() == at::kStrided && t.scalar_type() == type &&
           t.device() == dev && t.dim() == 1 && t.size(0) == n && t.is_contiguous();
}

// A tensor that a backward reads, as it comes back from the saved-tensor hooks,
// which may hand over any other one.
Tensor unpacked(const Tensor &t, at::ScalarType type, const at::Device &dev, int64_t numel,
                const char *what) {
    TORCH_CHECK(t.defined() && t.layout() == at::kStrided && t.scalar_type() == type &&
                    t.device() == dev && t.numel() == numel,
                what, ": expected ", numel, " values of scalar type ", type, " on ", dev);
    return t.contiguous();
}

// The device that a forward ran on, kept as its index.
at::Device gpu(int64_t index) {
    return at::Device(at::kCUDA, (at::DeviceIndex)index);
}

bool fits(int64_t D, int64_t H, int64_t W) {
    constexpr int64_t most = 1 << 20;
    return D > 0 && H > 0 && W > 0 && D <= most && H <= most && W <= most;
}

// ------------------------------------------------------------- projection --

struct Projected {
    Tensor pos_radii, conics, tile_min, tile_max, hits;
};

struct Project : public torch::autograd::Function<Project> {
    // The intensities get no gradient from here, but make the outputs require one.
    static variable_list forward(AutogradContext *ctx, const Tensor &pos, const Tensor &scale,
                                 const Tensor &quat, const Tensor &, const Volume *vol,
                                 const World *world, const Projected *out) {
        ctx->saved_data["vol"] =
            std::vector<int64_t>{vol->D, vol->H, vol->W, pos.size(0), pos.get_device()};
        ctx->saved_data["world"] = std::vector<double>{world->wz, world->wy, world->wx,
                                                       world->cz, world->cy, world->cx};
        ctx->save_for_backward({pos, scale, quat, out->pos_radii});
        ctx->mark_non_differentiable({out->tile_min, out->tile_max, out->hits});
        ctx->set_materialize_grads(false);
        return {out->pos_radii, out->conics, out->tile_min, out->tile_max, out->hits};
    }

    static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
        const auto saved = ctx->get_saved_variables();
        const auto vol = ctx->saved_data["vol"].toIntVector();
        const auto w = ctx->saved_data["world"].toDoubleVector();
        const int64_t n = vol[3];
        const at::Device dev = gpu(vol[4]);
        const c10::DeviceGuard guard(dev);
        const Tensor pos = unpacked(saved[0], at::kFloat, dev, n * 3, "pos3d");
        const Tensor scale = unpacked(saved[1], at::kFloat, dev, n * 3, "scale3d");
        const Tensor quat = unpacked(saved[2], at::kFloat, dev, n * 4, "quat");
        const Tensor pos_radii = unpacked(saved[3], at::kFloat, dev, n * 4, "pos3d_radii");
        const auto given = [&](const Tensor &g, int64_t width, const char *what) {
            if (!g.defined()) return at::zeros({n, width}, pos_radii.options());
            TORCH_CHECK(g.device() == dev && g.scalar_type() == at::kFloat && g.numel() == n * width,
                        what, ": expected ", n, " rows of ", width, " float32 values on the GPU");
            return g.contiguous();
        };
        const Tensor dpr = given(grads[0], 4, "pos3d_radii_grad_in");
        const Tensor dcn = given(grads[1], 6, "conics_grad_in");
        Tensor dpos = empty({n, 3}, pos, at::kFloat), dscale = empty({n, 3}, pos, at::kFloat);
        Tensor dquat = empty({n, 4}, pos, at::kFloat);
        check(lib.gsv_project_bwd((int)n, ptr<float>(pos), ptr<float>(scale),
                                  ptr<float>(quat), (int)vol[0], (int)vol[1], (int)vol[2],
                                  (float)w[0], (float)w[1], (float)w[2], (float)w[3], (float)w[4],
                                  (float)w[5], ptr<float>(dpr), ptr<float>(dcn),
                                  ptr<float>(pos_radii), ptr<float>(dpos), ptr<float>(dscale),
                                  ptr<float>(dquat), stream_of(pos)),
              "project_bwd");
        return {dpos, dscale, dquat, Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// optim_to_render's outputs, or nothing for a call that the Python class takes.
std::vector<Tensor> project(const Tensor &pos, const Tensor &scale, const Tensor &quat,
                            const Tensor &intens, int64_t D, int64_t H, int64_t W, double wz,
                            double wy, double wx, double cz, double cy, double cx) {
    if (!pos.defined() || !pos.is_cuda() || pos.dim() != 2 || !fits(D, H, W)) return {};
    const int64_t n = pos.size(0);
    const at::Device dev = pos.device();
    if (n < 1 || n > INT32_MAX || !is_rows(pos, at::kFloat, dev, n, 3) ||
        !is_rows(scale, at::kFloat, dev, n, 3) || !is_rows(quat, at::kFloat, dev, n, 4) ||
        intens.dim() != 2 || intens.size(1) < 1 || intens.size(1) > GSV_MAX_CHANNELS ||
        !is_rows(intens, at::kFloat, dev, n, intens.size(1)))
        return {};
    const c10::DeviceGuard guard(dev);
    const Volume vol{(int)D, (int)H, (int)W};
    const World world{(float)wz, (float)wy, (float)wx, (float)cz, (float)cy, (float)cx};
    Projected out;
    out.pos_radii = empty({n, 4}, pos, at::kFloat);
    out.conics = empty({n, 6}, pos, at::kFloat);
    out.tile_min = empty({n, 3}, pos, at::kInt);
    out.tile_max = empty({n, 3}, pos, at::kInt);
    out.hits = empty({n}, pos, at::kInt);
    check(lib.gsv_project_fwd((int)n, (int)intens.size(1), ptr<float>(pos), ptr<float>(scale),
                              ptr<float>(quat), ptr<float>(intens), vol.D, vol.H, vol.W, world.wz,
                              world.wy, world.wx, world.cz, world.cy, world.cx,
                              ptr<float>(out.pos_radii), ptr<float>(out.conics),
                              ptr<int32_t>(out.tile_min), ptr<int32_t>(out.tile_max),
                              ptr<int32_t>(out.hits), stream_of(pos)),
          "project_fwd");
    return Project::apply(pos, scale, quat, intens, &vol, &world, &out);
}

// ----------------------------------------------------------- voxelization --

struct Voxelized {
    Tensor volume, loss, sign;  // loss and sign: the fused L1 step only
    Tensor ids, bins, tiles, cum, live, tile_min, tile_max;
    int64_t count = -1;
};

// What a node keeps beside its tensors.
struct Kept {
    Volume vol;
    int64_t count, cap, n, channels, device;
    bool per_gaussian;

    explicit Kept(const std::vector<int64_t> &m)
        : vol{(int)m[0], (int)m[1], (int)m[2]}, count(m[3]), cap(m[4]), n(m[5]), channels(m[6]),
          device(m[7]), per_gaussian(m[8] != 0) {}
    int64_t voxels() const { return (int64_t)vol.D * vol.H * vol.W; }
};

// The backward of both nodes; grad_loss is undefined without the loss.
variable_list voxelize_backward(const Kept &k, const variable_list &saved, const Tensor &grad_loss,
                                const Tensor &grad_volume) {
    const Volume &vol = k.vol;
    const int64_t count = k.count;
    const int n = (int)k.n, C = (int)k.channels;
    const at::Device dev = gpu(k.device);
    const Tensor pr = unpacked(saved[0], at::kFloat, dev, k.n * 4, "pos3d_radii");
    const Tensor cn = unpacked(saved[1], at::kFloat, dev, k.n * 6, "conics");
    const Tensor intens = unpacked(saved[2], at::kFloat, dev, k.n * C, "intensities");
    const Tensor ids = unpacked(saved[3], at::kInt, dev, count, "gaussian_ids_sorted");
    const Tensor bins = unpacked(saved[4], at::kInt, dev, vol.tiles() * 2, "tile_bins");
    size_t next = 5;
    Tensor sign;
    if (grad_loss.defined()) sign = unpacked(saved[next++], at::kChar, dev, k.voxels() * C, "sign");
    const Tensor tile_min = unpacked(saved[next++], at::kInt, dev, k.n * 3, "tile_min");
    const Tensor tile_max = unpacked(saved[next++], at::kInt, dev, k.n * 3, "tile_max");
    const Tensor cum = unpacked(saved[next++], at::kInt, dev, k.n, "cum_tiles_hit");
    const Tensor tiles = unpacked(saved[next++], at::kInt, dev, count, "tiles_sorted");
    const Tensor live = unpacked(saved[next++], at::kByte, dev, k.cap, "pair_live");
    Tensor vg;
    if (grad_volume.defined()) {
        vg = grad_volume.contiguous();
        TORCH_CHECK(vg.device() == dev, "vol_grad_in must be a CUDA tensor on ", dev);
        TORCH_CHECK(vg.scalar_type() == at::kFloat, "vol_grad_in: expected scalar type float32");
        TORCH_CHECK(vg.numel() == k.voxels() * C,
                    "vol_grad_in must have D*H*W*channels elements");
    }
    Tensor dpos = empty({n, 4}, pr, at::kFloat), dconics = empty({n, 6}, pr, at::kFloat);
    Tensor dint = empty({n, C}, pr, at::kFloat);
    size_t bytes = 0;
    check(lib.gsv_voxelize_bwd_workspace_bytes(vol.D, vol.H, vol.W, C, n, count, 1, &bytes),
          "voxelize_bwd_workspace_bytes");
    const Tensor ws = workspace(bytes, pr);
    void *stream = stream_of(pr);
    const int variant = k.per_gaussian ? 1 : 0;
    if (sign.defined()) {
        TORCH_CHECK(grad_loss.device() == dev && grad_loss.scalar_type() == at::kFloat &&
                        grad_loss.numel() == 1,
                    "grad_loss must be one float32 value on the GPU");
        const Tensor gl = grad_loss.contiguous();
        check(lib.gsv_voxelize_bwd_l1(
                  vol.D, vol.H, vol.W, C, n, count, ptr<int32_t>(ids), ptr<int32_t>(bins),
                  ptr<float>(pr), ptr<float>(cn), ptr<float>(intens), ptr<int8_t>(sign),
                  ptr<float>(gl), ptr<float>(vg), ptr<int32_t>(tile_min), ptr<int32_t>(tile_max),
                  ptr<int32_t>(cum), ptr<int32_t>(tiles), nullptr, ptr<uint8_t>(live),
                  ptr<float>(dpos), ptr<float>(dconics), ptr<float>(dint), variant,
                  ptr<void>(ws), bytes, stream),
              "voxelize_bwd_l1");
    } else {
        check(lib.gsv_voxelize_bwd(
                  vol.D, vol.H, vol.W, C, n, count, ptr<int32_t>(ids), ptr<int32_t>(bins),
                  ptr<float>(pr), ptr<float>(cn), ptr<float>(intens), ptr<float>(vg),
                  ptr<int32_t>(tile_min), ptr<int32_t>(tile_max), ptr<int32_t>(cum),
                  ptr<int32_t>(tiles), nullptr, ptr<uint8_t>(live), ptr<float>(dpos),
                  ptr<float>(dconics), ptr<float>(dint), variant, ptr<void>(ws), bytes, stream),
              "voxelize_bwd");
    }
    return {dpos, dconics, dint};
}

variable_list zero_gradients(const Kept &k) {
    const auto options = at::TensorOptions().device(gpu(k.device)).dtype(at::kFloat);
    return {at::zeros({k.n, 4}, options), at::zeros({k.n, 6}, options),
            at::zeros({k.n, k.channels}, options)};
}

// The tensors, shapes and order that the classes save: a checkpointed forward on
// one route may be computed again on the other.
variable_list saved_tensors(const Tensor &pr, const Tensor &cn, const Tensor &intens,
                            const Voxelized &v) {
    if (v.count == 0) {
        if (v.sign.defined()) return {pr, cn, intens, empty({0}, pr, at::kInt), v.bins, v.sign};
        return {pr, cn, intens, empty({0, 1}, pr, at::kInt), empty({0, 3}, pr, at::kInt)};
    }
    // (no other tensor shares these two, so they shrink in place, without views)
    v.ids.unsafeGetTensorImpl()->set_sizes_contiguous({v.count});
    v.tiles.unsafeGetTensorImpl()->set_sizes_contiguous({v.count});
    if (v.sign.defined())
        return {pr, cn, intens, v.ids, v.bins, v.sign, v.tile_min, v.tile_max, v.cum, v.tiles,
                v.live};
    return {pr, cn, intens, v.ids, v.bins, v.tile_min, v.tile_max, v.cum, v.tiles, v.live};
}

void remember(AutogradContext *ctx, const Volume &vol, const Voxelized &v, const Tensor &intens,
              bool per_gaussian) {
    ctx->saved_data["kept"] = std::vector<int64_t>{
        vol.D, vol.H, vol.W, v.count, v.live.numel(), intens.size(0), intens.size(1),
        intens.get_device(), per_gaussian};
    ctx->set_materialize_grads(false);
}

struct Voxelize : public torch::autograd::Function<Voxelize> {
    static Tensor forward(AutogradContext *ctx, const Tensor &pr, const Tensor &cn,
                          const Tensor &intens, const Volume *vol, const Voxelized *v,
                          bool per_gaussian) {
        remember(ctx, *vol, *v, intens, per_gaussian);
        ctx->save_for_backward(saved_tensors(pr, cn, intens, *v));
        return v->volume;
    }

    static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
        const auto saved = ctx->get_saved_variables();
        const Kept k(ctx->saved_data["kept"].toIntVector());
        const c10::DeviceGuard guard(gpu(k.device));
        variable_list g = k.count > 0 && grads[0].defined()
                              ? voxelize_backward(k, saved, Tensor(), grads[0])
                              : zero_gradients(k);
        return {g[0], g[1], g[2], Tensor(), Tensor(), Tensor()};
    }
};

struct VoxelizeL1 : public torch::autograd::Function<VoxelizeL1> {
    // The target gets no gradient, but makes the outputs require one.
    static variable_list forward(AutogradContext *ctx, const Tensor &pr, const Tensor &cn,
                                 const Tensor &intens, const Tensor &, const Volume *vol,
                                 const Voxelized *v, bool per_gaussian) {
        remember(ctx, *vol, *v, intens, per_gaussian);
        ctx->save_for_backward(saved_tensors(pr, cn, intens, *v));
        return {v->loss, v->volume};
    }

    static variable_list backward(AutogradContext *ctx, const variable_list &grads) {
        const auto saved = ctx->get_saved_variables();
        const Kept k(ctx->saved_data["kept"].toIntVector());
        const c10::DeviceGuard guard(gpu(k.device));
        variable_list g;
        if (k.count < 1 || (!grads[0].defined() && !grads[1].defined())) {
            g = zero_gradients(k);
        } else {
            const Tensor gl =
                grads[0].defined()
                    ? grads[0]
                    : at::zeros({}, at::TensorOptions().device(gpu(k.device)).dtype(at::kFloat));
            g = voxelize_backward(k, saved, gl, grads[1]);
        }
        return {g[0], g[1], g[2], Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// The pair count that the prefix-sum kernel writes into pinned memory, read up to
// `reads` times and then once more behind the stream's work (a long queue ahead
// of this forward); negative when even that work left none.
int64_t await_count(const volatile int64_t *host, int64_t reads, const at::Device &dev) {
    int64_t v = *host;
    for (int64_t k = 1; v < 0 && k < reads; ++k) v = *host;
    if (v < 0) {
        c10::hip::getCurrentHIPStream(dev.index()).synchronize();
        v = *host;
    }
    std::atomic_thread_fence(std::memory_order_acquire);
    return v;
}

// Prefix sum, binning and forward at the capacity (target: the fused L1 step).
// False for a call that the Python class takes.
bool voxelize_forward(const Tensor &pr, const Tensor &cn, const Tensor &intens,
                      const Tensor &tile_min, const Tensor &tile_max, const Tensor &hits,
                      const Tensor &target, const Volume &vol, int64_t cap, const Tensor &slot,
                      int64_t reads, Voxelized &v) {
    const int64_t n = pr.size(0);
    const int C = (int)intens.size(1);
    int64_t *host = static_cast<int64_t *>(slot.data_ptr());
    *const_cast<volatile int64_t *>(host) = -1;
    v.tile_min = tile_min;
    v.tile_max = tile_max;
    v.cum = empty({n}, pr, at::kInt);
    v.bins = empty({vol.tiles(), 2}, pr, at::kInt);
    v.ids = empty({cap}, pr, at::kInt);
    v.tiles = empty({cap}, pr, at::kInt);
    v.live = empty({cap}, pr, at::kByte);
    v.volume = empty({vol.D, vol.H, vol.W, C}, pr, at::kFloat);
    size_t bytes = 0;
    check(lib.gsv_cumsum_bin_workspace_bytes((int)n, cap, vol.D, vol.H, vol.W, &bytes),
          "cumsum_bin_workspace_bytes");
    const Tensor total = empty({1}, pr, at::kLong), ws = workspace(bytes, pr);
    void *stream = stream_of(pr);
    check(lib.gsv_cumsum_bin_and_sort_device_count(
              (int)n, cap, ptr<int32_t>(hits), ptr<int32_t>(tile_min), ptr<int32_t>(tile_max),
              vol.D, vol.H, vol.W, ptr<int32_t>(v.cum), ptr<int64_t>(total), host, ptr<void>(ws),
              bytes, ptr<int32_t>(v.ids), ptr<int32_t>(v.bins), ptr<int32_t>(v.tiles), stream),
          "cumsum_bin_and_sort_device_count");
    if (target.defined()) {
        v.sign = empty({vol.D, vol.H, vol.W, C}, pr, at::kChar);
        v.loss = empty({}, pr, at::kFloat);
        check(lib.gsv_voxelize_fwd_l1_workspace_bytes(vol.D, vol.H, vol.W, &bytes),
              "voxelize_fwd_l1_workspace_bytes");
        const Tensor part = workspace(bytes, pr);
        check(lib.gsv_voxelize_fwd_l1(vol.D, vol.H, vol.W, C, (int)n, cap, ptr<int32_t>(v.ids),
                                      ptr<int32_t>(v.bins), ptr<float>(pr), ptr<float>(cn),
                                      ptr<float>(intens), ptr<float>(target),
                                      ptr<float>(v.volume), ptr<int8_t>(v.sign),
                                      ptr<float>(v.loss), ptr<uint8_t>(v.live), ptr<void>(part),
                                      bytes, stream),
              "voxelize_fwd_l1");
    } else {
        check(lib.gsv_voxelize_fwd(vol.D, vol.H, vol.W, C, (int)n, cap, ptr<int32_t>(v.ids),
                                   ptr<int32_t>(v.bins), ptr<float>(pr), ptr<float>(cn),
                                   ptr<float>(intens), ptr<float>(v.volume),
                                   ptr<uint8_t>(v.live), stream),
              "voxelize_fwd");
    }
    v.count = await_count(host, reads, pr.device());
    return v.count >= 0 && v.count <= cap;
}

// (count, outputs): the volume, or (loss, volume) with a target.  No outputs
// for a call that the Python class takes: inputs other than the plain ones, or
// more pairs than the capacity holds.  Without pairs every tile's range is empty:
// the volume is zero, and the gradients are.
std::tuple<int64_t, std::vector<Tensor>> voxelize(
    const Tensor &pr, const Tensor &cn, const Tensor &intens, const Tensor &tile_min,
    const Tensor &tile_max, const Tensor &hits, const c10::optional<Tensor> &target, int64_t D,
    int64_t H, int64_t W, bool per_gaussian, int64_t cap, const Tensor &slot, int64_t reads) {
    const std::tuple<int64_t, std::vector<Tensor>> none{-1, {}};
    if (!pr.defined() || !pr.is_cuda() || pr.dim() != 2 || !fits(D, H, W) || cap < 1) return none;
    const int64_t n = pr.size(0);
    const at::Device dev = pr.device();
    const Volume vol{(int)D, (int)H, (int)W};
    if (n < 1 || n > INT32_MAX || vol.tiles() > INT32_MAX || intens.dim() != 2 ||
        intens.size(1) < 1 || intens.size(1) > GSV_MAX_CHANNELS ||
        !is_rows(pr, at::kFloat, dev, n, 4) || !is_rows(cn, at::kFloat, dev, n, 6) ||
        !is_rows(intens, at::kFloat, dev, n, intens.size(1)) ||
        !is_rows(tile_min, at::kInt, dev, n, 3) || !is_rows(tile_max, at::kInt, dev, n, 3) ||
        !is_vector(hits, at::kInt, dev, n))
        return none;
    Tensor t;
    if (target.has_value()) {
        t = *target;
        const int64_t C = intens.size(1);
        const bool full = t.dim() == 4 && t.size(0) == D && t.size(1) == H && t.size(2) == W &&
                          t.size(3) == C;
        const bool single = t.dim() == 3 && C == 1 && t.size(0) == D && t.size(1) == H &&
                            t.size(2) == W;
        if (!(full || single) || t.device() != dev || t.scalar_type() != at::kFloat ||
            !t.is_contiguous())
            return none;
    }
    const c10::DeviceGuard guard(dev);
    Voxelized v;
    if (!voxelize_forward(pr, cn, intens, tile_min, tile_max, hits, t, vol, cap, slot,
                          reads, v))
        return {v.count, {}};
    if (t.defined()) return {v.count, VoxelizeL1::apply(pr, cn, intens, t, &vol, &v, per_gaussian)};
    return {v.count, {Voxelize::apply(pr, cn, intens, &vol, &v, per_gaussian)}};
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.attr("torch_version") = GSV_TORCH_VERSION;  // the torch it was compiled against
    m.def("bind", &bind);
    m.def("project", &project, py::call_guard<py::gil_scoped_release>());
    m.def("voxelize", &voxelize, py::call_guard<py::gil_scoped_release>());
}
