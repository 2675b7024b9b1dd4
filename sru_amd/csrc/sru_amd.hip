// C ABI of the SRU recurrence library: argument validation, kernel selection, launch.
// Everything before the launch is plain host logic, so bad arguments are rejected
// without touching the GPU.
#include "sru_amd.h"

#include <hip/hip_runtime.h>

#include "sru_launch.h"
#include "sru_layer.h"
#include "sru_reduce.h"

#include <mutex>

namespace {

using namespace sru_amd;

// Scratch of sru_amd_backward_static: the per-column partial sums (4 floats per column) of at most
// SRU_AMD_STATIC_MAX_COLUMNS columns. One copy of the array exists on every device the library runs
// on, at that device's own address, for the life of the process. In host code the array's name is
// only a handle for hipGetSymbolAddress, never a device address.
static __device__ __align__(256) float scratch[4 * SRU_AMD_STATIC_MAX_COLUMNS];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
float *g_scratch_ptr[kMaxDevices] = {};   // device address of `scratch`, per device ordinal

// Address of the current device's copy of `scratch`; resolved once per device, on the first
// call made with that device current. NULL if the runtime cannot tell.
float *static_scratch_of_current_device() {
    int dev = -1;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
    std::lock_guard<std::mutex> hold(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void *ptr = nullptr;
        if (hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)) != hipSuccess) return nullptr;
        g_scratch_ptr[dev] = static_cast<float *>(ptr);
    }
    return g_scratch_ptr[dev];
}

static_assert(SRU_AMD_STATE_INTERVAL == kCkptInterval, "header and kernels disagree");

size_t elem_size(int dtype) { return dtype == SRU_AMD_F64 ? 8 : dtype == SRU_AMD_F32 ? 4 : 2; }
// element size of the small tensors and of the partial sums: float, or double with double streams
size_t small_size(int dtype) { return dtype == SRU_AMD_F64 ? 8 : 4; }

bool aligned(const void *p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }

// x (and grad_x) is float while the other streams are 16-bit
bool x_is_float_beside_16bit(const sru_amd_shape &s) {
    return (s.dtype == SRU_AMD_F16 || s.dtype == SRU_AMD_BF16) && s.x_dtype == SRU_AMD_X_F32 && s.skip_type == 1;
}

// Shape and flag rules; those on k / skip_type are the device-side asserts of the
// reference's general kernels (sru/csrc/sru_cuda_kernel.cu:397-399).
int check_shape(const sru_amd_shape *s) {
    if (!s) return SRU_AMD_ERR_NULL_POINTER;
    if (s->length < 1 || s->batch < 1 || s->hidden < 1) return SRU_AMD_ERR_BAD_SHAPE;
    if (s->dirs != 1 && s->dirs != 2) return SRU_AMD_ERR_BAD_FLAGS;
    if (s->k != 3 && s->k != 4) return SRU_AMD_ERR_BAD_FLAGS;
    if (s->activation_type != 0 && s->activation_type != 1) return SRU_AMD_ERR_BAD_FLAGS;
    if (s->skip_type < 0 || s->skip_type > 2) return SRU_AMD_ERR_BAD_FLAGS;
    if (s->skip_type == 1 && s->k != 3) return SRU_AMD_ERR_BAD_FLAGS;
    if (s->skip_type == 2 && s->k != 4) return SRU_AMD_ERR_BAD_FLAGS;
    if (s->is_custom != 0 && s->is_custom != 1) return SRU_AMD_ERR_BAD_FLAGS;
    if (s->dtype != SRU_AMD_F32 && s->dtype != SRU_AMD_F16 && s->dtype != SRU_AMD_BF16 && s->dtype != SRU_AMD_F64)
        return SRU_AMD_ERR_BAD_DTYPE;
    if (s->state_interval != 0 && s->state_interval != 1 && s->state_interval != SRU_AMD_STATE_INTERVAL)
        return SRU_AMD_ERR_BAD_FLAGS;
    // checkpointed state exists only for the chunked kernels: not for four streams without a skip
    // term, not for a per-step weight_c together with tanh, and 16-bit streams need an even d
    // (their chunked kernels move two columns at a time); double streams run the general kernels
    if (s->state_interval == SRU_AMD_STATE_INTERVAL) {
        if (s->dtype == SRU_AMD_F64) return SRU_AMD_ERR_BAD_FLAGS;
        if (s->skip_type == 0 && s->k == 4) return SRU_AMD_ERR_BAD_FLAGS;
        if (s->is_custom != 0 && s->activation_type != 0) return SRU_AMD_ERR_BAD_FLAGS;
        if (elem_size(s->dtype) == 2 && s->hidden % 2 != 0) return SRU_AMD_ERR_BAD_FLAGS;
    }
    if (s->x_dtype != SRU_AMD_X_AS_STREAMS && s->x_dtype != SRU_AMD_X_F32) return SRU_AMD_ERR_BAD_DTYPE;
    // a float x next to 16-bit streams exists in the chunked kernels for the plain layer only
    // (and for the state as checkpoints or not at all, which the entry points check)
    if (x_is_float_beside_16bit(*s) && (s->is_custom != 0 || s->activation_type != 0 || s->hidden % 2 != 0))
        return SRU_AMD_ERR_BAD_FLAGS;
    // D' must fit an int, the grid must fit 2^31-1 workgroups and the largest stream
    // (L*B*D'*k elements) must stay far inside the 64-bit byte offsets the kernels use.
    const int64_t lim = INT64_C(1) << 31;
    if (s->hidden >= lim / 2) return SRU_AMD_ERR_BAD_SHAPE;
    const int64_t Dp = s->hidden * s->dirs;
    if (s->batch > (INT64_C(1) << 36) / Dp) return SRU_AMD_ERR_BAD_SHAPE;
    const int64_t ncols = s->batch * Dp;
    if (s->length > (INT64_C(1) << 56) / (ncols * 4)) return SRU_AMD_ERR_BAD_SHAPE;
    return SRU_AMD_OK;
}

// Small tensors in the stream type: only beside 16-bit streams, and weight_c only as a vector (a
// per-step weight_c is a stream).
int check_small(const sru_amd_shape &s, uint32_t small16) {
    if (small16 & ~(uint32_t)SRU_AMD_SMALL_ALL) return SRU_AMD_ERR_BAD_FLAGS;
    if (small16 && elem_size(s.dtype) != 2) return SRU_AMD_ERR_BAD_FLAGS;
    if ((small16 & SRU_AMD_SMALL_WEIGHT_C) && s.is_custom) return SRU_AMD_ERR_BAD_FLAGS;
    return SRU_AMD_OK;
}
static_assert(SRU_AMD_SMALL_WEIGHT_C == kSmallWeightC && SRU_AMD_SMALL_BIAS == kSmallBias && SRU_AMD_SMALL_INIT == kSmallInit &&
              SRU_AMD_SMALL_MASK == kSmallMask && SRU_AMD_SMALL_SCALE == kSmallScale && SRU_AMD_SMALL_LAST == kSmallLast, "header and kernels disagree");

// Everything sru_amd_backward and sru_amd_backward_static share: pointer checks, then the
// scan and the batch reduction enqueued on `stream`, with the per-column partial sums in
// `partial` (4 * B * D' floats of device memory).
int backward_core(const sru_amd_shape *shape, const void *u, const void *x, const void *weight_c,
                  const void *bias, const void *c_init, const void *mask_c, const uint8_t *mask_pad,
                  const void *scale_x, const void *c, const void *grad_h, const void *grad_last,
                  void *grad_u, void *grad_x, void *grad_wc, void *grad_bias, void *grad_init,
                  void *partial, void *stream, uint32_t small16 = 0) {
    const sru_amd_shape &s = *shape;
    if (const int rc = check_small(s, small16)) return rc;
    if (small16 & SRU_AMD_SMALL_INIT) return SRU_AMD_ERR_BAD_FLAGS;   // the chunk kernels select between it and a float checkpoint
    if (!u || !weight_c || !bias || !c || !grad_h || !grad_u || !grad_wc || !grad_bias || !grad_init)
        return SRU_AMD_ERR_NULL_POINTER;
    if (s.skip_type == 1 && (!x || !grad_x)) return SRU_AMD_ERR_NULL_POINTER;
    const size_t es = elem_size(s.dtype), ss = small_size(s.dtype);
    const size_t group = (s.k == 4) ? (es == 8 ? 16 : 4 * es) : es;
    const bool ckpt = s.state_interval == SRU_AMD_STATE_INTERVAL;
    const bool x_float = x_is_float_beside_16bit(s);
    if (x_float && !ckpt) return SRU_AMD_ERR_BAD_FLAGS;
    const size_t xs = x_float ? 4 : es;
    auto small_align = [&](uint32_t bit) { return (small16 & bit) ? es : ss; };
    if (!aligned(u, group) || !aligned(grad_u, group) || !aligned(c, ckpt ? 4 : es) || !aligned(grad_h, es) ||
        (s.skip_type == 1 && (!aligned(x, xs) || !aligned(grad_x, xs))) ||
        !aligned(weight_c, s.is_custom ? 2 * es : small_align(SRU_AMD_SMALL_WEIGHT_C)) || !aligned(grad_wc, s.is_custom ? 2 * es : ss) ||
        !aligned(bias, small_align(SRU_AMD_SMALL_BIAS)) || (c_init && !aligned(c_init, ss)) ||
        (grad_last && !aligned(grad_last, small_align(SRU_AMD_SMALL_LAST))) || !aligned(grad_bias, ss) || !aligned(grad_init, ss) ||
        (mask_c && !aligned(mask_c, small_align(SRU_AMD_SMALL_MASK))) || (scale_x && !aligned(scale_x, small_align(SRU_AMD_SMALL_SCALE))))
        return SRU_AMD_ERR_MISALIGNED;

    if (ckpt && es == 2 &&
        (!aligned(u, s.k == 4 ? 16 : 4) || !aligned(grad_u, s.k == 4 ? 16 : 4) ||
         (s.is_custom && (!aligned(weight_c, 8) || !aligned(grad_wc, 8))) || !aligned(grad_h, 4) ||
         (s.skip_type == 1 && (!aligned(x, 4) || !aligned(grad_x, 4)))))
        return SRU_AMD_ERR_MISALIGNED;

    // (the parameter block types what is always float or double as float; the double kernels know better)
    BwdParams p{};
    p.u = u; p.x = x; p.wc = weight_c; p.bias = bias; p.c0 = static_cast<const float *>(c_init); p.mask_c = mask_c;
    p.pad = mask_pad; p.scale_x = scale_x; p.gh = grad_h; p.glast = grad_last; p.small16 = small16;
    p.c = ckpt ? nullptr : c;
    p.ckpt = ckpt ? static_cast<const float *>(c) : nullptr;
    p.gu = grad_u; p.gx = grad_x; p.gwc_steps = s.is_custom ? grad_wc : nullptr;
    p.ginit = static_cast<float *>(grad_init); p.partial = static_cast<float *>(partial);
    p.L = s.length; p.B = s.batch; p.d = (int32_t)s.hidden; p.Dp = (int32_t)(s.hidden * s.dirs);
    p.ncols = s.batch * p.Dp; p.act = s.activation_type; p.custom = s.is_custom; p.x_float = x_float;

    hipStream_t st = static_cast<hipStream_t>(stream);
    const hipError_t err = s.dtype == SRU_AMD_F32    ? launch_backward<float>(s, p, st)
                           : s.dtype == SRU_AMD_F16  ? launch_backward<half_bits>(s, p, st)
                           : s.dtype == SRU_AMD_BF16 ? launch_backward<bf16_bits>(s, p, st)
                                                     : launch_backward<double>(s, p, st);
    if (err != hipSuccess) return SRU_AMD_ERR_LAUNCH;
    const hipError_t red =
        s.dtype == SRU_AMD_F64
            ? launch_reduce(static_cast<const double *>(partial), s.is_custom ? nullptr : static_cast<double *>(grad_wc),
                            static_cast<double *>(grad_bias), p.B, p.Dp, st)
            : launch_reduce(static_cast<const float *>(partial), s.is_custom ? nullptr : static_cast<float *>(grad_wc),
                            static_cast<float *>(grad_bias), p.B, p.Dp, st);
    return red == hipSuccess ? SRU_AMD_OK : SRU_AMD_ERR_LAUNCH;
}

}  // namespace

extern "C" {

int sru_amd_abi_version(void) { return SRU_AMD_ABI_VERSION; }

const char *sru_amd_status_string(int status) {
    switch (status) {
    case SRU_AMD_OK: return "ok";
    case SRU_AMD_ERR_NULL_POINTER: return "a required pointer is NULL";
    case SRU_AMD_ERR_BAD_SHAPE: return "length, batch or hidden is not positive, or the problem is too large";
    case SRU_AMD_ERR_BAD_FLAGS:
        return "inconsistent dirs / k / activation_type / skip_type / is_custom, or checkpointed state asked for a combination it does not exist for";
    case SRU_AMD_ERR_BAD_DTYPE: return "unknown dtype";
    case SRU_AMD_ERR_MISALIGNED: return "a pointer is not aligned as the header's alignment rules ask";
    case SRU_AMD_ERR_WORKSPACE: return "workspace is NULL, misaligned or too small";
    case SRU_AMD_ERR_LAUNCH: return "the HIP runtime refused the kernel launch";
    case SRU_AMD_ERR_STATIC_LIMIT:
        return "more than SRU_AMD_STATIC_MAX_COLUMNS (262144; half as many for double streams) columns: use sru_amd_backward with a workspace";
    default: return "unknown status";
    }
}

int sru_amd_forward(const sru_amd_shape *shape, const void *u, const void *x, const void *weight_c,
                    const void *bias, const void *c_init, const void *mask_c,
                    const uint8_t *mask_pad, const void *scale_x, void *h, void *c, void *c_last,
                    void *stream) {
    return sru_amd_forward_small(shape, 0, u, x, weight_c, bias, c_init, mask_c, mask_pad, scale_x, h, c, c_last, stream);
}

int sru_amd_forward_small(const sru_amd_shape *shape, uint32_t small16, const void *u, const void *x, const void *weight_c,
                          const void *bias, const void *c_init, const void *mask_c,
                          const uint8_t *mask_pad, const void *scale_x, void *h, void *c, void *c_last,
                          void *stream) {
    if (const int rc = check_shape(shape)) return rc;
    const sru_amd_shape &s = *shape;
    if (const int rc = check_small(s, small16)) return rc;
    if (!u || !weight_c || !bias || !h || !c_last) return SRU_AMD_ERR_NULL_POINTER;
    if (s.skip_type == 1 && !x) return SRU_AMD_ERR_NULL_POINTER;
    const size_t es = elem_size(s.dtype), ss = small_size(s.dtype);
    auto small_align = [&](uint32_t bit) { return (small16 & bit) ? es : ss; };
    const size_t group = (s.k == 4) ? (es == 8 ? 16 : 4 * es) : es;  // a k=4 group moves as one vector (doubles: as two)
    const bool ckpt = s.state_interval == SRU_AMD_STATE_INTERVAL;
    const bool x_float = x_is_float_beside_16bit(s);
    if (x_float && c && !ckpt) return SRU_AMD_ERR_BAD_FLAGS;
    // (a float x still travels with 16-bit streams that move two columns at a time)
    if (x_float && (!aligned(u, s.k == 4 ? 16 : 4) || !aligned(h, 4))) return SRU_AMD_ERR_MISALIGNED;
    if (!aligned(u, group) || !aligned(h, es) || (c && !aligned(c, ckpt ? 4 : es)) ||
        (s.skip_type == 1 && !aligned(x, x_float ? 4 : es)) ||
        !aligned(weight_c, s.is_custom ? 2 * es : small_align(SRU_AMD_SMALL_WEIGHT_C)) || !aligned(bias, small_align(SRU_AMD_SMALL_BIAS)) ||
        (c_init && !aligned(c_init, small_align(SRU_AMD_SMALL_INIT))) || !aligned(c_last, small_align(SRU_AMD_SMALL_LAST)) ||
        (mask_c && !aligned(mask_c, small_align(SRU_AMD_SMALL_MASK))) || (scale_x && !aligned(scale_x, small_align(SRU_AMD_SMALL_SCALE))))
        return SRU_AMD_ERR_MISALIGNED;

    // 16-bit streams with checkpoints move two columns at a time
    if (ckpt && es == 2 &&
        (!aligned(u, s.k == 4 ? 16 : 4) || (s.is_custom && !aligned(weight_c, 8)) || !aligned(h, 4) ||
         (s.skip_type == 1 && !aligned(x, 4))))
        return SRU_AMD_ERR_MISALIGNED;

    FwdParams p{};
    p.u = u; p.x = x; p.wc = weight_c; p.bias = bias; p.c0 = c_init; p.mask_c = mask_c;
    p.pad = mask_pad; p.scale_x = scale_x; p.h = h; p.c_last = c_last; p.small16 = small16;
    p.c = ckpt ? nullptr : c;
    p.ckpt = ckpt ? static_cast<float *>(c) : nullptr;
    p.L = s.length; p.B = s.batch; p.d = (int32_t)s.hidden; p.Dp = (int32_t)(s.hidden * s.dirs);
    p.ncols = s.batch * p.Dp; p.act = s.activation_type; p.custom = s.is_custom; p.x_float = x_float;

    hipStream_t st = static_cast<hipStream_t>(stream);
    const hipError_t err = s.dtype == SRU_AMD_F32    ? launch_forward<float>(s, p, st)
                           : s.dtype == SRU_AMD_F16  ? launch_forward<half_bits>(s, p, st)
                           : s.dtype == SRU_AMD_BF16 ? launch_forward<bf16_bits>(s, p, st)
                                                     : launch_forward<double>(s, p, st);
    return err == hipSuccess ? SRU_AMD_OK : SRU_AMD_ERR_LAUNCH;
}

size_t sru_amd_state_bytes(const sru_amd_shape *shape) {
    if (check_shape(shape) != SRU_AMD_OK) return 0;
    const size_t ncols = (size_t)(shape->batch * shape->hidden * shape->dirs);
    if (shape->state_interval == SRU_AMD_STATE_INTERVAL) {
        const size_t rows = (size_t)(shape->length / SRU_AMD_STATE_INTERVAL);
        return (rows ? rows : 1) * ncols * sizeof(float);
    }
    return (size_t)shape->length * ncols * elem_size(shape->dtype);
}

size_t sru_amd_backward_workspace_bytes(const sru_amd_shape *shape) {
    if (check_shape(shape) != SRU_AMD_OK) return 0;
    return (size_t)4 * small_size(shape->dtype) * (size_t)(shape->batch * shape->hidden * shape->dirs);
}

int sru_amd_backward(const sru_amd_shape *shape, const void *u, const void *x, const void *weight_c,
                     const void *bias, const void *c_init, const void *mask_c,
                     const uint8_t *mask_pad, const void *scale_x, const void *c,
                     const void *grad_h, const void *grad_last, void *grad_u, void *grad_x,
                     void *grad_wc, void *grad_bias, void *grad_init, void *workspace,
                     size_t workspace_bytes, void *stream) {
    return sru_amd_backward_small(shape, 0, u, x, weight_c, bias, c_init, mask_c, mask_pad, scale_x, c, grad_h, grad_last,
                                  grad_u, grad_x, grad_wc, grad_bias, grad_init, workspace, workspace_bytes, stream);
}

int sru_amd_backward_small(const sru_amd_shape *shape, uint32_t small16, const void *u, const void *x, const void *weight_c,
                           const void *bias, const void *c_init, const void *mask_c,
                           const uint8_t *mask_pad, const void *scale_x, const void *c,
                           const void *grad_h, const void *grad_last, void *grad_u, void *grad_x,
                           void *grad_wc, void *grad_bias, void *grad_init, void *workspace,
                           size_t workspace_bytes, void *stream) {
    if (const int rc = check_shape(shape)) return rc;
    if (!workspace || !aligned(workspace, 16) ||
        workspace_bytes < sru_amd_backward_workspace_bytes(shape))
        return SRU_AMD_ERR_WORKSPACE;
    return backward_core(shape, u, x, weight_c, bias, c_init, mask_c, mask_pad, scale_x, c, grad_h, grad_last,
                         grad_u, grad_x, grad_wc, grad_bias, grad_init, workspace, stream, small16);
}

int sru_amd_backward_static(const sru_amd_shape *shape, const void *u, const void *x, const void *weight_c,
                            const void *bias, const void *c_init, const void *mask_c,
                            const uint8_t *mask_pad, const void *scale_x, const void *c,
                            const void *grad_h, const void *grad_last, void *grad_u, void *grad_x,
                            void *grad_wc, void *grad_bias, void *grad_init, void *stream) {
    if (const int rc = check_shape(shape)) return rc;
    // the array holds 4 floats for SRU_AMD_STATIC_MAX_COLUMNS columns; double partial sums fill it with half as many
    if (sru_amd_backward_workspace_bytes(shape) > sizeof(float) * 4 * SRU_AMD_STATIC_MAX_COLUMNS) return SRU_AMD_ERR_STATIC_LIMIT;
    float *partial = static_scratch_of_current_device();
    if (!partial) return SRU_AMD_ERR_LAUNCH;
    return backward_core(shape, u, x, weight_c, bias, c_init, mask_c, mask_pad, scale_x, c, grad_h, grad_last,
                         grad_u, grad_x, grad_wc, grad_bias, grad_init, partial, stream);
}

int sru_amd_layer_route(const sru_amd_shape *shape, int64_t in_features, int64_t n_proj) {
    if (check_shape(shape) != SRU_AMD_OK || in_features < 1 || n_proj < 0) return 0;
    const sru_amd_shape &s = *shape;
    // (16-bit streams throughout; four streams per column only with the skip term among them)
    if (elem_size(s.dtype) != 2 || s.is_custom || x_is_float_beside_16bit(s) || (s.k == 4 && s.skip_type != 2)) return 0;
    if (s.length == 1 && step_sizes_ok(s.batch, s.hidden * s.dirs, in_features, n_proj)) return SRU_AMD_LAYER_STEP;
    // (the long-sequence kernel is built for the layers that a stack has: a skip term, the identity activation)
    if (n_proj == 0 && s.skip_type != 0 && s.activation_type == 0 && rows_sizes_ok(s.length, s.batch, s.hidden, s.dirs, in_features, s.k))
        return SRU_AMD_LAYER_ROWS;
    return 0;
}

int sru_amd_layer_forward(const sru_amd_shape *shape, uint32_t small16, int64_t in_features, int64_t n_proj,
                          const void *x, const void *skip, const void *weight_proj, const void *weight,
                          const void *weight_c, const void *bias, const void *c_init,
                          const uint8_t *mask_pad, const void *scale_x, void *projected,
                          void *h, void *c_last, void *stream) {
    if (const int rc = check_shape(shape)) return rc;
    const sru_amd_shape &s = *shape;
    const int route = sru_amd_layer_route(shape, in_features, n_proj);
    if (!route) return SRU_AMD_ERR_BAD_SHAPE;
    if (const int rc = check_small(s, small16)) return rc;
    if (!x || !weight || !weight_c || !bias || !h || !c_last || (s.skip_type == 1 && !skip) ||
        (n_proj > 0 && (!weight_proj || !projected)))
        return SRU_AMD_ERR_NULL_POINTER;
    for (const void *q : {x, s.skip_type == 1 ? skip : nullptr, weight_proj, weight, static_cast<const void *>(projected), static_cast<const void *>(h)})
        if (q && !aligned(q, 16)) return SRU_AMD_ERR_MISALIGNED;
    auto small_align = [&](uint32_t bit) { return (small16 & bit) ? (size_t)2 : (size_t)4; };
    if (!aligned(weight_c, small_align(SRU_AMD_SMALL_WEIGHT_C)) || !aligned(bias, small_align(SRU_AMD_SMALL_BIAS)) ||
        (c_init && !aligned(c_init, small_align(SRU_AMD_SMALL_INIT))) || !aligned(c_last, small_align(SRU_AMD_SMALL_LAST)) ||
        (scale_x && !aligned(scale_x, small_align(SRU_AMD_SMALL_SCALE))))
        return SRU_AMD_ERR_MISALIGNED;

    hipStream_t st = static_cast<hipStream_t>(stream);
    if (route == SRU_AMD_LAYER_ROWS) {
        RowsParams p{};
        p.x = x; p.weight = weight; p.wc = weight_c; p.bias = bias; p.c0 = c_init; p.scale_x = scale_x; p.skip = skip;
        p.pad = mask_pad; p.h = h; p.c_last = c_last; p.B = s.batch; p.Dp = s.hidden * s.dirs; p.L = (int32_t)s.length;
        p.d = (int32_t)s.hidden; p.dirs = s.dirs; p.inner = (int32_t)in_features; p.groups_per_dir = (p.d + 63) / 64;
        p.small16 = small16;
        return launch_layer_rows(p, s.dtype == SRU_AMD_F16, s.k, st) == hipSuccess ? SRU_AMD_OK : SRU_AMD_ERR_LAUNCH;
    }
    StepParams p{}, proj{};
    p.x = n_proj ? projected : x; p.weight = weight; p.wc = weight_c; p.bias = bias; p.c0 = c_init; p.scale_x = scale_x;
    p.skip = skip; p.pad = mask_pad; p.h = h; p.c_last = c_last; p.Dp = s.hidden * s.dirs; p.cols = p.Dp * s.k;
    p.rows = (int32_t)s.batch; p.inner = (int32_t)(n_proj ? n_proj : in_features); p.act = s.activation_type; p.small16 = small16;
    proj.x = x; proj.weight = weight_proj; proj.h = projected; proj.cols = n_proj;
    proj.rows = p.rows; proj.inner = (int32_t)in_features;
    const hipError_t err = launch_layer_step(p, n_proj ? &proj : nullptr, s.dtype == SRU_AMD_F16, s.k, s.skip_type, st);
    return err == hipSuccess ? SRU_AMD_OK : SRU_AMD_ERR_LAUNCH;
}

size_t sru_amd_stack_workspace_bytes(const sru_amd_shape *shape, int64_t layers, int64_t n_proj) {
    if (check_shape(shape) != SRU_AMD_OK || n_proj < 0) return 0;
    const sru_amd_shape &s = *shape;
    if (elem_size(s.dtype) != 2 || s.is_custom || x_is_float_beside_16bit(s) || s.k != 3 || (s.length > 1 && s.dirs != 1)) return 0;
    return stack_plan(layers, s.length, s.batch, s.hidden * s.dirs, n_proj).bytes;
}

int sru_amd_stack_wanted_in_graph(const sru_amd_shape *shape, int64_t layers, int64_t n_proj) {
    if (sru_amd_stack_workspace_bytes(shape, layers, n_proj) == 0) return 0;
    return shape->length > 1 || stack_wanted_in_graph(layers, shape->batch, shape->hidden * shape->dirs, n_proj);
}

int sru_amd_stack_forward(const sru_amd_shape *shape, uint32_t small16, int64_t layers, int64_t n_proj, const void *x,
                          const void *const *weight_proj, const void *const *weight, const void *const *weight_c,
                          const void *const *bias, const void *const *scale_x, const void *c_init, const uint8_t *mask_pad,
                          void *h, void *c_last, void *workspace, size_t workspace_bytes, void *stream) {
    if (const int rc = check_shape(shape)) return rc;
    const sru_amd_shape &s = *shape;
    const size_t need = sru_amd_stack_workspace_bytes(shape, layers, n_proj);
    if (need == 0) return SRU_AMD_ERR_BAD_SHAPE;
    if (const int rc = check_small(s, small16)) return rc;
    if (!x || !weight || !weight_c || !bias || !h || !c_last || (n_proj > 0 && !weight_proj)) return SRU_AMD_ERR_NULL_POINTER;
    if (!workspace || !aligned(workspace, 16) || workspace_bytes < need) return SRU_AMD_ERR_WORKSPACE;
    auto small_align = [&](uint32_t bit) { return (small16 & bit) ? (size_t)2 : (size_t)4; };
    StackParams p{};
    for (int64_t l = 0; l < layers; ++l) {
        StackLayer &to = p.layer[l];
        to = {weight[l], n_proj ? weight_proj[l] : nullptr, weight_c[l], bias[l], s.skip_type == 1 && scale_x ? scale_x[l] : nullptr};
        if (!to.weight || !to.wc || !to.bias || (n_proj > 0 && !to.weight_proj)) return SRU_AMD_ERR_NULL_POINTER;
        if (!aligned(to.weight, 16) || !aligned(to.weight_proj, 16) || !aligned(to.wc, small_align(SRU_AMD_SMALL_WEIGHT_C)) ||
            !aligned(to.bias, small_align(SRU_AMD_SMALL_BIAS)) || !aligned(to.scale_x, small_align(SRU_AMD_SMALL_SCALE)))
            return SRU_AMD_ERR_MISALIGNED;
    }
    if (!aligned(x, 16) || !aligned(h, 16) || !aligned(c_init, small_align(SRU_AMD_SMALL_INIT)) || !aligned(c_last, small_align(SRU_AMD_SMALL_LAST)))
        return SRU_AMD_ERR_MISALIGNED;
    p.x = x; p.c0 = c_init; p.pad = mask_pad; p.h = h; p.c_last = c_last;
    p.layers = (int32_t)layers; p.rows = (int32_t)(s.length * s.batch); p.Dp = (int32_t)(s.hidden * s.dirs); p.n_proj = (int32_t)n_proj;
    const StackPlan plan = stack_plan(layers, s.length, s.batch, p.Dp, n_proj);
    p.batch = (int32_t)s.batch; p.steps = plan.steps; p.chunks = plan.chunks; p.outputs_at = plan.outputs_at; p.states_at = plan.states_at;
    p.act = s.activation_type; p.skip = s.skip_type == 1; p.small16 = small16;
    const hipError_t err = (s.length == 1 ? launch_layer_stack : launch_prompt_stack)(p, workspace, need, s.dtype == SRU_AMD_F16, static_cast<hipStream_t>(stream));
    return err == hipSuccess ? SRU_AMD_OK : SRU_AMD_ERR_LAUNCH;
}

int sru_amd_product_wanted(int32_t dtype, int64_t rows, int64_t inner, int64_t cols) {
    return (dtype == SRU_AMD_F32 || dtype == SRU_AMD_F16 || dtype == SRU_AMD_BF16) && product_wanted((int)elem_size(dtype), rows, inner, cols);
}

int sru_amd_product(int32_t dtype, int64_t rows, int64_t inner, int64_t cols, const void *x, const void *weight, void *out, void *stream) {
    if (dtype != SRU_AMD_F32 && dtype != SRU_AMD_F16 && dtype != SRU_AMD_BF16) return SRU_AMD_ERR_BAD_SHAPE;
    const ProductTile tile = product_tile((int)elem_size(dtype), rows, inner, cols);
    if (tile.m == 0) return SRU_AMD_ERR_BAD_SHAPE;
    if (!x || !weight || !out) return SRU_AMD_ERR_NULL_POINTER;
    if (!aligned(x, 16) || !aligned(weight, 16) || !aligned(out, 16)) return SRU_AMD_ERR_MISALIGNED;
    const ProductParams p{x, weight, out, (int32_t)rows, (int32_t)inner, (int32_t)cols};
    const hipError_t err = launch_product(p, dtype, tile, static_cast<hipStream_t>(stream));
    return err == hipSuccess ? SRU_AMD_OK : SRU_AMD_ERR_LAUNCH;
}

size_t sru_amd_product_grad_workspace_bytes(int32_t dtype, int64_t rows, int64_t inner, int64_t cols) {
    if (dtype != SRU_AMD_F16 && dtype != SRU_AMD_BF16) return 0;
    return sizeof(float) * (size_t)product_grad_plan(rows, inner, cols).splits * (size_t)inner * (size_t)cols;
}

int sru_amd_product_grad(int32_t dtype, int64_t rows, int64_t inner, int64_t cols, const void *x, const void *grad_out, int32_t grad_dtype,
                         void *grad_weight, void *workspace, size_t workspace_bytes, void *stream) {
    const size_t need = sru_amd_product_grad_workspace_bytes(dtype, rows, inner, cols);
    if (need == 0) return SRU_AMD_ERR_BAD_SHAPE;
    if (grad_dtype != SRU_AMD_F32 && grad_dtype != dtype) return SRU_AMD_ERR_BAD_DTYPE;
    if (!x || !grad_out || !grad_weight) return SRU_AMD_ERR_NULL_POINTER;
    if (!workspace || !aligned(workspace, 16) || workspace_bytes < need) return SRU_AMD_ERR_WORKSPACE;
    if (!aligned(x, 16) || !aligned(grad_out, 16) || !aligned(grad_weight, 16)) return SRU_AMD_ERR_MISALIGNED;
    const GradPlan plan = product_grad_plan(rows, inner, cols);
    const GradParams p{x, grad_out, static_cast<float *>(workspace), (int32_t)rows, (int32_t)inner, (int32_t)cols, plan.splits};
    const hipError_t err = launch_product_grad(p, plan, dtype == SRU_AMD_F16, grad_dtype, grad_weight, static_cast<hipStream_t>(stream));
    return err == hipSuccess ? SRU_AMD_OK : SRU_AMD_ERR_LAUNCH;
}

}  // extern "C"
