// C ABI of the W4G64 backend (declared in include/w4g64.h).
//
// Host-side validation mirrors the fail-closed checks of the reference's
// GPU wrappers (src/qwen_int4/triton_kernels.py:128-139, :163-189,
// :224-256) for what a C caller can get wrong: null pointers, dtypes,
// dimensions, alignment and workspace size.  Tensor-level checks that need
// framework metadata (device, contiguity, shapes) live in the Python layer.
// Nothing is launched when a check fails.
#include <stdarg.h>
#include <stdio.h>
#include <string.h>

#include <mutex>

#include "../../include/w4g64.h"
#include "w4g64_device.h"
#include "w4g64_internal.h"

// The allocation-free entry point's scratch (w4g64_linear_static_scratch).
using w4g64::kScratchBytes;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {

thread_local char g_error[512] = "";

int fail(int status, const char* fmt, ...) {
    va_list args;
    va_start(args, fmt);
    vsnprintf(g_error, sizeof(g_error), fmt, args);
    va_end(args);
    return status;
}

int ok() {
    g_error[0] = '\0';
    return W4G64_STATUS_OK;
}

bool aligned(const void* p, uintptr_t bytes) { return (((uintptr_t)p) & (bytes - 1)) == 0; }

int element_bytes(int dtype) { return dtype == W4G64_DTYPE_F32 ? 4 : 2; }

int hip_status(hipError_t err, const char* what) {
    if (err != hipSuccess) return fail(W4G64_STATUS_HIP_ERROR, "%s launch failed: %s", what, hipGetErrorString(err));
    return ok();
}

// ---- the allocation-free entry point's scratch ----
// One file-scope device array per GPU, the workspace of
// w4g64_linear_static_scratch: the split-K partial sums (fp32), written in
// full by every call that uses them, so nothing in it needs clearing.  Every
// decode call (1..16 rows) of the Qwen2-1.5B shapes fits (at most 3.28 MiB,
// fp32 gate|up at 16 rows); larger needs are rejected.  In host
// code `scratch` names a host-side stand-in, never the device memory: the
// device address comes from hipGetSymbolAddress, once per device, and only
// that address is used.
constexpr int kMaxScratchDevices = 64;

std::mutex g_scratch_mutex;
void* g_scratch_ptr[kMaxScratchDevices] = {};

// The current device's scratch address: the symbol's device address, looked
// up on the first call on that device.
int device_scratch(void** out) {
    int device = -1;
    if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= kMaxScratchDevices)
        return fail(W4G64_STATUS_HIP_ERROR, "no usable current HIP device (got %d)", device);
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[device]) {
        void* ptr = nullptr;
        const hipError_t err = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (err != hipSuccess || !ptr)
            return fail(W4G64_STATUS_HIP_ERROR, "hipGetSymbolAddress(scratch) failed on device %d: %s", device,
                        hipGetErrorString(err));
        g_scratch_ptr[device] = ptr;
    }
    *out = g_scratch_ptr[device];
    return W4G64_STATUS_OK;
}

}  // namespace

int w4g64::set_error(int status, const char* fmt, ...) {
    va_list args;
    va_start(args, fmt);
    vsnprintf(g_error, sizeof(g_error), fmt, args);
    va_end(args);
    return status;
}

int w4g64::clear_error() {
    g_error[0] = '\0';
    return W4G64_STATUS_OK;
}

extern "C" {

int w4g64_abi_version(void) { return 3; }

const char* w4g64_last_error(void) { return g_error; }

int w4g64_unpack_canonical_int4(const uint8_t* packed, int64_t packed_bytes, int8_t* out, int64_t elements,
                                void* stream) {
    if (packed_bytes < 0) return fail(W4G64_STATUS_INVALID_VALUE, "packed byte count must be non-negative");
    if (elements < 0 || elements > 2 * packed_bytes)
        return fail(W4G64_STATUS_INVALID_VALUE, "elements must be in [0, %lld], got %lld", (long long)(2 * packed_bytes),
                    (long long)elements);
    if (elements == 0) return ok();
    if (!packed || !out) return fail(W4G64_STATUS_INVALID_VALUE, "packed and out must be non-null device pointers");
    return hip_status(w4g64::launch_unpack(packed, out, elements, (hipStream_t)stream), "unpack");
}

int w4g64_dequantize_canonical(const uint8_t* qweight, const uint16_t* scales, const uint8_t* zeros, float* out,
                               int64_t out_features, int64_t in_features, void* stream) {
    if (out_features <= 0) return fail(W4G64_STATUS_INVALID_VALUE, "out_features must be a positive integer");
    if (in_features <= 0 || in_features % 64)
        return fail(W4G64_STATUS_INVALID_VALUE,
                    "canonical W4G64 dequantization requires in_features divisible by 64, got %lld",
                    (long long)in_features);
    if (!qweight || !scales || !zeros || !out)
        return fail(W4G64_STATUS_INVALID_VALUE, "qweight, scales, zeros and out must be non-null device pointers");
    if (!aligned(qweight, 4)) return fail(W4G64_STATUS_INVALID_VALUE, "qweight must be 4-byte aligned");
    if (!aligned(out, 16)) return fail(W4G64_STATUS_INVALID_VALUE, "out must be 16-byte aligned");
    if (!aligned(scales, 2)) return fail(W4G64_STATUS_INVALID_VALUE, "scales must be 2-byte aligned");
    return hip_status(w4g64::launch_dequant(qweight, scales, zeros, out, out_features, in_features,
                                            (hipStream_t)stream),
                      "dequantize");
}

static bool fused_form(int x_dtype) { return x_dtype == W4G64_DTYPE_BF16_SWIGLU; }
// decode-only forms (1..16 rows): planes input, paired gate|up output
static bool decode_form(int x_dtype) {
    return x_dtype == W4G64_DTYPE_BF16_PLANES || x_dtype == W4G64_DTYPE_BF16_GATE_UP;
}
static w4g64::GemvPlan decode_form_plan(int64_t rows, int64_t out_features, int64_t in_features, int x_dtype) {
    return x_dtype == W4G64_DTYPE_BF16_GATE_UP ? w4g64::plan_gemv_paired(rows, out_features, in_features)
                                               : w4g64::plan_gemv(rows, out_features, in_features, w4g64::kPlanes);
}
// The pipelined kernel's plan for a decode form (planes in / paired gate|up
// out); it runs when the operands meet its alignment (16-byte x and
// qweight, 4-byte scales, 2-byte zeros).
static bool decode_form_pipe(int64_t rows, int64_t out_features, int64_t in_features, int x_dtype,
                             w4g64::GemvPlan& plan) {
    return x_dtype == W4G64_DTYPE_BF16_GATE_UP
               ? w4g64::plan_pipe_fused(w4g64::kPlain, true, rows, out_features, in_features, plan)
               : w4g64::plan_pipe_fused(w4g64::kPlanes3, false, rows, out_features, in_features, plan);
}

int64_t w4g64_linear_workspace_bytes(int64_t rows, int64_t out_features, int64_t in_features, int x_dtype) {
    if (rows <= 0 || out_features <= 0 || in_features <= 0 || in_features % 64) return 0;
    if (decode_form(x_dtype)) {
        if (rows > w4g64::kGemvMaxRows) return 0;
        int64_t need = decode_form_plan(rows, out_features, in_features, x_dtype).workspace_bytes;
        w4g64::GemvPlan pipe;
        if (decode_form_pipe(rows, out_features, in_features, x_dtype, pipe) && pipe.workspace_bytes > need)
            need = pipe.workspace_bytes;
        return need;
    }
    if (fused_form(x_dtype))
        return rows <= w4g64::kGemvMaxRows
                   ? w4g64::plan_gemv(rows, out_features, in_features, x_dtype).workspace_bytes
                   : w4g64::gemm_workspace_bytes(rows, out_features, in_features, x_dtype);
    if (x_dtype != W4G64_DTYPE_F16 && x_dtype != W4G64_DTYPE_BF16 && x_dtype != W4G64_DTYPE_F32) return 0;
    if (rows > w4g64::kGemvMaxRows) {
        w4g64::LinearProblem p{nullptr, x_dtype, nullptr, nullptr, nullptr, nullptr, 0, nullptr, rows, out_features,
                               in_features};
        return w4g64::gemm_supported(p) ? w4g64::gemm_workspace_bytes(rows, out_features, in_features, x_dtype) : 0;
    }
    // the larger of the pipelined plan's and the other decode kernels' needs
    // (which kernel runs also depends on pointer alignment)
    int64_t need = w4g64::plan_gemv(rows, out_features, in_features, x_dtype).workspace_bytes;
    w4g64::GemvPlan pipe;
    if (w4g64::plan_pipe(rows, out_features, in_features, x_dtype, pipe) && pipe.workspace_bytes > need)
        need = pipe.workspace_bytes;
    return need;
}

const char* w4g64_linear_kernel_name(int64_t rows, int64_t out_features, int64_t in_features, int x_dtype) {
    if (rows <= 0 || out_features <= 0 || in_features <= 0 || in_features % 64) return "none";
    if (decode_form(x_dtype)) {
        if (rows > w4g64::kGemvMaxRows) return "none";
        const int kind = x_dtype == W4G64_DTYPE_BF16_GATE_UP ? w4g64::kBF16 : w4g64::kPlanes;
        w4g64::GemvPlan pipe;
        if (decode_form_pipe(rows, out_features, in_features, x_dtype, pipe))
            return w4g64::gemv_kernel_name(pipe, kind);  // with aligned operands
        return w4g64::gemv_kernel_name(decode_form_plan(rows, out_features, in_features, x_dtype), kind);
    }
    if (fused_form(x_dtype))
        return rows <= w4g64::kGemvMaxRows
                   ? w4g64::gemv_kernel_name(w4g64::plan_gemv(rows, out_features, in_features, x_dtype), x_dtype)
                   : w4g64::gemm_kernel_name(rows, out_features, in_features, x_dtype);
    if (x_dtype != W4G64_DTYPE_F16 && x_dtype != W4G64_DTYPE_BF16 && x_dtype != W4G64_DTYPE_F32) return "none";
    if (rows <= w4g64::kGemvMaxRows) {
        w4g64::GemvPlan lean;
        if (in_features % 256 == 0 && w4g64::plan_pipe(rows, out_features, in_features, x_dtype, lean))
            return w4g64::gemv_kernel_name(lean, x_dtype);  // with aligned operands
        if (w4g64::plan_seg(rows, out_features, in_features, x_dtype, lean))
            return w4g64::gemv_kernel_name(lean, x_dtype);  // with 16-byte aligned operands
        return w4g64::gemv_kernel_name(w4g64::plan_gemv(rows, out_features, in_features, x_dtype), x_dtype);
    }
    return w4g64::gemm_kernel_name(rows, out_features, in_features, x_dtype);
}

static int check_workspace(const void* workspace, int64_t have, int64_t need) {
    if (need <= 0) return W4G64_STATUS_OK;
    if (!workspace || have < need)
        return fail(W4G64_STATUS_WORKSPACE, "workspace of %lld bytes required, got %lld", (long long)need,
                    (long long)(workspace ? have : 0));
    if (!aligned(workspace, 16)) return fail(W4G64_STATUS_WORKSPACE, "workspace must be 16-byte aligned");
    return W4G64_STATUS_OK;
}

static int linear_impl(const void* x, int x_dtype, const uint8_t* qweight, const uint16_t* scales,
                       const uint8_t* zeros, const void* bias, int bias_dtype, void* y, int64_t rows,
                       int64_t out_features, int64_t in_features, void* workspace, int64_t workspace_bytes, void* stream, void* start_event, void* stop_event) {
    const bool planes = x_dtype == W4G64_DTYPE_BF16_PLANES;
    if (x_dtype != W4G64_DTYPE_F16 && x_dtype != W4G64_DTYPE_BF16 && x_dtype != W4G64_DTYPE_F32 && !planes)
        return fail(W4G64_STATUS_INVALID_DTYPE, "activations must have dtype float16, bfloat16, or float32");
    if (planes && rows > w4g64::kGemvMaxRows)
        return fail(W4G64_STATUS_INVALID_VALUE, "the bf16-planes activation form takes 1..%d rows, got %lld",
                    w4g64::kGemvMaxRows, (long long)rows);
    if (bias_dtype != W4G64_DTYPE_NONE && bias_dtype != W4G64_DTYPE_F16 && bias_dtype != W4G64_DTYPE_BF16 &&
        bias_dtype != W4G64_DTYPE_F32)
        return fail(W4G64_STATUS_INVALID_DTYPE, "bias must have dtype float16, bfloat16, or float32");
    if ((bias_dtype == W4G64_DTYPE_NONE) != (bias == nullptr))
        return fail(W4G64_STATUS_INVALID_VALUE, "bias pointer and bias dtype disagree");
    if (rows <= 0 || in_features <= 0 || in_features % 64)
        return fail(W4G64_STATUS_INVALID_VALUE,
                    "activations require a positive W4G64-compatible feature dimension (rows=%lld, in_features=%lld)",
                    (long long)rows, (long long)in_features);
    if (out_features <= 0) return fail(W4G64_STATUS_INVALID_VALUE, "out_features must be a positive integer");
    if (out_features > (1ll << 30) || in_features > (1ll << 30) || rows > (1ll << 30) ||
        rows * in_features > (1ll << 40) || rows * out_features > (1ll << 40))
        return fail(W4G64_STATUS_UNSUPPORTED, "problem size exceeds the supported index range");
    if (!x || !qweight || !scales || !zeros || !y)
        return fail(W4G64_STATUS_INVALID_VALUE, "x, qweight, scales, zeros and y must be non-null device pointers");
    if (!aligned(x, 16) || !aligned(qweight, 16))
        return fail(W4G64_STATUS_INVALID_VALUE, "x and qweight must be 16-byte aligned");
    if (!aligned(y, (uintptr_t)(planes ? 4 : element_bytes(x_dtype))) || !aligned(scales, 2))
        return fail(W4G64_STATUS_INVALID_VALUE, "y and scales must be element aligned");
    if (bias && !aligned(bias, (uintptr_t)element_bytes(bias_dtype)))
        return fail(W4G64_STATUS_INVALID_VALUE, "bias must be element aligned");

    w4g64::LinearProblem p{x, planes ? (int)w4g64::kPlanes : x_dtype, qweight, scales, zeros, bias, bias_dtype, y, rows,
                           out_features, in_features};
    hipStream_t s = (hipStream_t)stream;
    if (rows <= w4g64::kGemvMaxRows) {
        if (out_features > w4g64::kGemvMaxOutFeatures)
            return fail(W4G64_STATUS_UNSUPPORTED, "decode path supports at most %lld output features",
                        (long long)(w4g64::kGemvMaxOutFeatures));
        w4g64::GemvPlan lean;
        const bool pipe_plan = planes ? w4g64::plan_pipe_fused(w4g64::kPlanes3, false, rows, out_features,
                                                                in_features, lean)
                                      : w4g64::plan_pipe(rows, out_features, in_features, p.x_kind, lean);
        if (pipe_plan && w4g64::pipe_supported(p)) {
            if (int st = check_workspace(workspace, workspace_bytes, lean.workspace_bytes)) return st;
            return hip_status(w4g64::launch_gemv_pipe(p, lean, workspace, s, (hipEvent_t)start_event,
                                                      (hipEvent_t)stop_event),
                              "gemv");
        }
        if (w4g64::plan_seg(rows, out_features, in_features, p.x_kind, lean) && w4g64::seg_supported(p))
            return hip_status(w4g64::launch_gemv_seg(p, lean, s, (hipEvent_t)start_event, (hipEvent_t)stop_event),
                              "gemv");
        const w4g64::GemvPlan plan = w4g64::plan_gemv(rows, out_features, in_features, p.x_kind);
        if (int st = check_workspace(workspace, workspace_bytes, plan.workspace_bytes)) return st;
        return hip_status(w4g64::launch_gemv(p, plan, workspace, s, (hipEvent_t)start_event, (hipEvent_t)stop_event),
                          "gemv");
    }
    if (!w4g64::gemm_supported(p))
        return fail(W4G64_STATUS_UNSUPPORTED, "GEMM path supports rows * in_features below 2^31 (2^30 for float32) "
                    "and out_features * in_features below 2^32");
    const int64_t need = w4g64::gemm_least_workspace_bytes(rows, out_features, in_features, x_dtype);
    if (int st = check_workspace(workspace, workspace_bytes, need)) return st;
    return hip_status(w4g64::launch_gemm(p, workspace, workspace_bytes, s, (hipEvent_t)start_event,
                                         (hipEvent_t)stop_event),
                      "gemm");
}

int w4g64_linear(const void* x, int x_dtype, const uint8_t* qweight, const uint16_t* scales, const uint8_t* zeros,
                 const void* bias, int bias_dtype, void* y, int64_t rows, int64_t out_features, int64_t in_features,
                 void* workspace, int64_t workspace_bytes, void* stream) {
    return linear_impl(x, x_dtype, qweight, scales, zeros, bias, bias_dtype, y, rows, out_features, in_features,
                       workspace, workspace_bytes, stream, nullptr, nullptr);
}

int w4g64_linear_timed(const void* x, int x_dtype, const uint8_t* qweight, const uint16_t* scales,
                       const uint8_t* zeros, const void* bias, int bias_dtype, void* y, int64_t rows,
                       int64_t out_features, int64_t in_features, void* workspace, int64_t workspace_bytes,
                       void* stream, void* start_event, void* stop_event) {
    return linear_impl(x, x_dtype, qweight, scales, zeros, bias, bias_dtype, y, rows, out_features, in_features,
                       workspace, workspace_bytes, stream, start_event, stop_event);
}

int w4g64_linear_static_scratch(const void* x, int x_dtype, const uint8_t* qweight, const uint16_t* scales,
                                 const uint8_t* zeros, const void* bias, int bias_dtype, void* y, int64_t rows,
                                 int64_t out_features, int64_t in_features, void* stream) {
    // the problem's own checks first, then the scratch bound (its planner
    // needs sane sizes), then the set-up, and nothing that allocates
    if (rows <= 0 || in_features <= 0 || in_features % 64 || out_features <= 0 || rows > (1ll << 30) ||
        in_features > (1ll << 30) || out_features > (1ll << 30))
        return linear_impl(x, x_dtype, qweight, scales, zeros, bias, bias_dtype, y, rows, out_features, in_features,
                           nullptr, 0, stream, nullptr, nullptr);
    const int64_t need = w4g64_linear_workspace_bytes(rows, out_features, in_features, x_dtype);
    if (need > kScratchBytes)
        return fail(W4G64_STATUS_UNSUPPORTED,
                    "this problem needs %lld bytes of scratch; the allocation-free entry point holds at most %lld "
                    "(use w4g64_linear with a caller-owned workspace)",
                    (long long)need, (long long)kScratchBytes);
    void* ptr = nullptr;
    if (int st = device_scratch(&ptr)) return st;
    return linear_impl(x, x_dtype, qweight, scales, zeros, bias, bias_dtype, y, rows, out_features, in_features, ptr,
                       kScratchBytes, stream, nullptr, nullptr);
}

int64_t w4g64_static_scratch_bytes(void) { return kScratchBytes; }

// Shared checks of the fused decode entry points (weights, bias, sizes).
static int fused_common_checks(const uint8_t* qweight, const uint16_t* scales, const uint8_t* zeros,
                               const void* bias, int bias_dtype, const void* y, int y_bytes, int64_t rows,
                               int64_t out_features, int64_t in_features) {
    if (bias_dtype != W4G64_DTYPE_NONE && bias_dtype != W4G64_DTYPE_F16 && bias_dtype != W4G64_DTYPE_BF16 &&
        bias_dtype != W4G64_DTYPE_F32)
        return fail(W4G64_STATUS_INVALID_DTYPE, "bias must have dtype float16, bfloat16, or float32");
    if ((bias_dtype == W4G64_DTYPE_NONE) != (bias == nullptr))
        return fail(W4G64_STATUS_INVALID_VALUE, "bias pointer and bias dtype disagree");
    if (rows <= 0 || rows > (1ll << 30))
        return fail(W4G64_STATUS_INVALID_VALUE, "rows must be positive, got %lld", (long long)rows);
    if (in_features <= 0 || in_features % 64 || in_features > (1ll << 24))
        return fail(W4G64_STATUS_INVALID_VALUE, "in_features must be a positive multiple of 64, got %lld",
                    (long long)in_features);
    if (out_features <= 0 || out_features > w4g64::kGemvMaxOutFeatures)
        return fail(W4G64_STATUS_INVALID_VALUE, "out_features must be in [1, %lld], got %lld",
                    (long long)(w4g64::kGemvMaxOutFeatures), (long long)out_features);
    if (!qweight || !scales || !zeros || !y)
        return fail(W4G64_STATUS_INVALID_VALUE, "qweight, scales, zeros and y must be non-null device pointers");
    if (!aligned(qweight, 16)) return fail(W4G64_STATUS_INVALID_VALUE, "qweight must be 16-byte aligned");
    if (!aligned(y, (uintptr_t)y_bytes) || !aligned(scales, 2))
        return fail(W4G64_STATUS_INVALID_VALUE, "y and scales must be element aligned");
    if (bias && !aligned(bias, (uintptr_t)element_bytes(bias_dtype)))
        return fail(W4G64_STATUS_INVALID_VALUE, "bias must be element aligned");
    return W4G64_STATUS_OK;
}

int w4g64_linear_swiglu(const void* gate_up, const uint8_t* qweight, const uint16_t* scales, const uint8_t* zeros,
                        const void* bias, int bias_dtype, float* y, int64_t rows, int64_t out_features,
                        int64_t in_features, void* workspace, int64_t workspace_bytes, void* stream) {
    if (int st = fused_common_checks(qweight, scales, zeros, bias, bias_dtype, y, 4, rows, out_features, in_features))
        return st;
    if (!gate_up) return fail(W4G64_STATUS_INVALID_VALUE, "gate_up must be a non-null device pointer");
    if (!aligned(gate_up, 16)) return fail(W4G64_STATUS_INVALID_VALUE, "gate_up must be 16-byte aligned");
    w4g64::LinearProblem p{gate_up, w4g64::kSwiGLU, qweight, scales, zeros, bias, bias_dtype, y, rows, out_features,
                           in_features};
    if (rows > w4g64::kGemvMaxRows) {
        if (!w4g64::gemm_supported(p))
            return fail(W4G64_STATUS_UNSUPPORTED, "GEMM path supports rows * in_features below 2^30 and "
                        "out_features * in_features below 2^32");
        const int64_t need = w4g64::gemm_least_workspace_bytes(rows, out_features, in_features, w4g64::kSwiGLU);
        if (int st = check_workspace(workspace, workspace_bytes, need)) return st;
        return hip_status(w4g64::launch_gemm(p, workspace, workspace_bytes, (hipStream_t)stream), "gemm");
    }
    const w4g64::GemvPlan plan = w4g64::plan_gemv(rows, out_features, in_features, w4g64::kSwiGLU);
    if (int st = check_workspace(workspace, workspace_bytes, plan.workspace_bytes)) return st;
    return hip_status(w4g64::launch_gemv(p, plan, workspace, (hipStream_t)stream), "gemv");
}

int w4g64_linear_rmsnorm(const void* residual, const void* delta, int delta_dtype, const void* norm_weight, float eps,
                         void* out_sum, const uint8_t* qweight, const uint16_t* scales, const uint8_t* zeros,
                         const void* bias, int bias_dtype, void* y, int gate_up_planes, int64_t rows,
                         int64_t out_features, int64_t in_features, void* workspace, int64_t workspace_bytes,
                         void* stream) {
    if (int st = fused_common_checks(qweight, scales, zeros, bias, bias_dtype, y, 2, rows, out_features, in_features))
        return st;
    if (rows != 1)
        return fail(W4G64_STATUS_INVALID_VALUE, "the fused RMSNorm linear takes one row, got %lld", (long long)rows);
    const int parts = W4G64_DTYPE_F32_PARTS_OF(delta_dtype);
    if (delta_dtype != W4G64_DTYPE_BF16 && delta_dtype != W4G64_DTYPE_F32 && parts == 0)
        return fail(W4G64_STATUS_INVALID_DTYPE, "delta must have dtype bfloat16, float32 or fp32 partial sums");
    if (parts > w4g64::kMaxDeltaParts)
        return fail(W4G64_STATUS_UNSUPPORTED, "the fused RMSNorm linear adds at most %d partial sums, got %d",
                    w4g64::kMaxDeltaParts, parts);
    if (!residual || !delta || !norm_weight || !out_sum)
        return fail(W4G64_STATUS_INVALID_VALUE, "residual, delta, norm_weight and out_sum must be non-null");
    if (!aligned(residual, 16) || !aligned(delta, 16) || !aligned(norm_weight, 16) || !aligned(out_sum, 16))
        return fail(W4G64_STATUS_INVALID_VALUE, "residual, delta, norm_weight and out_sum must be 16-byte aligned");
    const int64_t row_bytes = rows * in_features * 2;
    const char* r0 = (const char*)residual;
    const char* o0 = (const char*)out_sum;
    if (o0 < r0 + row_bytes && r0 < o0 + row_bytes)
        return fail(W4G64_STATUS_INVALID_VALUE, "out_sum must not overlap residual (every workgroup reads it)");
    if (gate_up_planes && out_features % 2)
        return fail(W4G64_STATUS_INVALID_VALUE, "out_features must be even (gate rows then up rows), got %lld",
                    (long long)out_features);
    const int kind = delta_dtype == W4G64_DTYPE_BF16 ? w4g64::kNormB : (parts ? w4g64::kNormP : w4g64::kNormF);
    w4g64::LinearProblem p{residual, kind, qweight, scales, zeros, bias, bias_dtype, y, rows, out_features,
                           in_features, gate_up_planes ? 1 : 0};
    p.norm_delta = delta;
    p.norm_delta_parts = parts ? parts : 1;
    p.norm_weight = (const uint16_t*)norm_weight;
    p.norm_eps = eps;
    p.norm_out_sum = out_sum;
    w4g64::GemvPlan lean;
    // the pipelined kernel: bf16 delta with the paired gate|up epilogue, fp32
    // delta or partial sums with a plain bf16 output
    const bool pipe_plan =
        gate_up_planes ? kind == w4g64::kNormB && w4g64::plan_pipe_fused(w4g64::kNormBf16, true, rows, out_features,
                                                                         in_features, lean)
                       : kind != w4g64::kNormB && w4g64::plan_pipe_fused(w4g64::kNormParts, false, rows,
                                                                         out_features, in_features, lean);
    if (pipe_plan && w4g64::pipe_supported(p))
        return hip_status(w4g64::launch_gemv_pipe(p, lean, nullptr, (hipStream_t)stream), "gemv");
    if (gate_up_planes && w4g64::plan_seg_norm_planes(p, lean))
        return hip_status(w4g64::launch_gemv_seg_norm_planes(p, lean, (hipStream_t)stream), "gemv");
    const w4g64::GemvPlan plan = gate_up_planes ? w4g64::plan_gemv_paired(rows, out_features, in_features, kind)
                                                : w4g64::plan_gemv(rows, out_features, in_features, kind);
    if (plan.kind != 0 || plan.splits != 1)
        return fail(W4G64_STATUS_UNSUPPORTED,
                    "the fused RMSNorm linear needs the whole row in one workgroup (in_features %lld too long)",
                    (long long)in_features);
    if (int st = check_workspace(workspace, workspace_bytes, plan.workspace_bytes)) return st;
    return hip_status(w4g64::launch_gemv(p, plan, workspace, (hipStream_t)stream), "gemv");
}

int w4g64_linear_attention_merge(const void* attention_workspace, int64_t attention_workspace_bytes,
                                 int64_t max_length, int64_t num_heads, int64_t num_kv_heads, const uint8_t* qweight,
                                 const uint16_t* scales, const uint8_t* zeros, const void* bias, int bias_dtype,
                                 void* y, int64_t rows, int64_t out_features, void* stream) {
    if (num_kv_heads <= 0 || num_heads <= 0 || num_heads % num_kv_heads != 0 ||
        num_heads / num_kv_heads > w4g64::kAttnMaxGroup)
        return fail(W4G64_STATUS_INVALID_VALUE,
                    "num_heads (%lld) must be a positive multiple of num_kv_heads (%lld), at most %d times",
                    (long long)num_heads, (long long)num_kv_heads, w4g64::kAttnMaxGroup);
    if (num_heads > (1 << 16)) return fail(W4G64_STATUS_INVALID_VALUE, "num_heads too large");
    const int64_t in_features = num_heads * w4g64::kAttnHeadDim;
    if (int st = fused_common_checks(qweight, scales, zeros, bias, bias_dtype, y, 2, rows, out_features, in_features))
        return st;
    if (rows != 1)
        return fail(W4G64_STATUS_INVALID_VALUE, "the attention-merge linear takes one row, got %lld", (long long)rows);
    if (max_length <= 0) return fail(W4G64_STATUS_INVALID_VALUE, "max_length must be positive");
    const int64_t chunks = (max_length + w4g64::kAttnChunk - 1) / w4g64::kAttnChunk;
    if (!attention_workspace || !aligned(attention_workspace, 16))
        return fail(W4G64_STATUS_WORKSPACE, "the attention workspace must be a 16-byte aligned device pointer");
    const int64_t counters = w4g64::attention_counter_bytes(rows, num_kv_heads);
    const int64_t need = counters + rows * num_kv_heads * chunks * w4g64::kAttnPartFloats * (int64_t)sizeof(float);
    if (attention_workspace_bytes < need)
        return fail(W4G64_STATUS_WORKSPACE, "attention workspace of %lld bytes required, got %lld", (long long)need,
                    (long long)attention_workspace_bytes);
    w4g64::LinearProblem p{(const char*)attention_workspace + counters, w4g64::kAttnM, qweight, scales, zeros, bias,
                           bias_dtype, y, rows, out_features, in_features};
    p.att_chunks = (int)chunks;
    p.att_group = (int)(num_heads / num_kv_heads);
    p.att_kv_heads = (int)num_kv_heads;
    w4g64::GemvPlan plan;
    if (chunks > w4g64::kAttnMergeMaxChunks ||
        !w4g64::plan_pipe_fused(w4g64::kAttnMerge, false, rows, out_features, in_features, plan) ||
        !w4g64::pipe_supported(p))
        return fail(W4G64_STATUS_UNSUPPORTED,
                    "the attention-merge linear takes max_length <= %d, in_features a multiple of 256 up to 1536 "
                    "and 16-byte aligned weights (max_length %lld, in_features %lld): use qwen2_decode_attention "
                    "and w4g64_linear",
                    w4g64::kAttnMergeMaxChunks * w4g64::kAttnChunk, (long long)max_length, (long long)in_features);
    return hip_status(w4g64::launch_gemv_pipe(p, plan, nullptr, (hipStream_t)stream), "gemv");
}

int64_t w4g64_linear_partial_count(int64_t rows, int64_t out_features, int64_t in_features, int x_dtype) {
    if (rows < 1 || rows > w4g64::kGemvMaxRows || out_features <= 0 || out_features > w4g64::kGemvMaxOutFeatures ||
        in_features <= 0 || in_features % 64 || in_features > (1ll << 24))
        return 0;
    if (x_dtype != W4G64_DTYPE_BF16_PLANES && x_dtype != W4G64_DTYPE_F32) return 0;
    w4g64::GemvPlan pipe;
    if (x_dtype == W4G64_DTYPE_BF16_PLANES &&
        w4g64::plan_pipe_fused(w4g64::kPlanes3, false, rows, out_features, in_features, pipe))
        return pipe.splits;
    const w4g64::GemvPlan plan =
        w4g64::plan_gemv(rows, out_features, in_features, x_dtype == W4G64_DTYPE_F32 ? w4g64::kF32 : w4g64::kPlanes);
    return plan.kind == 0 ? plan.splits : 0;
}

int w4g64_linear_partials(const void* x, int x_dtype, const uint8_t* qweight, const uint16_t* scales,
                          const uint8_t* zeros, float* partials, int64_t partials_bytes, int64_t rows,
                          int64_t out_features, int64_t in_features, void* stream) {
    if (int st = fused_common_checks(qweight, scales, zeros, nullptr, W4G64_DTYPE_NONE, partials, 16, rows,
                                     out_features, in_features))
        return st;
    if (x_dtype != W4G64_DTYPE_BF16_PLANES && x_dtype != W4G64_DTYPE_F32)
        return fail(W4G64_STATUS_INVALID_DTYPE, "partial sums take bf16-planes or float32 activations");
    const int64_t count = w4g64_linear_partial_count(rows, out_features, in_features, x_dtype);
    if (count <= 0)
        return fail(W4G64_STATUS_UNSUPPORTED, "partial sums are a decode form (1..%d rows), got %lld rows",
                    w4g64::kGemvMaxRows, (long long)rows);
    if (!x) return fail(W4G64_STATUS_INVALID_VALUE, "x must be a non-null device pointer");
    if (!aligned(x, 16)) return fail(W4G64_STATUS_INVALID_VALUE, "x must be 16-byte aligned");
    const int64_t need = count * rows * out_features * 4;
    if (partials_bytes < need)
        return fail(W4G64_STATUS_INVALID_VALUE, "partials must hold %lld bytes (%lld partial sums), got %lld",
                    (long long)need, (long long)count, (long long)partials_bytes);
    const int kind = x_dtype == W4G64_DTYPE_F32 ? w4g64::kF32 : w4g64::kPlanes;
    w4g64::LinearProblem p{x, kind, qweight, scales, zeros, nullptr, W4G64_DTYPE_NONE, partials, rows, out_features,
                           in_features};
    p.partials_out = partials;
    w4g64::GemvPlan pipe;
    if (kind == w4g64::kPlanes &&
        w4g64::plan_pipe_fused(w4g64::kPlanes3, false, rows, out_features, in_features, pipe)) {
        // the count above came from this plan: its operand alignment is required
        if (!aligned(scales, 4) || !aligned(zeros, 2))
            return fail(W4G64_STATUS_INVALID_VALUE,
                        "partial sums over in_features %lld need 4-byte aligned scales and 2-byte aligned zeros",
                        (long long)in_features);
        return hip_status(w4g64::launch_gemv_pipe(p, pipe, nullptr, (hipStream_t)stream), "gemv");
    }
    const w4g64::GemvPlan plan = w4g64::plan_gemv(rows, out_features, in_features, kind);
    return hip_status(w4g64::launch_gemv(p, plan, nullptr, (hipStream_t)stream), "gemv");
}

int w4g64_linear_gate_up_planes(const void* x, const uint8_t* qweight, const uint16_t* scales, const uint8_t* zeros,
                                const void* bias, int bias_dtype, void* planes, int64_t rows, int64_t out_features,
                                int64_t in_features, void* workspace, int64_t workspace_bytes, void* stream) {
    if (int st = fused_common_checks(qweight, scales, zeros, bias, bias_dtype, planes, 2, rows, out_features,
                                     in_features))
        return st;
    if (rows > w4g64::kGemvMaxRows)
        return fail(W4G64_STATUS_INVALID_VALUE, "the paired gate|up projection takes 1..%d rows, got %lld",
                    w4g64::kGemvMaxRows, (long long)rows);
    if (out_features % 2)
        return fail(W4G64_STATUS_INVALID_VALUE, "out_features must be even (gate rows then up rows), got %lld",
                    (long long)out_features);
    if (!x) return fail(W4G64_STATUS_INVALID_VALUE, "x must be a non-null device pointer");
    if (!aligned(x, 16)) return fail(W4G64_STATUS_INVALID_VALUE, "x must be 16-byte aligned");
    w4g64::LinearProblem p{x, w4g64::kBF16, qweight, scales, zeros, bias, bias_dtype, planes, rows, out_features,
                           in_features, 1};
    w4g64::GemvPlan pipe;
    if (w4g64::plan_pipe_fused(w4g64::kPlain, true, rows, out_features, in_features, pipe) &&
        w4g64::pipe_supported(p))
        return hip_status(w4g64::launch_gemv_pipe(p, pipe, nullptr, (hipStream_t)stream), "gemv");
    const w4g64::GemvPlan plan = w4g64::plan_gemv_paired(rows, out_features, in_features);
    if (int st = check_workspace(workspace, workspace_bytes, plan.workspace_bytes)) return st;
    return hip_status(w4g64::launch_gemv(p, plan, workspace, (hipStream_t)stream), "gemv");
}

}  // extern "C"


#ifdef W4G64_TIMELINE
// ---- profiling builds only: workgroup timelines ----
namespace w4g64 {
unsigned long long* g_timeline_stamps = nullptr;
int g_timeline_workgroups = 0;
}  // namespace w4g64

// Registers the stamp buffer ([workgroups][8] uint64) read by the
// instrumented kernels launched after this call (NULL: none).
extern "C" int w4g64_timeline_register(void* stamps, int64_t workgroups) {
    w4g64::g_timeline_stamps = (unsigned long long*)stamps;
    w4g64::g_timeline_workgroups = stamps ? (int)workgroups : 0;
    return ok();
}
#endif

// ---- the bare-stream probe (measurement aid) ----
namespace w4g64 {
namespace {
struct StreamArgs {
    const u32x4* src;
    uint32_t* sink;
    W4G64_TIMELINE_FIELDS
};
// One 16-byte nontemporal load per lane over exactly `bytes` (a multiple of
// 4096) and a store that practically never happens (it keeps the loads):
// the floor a decode GEMV launch over the same bytes is measured against.
__global__ __launch_bounds__(256) void stream_probe_kernel(StreamArgs a) {
    W4G64_TIMELINE_DECL;
    W4G64_STAMP(0);
    const u32x4 v = __builtin_nontemporal_load(a.src + (int64_t)blockIdx.x * 256 + threadIdx.x);
    W4G64_STAMP(1);
    const uint32_t t = v[0] ^ v[1] ^ v[2] ^ v[3];
    if (t == 0x9E3779B9u) a.sink[threadIdx.x] = t;
    W4G64_STAMP(2);
    W4G64_TIMELINE_STORE(a);
}
}  // namespace
}  // namespace w4g64

extern "C" int w4g64_stream_probe(const void* src, int64_t bytes, void* sink, void* stream) {
    if (!src || !sink || bytes <= 0 || bytes % 4096 || bytes > (int64_t(1) << 40) || !aligned(src, 16))
        return fail(W4G64_STATUS_INVALID_VALUE, "stream probe needs a 16-byte aligned source of 4096-byte blocks");
    w4g64::StreamArgs a{};
    a.src = (const w4g64::u32x4*)src;
    a.sink = (uint32_t*)sink;
    W4G64_TIMELINE_SET(a);
    hipLaunchKernelGGL(w4g64::stream_probe_kernel, dim3((unsigned)(bytes / 4096)), dim3(256), 0,
                       (hipStream_t)stream, a);
    return hip_status(hipGetLastError(), "stream probe");
}

#ifdef W4G64_TIMELINE
// The timelines' reference stream: the probe, with its stamps recorded.
extern "C" int w4g64_timeline_stream(const void* src, int64_t bytes, void* sink, void* stream) {
    return w4g64_stream_probe(src, bytes, sink, stream);
}
#endif
