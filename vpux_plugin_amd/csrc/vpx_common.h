// Shared host/device helpers of the execution library.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <tuple>

#include "vpx_runtime.h"

namespace vpx {

// ---- error channel -------------------------------------------------------------------------
const char* last_error();
void clear_error();
int fail(int code, const char* fmt, ...) __attribute__((format(printf, 2, 3)));

#define VPX_HIP_CHECK(expr)                                                                              \
    do {                                                                                                 \
        hipError_t _e = (expr);                                                                          \
        if (_e != hipSuccess)                                                                            \
            return ::vpx::fail(_e == hipErrorOutOfMemory ? VPX_RESULT_ERROR_OUT_OF_MEMORY                \
                                                         : VPX_RESULT_ERROR_UNKNOWN,                     \
                               "%s failed: %s (%s:%d)", #expr, hipGetErrorString(_e), __FILE__, __LINE__); \
    } while (0)

#define VPX_REQUIRE(cond, code, ...)                   \
    do {                                               \
        if (!(cond)) return ::vpx::fail(code, __VA_ARGS__); \
    } while (0)

// ---- a kernel's arguments -------------------------------------------------------------------
// They lie in memory, and a wave reads a line of 64 bytes when it comes to the first value in it.  Kernels whose first load waits for values of several
// lines, come to one after another, name a value of each in an empty asm at their start, in front of which all of them are asked for together (us in a
// HIP graph, without / with it: softmax of 4 x 512 x 512 2.40 / 2.28, add with one value a channel [2,64,56,56] 2.18 / 2.08, [2,160,160,16] -> 32 3x3
// on nce_direct 3.20 / 3.05; where the set-up does not wait for them it is none of these or, registers held from the start, a loss: [16,7,7,512] -> 512
// 3x3 on nce_conv_stream 12.5 / 13.1).

// ---- launches --------------------------------------------------------------------------------
// The arguments go straight to hipLaunchKernel, which says whether the launch was taken: the triple-chevron form keeps the launch's shape in a stack of
// the runtime's and takes it from there again, and its result has to be asked for, three calls into the runtime of 0.04 ... 0.05 us each.
// A launch holds fewer than 2^32 lanes; what is beyond them would be dropped without an error.
template <class... P, class... A>
int launch(void (*kernel)(P...), const dim3& grid, const dim3& block, size_t lds, hipStream_t s, const A&... args) {
    static_assert(sizeof...(P) == sizeof...(A), "a launch gives every argument of its kernel");
    if ((uint64_t)grid.x * block.x >= (1ull << 32))
        return fail(VPX_RESULT_ERROR_UNSUPPORTED_FEATURE, "%u workgroups of %u lanes exceed the launch limit", grid.x, block.x);
    const std::tuple<P...> held(static_cast<P>(args)...);  // (of the kernel's own types: the runtime copies bytes)
    return std::apply(
            [&](const P&... p) -> int {
                void* at[] = {const_cast<void*>(static_cast<const void*>(&p))...};
                const hipError_t e = hipLaunchKernel(reinterpret_cast<const void*>(kernel), grid, block, at, lds, s);
                if (e == hipSuccess) return VPX_RESULT_SUCCESS;
                (void)hipGetLastError();  // (reported here: not to the next one who asks)
                return fail(e == hipErrorOutOfMemory ? VPX_RESULT_ERROR_OUT_OF_MEMORY : VPX_RESULT_ERROR_UNKNOWN, "a kernel launch failed: %s",
                            hipGetErrorString(e));
            },
            held);
}

#define VPX_LAUNCH(kernel, grid, block, lds, stream, ...)                                                    \
    do {                                                                                                     \
        if (const int _rc = ::vpx::launch(kernel, grid, block, lds, stream, __VA_ARGS__)) return _rc; \
    } while (0)

// ---- divisions ---------------------------------------------------------------------------------
// n / d for any n and d of 32 bits: magic = floor((2^32 - 1) / d) lies at most one below 2^32 / d (one where d is a power of two), so n * magic
// falls short of 2^32 * n / d by at most n < 2^32, and its high half is the quotient or one less.
inline unsigned quotient_magic(unsigned d) { return 0xffffffffu / d; }
__device__ __forceinline__ unsigned quotient(unsigned n, unsigned d, unsigned magic) {
    const unsigned q = __umulhi(n, magic);
    return q + (n - q * d >= d ? 1u : 0u);
}

// ---- tensor views parsed from a params blob ---------------------------------------------------
constexpr int kMaxDims = 8;  // deepest rank the strided kernels accept

struct MemRef {
    void* data = nullptr;
    uint32_t dtype = VPX_NN_UNDEFINED;
    uint64_t order = 0;
    int nd = 0;
    int64_t dims[VPX_MAX_ND_DIMS] = {};     // innermost first
    int64_t strides[VPX_MAX_ND_DIMS] = {};  // in elements, innermost first
    int elem_bits = 0;
    bool compact = false;
    // A memref whose MemRefData says isStatic = 0 (a bounded dynamic shape): dims / strides above are the bounds the blob
    // holds; the live ones sit in device memory (int32 dims, int64 strides in bits, innermost first), where the producer
    // of the shape wrote them, and only a kernel can read them.
    const int32_t* live_dims = nullptr;
    const int64_t* live_strides = nullptr;

    int64_t numel() const {
        int64_t n = 1;
        for (int i = 0; i < nd; i++) n *= dims[i];
        return n;
    }
};

inline int dtype_bits(uint32_t t) {
    switch (t) {
    case VPX_NN_FP32:
    case VPX_NN_I32:
    case VPX_NN_U32: return 32;
    case VPX_NN_FP16:
    case VPX_NN_BF16:
    case VPX_NN_I16:
    case VPX_NN_U16: return 16;
    case VPX_NN_U8:
    case VPX_NN_I8: return 8;
    case VPX_NN_FP64:
    case VPX_NN_I64:
    case VPX_NN_U64: return 64;
    default: return 0;
    }
}

const char* dtype_name(uint32_t t);

// Device-side view for the generic strided kernels.
struct NdIndex {
    int nd;
    int32_t dims[kMaxDims];     // output dims, innermost first
    int64_t stride[4][kMaxDims];  // element strides of up to 4 operands (0 where broadcast)
};

// Library-owned scratch memory, one buffer per (device, stream): calls on one stream are ordered,
// so they can share it; calls on different streams get different buffers.
int get_workspace(hipStream_t stream, size_t bytes, void** out);
// A small area, zero at first, per (device, stream handle) for kernels whose workgroups meet inside a launch: each such
// kernel has a part of its own and keeps its counters and tagged records there from launch to launch.
constexpr size_t kSyncCminor = 128 * 1024;  // the channel-minor MVN's part: 128 groups of 2048 records of 16 bytes and 16 of
                                            // 16384, 256 launch counts of 16 bytes for each group
constexpr size_t kSyncBytes = kSyncCminor + (128 + 16) * (256 * 16) + 128 * (2048 * 16) + 16 * (16384 * 16);
int get_sync_area(hipStream_t stream, void** out, bool* absent = nullptr);
// Compute units of the current device (cached per device).
int device_compute_units(int* out);
// True while the calling thread is inside the entry point that may not allocate: get_workspace() then hands out the
// fixed scratch array (at most VPX_NOALLOC_SCRATCH_BYTES), and launchers must not call hipMalloc for caches of their own.
bool noalloc_call();
// Frees the per-axis quantization tables cached for (device, stream); the caller has drained the stream.
int release_axis_tables(int dev, hipStream_t stream);

// Register-only int8 MFMA loop over every compute unit (calibration of the MFMA roofline); *ops = operations enqueued.
int calib_mfma_i8(const void* operands, void* sink, int iters, int fragment_reads, int64_t* ops, hipStream_t s);
int calib_coissue(int valu_kind, int wide_mfma, int mode, int iters, void* sink, hipStream_t s);

// Dispatch override for tests and tuning (knob names are those of the VPX_* environment variables, read once).
int set_tuning(const char* knob, const char* value);
// VPX_MVN_FUSED: 0 = never take the one-launch MVN kernels, 1 = default, 2 = their workgroups do not wait for each other
// (each computes and publishes what it finds missing: the path a workgroup takes when the others are not resident)
int tuning_mvn_fused();
// VPX_CALIB_BLOCKS: workgroups of the MFMA calibration loop (0: one per compute unit); fewer leave compute units free
// for whatever another stream launches beside it
int tuning_calib_blocks();

// ---- kernel launchers (defined in the .hip files) ------------------------------------------
int launch_convert(const MemRef& in, const MemRef& out, hipStream_t s);
int launch_eltwise(int op, const MemRef& a, const MemRef& b, const MemRef& out, hipStream_t s);
int launch_fake_quantize(const MemRef& in, const MemRef lims[4], const MemRef& out, int64_t levels, hipStream_t s);
int launch_quantize(const MemRef& in, const MemRef& out, double scale, int64_t zp, hipStream_t s);
int launch_dequantize(const MemRef& in, const MemRef& out, double scale, int64_t zp, hipStream_t s);
// per-axis forms: n scales / zero points along the dimension of size n (see the definition for how it is chosen)
int launch_quantize_per_axis(const MemRef& in, const MemRef& out, const double* scales, const int64_t* zps, int64_t n,
                             hipStream_t s);
int launch_dequantize_per_axis(const MemRef& in, const MemRef& out, const double* scales, const int64_t* zps, int64_t n,
                               hipStream_t s);

struct SoftmaxPlan {
    int axis;  // index into dims (innermost first)
    int pad;
    int nd;
    int64_t dims[VPX_MAX_ND_DIMS];
    int64_t in_stride[VPX_MAX_ND_DIMS];
    int64_t out_stride[VPX_MAX_ND_DIMS];
};
int launch_softmax(const SoftmaxPlan& p, uint32_t dtype, const void* in, void* out, hipStream_t s);
// bounded dynamic shapes (SoftmaxModeDynamic): the live dims and strides are read on the device; `axis` counts from the
// innermost dimension of the memrefs as they are (no packing)
int launch_softmax_dynamic(const MemRef& in, const MemRef& out, int axis, int pad, hipStream_t s);

int launch_mvn(const MemRef& in, const MemRef& out, bool across_channels, bool normalize_variance, float eps,
               hipStream_t s);

// mvn1 with per-channel statistics on a channel-minor layout in one launch, where the tensor fits the registers of the
// chip (*done says whether it was launched)
int launch_mvn_cminor_resident(const void* in, void* out, int64_t N, int64_t S, int64_t C, int nv, float eps, hipStream_t s, bool* done);

// whole-tensor range -> one scale and zero point -> u8 values (ONNX DynamicQuantizeLinear arithmetic)
int launch_dynamic_quantize(const MemRef& in, const MemRef& out, const MemRef& scale, const MemRef& zp, hipStream_t s);

// y = (q - zp) * scale with tensor scale / zero point that broadcast onto the input; zp may be null
int launch_dynamic_dequantize(const MemRef& in, const MemRef& scale, const MemRef* zp, const MemRef& out, hipStream_t s);

// MVN-1 decomposition (mvn1_sum -> mvn1_mean_var -> mvn1_norm)
int launch_mvn_sum(const MemRef& in, const MemRef& out, bool across_channels, bool normalize_variance, hipStream_t s);
int launch_mvn_mean_var(const MemRef& sum, const MemRef& out, const int64_t orig_shape[4], bool across_channels,
                        bool normalize_variance, int64_t group_c, float eps, hipStream_t s);
int launch_mvn_norm(const MemRef& in, const MemRef& mean_var, const MemRef& out, bool across_channels, bool normalize_variance,
                    hipStream_t s);

// mem_axes: normalised dimensions counted from the innermost memory dimension; scale / bias may be null
int launch_mvn6(const MemRef& in, const MemRef* scale, const MemRef* bias, const MemRef& out, bool normalize_variance, int eps_mode,
                float eps, const int64_t* mem_axes, int n_axes, hipStream_t s);

enum EltOp { ELT_ADD = 0, ELT_SUB, ELT_MUL, ELT_MIN, ELT_MAX, ELT_DIV, ELT_PRELU };

// Unary activations; p0 / p1 are the kernel's float attributes in the order the compiler serialises them.
enum ActOp {
    ACT_RELU = 0,
    ACT_LEAKY_RELU,   // p0 = negative slope
    ACT_CLAMP,        // p0 = min, p1 = max
    ACT_NEGATIVE,
    ACT_ABS,
    ACT_HSWISH,
    ACT_HSIGMOID,
    ACT_HARDSIGMOID,  // p0 = alpha, p1 = beta
    ACT_SIGMOID,
    ACT_TANH,
    ACT_EXP,
    ACT_SQRT,
    ACT_LOG,
    ACT_FLOOR,
    ACT_CEIL,
    ACT_SIGN,
    ACT_ELU,          // p0 = alpha
    ACT_SELU,         // p0 = alpha, p1 = lambda
    ACT_SWISH,        // p0 = beta
    ACT_MISH,
    ACT_SOFTPLUS,
    ACT_GELU,
    ACT_ERF,
    ACT_COUNT
};
int launch_activation(int op, float p0, float p1, const MemRef& in, const MemRef& out, hipStream_t s);

}  // namespace vpx
