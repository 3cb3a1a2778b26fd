// Several tensors between fp32 and one 16-bit type in one launch, for gfx950: what a linear layer under autocast casts on its way
// in (input, weight, bias) and out (their gradients).
// Bound by memory (4096 x 1024 and 1024 x 4096 fp32 elements to 16 bits: 12 us, 50 MB; the way back 9) and, for the biases, by being
// launches at all: one of a few KB took 4 us. us, kernels of a block's step of 4096 tokens at 1024 in such a region: the casts of four
// layers as 20 launches of torch's 91, as 8 launches here 62.
#include "cw_common.h"

namespace cw {

namespace {

constexpr int kCastThreads = 256, kCastUnroll = 4;
constexpr int kCastBlock = kCastThreads * kCastUnroll * 4;  // elements of a block

struct CastArgs {
    const void* src[CW_MAX_CASTS];
    void* dst[CW_MAX_CASTS];
    int64_t n[CW_MAX_CASTS];
    uint32_t first[CW_MAX_CASTS];  // block of the tensor's first element
    int count;
};

typedef uint32_t half4_t __attribute__((ext_vector_type(2)));
template <typename T>
struct quad {
    using raw = half4_t;
};
template <>
struct quad<float> {
    using raw = raw16_t;
};
template <typename H>
__device__ __forceinline__ half4_t convert(raw16_t q, H*) {
    return half4_t{half_conv<H>::pack2(__uint_as_float(q.x), __uint_as_float(q.y)), half_conv<H>::pack2(__uint_as_float(q.z), __uint_as_float(q.w))};
}
template <typename H>
__device__ __forceinline__ raw16_t convert(half4_t q, H*) {
    return raw16_t{__float_as_uint(half_conv<H>::lo(q.x)), __float_as_uint(half_conv<H>::hi(q.x)), __float_as_uint(half_conv<H>::lo(q.y)),
                   __float_as_uint(half_conv<H>::hi(q.y))};
}

// A lane moves 4 elements at a time, so that the loads and the stores of an instruction are both contiguous.
template <typename S, typename D, typename H>
__global__ __launch_bounds__(kCastThreads) void cast_many_kernel(const CastArgs args) {
    int t = 0;
    while (t + 1 < args.count && blockIdx.x >= args.first[t + 1]) ++t;
    const int64_t base = (int64_t)(blockIdx.x - args.first[t]) * kCastBlock, left = args.n[t] - base;
    const S* src = reinterpret_cast<const S*>(args.src[t]) + base;
    D* dst = reinterpret_cast<D*>(args.dst[t]) + base;
    using Q = typename quad<S>::raw;
    using R = typename quad<D>::raw;
    Q q[kCastUnroll];
#pragma unroll
    for (int u = 0; u < kCastUnroll; ++u) {
        const int i = (u * kCastThreads + (int)threadIdx.x) * 4;
        if (i + 4 <= left) q[u] = *reinterpret_cast<const Q*>(src + i);
    }
#pragma unroll
    for (int u = 0; u < kCastUnroll; ++u) {
        const int i = (u * kCastThreads + (int)threadIdx.x) * 4;
        if (i + 4 <= left) *reinterpret_cast<R*>(dst + i) = convert(q[u], (H*)nullptr);
    }
    if (left < kCastBlock) {
        const int64_t i = (left & ~(int64_t)3) + threadIdx.x;
        if (i < left) store_elem(dst + i, load_elem(src + i));
    }
}

}  // namespace
}  // namespace cw

using namespace cw;

extern "C" int cw_cast_many(int count, const void* const* src, void* const* dst, const int64_t* numels, int src_dtype, int dst_dtype, void* stream) {
    if (count < 0 || count > CW_MAX_CASTS) return fail(CW_ERR_INVALID, "cw_cast_many: bad count %d", count);
    const int half = src_dtype == CW_F32 ? dst_dtype : src_dtype;
    if ((src_dtype == CW_F32) == (dst_dtype == CW_F32) || (half != CW_BF16 && half != CW_F16) || (src_dtype != half && dst_dtype != half))
        return fail(CW_ERR_UNSUPPORTED, "cw_cast_many: casts are between float32 and a 16-bit type (%d -> %d)", src_dtype, dst_dtype);
    if (count > 0 && (src == nullptr || dst == nullptr || numels == nullptr)) return fail(CW_ERR_INVALID, "cw_cast_many: null pointer");
    CastArgs a{};
    int64_t blocks = 0;
    for (int i = 0; i < count; ++i) {
        if (numels[i] < 0) return fail(CW_ERR_INVALID, "cw_cast_many: negative size of tensor %d", i);
        if (numels[i] == 0) continue;
        if (src[i] == nullptr || dst[i] == nullptr) return fail(CW_ERR_INVALID, "cw_cast_many: null pointer of tensor %d", i);
        if (!aligned16(src[i]) || !aligned16(dst[i])) return fail(CW_ERR_ALIGNMENT, "cw_cast_many: tensor %d is not 16-byte aligned", i);
        a.src[a.count] = src[i];
        a.dst[a.count] = dst[i];
        a.n[a.count] = numels[i];
        a.first[a.count++] = (uint32_t)blocks;
        blocks += (numels[i] + kCastBlock - 1) / kCastBlock;
        if (blocks >= (int64_t)1 << 24) return fail(CW_ERR_UNSUPPORTED, "cw_cast_many: more than 2^36 elements");  // fewer than 2^32 work-items
    }
    if (blocks == 0) return CW_OK;
    if (const int drc = require_gfx950("cw_cast_many"); drc != CW_OK) return drc;
    return with_elem_type(half, [&](auto* tag) {
        using H = std::remove_pointer_t<decltype(tag)>;
        if constexpr (!std::is_same<H, float>::value) {
            if (src_dtype == CW_F32)
                hipLaunchKernelGGL((cast_many_kernel<float, H, H>), dim3((unsigned)blocks), dim3(kCastThreads), 0, (hipStream_t)stream, a);
            else
                hipLaunchKernelGGL((cast_many_kernel<H, float, H>), dim3((unsigned)blocks), dim3(kCastThreads), 0, (hipStream_t)stream, a);
        }
        return check_launch("cast_many_kernel");
    });
}
