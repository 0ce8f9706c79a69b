// Gated SwiGLU product of the LM's feed-forward blocks, in one pass.
//
// Reference: SwiGLUFFN.forward (dsalt/modules/dsalt_transformer.py:20-21):
//   F.silu(gate_proj(x)) * up_proj(x)
// which torch runs as two elementwise passes: silu(g) = g / (1 + exp(-g)) in fp32, rounded
// to the tensor dtype, then the product with u in fp32, rounded again. This kernel reads
// g and u once and writes the product once, with the same two roundings (bit for bit
// torch's result): 3 bytes moved per 5 of the two passes.
//
// The pass is VALU-bound, not HBM-bound: expf and the IEEE division take ~25 instructions
// per element, and a wave64 instruction occupies a 16-lane SIMD for 4 cycles. The 16-bit
// roundings therefore use the hardware round-to-nearest-even conversions
// (v_cvt_pk_bf16_f32, v_cvt_f16_f32: one instruction per pair or value) rather than
// integer arithmetic. This file is built with hipcc's default contraction: under
// -ffp-contract=fast the backend fuses the range reduction inside expf into one fma and
// exp's last bit no longer matches torch's build.
#include "common.h"
#include "launch.h"
#include "rotary.h"  // the F32 element tag

#include <algorithm>
#include <type_traits>

namespace dsalt {
namespace {

// silu(g) rounded to the tensor dtype, as fp32. The fp32 quotient is made opaque before the
// conversion: otherwise the backend may fold the last step of the division and the
// conversion into one mixed-precision instruction that rounds the exact value once
// instead of to fp32 first.
template <typename DT>
__device__ __forceinline__ float silu_rounded(float g) {
    float s = g / (1.f + expf(-g));
    asm volatile("" : "+v"(s));
    if constexpr (std::is_same<DT, F32>::value)
        return s;
    else
        return DT::round(s);
}

// The fp32 product, opaque for the same reason, before its rounding by the caller's pack.
__device__ __forceinline__ float product(float s, float u) {
    float r = s * u;
    asm volatile("" : "+v"(r));
    return r;
}

// One 32-bit word of a 16-bit tensor: two elements, lo and hi.
template <typename DT>
__device__ __forceinline__ uint32_t swiglu_pair(uint32_t g, uint32_t u) {
    const float r0 = product(silu_rounded<DT>(DT::lo_f32(g)), DT::lo_f32(u));
    const float r1 = product(silu_rounded<DT>(DT::hi_f32(g)), DT::hi_f32(u));
    return DT::pack2(r0, r1);
}

// One 16-byte word: 8 elements of a 16-bit tensor, 4 of an fp32 one.
template <typename DT>
__device__ __forceinline__ uint4 swiglu_word(uint4 g, uint4 u) {
    if constexpr (std::is_same<DT, F32>::value) {
        float4 a = bitcast<float4>(g), b = bitcast<float4>(u), r;
        r.x = product(silu_rounded<F32>(a.x), b.x);
        r.y = product(silu_rounded<F32>(a.y), b.y);
        r.z = product(silu_rounded<F32>(a.z), b.z);
        r.w = product(silu_rounded<F32>(a.w), b.w);
        return bitcast<uint4>(r);
    } else {
        return make_uint4(swiglu_pair<DT>(g.x, u.x), swiglu_pair<DT>(g.y, u.y), swiglu_pair<DT>(g.z, u.z),
                          swiglu_pair<DT>(g.w, u.w));
    }
}

// n16: 16-byte words of each tensor; grid-stride over them, two words in flight per
// iteration (the loads of both issued before either's arithmetic).
template <typename DT>
__global__ void __launch_bounds__(256) swiglu_kernel(const uint4 *__restrict__ g, const uint4 *__restrict__ u,
                                                     uint4 *__restrict__ o, int64_t n16) {
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    for (; i + stride < n16; i += 2 * stride) {
        const uint4 g0 = g[i], u0 = u[i], g1 = g[i + stride], u1 = u[i + stride];
        o[i] = swiglu_word<DT>(g0, u0);
        o[i + stride] = swiglu_word<DT>(g1, u1);
    }
    if (i < n16) o[i] = swiglu_word<DT>(g[i], u[i]);
}

// Training: gu [rows, 2F] holds gate | up, the output of one GEMM against both weights
// concatenated. Forward: out [rows, F] as above. Backward, with da = d out: dgu [rows, 2F] =
//   dgate = da * u * sig * (1 + g * (1 - sig)),  dup = da * silu(g)
// each formed in fp32 and rounded once (torch rounds silu, da * u and each factor's gradient
// to 16 bits on the way); dup takes the rounded silu(g) that the forward multiplied with.
// A thread takes one 16-byte word of each half. 6473 x 2816 in bf16: forward 21.5 us (109 MB,
// 5.1 TB/s), backward 35.5 us (182 MB, 5.1 TB/s), as fast as a copy of the bytes; torch's
// passes took 18 + 17 and 21 + 17 + 17 us.
template <typename DT>
__device__ __forceinline__ void swiglu_grad(float g, float u, float da, float &dg, float &du) {
    const float sig = 1.f / (1.f + expf(-g));
    // where g * (1 - sig) is inf * 0 (g = +inf) or sig * g is 0 * inf (g = -inf) this is NaN,
    // as torch's formula is
    dg = da * u * (sig * (1.f + g * (1.f - sig)));
    du = da * silu_rounded<DT>(g);
    asm volatile("" : "+v"(dg), "+v"(du));
}

template <typename DT>
__device__ __forceinline__ void swiglu_grad_word(uint4 g, uint4 u, uint4 da, uint4 &dg, uint4 &du) {
    const uint32_t gw[4] = {g.x, g.y, g.z, g.w}, uw[4] = {u.x, u.y, u.z, u.w}, aw[4] = {da.x, da.y, da.z, da.w};
    uint32_t og[4], ou[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if constexpr (std::is_same<DT, F32>::value) {
            float a, b;
            swiglu_grad<F32>(__uint_as_float(gw[e]), __uint_as_float(uw[e]), __uint_as_float(aw[e]), a, b);
            og[e] = __float_as_uint(a);
            ou[e] = __float_as_uint(b);
        } else {
            float a0, b0, a1, b1;
            swiglu_grad<DT>(DT::lo_f32(gw[e]), DT::lo_f32(uw[e]), DT::lo_f32(aw[e]), a0, b0);
            swiglu_grad<DT>(DT::hi_f32(gw[e]), DT::hi_f32(uw[e]), DT::hi_f32(aw[e]), a1, b1);
            og[e] = DT::pack2(a0, a1);
            ou[e] = DT::pack2(b0, b1);
        }
    }
    dg = make_uint4(og[0], og[1], og[2], og[3]);
    du = make_uint4(ou[0], ou[1], ou[2], ou[3]);
}

// fw: words of F elements; n = rows * fw. The row of a workgroup's first word is a scalar
// division, the row of a thread's word from there a 32-bit one.
template <typename DT, bool BWD>
__global__ void __launch_bounds__(256) swiglu_rows_kernel(const uint4 *__restrict__ gu, const uint4 *__restrict__ da,
                                                          uint4 *__restrict__ o, int64_t n, uint32_t fw) {
    const int64_t first = (int64_t)blockIdx.x * 256;
    const int64_t row0 = first / fw;
    const uint32_t w = (uint32_t)(first - row0 * fw) + threadIdx.x, r = w / fw, col = w - r * fw;
    const int64_t i = first + threadIdx.x, row = row0 + r;
    if (i >= n) return;
    const int64_t at = row * 2 * fw + col;
    const uint4 g = gu[at], u = gu[at + fw];
    if constexpr (BWD) {
        uint4 dg, du;
        swiglu_grad_word<DT>(g, u, da[i], dg, du);
        o[at] = dg;
        o[at + fw] = du;
    } else {
        o[i] = swiglu_word<DT>(g, u);
    }
}

template <typename DT>
void launch_rows(const uint4 *gu, const uint4 *da, uint4 *o, int64_t n, uint32_t fw, hipStream_t stream) {
    const dim3 grid((unsigned)((n + 255) / 256));
    if (da) hipLaunchKernelGGL((swiglu_rows_kernel<DT, true>), grid, dim3(256), 0, stream, gu, da, o, n, fw);
    else hipLaunchKernelGGL((swiglu_rows_kernel<DT, false>), grid, dim3(256), 0, stream, gu, da, o, n, fw);
}

}  // namespace

hipError_t launch_swiglu_rows(const void *gate_up, const void *d_out, void *out, int64_t rows, int f, int dtype,
                              hipStream_t stream) {
    if (rows == 0) return hipSuccess;
    const int fw = f / (dtype == DSALT_DTYPE_F32 ? 4 : 8);
    const uint4 *gu = static_cast<const uint4 *>(gate_up), *da = static_cast<const uint4 *>(d_out);
    uint4 *o = static_cast<uint4 *>(out);
    if (dtype == DSALT_DTYPE_BF16) launch_rows<BF16>(gu, da, o, rows * fw, fw, stream);
    else if (dtype == DSALT_DTYPE_F16) launch_rows<F16>(gu, da, o, rows * fw, fw, stream);
    else launch_rows<F32>(gu, da, o, rows * fw, fw, stream);
    return hipGetLastError();
}

hipError_t launch_swiglu(const void *gate, const void *up, void *out, int64_t n, int dtype, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    const int per = dtype == DSALT_DTYPE_F32 ? 4 : 8;  // elements per 16-byte word
    const int64_t n16 = n / per;
    const int64_t blocks = std::min<int64_t>((n16 + 255) / 256, 8192);
    const uint4 *g = static_cast<const uint4 *>(gate), *u = static_cast<const uint4 *>(up);
    uint4 *o = static_cast<uint4 *>(out);
    if (dtype == DSALT_DTYPE_BF16)
        hipLaunchKernelGGL(swiglu_kernel<BF16>, dim3((unsigned)blocks), dim3(256), 0, stream, g, u, o, n16);
    else if (dtype == DSALT_DTYPE_F16)
        hipLaunchKernelGGL(swiglu_kernel<F16>, dim3((unsigned)blocks), dim3(256), 0, stream, g, u, o, n16);
    else
        hipLaunchKernelGGL(swiglu_kernel<F32>, dim3((unsigned)blocks), dim3(256), 0, stream, g, u, o, n16);
    return hipGetLastError();
}

}  // namespace dsalt
