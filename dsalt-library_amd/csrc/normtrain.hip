// Residual add and RMSNorm of a training step, forward and backward, one pass each.
//
// Reference: x = x + x_attn, h = norm(x) of DSALTTransformerBlock.forward
// (dsalt/modules/dsalt_transformer.py:81-84; RMSENorm, dsalt/kernels/RMSENorm.py:21-23) with
// torch's autograd. Under autocast the residual stream is fp32 and the branch h 16-bit.
// Forward, per row of d:
//   x_out = x + h                              fp32 sum, rounded to x's dtype (torch's add)
//   rstd  = rsqrt(sum(x_out^2) / d + eps)      kept for the backward
//   y     = (x_out * rstd) * w                 in x's dtype and/or rounded to a 16-bit type
// Backward, with a = dy * w and n = x_out * rstd:
//   dx = dx_out + rstd * (a - n * sum(a n) / d), also rounded to h's dtype as dh
//   dw = sum over rows of dy * n               fp32: per lane over a workgroup's rows, over
//        the workgroup in LDS, then over the workgroups in order (deterministic)
//
// Bound by HBM bytes. A row is held in the registers of one wave (d <= 1024) or of four (d <=
// 4096, sums joined through LDS; one wave would need more registers than keep three
// workgroups on a CU), so that every tensor is read and written once. 6473 x 1024, fp32
// stream and bf16 branch: forward 14.3 us (80 MB, 5.6 TB/s), backward 20.4-22.5 us (106 MB,
// 4.7-5.2 TB/s) and 4.9 us for the weight's sums, against torch's 75 (mixed-dtype add) + 12
// (norm) forward and 28 + 24 (norm's two backward passes) + 13 (cast of the branch's
// gradient) + 13 (addition of the residual's) backward.
#include "launch.h"
#include "lanes.h"
#include "rotary.h"  // the F32 element tag

#include <algorithm>
#include <type_traits>

namespace dsalt {
namespace {

constexpr int kNormWaves = 4;        // waves per workgroup
constexpr int kNormMaxGroups = 768;  // workgroups of the backward: three per CU, what its registers allow

struct NormParams {
    const void *x, *h, *w, *dy, *dx_out;
    void *x_out, *y, *y_cast, *dx, *dh;
    float *rstd, *part;
    int64_t rows;
    int nch;  // chunks of 8 elements per row
    int cast_dtype, dh_dtype;
    float d, eps;
};

// Eight consecutive elements as loaded.
template <typename DT>
struct Raw8 {
    uint4 v;
    __device__ __forceinline__ void load(const void *p, int64_t chunk) { v = static_cast<const uint4 *>(p)[chunk]; }
    __device__ __forceinline__ void get(float *f) const {
        const uint32_t a[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            f[2 * e] = DT::lo_f32(a[e]);
            f[2 * e + 1] = DT::hi_f32(a[e]);
        }
    }
};
template <>
struct Raw8<F32> {
    float4 a, b;
    __device__ __forceinline__ void load(const void *p, int64_t chunk) {
        a = static_cast<const float4 *>(p)[2 * chunk];
        b = static_cast<const float4 *>(p)[2 * chunk + 1];
    }
    __device__ __forceinline__ void get(float *f) const {
        f[0] = a.x; f[1] = a.y; f[2] = a.z; f[3] = a.w;
        f[4] = b.x; f[5] = b.y; f[6] = b.z; f[7] = b.w;
    }
};

template <typename DT>
__device__ __forceinline__ void store8(void *p, int64_t chunk, const float *f) {
    if constexpr (std::is_same<DT, F32>::value) {
        float4 *o = static_cast<float4 *>(p) + 2 * chunk;
        o[0] = make_float4(f[0], f[1], f[2], f[3]);
        o[1] = make_float4(f[4], f[5], f[6], f[7]);
    } else {
        static_cast<uint4 *>(p)[chunk] = make_uint4(DT::pack2(f[0], f[1]), DT::pack2(f[2], f[3]),
                                                    DT::pack2(f[4], f[5]), DT::pack2(f[6], f[7]));
    }
}
__device__ __forceinline__ void store8_dt(void *p, int64_t chunk, const float *f, int dtype) {
    if (dtype == DSALT_DTYPE_BF16) store8<BF16>(p, chunk, f);
    else if (dtype == DSALT_DTYPE_F16) store8<F16>(p, chunk, f);
    else store8<F32>(p, chunk, f);
}

// fp32 value made opaque: rounded to fp32 before a 16-bit conversion.
__device__ __forceinline__ float opaque(float v) {
    asm volatile("" : "+v"(v));
    return v;
}
template <typename DT>
__device__ __forceinline__ float rounded(float v) {
    if constexpr (std::is_same<DT, F32>::value) return v;
    else return DT::round(opaque(v));
}

// Sum over the WPR waves of a row; every lane receives it. With WPR > 1 all waves of the
// workgroup call it together.
template <int WPR>
__device__ __forceinline__ float row_sum(float v, float *lds, int wave) {
    v = group_sum_lanes(v, 64);
    if constexpr (WPR > 1) {
        __syncthreads();  // the previous sum has been read
        if ((threadIdx.x & 63) == 0) lds[wave] = v;
        __syncthreads();
        const float *g = lds + wave / WPR * WPR;
        v = (g[0] + g[1]) + (g[2] + g[3]);
        static_assert(WPR == 4, "four waves per row");
    }
    return v;
}

// Lane `l` of a row's 64 * WPR lanes holds chunks l, l + 64 WPR, ... (NCH of them).
template <typename DX, typename DH, typename DW, int NCH, int WPR>
__global__ void __launch_bounds__(64 * kNormWaves) norm_fwd_kernel(const NormParams p) {
    __shared__ float lds[kNormWaves];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l = (wave % WPR) * 64 + (threadIdx.x & 63);
    const int64_t row = (int64_t)blockIdx.x * (kNormWaves / WPR) + wave / WPR;
    const bool live = row < p.rows;  // wave-uniform; with WPR > 1 a dead wave keeps the barriers
    if (WPR == 1 && !live) return;
    const int64_t base = row * p.nch;
    const bool norm = p.rstd || p.y || p.y_cast;
    Raw8<DX> xv[NCH];
    Raw8<DH> hv[NCH];
    Raw8<DW> wv[NCH];
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int ch = c * 64 * WPR + l;
        if (live && ch < p.nch) {
            xv[c].load(p.x, base + ch);
            if (p.h) hv[c].load(p.h, base + ch);
            if (norm) wv[c].load(p.w, ch);
        }
    }
    float s[NCH][8], ss = 0.f;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int ch = c * 64 * WPR + l;
        if (live && ch < p.nch) {
            xv[c].get(s[c]);
            if (p.h) {
                float b[8];
                hv[c].get(b);
#pragma unroll
                for (int e = 0; e < 8; ++e) s[c][e] = rounded<DX>(s[c][e] + b[e]);
                store8<DX>(p.x_out, base + ch, s[c]);
            }
#pragma unroll
            for (int e = 0; e < 8; ++e) ss = fmaf(s[c][e], s[c][e], ss);
        }
    }
    if (!norm) return;  // uniform over the grid
    ss = row_sum<WPR>(ss, lds, wave);
    const float rstd = rsqrtf(ss / p.d + p.eps);
    if (!live) return;
    if (l == 0 && p.rstd) p.rstd[row] = rstd;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int ch = c * 64 * WPR + l;
        if (ch < p.nch) {
            float wf[8], o[8];
            wv[c].get(wf);
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = opaque((s[c][e] * rstd) * wf[e]);
            if (p.y) store8<DX>(p.y, base + ch, o);
            if (p.y_cast) store8_dt(p.y_cast, base + ch, o, p.cast_dtype);
        }
    }
}

template <typename DX, typename DY, typename DW, int NCH, int WPR>
__global__ void __launch_bounds__(64 * kNormWaves) norm_bwd_kernel(const NormParams p) {
    __shared__ float lds[kNormWaves];
    __shared__ float4 acc[kNormWaves][NCH * 2][64];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int l = (wave % WPR) * 64 + lane;
    constexpr int kRows = kNormWaves / WPR;  // rows of a workgroup at a time
    float wf[NCH][8], dw[NCH][8];
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        const int ch = c * 64 * WPR + l;
        Raw8<DW> wv = {};
        if (ch < p.nch) wv.load(p.w, ch);
        wv.get(wf[c]);
#pragma unroll
        for (int e = 0; e < 8; ++e) dw[c][e] = 0.f;
    }
    for (int64_t r0 = (int64_t)blockIdx.x * kRows; r0 < p.rows; r0 += (int64_t)gridDim.x * kRows) {
        const int64_t row = r0 + wave / WPR;
        const bool live = row < p.rows;
        if (WPR == 1 && !live) break;
        const int64_t base = row * p.nch;
        Raw8<DX> xv[NCH], rv[NCH];
        Raw8<DY> yv[NCH];
        float rstd = 0.f;
        if (live) rstd = p.rstd[row];
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const int ch = c * 64 * WPR + l;
            if (live && ch < p.nch) {
                xv[c].load(p.x, base + ch);
                yv[c].load(p.dy, base + ch);
                if (p.dx_out) rv[c].load(p.dx_out, base + ch);
            }
        }
        float n[NCH][8], a[NCH][8], dot = 0.f;
#pragma unroll
        for (int c = 0; c < NCH; ++c) {
            const int ch = c * 64 * WPR + l;
            if (live && ch < p.nch) {
                xv[c].get(n[c]);
                yv[c].get(a[c]);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    n[c][e] *= rstd;
                    dw[c][e] = fmaf(a[c][e], n[c][e], dw[c][e]);
                    a[c][e] *= wf[c][e];
                    dot = fmaf(a[c][e], n[c][e], dot);
                }
            }
        }
        dot = row_sum<WPR>(dot, lds, wave) / p.d;
        if (live) {
#pragma unroll
            for (int c = 0; c < NCH; ++c) {
                const int ch = c * 64 * WPR + l;
                if (ch < p.nch) {
                    float o[8];
#pragma unroll
                    for (int e = 0; e < 8; ++e) o[e] = rstd * fmaf(-n[c][e], dot, a[c][e]);
                    if (p.dx_out) {
                        float r[8];
                        rv[c].get(r);
#pragma unroll
                        for (int e = 0; e < 8; ++e) o[e] += r[e];
                    }
#pragma unroll
                    for (int e = 0; e < 8; ++e) o[e] = opaque(o[e]);
                    if (p.dx) store8<DX>(p.dx, base + ch, o);
                    if (p.dh) store8_dt(p.dh, base + ch, o, p.dh_dtype);
                }
            }
        }
    }
    if (!p.part) return;
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
        acc[wave][2 * c][lane] = make_float4(dw[c][0], dw[c][1], dw[c][2], dw[c][3]);
        acc[wave][2 * c + 1][lane] = make_float4(dw[c][4], dw[c][5], dw[c][6], dw[c][7]);
    }
    __syncthreads();
    // wave `wave` sums the kRows copies of half-chunks; each (lane, half-chunk) of a row's WPR
    // waves is summed once, in the order of the rows
    float4 *out = reinterpret_cast<float4 *>(p.part) + (int64_t)blockIdx.x * p.nch * 2;
    for (int i = threadIdx.x; i < WPR * NCH * 2 * 64; i += 64 * kNormWaves) {
        const int ln = i & 63, hc = (i >> 6) % (NCH * 2), wv = (i >> 6) / (NCH * 2);
        float4 t = acc[wv][hc][ln];
#pragma unroll
        for (int r = 1; r < kRows; ++r) {
            const float4 b = acc[r * WPR + wv][hc][ln];
            t.x += b.x; t.y += b.y; t.z += b.z; t.w += b.w;
        }
        const int ch = (hc >> 1) * 64 * WPR + wv * 64 + ln;
        if (ch < p.nch) out[2 * ch + (hc & 1)] = t;
    }
}

// d_weight[c] = sum over the workgroups' partial rows: 32 columns per workgroup, 32 threads
// per column, each over every 32nd partial.
__global__ void __launch_bounds__(1024) norm_dw_kernel(const float *__restrict__ part, void *out, int groups, int d,
                                                       int dtype) {
    __shared__ float lds[32][33];
    const int col = blockIdx.x * 32 + (threadIdx.x & 31), r = threadIdx.x >> 5;
    float t = 0.f;
    if (col < d) {
        for (int g = r; g < groups; g += 32 * 4) {
            float v[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) v[u] = g + 32 * u < groups ? part[(int64_t)(g + 32 * u) * d + col] : 0.f;
            t += (v[0] + v[1]) + (v[2] + v[3]);
        }
    }
    lds[r][threadIdx.x & 31] = t;
    __syncthreads();
    if (r == 0 && col < d) {
        float s = 0.f;
#pragma unroll
        for (int i = 0; i < 32; ++i) s += lds[i][threadIdx.x];
        if (dtype == DSALT_DTYPE_F32) static_cast<float *>(out)[col] = s;
        else if (dtype == DSALT_DTYPE_BF16) static_cast<uint16_t *>(out)[col] = (uint16_t)BF16::pack2(s, s);
        else static_cast<uint16_t *>(out)[col] = (uint16_t)F16::pack2(s, s);
    }
}

int bwd_groups(int64_t rows, int d) {
    const int per = d <= 1024 ? kNormWaves : kNormWaves / 4;
    return (int)std::min<int64_t>((rows + per - 1) / per, kNormMaxGroups);
}

template <typename DX, typename DB, typename DW, int NCH, int WPR>
void launch_shape(const NormParams &p, bool bwd, hipStream_t stream) {
    if (bwd) {
        const int groups = bwd_groups(p.rows, p.nch * 8);
        hipLaunchKernelGGL((norm_bwd_kernel<DX, DB, DW, NCH, WPR>), dim3(groups), dim3(64 * kNormWaves), 0, stream, p);
    } else {
        const int64_t groups = (p.rows + kNormWaves / WPR - 1) / (kNormWaves / WPR);
        hipLaunchKernelGGL((norm_fwd_kernel<DX, DB, DW, NCH, WPR>), dim3((unsigned)groups), dim3(64 * kNormWaves), 0,
                           stream, p);
    }
}

template <typename DX, typename DB, typename DW>
void launch_types(const NormParams &p, bool bwd, hipStream_t stream) {
    if (p.nch <= 64) launch_shape<DX, DB, DW, 1, 1>(p, bwd, stream);
    else if (p.nch <= 128) launch_shape<DX, DB, DW, 2, 1>(p, bwd, stream);
    else if (p.nch <= 256) launch_shape<DX, DB, DW, 1, 4>(p, bwd, stream);
    else launch_shape<DX, DB, DW, 2, 4>(p, bwd, stream);
}

// DB: the dtype of the branch, h forward and dy backward.
void launch_norm(const NormParams &p, int x_dtype, int b_dtype, int w_dtype, bool bwd, hipStream_t stream) {
    if (x_dtype == DSALT_DTYPE_F32) {
        if (b_dtype == DSALT_DTYPE_BF16) launch_types<F32, BF16, F32>(p, bwd, stream);
        else if (b_dtype == DSALT_DTYPE_F16) launch_types<F32, F16, F32>(p, bwd, stream);
        else launch_types<F32, F32, F32>(p, bwd, stream);
    } else if (x_dtype == DSALT_DTYPE_BF16) {
        if (w_dtype == DSALT_DTYPE_F32) launch_types<BF16, BF16, F32>(p, bwd, stream);
        else launch_types<BF16, BF16, BF16>(p, bwd, stream);
    } else {
        if (w_dtype == DSALT_DTYPE_F32) launch_types<F16, F16, F32>(p, bwd, stream);
        else launch_types<F16, F16, F16>(p, bwd, stream);
    }
}

}  // namespace

int64_t norm_train_workspace_bytes(int64_t rows, int d) { return (int64_t)bwd_groups(rows, d) * d * 4; }

hipError_t launch_norm_train(const dsalt_norm_train_args &a, hipStream_t stream) {
    if (a.rows == 0) return hipSuccess;
    NormParams p = {};
    p.x = a.x;
    p.h = a.h;
    p.w = a.weight;
    p.x_out = a.x_out;
    p.y = a.y;
    p.y_cast = a.y_cast;
    p.rstd = a.rstd;
    p.rows = a.rows;
    p.nch = a.d / 8;
    p.cast_dtype = a.cast_dtype;
    p.d = (float)a.d;
    p.eps = a.eps;
    launch_norm(p, a.x_dtype, a.h ? a.h_dtype : a.x_dtype, a.w_dtype, false, stream);
    return hipGetLastError();
}

hipError_t launch_norm_train_bwd(const dsalt_norm_train_args &a, hipStream_t stream) {
    if (a.rows == 0) return hipSuccess;
    NormParams p = {};
    p.x = a.x;
    p.w = a.weight;
    p.dy = a.dy;
    p.dx_out = a.dx_out;
    p.dx = a.dx;
    p.dh = a.dh;
    p.dh_dtype = a.h_dtype;
    p.rstd = a.rstd;
    p.part = a.d_weight ? static_cast<float *>(a.workspace) : nullptr;
    p.rows = a.rows;
    p.nch = a.d / 8;
    p.d = (float)a.d;
    launch_norm(p, a.x_dtype, a.dy_dtype, a.w_dtype, true, stream);
    if (a.d_weight)
        hipLaunchKernelGGL(norm_dw_kernel, dim3((a.d + 31) / 32), dim3(1024), 0, stream,
                           static_cast<const float *>(a.workspace), a.d_weight, bwd_groups(a.rows, a.d), a.d, a.w_dtype);
    return hipGetLastError();
}

}  // namespace dsalt
