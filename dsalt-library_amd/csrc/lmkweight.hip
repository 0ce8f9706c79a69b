// Differentiable landmark weights from the norms pass, forward and backward.
//
// Reference: hybrid_scores_per_head (dsalt/kernels/landmark_tokens_ker.py:45-61) followed by
// the weight of a selected landmark, log(max(sigmoid(s / tau), 1e-20)), gathered per (head,
// sequence, slot) in _train_selectors (dsalt/modules/dsalt_attention.py:457-487) and laid
// out as an [H, T] table (-inf off the landmarks) in _diff_logbias (:403-438). In torch
// that is ~35 elementwise, reduction and gather launches forward and ~70 backward, each
// over [T, H] or [T, d]: at 9290 tokens x 1024 about 600 us of GPU time and most of the
// host time of a training step. The selection has computed the norms and their fp64
// partial sums already, so:
//   weight_kernel   one workgroup per (head, sequence): the head's statistics from the
//                   partials (hybrid.h, the bits that the selection used), then the weight of
//                   each selected slot (packed) or the head's whole table row (dense).
//   reduce_kernel   (backward) one workgroup per head: the score gradient of each selected
//                   token into the head's dense [T] row, and its sums against 1, z_v, z_x.
//   apply_kernel    (backward) one wave per token: the gradient of its norms (the
//                   standardisation's mean and std terms from the heads' sums), then
//                   d_x = c_x x and d_v = d_v_in + c_g v in one pass over the rows.
// The statistics' sums run over fp64 partials, the rest in fp32 with one rounding of each
// result. Deterministic: no atomics, every element is written by one thread. Bound: the
// apply pass streams x, v and d_v_in (read), d_x and d_v (written): 95 MB in 24.0 us (4.0
// TB/s) at 9290 tokens x 1024 in bf16; weight_kernel (4.7 us) and reduce_kernel (5.3 us) are
// latency. A training step of the module at that shape went 1985 -> 1146 us (152 -> 46
// launches, GPU busy 1391 -> 888 us).
#include "common.h"
#include "hybrid.h"
#include "launch.h"
#include "rotary.h"

#include <type_traits>

namespace dsalt {
namespace {

constexpr int kWThreads = 256;
constexpr int kTableThreads = 1024;
constexpr int kApplyWaves = 4;   // tokens (= waves) per workgroup of apply_kernel
constexpr int kMaxKvW = 128;     // = scores_max_kv()
constexpr float kSigClamp = 1e-20f;

struct WeightParams {
    const float *xn, *vn;   // norms [T], [T, n_kv]
    const double *part;     // [nblk][1 + n_kv][2]
    const float *alpha;     // [H]
    const int64_t *pos;     // [H, S, k]
    const int32_t *cu;
    float *weight;          // [H, S, k] or (table) [H, T]
    float *stats;           // [1 + n_kv][2]: mean, std as used
    int T, S, H, n_kv, rep, k, nblk, table;
    float tau, inv_tau;
    // backward
    const float *g;         // gradient of `weight`, its layout
    float *gz;              // [H][T] score gradients
    double *hsum;           // [H][3]: sums of ds, ds z_v, ds z_x
    float *d_alpha;         // [H] or null
    const void *x, *v, *dv_in;
    void *dx, *dv;
    int64_t x_st, v_st, v_sh, di_st, di_sh;
    int d, D;
};

// log(max(sigmoid(s / tau), 1e-20)) as torch's fp32 ops form it.
__device__ __forceinline__ float lmk_weight(float s, float tau) {
    const float sg = 1.f / (1.f + expf(-s / tau));
    return logf(fmaxf(sg, kSigClamp));
}

__global__ void __launch_bounds__(kTableThreads) weight_kernel(const WeightParams p) {
    __shared__ float st[4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int head = blockIdx.x / p.S, seq = blockIdx.x - head * p.S;
    const int g = head / p.rep;
    if (wave < 2) {
        float m, sd;
        const int q = wave == 0 ? 0 : 1 + g;
        hybrid_stat(p.part, p.nblk, 1 + p.n_kv, q, (double)p.T, lane, m, sd);
        if (lane == 0) {
            st[2 * wave] = m;
            st[2 * wave + 1] = sd;
            // published once per quantity: by sequence 0 of the group's first head
            if (seq == 0 && (q == 0 ? head == 0 : head == g * p.rep)) {
                p.stats[2 * q] = m;
                p.stats[2 * q + 1] = sd;
            }
        }
    }
    float *row = p.weight + (p.table ? (int64_t)head * p.T : ((int64_t)head * p.S + seq) * p.k);
    if (p.table)
        for (int t = tid; t < p.T; t += blockDim.x) row[t] = -INFINITY;
    __syncthreads();  // the statistics; and every -inf of the row before its landmarks
    int c0, c1;
    seq_bounds(p.cu, seq, p.T, c0, c1);
    const float alpha = p.alpha[head];
    const int64_t *pos = p.pos + ((int64_t)head * p.S + seq) * p.k;
    for (int j = tid; j < p.k; j += blockDim.x) {
        const int64_t o = pos[j];
        const bool ok = o >= 0 && o < c1 - c0;
        float w = -INFINITY;
        if (ok) {
            const int64_t t = c0 + o;
            const float s = hybrid_mix(hybrid_z(p.xn[t], st[0], st[1]),
                                       hybrid_z(p.vn[t * p.n_kv + g], st[2], st[3]), alpha);
            w = lmk_weight(s, p.tau);
            if (p.table) row[t] = w;
        }
        if (!p.table) row[j] = w;
    }
}

__device__ __forceinline__ double wave_sumd(double x) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o);
    return x;
}

__global__ void __launch_bounds__(kTableThreads) reduce_kernel(const WeightParams p) {
    __shared__ double s_sum[kTableThreads / 64][3];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int head = blockIdx.x, g = head / p.rep;
    float *gz = p.gz + (int64_t)head * p.T;
    for (int t = tid; t < p.T; t += blockDim.x) gz[t] = 0.f;
    __syncthreads();  // every zero of the row before its landmarks
    const float alpha = p.alpha[head];
    const float mx = p.stats[0], sx = p.stats[1], mv = p.stats[2 + 2 * g], sv = p.stats[3 + 2 * g];
    double a0 = 0.0, a1 = 0.0, a2 = 0.0;
    for (int e = tid; e < p.S * p.k; e += blockDim.x) {
        const int seq = e / p.k;
        int c0, c1;
        seq_bounds(p.cu, seq, p.T, c0, c1);
        const int64_t o = p.pos[(int64_t)head * p.S * p.k + e];
        if (o < 0 || o >= c1 - c0) continue;
        const int64_t t = c0 + o;
        const float zx = hybrid_z(p.xn[t], mx, sx), zv = hybrid_z(p.vn[t * p.n_kv + g], mv, sv);
        const float s = hybrid_mix(zx, zv, alpha);
        const float sg = 1.f / (1.f + expf(-s / p.tau));
        const float gw = p.g[p.table ? (int64_t)head * p.T + t : (int64_t)head * p.S * p.k + e];
        // d log(max(sg, c)) / ds = (1 - sg) / tau above the clamp, 0 below it
        const float ds = sg >= kSigClamp ? gw * (1.f - sg) * p.inv_tau : 0.f;
        gz[t] = ds;
        a0 += ds;
        a1 += (double)ds * zv;
        a2 += (double)ds * zx;
    }
    a0 = wave_sumd(a0);
    a1 = wave_sumd(a1);
    a2 = wave_sumd(a2);
    if (lane == 0) {
        s_sum[wave][0] = a0;
        s_sum[wave][1] = a1;
        s_sum[wave][2] = a2;
    }
    __syncthreads();
    if (tid == 0) {
        double t0 = 0.0, t1 = 0.0, t2 = 0.0;
        for (int w = 0; w < (int)(blockDim.x >> 6); ++w) {
            t0 += s_sum[w][0];
            t1 += s_sum[w][1];
            t2 += s_sum[w][2];
        }
        p.hsum[3 * head] = t0;
        p.hsum[3 * head + 1] = t1;
        p.hsum[3 * head + 2] = t2;
        if (p.d_alpha) p.d_alpha[head] = (float)(t1 - t2);
    }
}

// Gradient of norm n (standardised to z = (n - mean) / sd over T tokens) divided by n, from
// z's gradient dz and the sums A = sum dz, B = sum dz z over the tokens: the row's own
// gradient is this times the row (0 for a zero row, as torch masks it). A clamped std
// takes no gradient.
__device__ __forceinline__ float norm_coef(float n, float mean, float sd, float dz, double A, double B, int T) {
    if (n == 0.f) return 0.f;
    const float z = hybrid_z(n, mean, sd);
    float dn = dz - (float)(A / T);
    if (sd > 1e-6f) dn -= z * (float)(B / (T - 1));
    return dn / sd / n;
}

template <typename DX, typename DV>
__global__ void __launch_bounds__(64 * kApplyWaves) apply_kernel(const WeightParams p) {
    constexpr int EX = std::is_same<DX, F32>::value ? 4 : 8, EV = std::is_same<DV, F32>::value ? 4 : 8;
    __shared__ double s_ab[1 + kMaxKvW][2];
    __shared__ float s_c[kApplyWaves][kMaxKvW];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // the quantities' sums from the heads' sums, in head order
    for (int q = tid; q <= p.n_kv; q += blockDim.x) {
        double A = 0.0, B = 0.0;
        const int h0 = q == 0 ? 0 : (q - 1) * p.rep, h1 = q == 0 ? p.H : h0 + p.rep;
        for (int h = h0; h < h1; ++h) {
            const double a = q == 0 ? 1.0 - (double)p.alpha[h] : (double)p.alpha[h];
            A += a * p.hsum[3 * h];
            B += a * p.hsum[3 * h + (q == 0 ? 2 : 1)];
        }
        s_ab[q][0] = A;
        s_ab[q][1] = B;
    }
    __syncthreads();
    const int t = blockIdx.x * kApplyWaves + wave;
    const bool live = t < p.T;  // wave-uniform
    float dzx = 0.f;
    for (int g = lane; live && g < p.n_kv; g += 64) {
        float dzv = 0.f;
        for (int r = 0; r < p.rep; ++r) {
            const int h = g * p.rep + r;
            const float gz = p.gz[(int64_t)h * p.T + t], a = p.alpha[h];
            dzv += a * gz;
            dzx += (1.f - a) * gz;
        }
        s_c[wave][g] = norm_coef(p.vn[(int64_t)t * p.n_kv + g], p.stats[2 + 2 * g], p.stats[3 + 2 * g], dzv,
                                 s_ab[1 + g][0], s_ab[1 + g][1], p.T);
    }
    __syncthreads();
    if (!live) return;
    if (p.dx) {
        dzx = wave_sumf(dzx);
        const float cx = norm_coef(p.xn[t], p.stats[0], p.stats[1], dzx, s_ab[0][0], s_ab[0][1], p.T);
        for (int c = lane * EX; c < p.d; c += 64 * EX) {
            float a[EX];
            Elem<DX>::template ldv<EX>(p.x, (int64_t)t * p.x_st + c, a);
#pragma unroll
            for (int e = 0; e < EX; ++e) a[e] *= cx;
            Elem<DX>::template stv<EX>(p.dx, (int64_t)t * p.d + c, a);
        }
    }
    if (p.dv) {
        const int G = p.D / EV;
        for (int c = lane; c < p.n_kv * G; c += 64) {
            const int g = c / G, j = (c - g * G) * EV;
            const float cg = s_c[wave][g];
            float a[EV];
            Elem<DV>::template ldv<EV>(p.v, (int64_t)t * p.v_st + (int64_t)g * p.v_sh + j, a);
            if (p.dv_in) {
                float b[EV];
                Elem<DV>::template ldv<EV>(p.dv_in, (int64_t)t * p.di_st + (int64_t)g * p.di_sh + j, b);
#pragma unroll
                for (int e = 0; e < EV; ++e) a[e] = fmaf(cg, a[e], b[e]);
            } else {
#pragma unroll
                for (int e = 0; e < EV; ++e) a[e] *= cg;
            }
            Elem<DV>::template stv<EV>(p.dv, ((int64_t)t * p.n_kv + g) * p.D + j, a);
        }
    }
}

template <typename DX>
void launch_apply(int v_dtype, const WeightParams &p, hipStream_t stream) {
    const dim3 grid((unsigned)((p.T + kApplyWaves - 1) / kApplyWaves)), block(64 * kApplyWaves);
    if (v_dtype == DSALT_DTYPE_BF16) hipLaunchKernelGGL((apply_kernel<DX, BF16>), grid, block, 0, stream, p);
    else if (v_dtype == DSALT_DTYPE_F16) hipLaunchKernelGGL((apply_kernel<DX, F16>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((apply_kernel<DX, F32>), grid, block, 0, stream, p);
}

WeightParams make_params(const dsalt_lmk_weights_args &a) {
    WeightParams p{};
    const NormsView n = scores_workspace_view(const_cast<void *>(a.norms), a.total_len, a.n_kv_heads);
    p.xn = n.xn;
    p.vn = n.vn;
    p.part = n.part;
    p.nblk = n.nblk;
    p.stats = n.stats;
    p.alpha = a.alpha;
    p.pos = a.lmk_pos;
    p.cu = a.cu_seqlens;
    p.weight = a.weight;
    p.T = a.total_len;
    p.S = a.num_seqs;
    p.H = a.n_heads;
    p.n_kv = a.n_kv_heads;
    p.rep = a.n_heads / a.n_kv_heads;
    p.k = a.k_lmk;
    p.table = a.table != 0;
    p.tau = a.tau;
    p.inv_tau = 1.f / a.tau;
    return p;
}

}  // namespace

int64_t lmk_weights_workspace_bytes(int total_len, int n_heads) {
    auto al = [](int64_t b) { return (b + 255) & ~(int64_t)255; };
    return al((int64_t)n_heads * total_len * 4) + al((int64_t)n_heads * 3 * 8);
}

hipError_t launch_lmk_weights(const dsalt_lmk_weights_args &a, hipStream_t stream) {
    if (a.total_len == 0) return hipSuccess;
    const WeightParams p = make_params(a);
    const int threads = p.table ? kTableThreads : kWThreads;
    hipLaunchKernelGGL(weight_kernel, dim3((unsigned)(p.H * p.S)), dim3(threads), 0, stream, p);
    return hipGetLastError();
}

hipError_t launch_lmk_weights_bwd(const dsalt_lmk_weights_args &a, hipStream_t stream) {
    if (a.total_len == 0) return hipSuccess;
    WeightParams p = make_params(a);
    p.g = a.d_weight;
    char *ws = static_cast<char *>(a.workspace);
    p.gz = reinterpret_cast<float *>(ws);
    p.hsum = reinterpret_cast<double *>(ws + (((int64_t)p.H * p.T * 4 + 255) & ~(int64_t)255));
    p.d_alpha = a.d_alpha;
    p.x = a.x;
    p.v = a.v;
    p.dv_in = a.dv_in;
    p.dx = a.dx;
    p.dv = a.dv;
    p.x_st = a.x_stride_t;
    p.v_st = a.v_stride_t;
    p.v_sh = a.v_stride_h;
    p.di_st = a.dv_in_stride_t;
    p.di_sh = a.dv_in_stride_h;
    p.d = a.d_model;
    p.D = a.head_dim;
    hipLaunchKernelGGL(reduce_kernel, dim3((unsigned)p.H), dim3(kTableThreads), 0, stream, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || (!p.dx && !p.dv)) return e;
    if (a.x_dtype == DSALT_DTYPE_BF16) launch_apply<BF16>(a.v_dtype, p, stream);
    else if (a.x_dtype == DSALT_DTYPE_F16) launch_apply<F16>(a.v_dtype, p, stream);
    else launch_apply<F32>(a.v_dtype, p, stream);
    return hipGetLastError();
}

}  // namespace dsalt
