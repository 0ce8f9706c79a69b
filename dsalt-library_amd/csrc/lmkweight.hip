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
// latency. Both walk the sequences: 4.7 and 6.5 us up to 8 of them, 25 and 32 at 300 (9300
// tokens), 148 and 198 at 2000 (10000 tokens; each of H x S workgroups re-sums the partials).
// The module's own function (dsalt_module_grads_v / _x) splits the apply pass around the
// projections' GEMMs:
//   grads_v_kernel  one wave per token: dv = value-norm share + the attention's dv (summed over
//                   grouped heads; dk likewise), written where the GEMMs read them.
//   grads_x_kernel  8 to 32 tokens per workgroup, threads own columns: dx = the GEMM's dx + norm
//                   share + d_logit w of the window gate, and the gate weight's partial
//                   gradient sums (one row per workgroup), summed by gate_kernel.
// One pass over x, dx_in and dx (19.3 us at that shape; grads_v 13.0, gate 8.8) instead of
// torch's outer-product GEMM, GEMV, bias sum and three additions over [T, d].
// A training step of the module at that shape: 1985 us with torch's ops (152 launches, GPU
// busy 1391 us), 1146 with the weights here (46, 888), 716 with everything between x and
// the attention's output as one function (23, 662).
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
    int alpha_sigmoid;      // d_alpha is that of alpha_w, alpha = sigmoid(alpha_w)
    // module gradients
    const void *kh, *vh;    // per-query-head dk, dv [T, H, D]
    void *dk;
    int64_t kh_st, kh_sh, vh_st, vh_sh, dk_st, dk_sh, dv_st, dv_sh;
    const void *dx_in;      // [T, d] or null
    const void *win_w;      // [d] in x's dtype or null (no gate)
    const float *win_logit, *d_w;
    float *part_w;          // [n_xblk][d + 1]: the workgroups' sums of d_win_w, d_win_b
    void *d_win_w, *d_win_b;
    int n_xblk, x_tok, win_dt;
    float n_min, span;
};

// log(max(sigmoid(s / tau), 1e-20)) as torch's fp32 ops form it (a NaN score gives NaN).
__device__ __forceinline__ float lmk_weight(float s, float tau) {
    const float sg = 1.f / (1.f + expf(-s / tau));
    return logf(sg < kSigClamp ? kSigClamp : sg);
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
        // where a norm is not finite torch's std, and with it every score, is NaN
        if (!(fabsf(m) < INFINITY)) sd = NAN;
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
        const float ds = sg < kSigClamp ? 0.f : gw * (1.f - sg) * p.inv_tau;
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
        // NaN scores are never selected, but through an empty slot's (or an unselected key's) zero
        // gradient they still make every gradient NaN, as in torch: 0 times NaN
        if ((sx != sx || sv != sv) && (p.k > 0 || p.table)) t0 = t1 = t2 = NAN;
        p.hsum[3 * head] = t0;
        p.hsum[3 * head + 1] = t1;
        p.hsum[3 * head + 2] = t2;
        if (p.d_alpha) {
            const float da = (float)(t1 - t2);
            p.d_alpha[head] = p.alpha_sigmoid ? da * (1.f - alpha) * alpha : da;
        }
    }
}

// Gradient of norm n (standardised to z = (n - mean) / sd over T tokens) divided by n, from
// z's gradient dz and the sums A = sum dz, B = sum dz z over the tokens: the row's own
// gradient is this times the row (0 for a zero row, as torch masks it, and where no
// gradient comes in, whatever the std). A clamped std takes no gradient.
__device__ __forceinline__ float norm_coef(float n, float mean, float sd, float dz, double A, double B, int T) {
    if (n == 0.f || (dz == 0.f && A == 0.0 && B == 0.0)) return 0.f;
    const float z = hybrid_z(n, mean, sd);
    float dn = dz - (float)(A / T);
    if (sd > 1e-6f) dn -= z * (float)(B / (T - 1));
    return dn / sd / n;
}

// The quantities' sums (A = sum dz, B = sum dz z) from the heads' sums, in head order.
__device__ __forceinline__ void quantity_sums(const WeightParams &p, int q, double &A, double &B) {
    A = 0.0;
    B = 0.0;
    const int h0 = q == 0 ? 0 : (q - 1) * p.rep, h1 = q == 0 ? p.H : h0 + p.rep;
    for (int h = h0; h < h1; ++h) {
        const double a = q == 0 ? 1.0 - (double)p.alpha[h] : (double)p.alpha[h];
        A += a * p.hsum[3 * h];
        B += a * p.hsum[3 * h + (q == 0 ? 2 : 1)];
    }
}

template <typename DX, typename DV>
__global__ void __launch_bounds__(64 * kApplyWaves) apply_kernel(const WeightParams p) {
    constexpr int EX = std::is_same<DX, F32>::value ? 4 : 8, EV = std::is_same<DV, F32>::value ? 4 : 8;
    __shared__ double s_ab[1 + kMaxKvW][2];
    __shared__ float s_c[kApplyWaves][kMaxKvW];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int q = tid; q <= p.n_kv; q += blockDim.x) quantity_sums(p, q, s_ab[q][0], s_ab[q][1]);
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

// 8 (or 4) consecutive elements of an array of element type DI as fp32.
template <typename DI, int N>
__device__ __forceinline__ void load_f32(const void *p, int64_t i, float (&x)[N]) {
    if constexpr (std::is_same<DI, F32>::value && N == 8) {
        Elem<F32>::template ldv<4>(p, i, x);
        Elem<F32>::template ldv<4>(p, i + 4, x + 4);
    } else {
        Elem<DI>::template ldv<N>(p, i, x);
    }
}

template <typename DV, typename DH>
__global__ void __launch_bounds__(64 * kApplyWaves) grads_v_kernel(const WeightParams p) {
    constexpr int EV = std::is_same<DV, F32>::value ? 4 : 8;
    __shared__ double s_ab[kMaxKvW][2];
    __shared__ float s_c[kApplyWaves][kMaxKvW];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    for (int g = tid; g < p.n_kv; g += blockDim.x) quantity_sums(p, 1 + g, s_ab[g][0], s_ab[g][1]);
    __syncthreads();
    const int t = blockIdx.x * kApplyWaves + wave;
    const bool live = t < p.T;  // wave-uniform
    for (int g = lane; live && g < p.n_kv; g += 64) {
        float dzv = 0.f;
        for (int r = 0; r < p.rep; ++r) {
            const int h = g * p.rep + r;
            dzv += p.alpha[h] * p.gz[(int64_t)h * p.T + t];
        }
        s_c[wave][g] = norm_coef(p.vn[(int64_t)t * p.n_kv + g], p.stats[2 + 2 * g], p.stats[3 + 2 * g], dzv,
                                 s_ab[g][0], s_ab[g][1], p.T);
    }
    __syncthreads();
    if (!live) return;
    const int G = p.D / EV;
    for (int c = lane; c < p.n_kv * G; c += 64) {
        const int g = c / G, j = (c - g * G) * EV;
        float a[EV], b[EV];
        Elem<DV>::template ldv<EV>(p.v, (int64_t)t * p.v_st + (int64_t)g * p.v_sh + j, a);
        const int64_t vb = (int64_t)t * p.vh_st + (int64_t)g * p.rep * p.vh_sh + j;
        load_f32<DH>(p.vh, vb, b);
        for (int r = 1; r < p.rep; ++r) {
            float x[EV];
            load_f32<DH>(p.vh, vb + (int64_t)r * p.vh_sh, x);
#pragma unroll
            for (int e = 0; e < EV; ++e) b[e] += x[e];
        }
        const float cg = s_c[wave][g];
#pragma unroll
        for (int e = 0; e < EV; ++e) a[e] = fmaf(cg, a[e], b[e]);
        Elem<DV>::template stv<EV>(p.dv, (int64_t)t * p.dv_st + (int64_t)g * p.dv_sh + j, a);
        if (p.kh) {
            const int64_t kb = (int64_t)t * p.kh_st + (int64_t)g * p.rep * p.kh_sh + j;
            load_f32<DH>(p.kh, kb, b);
            for (int r = 1; r < p.rep; ++r) {
                float x[EV];
                load_f32<DH>(p.kh, kb + (int64_t)r * p.kh_sh, x);
#pragma unroll
                for (int e = 0; e < EV; ++e) b[e] += x[e];
            }
            Elem<DV>::template stv<EV>(p.dk, (int64_t)t * p.dk_st + (int64_t)g * p.dk_sh + j, b);
        }
    }
}

constexpr int kXTokens = 32;    // most tokens per workgroup of grads_x_kernel
constexpr int kXThreads = 256;
constexpr int kXBatch = 4;      // tokens whose rows a thread loads together

// Tokens per workgroup: a thread walks its share of them in latency-bound steps, so small
// batches take few (1001 tokens x 1024: 126 workgroups), large ones more (fewer rows of
// partial sums for gate_kernel). With 8 / 16 / 32 the two kernels take, at d = 1024 in bf16, 2048
// tokens 14.4 / 16.2 / 20.4 us, 4096 18.3 / 16.6 / 21.9, 9290 37.4 / 27.8 / 26.7, 16384 53.3 /
// 36.8 / 32.4; at d = 4096, 2048 29 / 39 / 64, 9290 75 / 56 / 75, 16384 125 / 105 / 112.
inline int x_tokens(int T) { return T >= 16384 ? 32 : T >= 4096 ? 16 : 8; }

__device__ __forceinline__ float round_win(float v, int dt) {
    return dt == DSALT_DTYPE_BF16 ? BF16::round(v) : dt == DSALT_DTYPE_F16 ? F16::round(v) : v;
}

template <typename DX, typename DI>
__global__ void __launch_bounds__(kXThreads) grads_x_kernel(const WeightParams p) {
    constexpr int E = std::is_same<DX, F32>::value ? 4 : 8;
    __shared__ double s_ab[2];
    __shared__ float s_cx[kXTokens], s_dl[kXTokens];
    __shared__ float s_acc[kXThreads][E + 1];
    const int tid = threadIdx.x;
    const int t0 = blockIdx.x * p.x_tok, nt = min(p.x_tok, p.T - t0);
    if (tid == 0) quantity_sums(p, 0, s_ab[0], s_ab[1]);
    // 8 threads per token sum its heads' score gradients
    const int tk = tid >> 3, sub = tid & 7;
    float dz = 0.f;
    if (tk < nt)
        for (int h = sub; h < p.H; h += 8) dz += (1.f - p.alpha[h]) * p.gz[(int64_t)h * p.T + t0 + tk];
#pragma unroll
    for (int o = 1; o < 8; o <<= 1) dz += __shfl_xor(dz, o);
    __syncthreads();
    if (sub == 0) {
        float cx = 0.f, dl = 0.f;
        if (tk < nt) {
            cx = norm_coef(p.xn[t0 + tk], p.stats[0], p.stats[1], dz, s_ab[0], s_ab[1], p.T);
            if (p.win_w) {
                const float sg = round_win(1.f / (1.f + expf(-p.win_logit[t0 + tk])), p.win_dt);
                dl = p.d_w[t0 + tk] * p.span * ((1.f - sg) * sg);
            }
        }
        s_cx[tk] = cx;
        s_dl[tk] = dl;
    }
    __syncthreads();
    // columns: chunk `ch` of E elements; tp threads share it, each with every tp-th token
    const int nch = p.d / E, per = min(nch, kXThreads), tp = kXThreads / per;
    const int grp = tid / per, ch0 = tid - grp * per;
    float *part = p.part_w + (int64_t)blockIdx.x * (p.d + 1);
    for (int cb = 0; cb < nch; cb += per) {  // workgroup-uniform
        const int ch = cb + ch0;
        const bool on = grp < tp && ch < nch;
        float acc[E], w[E];
#pragma unroll
        for (int e = 0; e < E; ++e) acc[e] = w[e] = 0.f;
        if (on) {
            if (p.win_w) {
                Elem<DX>::template ldv<E>(p.win_w, (int64_t)ch * E, w);
#pragma unroll
                for (int e = 0; e < E; ++e) w[e] = round_win(w[e], p.win_dt);
            }
            for (int k0 = grp; k0 < nt; k0 += kXBatch * tp) {
                float x[kXBatch][E], y[kXBatch][E];
#pragma unroll
                for (int u = 0; u < kXBatch; ++u) {  // every load of the batch first
                    const int64_t t = t0 + min(k0 + u * tp, nt - 1);
                    Elem<DX>::template ldv<E>(p.x, t * p.x_st + (int64_t)ch * E, x[u]);
                    if (p.dx_in) {
                        load_f32<DI>(p.dx_in, t * p.d + (int64_t)ch * E, y[u]);
                    } else {
#pragma unroll
                        for (int e = 0; e < E; ++e) y[u][e] = 0.f;
                    }
                }
#pragma unroll
                for (int u = 0; u < kXBatch; ++u) {
                    const int k = k0 + u * tp;
                    if (k >= nt) break;
                    const float cx = s_cx[k], dl = s_dl[k];
                    if (p.dx) {
#pragma unroll
                        for (int e = 0; e < E; ++e) y[u][e] += fmaf(cx, x[u][e], dl * w[e]);
                        Elem<DX>::template stv<E>(p.dx, (int64_t)(t0 + k) * p.d + (int64_t)ch * E, y[u]);
                    }
                    // the products that win_gate's forward took: x rounded to its compute type
#pragma unroll
                    for (int e = 0; e < E; ++e) acc[e] = fmaf(dl, round_win(x[u][e], p.win_dt), acc[e]);
                }
            }
        }
        if (p.win_w) {  // sums over the tp token groups, in group order
#pragma unroll
            for (int e = 0; e < E; ++e) s_acc[tid][e] = acc[e];
            __syncthreads();
            if (on && grp == 0) {
                for (int g = 1; g < tp; ++g)
#pragma unroll
                    for (int e = 0; e < E; ++e) acc[e] += s_acc[g * per + ch0][e];
#pragma unroll
                for (int e = 0; e < E; ++e) part[(int64_t)ch * E + e] = acc[e];
            }
            __syncthreads();
        }
    }
    if (p.win_w && tid == 0) {
        float b = 0.f;
        for (int k = 0; k < nt; ++k) b += s_dl[k];
        part[p.d] = b;
    }
}

// d_win_w (columns) and d_win_b (column d) from the workgroups' rows: 64 columns per
// workgroup, 4 waves over the rows, their sums added in wave order.
template <typename DX>
__global__ void __launch_bounds__(256) gate_kernel(const WeightParams p) {
    __shared__ float s_sum[4][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int c = blockIdx.x * 64 + lane;
    float a = 0.f;
    if (c <= p.d) {
#pragma unroll 8
        for (int b = wave; b < p.n_xblk; b += 4) a += p.part_w[(int64_t)b * (p.d + 1) + c];
    }
    s_sum[wave][lane] = a;
    __syncthreads();
    if (wave == 0 && c <= p.d) {
        a = ((s_sum[0][lane] + s_sum[1][lane]) + s_sum[2][lane]) + s_sum[3][lane];
        if (c < p.d) {
            if (p.d_win_w) Elem<DX>::st(p.d_win_w, c, a);
        } else if (p.d_win_b) {
            Elem<DX>::st(p.d_win_b, 0, a);
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

namespace {

WeightParams make_bwd_params(const dsalt_lmk_weights_args &a) {
    WeightParams p = make_params(a);
    p.g = a.d_weight;
    char *ws = static_cast<char *>(a.workspace);
    p.gz = reinterpret_cast<float *>(ws);
    p.hsum = reinterpret_cast<double *>(ws + (((int64_t)p.H * p.T * 4 + 255) & ~(int64_t)255));
    p.x = a.x;
    p.v = a.v;
    p.x_st = a.x_stride_t;
    p.v_st = a.v_stride_t;
    p.v_sh = a.v_stride_h;
    p.d = a.d_model;
    p.D = a.head_dim;
    return p;
}

template <typename DV>
void launch_grads_v(int heads_dtype, const WeightParams &p, hipStream_t stream) {
    const dim3 grid((unsigned)((p.T + kApplyWaves - 1) / kApplyWaves)), block(64 * kApplyWaves);
    if (heads_dtype == DSALT_DTYPE_F32) hipLaunchKernelGGL((grads_v_kernel<DV, F32>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((grads_v_kernel<DV, DV>), grid, block, 0, stream, p);
}

template <typename DX>
void launch_grads_x(int in_dtype, const WeightParams &p, hipStream_t stream) {
    const dim3 grid((unsigned)p.n_xblk), block(kXThreads);
    if (in_dtype == DSALT_DTYPE_BF16) hipLaunchKernelGGL((grads_x_kernel<DX, BF16>), grid, block, 0, stream, p);
    else if (in_dtype == DSALT_DTYPE_F16) hipLaunchKernelGGL((grads_x_kernel<DX, F16>), grid, block, 0, stream, p);
    else hipLaunchKernelGGL((grads_x_kernel<DX, F32>), grid, block, 0, stream, p);
    if (p.win_w && (p.d_win_w || p.d_win_b))
        hipLaunchKernelGGL((gate_kernel<DX>), dim3((unsigned)((p.d + 64) / 64)), dim3(256), 0, stream, p);
}

}  // namespace

int64_t module_grads_workspace_bytes(int total_len, int n_heads, int d_model) {
    const int64_t nblk = (total_len + x_tokens(total_len) - 1) / x_tokens(total_len);
    return lmk_weights_workspace_bytes(total_len, n_heads) + ((nblk * (d_model + 1) * 4 + 255) & ~(int64_t)255);
}

hipError_t launch_module_grads_v(const dsalt_module_grads_args &a, hipStream_t stream) {
    const dsalt_lmk_weights_args &w = a.weights;
    if (w.total_len == 0) return hipSuccess;
    WeightParams p = make_bwd_params(w);
    p.d_alpha = a.d_alpha;
    p.alpha_sigmoid = a.alpha_sigmoid;
    p.kh = p.rep > 1 ? a.dk_heads : nullptr;
    p.vh = a.dv_heads;
    p.kh_st = a.dkh_stride_t;
    p.kh_sh = a.dkh_stride_h;
    p.vh_st = a.dvh_stride_t;
    p.vh_sh = a.dvh_stride_h;
    p.dk = a.dk;
    p.dk_st = a.dk_stride_t;
    p.dk_sh = a.dk_stride_h;
    p.dv = a.dv;
    p.dv_st = a.dv_stride_t;
    p.dv_sh = a.dv_stride_h;
    hipLaunchKernelGGL(reduce_kernel, dim3((unsigned)p.H), dim3(kTableThreads), 0, stream, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (w.v_dtype == DSALT_DTYPE_BF16) launch_grads_v<BF16>(a.heads_dtype, p, stream);
    else if (w.v_dtype == DSALT_DTYPE_F16) launch_grads_v<F16>(a.heads_dtype, p, stream);
    else launch_grads_v<F32>(a.heads_dtype, p, stream);
    return hipGetLastError();
}

hipError_t launch_module_grads_x(const dsalt_module_grads_args &a, hipStream_t stream) {
    const dsalt_lmk_weights_args &w = a.weights;
    if (w.total_len == 0) return hipSuccess;
    WeightParams p = make_bwd_params(w);
    p.dx_in = a.dx_in;
    p.dx = a.dx;
    p.win_w = a.win_w;
    p.win_logit = a.win_logit;
    p.d_w = a.d_w;
    p.d_win_w = a.d_win_w;
    p.d_win_b = a.d_win_b;
    p.win_dt = a.win_dtype;
    p.n_min = a.n_min;
    p.span = a.n_max - a.n_min;
    p.x_tok = x_tokens(p.T);
    p.n_xblk = (p.T + p.x_tok - 1) / p.x_tok;
    p.part_w = reinterpret_cast<float *>(static_cast<char *>(w.workspace) + lmk_weights_workspace_bytes(p.T, p.H));
    if (w.x_dtype == DSALT_DTYPE_BF16) launch_grads_x<BF16>(a.in_dtype, p, stream);
    else if (w.x_dtype == DSALT_DTYPE_F16) launch_grads_x<F16>(a.in_dtype, p, stream);
    else launch_grads_x<F32>(a.in_dtype, p, stream);
    return hipGetLastError();
}

hipError_t launch_lmk_weights_bwd(const dsalt_lmk_weights_args &a, hipStream_t stream) {
    if (a.total_len == 0) return hipSuccess;
    WeightParams p = make_bwd_params(a);
    p.d_alpha = a.d_alpha;
    p.dv_in = a.dv_in;
    p.dx = a.dx;
    p.dv = a.dv;
    p.di_st = a.dv_in_stride_t;
    p.di_sh = a.dv_in_stride_h;
    hipLaunchKernelGGL(reduce_kernel, dim3((unsigned)p.H), dim3(kTableThreads), 0, stream, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || (!p.dx && !p.dv)) return e;
    if (a.x_dtype == DSALT_DTYPE_BF16) launch_apply<BF16>(a.v_dtype, p, stream);
    else if (a.x_dtype == DSALT_DTYPE_F16) launch_apply<F16>(a.v_dtype, p, stream);
    else launch_apply<F32>(a.v_dtype, p, stream);
    return hipGetLastError();
}

}  // namespace dsalt
