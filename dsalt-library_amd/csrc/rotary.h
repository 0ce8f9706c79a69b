// Rotary position embedding helpers shared by the RoPE kernel (rope.hip) and the score
// pass that rotates k alongside the selector norms (scores.hip).
//
// Reference: apply_rotary_emb (dsalt/kernels/window_utils.py:73-88), half-split, per
// head, for j < D/2 with cos/sin rows rounded to the tensor dtype:
//   out[j]       = x[j] c[j]             - x[j + D/2] s[j]
//   out[j + D/2] = x[j + D/2] c[j + D/2] + x[j] s[j + D/2]
// products and sum in fp32 without FMA contraction, one rounding of the result. The
// transposed rotation (the backward) swaps the signs: g -> dx with
//   dx[j]       = g[j] c[j]             + g[j + D/2] s[j + D/2]
//   dx[j + D/2] = g[j + D/2] c[j + D/2] - g[j] s[j]
#pragma once

#include "../../include/dsalt_hip.h"
#include "common.h"

#include <type_traits>

namespace dsalt {

struct F32 {};  // element tag of fp32 tensors

template <typename DT>
struct Elem;
template <>
struct Elem<BF16> {
    static __device__ __forceinline__ float ld(const void *p, int64_t i) {
        return __uint_as_float((uint32_t)static_cast<const uint16_t *>(p)[i] << 16);
    }
    // round to nearest even with the hardware conversion (v_cvt_pk_bf16_f32; NaN stays NaN): in
    // software it takes five VALU operations an element, and the rotations are VALU work
    static __device__ __forceinline__ float round(float x) { return BF16::round(x); }
    static __device__ __forceinline__ void st(void *p, int64_t i, float x) {
        static_cast<uint16_t *>(p)[i] = (uint16_t)(BF16::pack2(x, x) & 0xffffu);
    }
    template <int VW>
    static __device__ __forceinline__ void ldv(const void *p, int64_t i, float *x) {
        if constexpr (VW == 8) {
            const uint4 u = *reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(p) + i);
            const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                x[2 * e] = __uint_as_float(w[e] << 16);
                x[2 * e + 1] = __uint_as_float(w[e] & 0xffff0000u);
            }
        } else {
#pragma unroll
            for (int e = 0; e < VW; ++e) x[e] = ld(p, i + e);
        }
    }
    template <int VW>
    static __device__ __forceinline__ void stv(void *p, int64_t i, const float *x) {
        if constexpr (VW == 8) {
            uint32_t w[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                w[e] = BF16::pack2(x[2 * e], x[2 * e + 1]);
            *reinterpret_cast<uint4 *>(static_cast<uint16_t *>(p) + i) = make_uint4(w[0], w[1], w[2], w[3]);
        } else {
#pragma unroll
            for (int e = 0; e < VW; ++e) st(p, i + e, x[e]);
        }
    }
};
template <>
struct Elem<F16> {
    static __device__ __forceinline__ float ld(const void *p, int64_t i) {
        return (float)static_cast<const _Float16 *>(p)[i];
    }
    static __device__ __forceinline__ float round(float x) { return (float)(_Float16)x; }
    static __device__ __forceinline__ void st(void *p, int64_t i, float x) { static_cast<_Float16 *>(p)[i] = (_Float16)x; }
    template <int VW>
    static __device__ __forceinline__ void ldv(const void *p, int64_t i, float *x) {
        if constexpr (VW == 8) {  // one 16-byte load
            const uint4 u = *reinterpret_cast<const uint4 *>(static_cast<const _Float16 *>(p) + i);
            const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                x[2 * e] = F16::lo_f32(w[e]);
                x[2 * e + 1] = F16::hi_f32(w[e]);
            }
        } else {
#pragma unroll
            for (int e = 0; e < VW; ++e) x[e] = ld(p, i + e);
        }
    }
    template <int VW>
    static __device__ __forceinline__ void stv(void *p, int64_t i, const float *x) {
        if constexpr (VW == 8) {  // one 16-byte store
            uint32_t w[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) w[e] = F16::pack2(x[2 * e], x[2 * e + 1]);
            *reinterpret_cast<uint4 *>(static_cast<_Float16 *>(p) + i) = make_uint4(w[0], w[1], w[2], w[3]);
        } else {
#pragma unroll
            for (int e = 0; e < VW; ++e) st(p, i + e, x[e]);
        }
    }
};
template <>
struct Elem<F32> {
    static __device__ __forceinline__ float ld(const void *p, int64_t i) { return static_cast<const float *>(p)[i]; }
    static __device__ __forceinline__ float round(float x) { return x; }
    static __device__ __forceinline__ void st(void *p, int64_t i, float x) { static_cast<float *>(p)[i] = x; }
    template <int VW>
    static __device__ __forceinline__ void ldv(const void *p, int64_t i, float *x) {
        if constexpr (VW == 4) {  // one 16-byte load
            const float4 v = *reinterpret_cast<const float4 *>(static_cast<const float *>(p) + i);
            x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
        } else {
#pragma unroll
            for (int e = 0; e < VW; ++e) x[e] = ld(p, i + e);
        }
    }
    template <int VW>
    static __device__ __forceinline__ void stv(void *p, int64_t i, const float *x) {
        if constexpr (VW == 4) {  // one 16-byte store
            *reinterpret_cast<float4 *>(static_cast<float *>(p) + i) = make_float4(x[0], x[1], x[2], x[3]);
        } else {
#pragma unroll
            for (int e = 0; e < VW; ++e) st(p, i + e, x[e]);
        }
    }
};

template <int VW>
__device__ __forceinline__ void ldv_f32(const float *p, float *x) {
#pragma unroll
    for (int e = 0; e < VW; ++e) x[e] = p[e];
}


// Offset of token t inside its sequence (binary search over cu_seqlens[0 .. S], its
// entries clamped to [0, T] as seq_bounds clamps them). Negative for a token before the
// first sequence.
__device__ __forceinline__ int seq_offset(const int32_t *cu, int S, int T, int t) {
    auto at = [&](int s) { return min(max(cu[s], 0), T); };
    int lo = 0, hi = S;  // cu[lo] <= t < cu[hi]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (at(mid) <= t) lo = mid;
        else hi = mid;
    }
    return t - at(lo);
}

// The table entries of VW pairs (j0 + e, j0 + e + half), rounded to DT (NaN when !in_table).
// `rep`: the row repeats its first half, which alone is read. Entries of 16-bit types are
// held in pairs (16 registers for 8 pairs instead of 32).
template <typename DT, int VW>
struct RopeVec {
    static constexpr bool PACK = VW % 2 == 0 && !std::is_same<DT, F32>::value;
    static constexpr int N = PACK ? VW / 2 : VW;
    uint32_t c0[N], c1[N], s0[N], s1[N];
    static __device__ __forceinline__ void put(const float *p, bool in_table, uint32_t (&o)[N]) {
        float x[VW];
        ldv_f32<VW>(p, x);
#pragma unroll
        for (int e = 0; e < VW; ++e) x[e] = in_table ? x[e] : NAN;
#pragma unroll
        for (int e = 0; e < N; ++e) {
            if constexpr (PACK) o[e] = DT::pack2(x[2 * e], x[2 * e + 1]);
            else o[e] = __float_as_uint(Elem<DT>::round(x[e]));
        }
    }
    static __device__ __forceinline__ float get(const uint32_t (&o)[N], int e) {
        if constexpr (PACK) return (e & 1) ? DT::hi_f32(o[e / 2]) : DT::lo_f32(o[e / 2]);
        else return __uint_as_float(o[e]);
    }
    // The entries made opaque where a loop uses them: nothing unpacked from them is kept
    // across its iterations.
    __device__ __forceinline__ void pin() {
#pragma unroll
        for (int e = 0; e < N; ++e) asm volatile("" : "+v"(c0[e]), "+v"(c1[e]), "+v"(s0[e]), "+v"(s1[e]));
    }
    // LEAN: the second halves are read after the first are packed (fewer registers at once)
    template <bool LEAN = false>
    __device__ __forceinline__ void load(const float *cr, const float *sr, int half, int j0, bool in_table, bool rep) {
        put(cr + j0, in_table, c0);
        put(sr + j0, in_table, s0);
        if constexpr (LEAN) __builtin_amdgcn_sched_barrier(0);
        if (rep) {
#pragma unroll
            for (int e = 0; e < N; ++e) {
                c1[e] = c0[e];
                s1[e] = s0[e];
            }
        } else {
            put(cr + j0 + half, in_table, c1);
            put(sr + j0 + half, in_table, s1);
        }
    }
};

// Rotate the VW pairs (j0 + e, j0 + e + half) of one head row: reads in[ib + ...], writes
// out[ob + ...] (out may alias in: each pair is read before it is written).
// The products are never contracted into an FMA with the sum, and each fp32 result is made
// opaque before its conversion to the 16-bit type: otherwise the backend may fold the sum
// and the conversion into one mixed-precision v_fma_mix{lo,hi}_f16, which rounds the exact
// sum once instead of to fp32 first.
// DO: element type of the output (the rotated value rounded to DT, then to DO).
template <typename DT, int VW, typename DO = DT>
__device__ __forceinline__ void rotate_pairs(const void *in, int64_t ib, void *out, int64_t ob, const RopeVec<DT, VW> &t,
                                             int half, int j0, bool transpose) {
    // element e of the pair (a, b): its two rotated values, each rounded to fp32 once
    auto rot = [&](float a, float b, int e, float &o0, float &o1) {
        const float c0 = t.get(t.c0, e), c1 = t.get(t.c1, e), s0 = t.get(t.s0, e), s1 = t.get(t.s1, e);
        // the four products; those of 16-bit values are exact in fp32, fp32 ones are made opaque
        // so that the backend (-ffp-contract=fast) fuses none into the sums
        float ac = a * c0, bc = b * c1, as = a * (transpose ? s0 : s1), bs = b * (transpose ? s1 : s0);
        if constexpr (std::is_same<DT, F32>::value) asm volatile("" : "+v"(ac), "+v"(bc), "+v"(as), "+v"(bs));
        o0 = transpose ? ac + bs : ac - bs;
        o1 = transpose ? bc - as : bc + as;
        asm volatile("" : "+v"(o0), "+v"(o1));
    };
    if constexpr (VW == 8 && !std::is_same<DT, F32>::value && std::is_same<DT, DO>::value) {
        // 16-bit rows stay packed: two pairs unpacked at a time (half the registers)
        const uint16_t *src = static_cast<const uint16_t *>(in) + ib + j0;
        const uint4 a4 = *reinterpret_cast<const uint4 *>(src), b4 = *reinterpret_cast<const uint4 *>(src + half);
        const uint32_t aw[4] = {a4.x, a4.y, a4.z, a4.w}, bw[4] = {b4.x, b4.y, b4.z, b4.w};
        uint32_t ow0[4], ow1[4];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            float p0, p1, q0, q1;
            rot(DT::lo_f32(aw[w]), DT::lo_f32(bw[w]), 2 * w, p0, q0);
            rot(DT::hi_f32(aw[w]), DT::hi_f32(bw[w]), 2 * w + 1, p1, q1);
            ow0[w] = DT::pack2(p0, p1);
            ow1[w] = DT::pack2(q0, q1);
        }
        uint16_t *dst = static_cast<uint16_t *>(out) + ob + j0;
        *reinterpret_cast<uint4 *>(dst) = make_uint4(ow0[0], ow0[1], ow0[2], ow0[3]);
        *reinterpret_cast<uint4 *>(dst + half) = make_uint4(ow1[0], ow1[1], ow1[2], ow1[3]);
    } else {
        float a[VW], b[VW], o0[VW], o1[VW];
        Elem<DT>::template ldv<VW>(in, ib + j0, a);
        Elem<DT>::template ldv<VW>(in, ib + j0 + half, b);
#pragma unroll
        for (int e = 0; e < VW; ++e) rot(a[e], b[e], e, o0[e], o1[e]);
        Elem<DO>::template stv<VW>(out, ob + j0, o0);
        Elem<DO>::template stv<VW>(out, ob + j0 + half, o1);
    }
}
template <typename DT, int VW>
__device__ __forceinline__ void rotate_vec(const void *in, int64_t ib, void *out, int64_t ob, const float *cr,
                                           const float *sr, int half, int j0, bool in_table, bool transpose) {
    RopeVec<DT, VW> t;
    t.load(cr, sr, half, j0, in_table, false);
    rotate_pairs<DT, VW>(in, ib, out, ob, t, half, j0, transpose);
}

// RoPE tables of a gradient epilogue (dsalt_rope_tables): rows of head_dim fp32 entries,
// each rounded to `round_dtype` as it is read; cos = null: no rotation.
struct RopeRows {
    const float *cos, *sin;
    int64_t st;
    int rows, half, round_dtype;
};

// The RopeRows at byte offset `off` of the kernel's argument block, read here: through the
// parameter itself the compiler loads the six fields at kernel entry and holds them in
// scalar registers across the tile loops, which have none to spare.
__device__ __forceinline__ RopeRows late_rope_rows(size_t off) {
    typedef const __attribute__((address_space(4))) char *kptr;
    uint64_t a = (uint64_t)(kptr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(a));
    const __attribute__((address_space(4))) RopeRows *r = (const __attribute__((address_space(4))) RopeRows *)(a + off);
    RopeRows t;
    t.cos = r->cos;
    t.sin = r->sin;
    t.st = r->st;
    t.rows = r->rows;
    t.half = r->half;
    t.round_dtype = r->round_dtype;
    return t;
}

inline RopeRows rope_rows(const dsalt_rope_tables *t) {
    RopeRows r{};
    if (t) {
        r.cos = t->cos;
        r.sin = t->sin;
        r.st = t->stride;
        r.rows = t->rows;
        r.half = t->half;
        r.round_dtype = t->round_dtype;
    }
    return r;
}

// The transposed rotation of one gradient row held as D/32 transposed 32x32 accumulator
// blocks (registers = head-dim d*32 + (r/4)*8 + hh*4 + r%4: a lane holds both elements of
// each of its pairs, in blocks d and d + ND/2), scaled by `mul` first; `pos` the row's
// position in its sequence (NaN outside the table, as rotate_vec). fp32 throughout: the
// caller's store rounds once.
template <typename DT, bool ROUND, int ND>
__device__ __forceinline__ void rotate_acc_rounded(f32x16 (&acc)[ND], float mul, const RopeRows &t, int pos, int hh) {
    const bool in_table = pos >= 0 && pos < t.rows;
    const float *cr = t.cos + (int64_t)(in_table ? pos : 0) * t.st, *sr = t.sin + (int64_t)(in_table ? pos : 0) * t.st;
    if (!in_table) mul = NAN;
    auto ld4 = [](const float *p, float (&o)[4]) {
        const float4 v = *reinterpret_cast<const float4 *>(p);
        if constexpr (ROUND) {
            const uint32_t a = DT::pack2(v.x, v.y), b = DT::pack2(v.z, v.w);
            o[0] = DT::lo_f32(a); o[1] = DT::hi_f32(a); o[2] = DT::lo_f32(b); o[3] = DT::hi_f32(b);
        } else {
            o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
        }
    };
#pragma unroll
    for (int d = 0; d < ND / 2; ++d) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            // one block pair's table loads in flight at a time: all of them at D = 128 cost
            // the kernels around this a wave per SIMD
            if (g == 0) __builtin_amdgcn_sched_barrier(0);
            const int lo = d * 32 + g * 8 + hh * 4;
            float ca[4], sa[4], cb[4], sb[4];
            ld4(cr + lo, ca);
            ld4(sr + lo, sa);
            if (t.half) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    cb[e] = ca[e];
                    sb[e] = sa[e];
                }
            } else {
                ld4(cr + lo + ND * 16, cb);
                ld4(sr + lo + ND * 16, sb);
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float a = acc[d][g * 4 + e] * mul, b = acc[d + ND / 2][g * 4 + e] * mul;
                acc[d][g * 4 + e] = a * ca[e] + b * sb[e];
                acc[d + ND / 2][g * 4 + e] = b * cb[e] - a * sa[e];
            }
        }
    }
}
// round_dtype is DT's or fp32 (checked on the host). A run-time choice per table entry
// (three conversions and two selects each) made this epilogue 12 us of the dq pass and
// 16 us of the band pass at 9290 tokens x 16 x 64.
template <typename DT, int ND>
__device__ __forceinline__ void rotate_acc_transposed(f32x16 (&acc)[ND], float mul, const RopeRows &t, int pos, int hh) {
    if (t.round_dtype == DSALT_DTYPE_F32) rotate_acc_rounded<DT, false, ND>(acc, mul, t, pos, hh);
    else rotate_acc_rounded<DT, true, ND>(acc, mul, t, pos, hh);
}

}  // namespace dsalt
