// Gates on 16 amplitudes that a thread holds in registers (4 index bits are
// its register slots), and the padding of the LDS tile they come from: shared
// by the tile passes of compiled schedules (tile.hip) and the runs of
// uncompiled ops (runs.hip).
#ifndef AQS_REGOPS_H
#define AQS_REGOPS_H

#include <hip/hip_runtime.h>

#include <cstdint>

namespace aqs_hip {

// Two padding amplitudes after every 32 keep LDS accesses of strided layouts
// spread over the banks and keep amplitude pairs 16-byte aligned.
__device__ __forceinline__ uint32_t lds_pad(uint32_t l) { return l + ((l >> 5) << 1); }
constexpr uint32_t lds_len(uint32_t tile) { return tile + (tile >> 4); }

template <typename T2>
struct Cplx;
template <>
struct Cplx<float2> {
    using R = float;
};
template <>
struct Cplx<double2> {
    using R = double;
};

template <typename T2, typename R>
__device__ __forceinline__ T2 cmul(R fr, R fi, T2 x) {
    T2 y;
    y.x = fr * x.x - fi * x.y;
    y.y = fr * x.y + fi * x.x;
    return y;
}

template <typename T2, typename R>
__device__ __forceinline__ void butterfly(T2& p, T2& q, const R (&m)[8]) {
    T2 u, v;
    u.x = m[0] * p.x - m[1] * p.y + m[2] * q.x - m[3] * q.y;
    u.y = m[0] * p.y + m[1] * p.x + m[2] * q.y + m[3] * q.x;
    v.x = m[4] * p.x - m[5] * p.y + m[6] * q.x - m[7] * q.y;
    v.y = m[4] * p.y + m[5] * p.x + m[6] * q.y + m[7] * q.x;
    p = u;
    q = v;
}

// Real 2x2 (m[0..3] row-major) on complex amplitudes: 8 multiplies per pair
// instead of 16, for one-qubit gates whose matrix is real (H, RotY).
template <typename T2, typename R>
__device__ __forceinline__ void butterfly_real(T2& p, T2& q, const R (&m)[8]) {
    T2 u, v;
    u.x = m[0] * p.x + m[1] * q.x;
    u.y = m[0] * p.y + m[1] * q.y;
    v.x = m[2] * p.x + m[3] * q.x;
    v.y = m[2] * p.y + m[3] * q.y;
    p = u;
    q = v;
}

// q times z (m[4], m[5]), then the rotation [[c, -s], [s, c]] (c, s >= 0)
// as three shears, t = m[0] = s / (1 + c), s = m[1]: p -= t q, q += s p,
// p -= t q.  A one-qubit gate factored as a rotation between phases in 10
// multiply-adds per pair (a complex 2x2 takes 16).
template <typename T2, typename R>
__device__ __forceinline__ void butterfly_rotp(T2& p, T2& q, const R (&m)[8]) {
    T2 w;
    w.x = m[4] * q.x - m[5] * q.y;
    w.y = m[4] * q.y + m[5] * q.x;
    p.x -= m[0] * w.x;
    p.y -= m[0] * w.y;
    w.x += m[1] * p.x;
    w.y += m[1] * p.y;
    p.x -= m[0] * w.x;
    p.y -= m[0] * w.y;
    q = w;
}

// Pair operations across register slot SL (OP: 0 complex 2x2, 1 exchange,
// 2 real 2x2, 3 phase then real 2x2).  Form 0: every pair.  Form 1:
// pairs whose register index holds the control slots `creg` (uniform test,
// the partner has the same control bits since a control is never the
// target).  Form 2: per-thread predicate `ok(j)`, results selected.
template <int SL, int OP, int FORM, typename T2, typename R, typename OK>
__device__ __forceinline__ void pairs(T2 (&x)[16], const R (&m)[8], uint32_t creg, OK ok) {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
        if (j & (1 << SL)) continue;
        const int k = j | (1 << SL);
        if (FORM == 1 && ((uint32_t)j & creg) != creg) continue;
        T2 p = x[j], q = x[k];
        if (OP == 1) {
            const T2 t = p;
            p = q;
            q = t;
        } else if (OP == 2) {
            butterfly_real(p, q, m);
        } else if (OP == 3) {
            butterfly_rotp(p, q, m);
        } else {
            butterfly(p, q, m);
        }
        if (FORM == 2) {
            // component by component: a select of whole double2 values is one
            // of addresses, which keeps the array out of registers
            const bool c = ok(j);
            x[j].x = c ? p.x : x[j].x;
            x[j].y = c ? p.y : x[j].y;
            x[k].x = c ? q.x : x[k].x;
            x[k].y = c ? q.y : x[k].y;
        } else {
            x[j] = p;
            x[k] = q;
        }
    }
}

template <typename R>
__device__ __forceinline__ void cmul_acc(R& ar, R& ai, R zr, R zi) {
    const R t = ar * zr - ai * zi;
    ai = ar * zi + ai * zr;
    ar = t;
}

}  // namespace aqs_hip

#endif
