// rb_fft64.h -- complex FP64 convolution of length L = 2^LOG2L in LDS, sixteen points per thread.
//
// Both transforms use the butterfly (a + w b, a - w b), six FMAs: the sum in four, the difference as
// 2 a minus the sum.  Forward, from natural to bit-reversed order, as the reduction of
// x(z) mod z^L - 1 by its factors: the stage of distance 2^s maps x mod z^(2^(s+1)) - c^2 to
// x mod z^(2^s) -+ c, so that its twiddle c depends on the block alone (c = e^(-i pi f),
// f = rev(block) / blocks) and the first pass, one block, multiplies by sixteenth roots of unity
// only.  Backward, from bit-reversed to natural order, by decimation in time (twiddles by position;
// the last R stages' sixteen points start at position 0: constants again).
//
// Stages run in passes over groups of 16 points in registers, thread t's points at i0 + k 2^SB:
// forward SB = LOG2L - 4, LOG2L - 8, ..., then the middle pass on 16 consecutive points (the last
// R = 1..4 stages, the product with the spectrum, the first R stages back), then the passes in
// reverse.  Element i sits in slot i + i / 16: every pass's accesses spread over the banks.
#pragma once
#include <hip/hip_runtime.h>

namespace rb {

template <int LOG2L>
struct Fft64 {
    static constexpr int L = 1 << LOG2L, TP = L / 16;                  // points, threads
    static constexpr int R = LOG2L % 4 == 0 ? 4 : LOG2L % 4;           // stages of the middle pass
    static constexpr int PASSES = (LOG2L - R) / 4;                     // full passes each way
    static constexpr int SLOTS = L + L / 16;
    // tables: forward passes 1 .. PASSES - 1 and the middle pass ([8][blocks] each; pass 0 has
    // constants), then backward passes PASSES - 1 .. 0 ([8][2^SB])
    static constexpr int sb(int pass) { return LOG2L - 4 * (pass + 1); }
    static constexpr int fwd_off(int pass) {  // pass = PASSES: the middle pass
        int o = 0;
        for (int p = 1; p < pass; ++p) o += 8 << (4 * p);
        return o;
    }
    static constexpr int mid_off() { return fwd_off(PASSES); }
    static constexpr int inv_off(int pass) {
        int o = mid_off() + 8 * TP;
        for (int p = PASSES - 1; p > pass; --p) o += 8 << sb(p);
        return o;
    }
    static constexpr int TABLE = inv_off(0) + (8 << (LOG2L - 4));
};

__device__ __forceinline__ int fpad64(int i) { return i + (i >> 4); }

__device__ __forceinline__ void bfly64(double2& a, double2& b, double2 w) {
    const double2 t = a;
    a.x = fma(-w.y, b.y, fma(w.x, b.x, t.x));
    a.y = fma(w.y, b.x, fma(w.x, b.y, t.y));
    b.x = fma(2.0, t.x, -a.x);
    b.y = fma(2.0, t.y, -a.y);
}
// w = 1, and w = -i (SIGN = -1) or i
__device__ __forceinline__ void bfly64_one(double2& a, double2& b) {
    const double2 t = a, u = b;
    a = make_double2(t.x + u.x, t.y + u.y);
    b = make_double2(t.x - u.x, t.y - u.y);
}
template <int SIGN>
__device__ __forceinline__ void bfly64_rot(double2& a, double2& b) {
    const double2 t = a, u = SIGN < 0 ? make_double2(b.y, -b.x) : make_double2(-b.y, b.x);
    a = make_double2(t.x + u.x, t.y + u.y);
    b = make_double2(t.x - u.x, t.y - u.y);
}

constexpr double C8 = 0.92387953251128673848, S8 = 0.38268343236508978178, C4 = 0.70710678118654752440;

// Forward stage r (distance 2^r in the group): its block kb = k >> (r + 1) of 2^(3 - r) has the
// twiddle in slot base + kb / 2 for even kb, -i times that for odd.  Bases: r = 3, 2, 1, 0 at
// 0, 1, 2, 4.  UNIT: the group is the transform's first (constants).
template <int r, bool UNIT>
__device__ __forceinline__ void fft64_fwd_stage(double2 (&x)[16], const double2* w) {
    constexpr int base = r == 3 ? 0 : r == 2 ? 1 : r == 1 ? 2 : 4;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        if (k & (1 << r)) continue;
        const int kb = k >> (r + 1), s = kb >> 1;
        double2 &a = x[k], &b = x[k + (1 << r)];
        if constexpr (UNIT) {
            // f of block 2 s: rev(2 s) / blocks = 0, 1/4, 1/8, 3/8
            if (s == 0) {
                if (kb & 1) bfly64_rot<-1>(a, b);
                else bfly64_one(a, b);
            } else {
                const double2 c = s == 1 ? make_double2(C4, -C4) : s == 2 ? make_double2(C8, -S8) : make_double2(S8, -C8);
                bfly64(a, b, kb & 1 ? make_double2(c.y, -c.x) : c);
            }
        } else {
            const double2 c = w[base + s];
            bfly64(a, b, kb & 1 ? make_double2(c.y, -c.x) : c);
        }
    }
}

// Backward stage r: twiddle e^(i pi (pos + 2^SB m) / 2^(SB + r)) of m = k mod 2^r: slot base + m
// for m below half, i times that of m - half above.  Bases: r = 0, 1, 2, 3 at 0, 1, 2, 4.  UNIT:
// pos = 0 and SB = 0.  HALF: only the lower outputs are wanted.
template <int r, bool UNIT, bool HALF>
__device__ __forceinline__ void fft64_inv_stage(double2 (&x)[16], const double2* w) {
    constexpr int base = r == 0 ? 0 : r == 1 ? 1 : r == 2 ? 2 : 4, half = r == 0 ? 1 : 1 << (r - 1);
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        if (k & (1 << r)) continue;
        const int m = k & ((1 << r) - 1), s = m >= half ? m - half : m;
        const bool rot = m >= half;
        double2 &a = x[k], &b = x[k + (1 << r)];
        if constexpr (UNIT) {
            if (s == 0) {
                if (rot) bfly64_rot<1>(a, b);
                else bfly64_one(a, b);
            } else {
                const double2 c = r == 2 || s == 2 ? make_double2(C4, C4) : s == 1 ? make_double2(C8, S8) : make_double2(S8, C8);
                bfly64(a, b, rot ? make_double2(-c.y, c.x) : c);
            }
        } else {
            const double2 c = w[base + s], v = rot ? make_double2(-c.y, c.x) : c;
            if constexpr (HALF) {
                a.x = fma(-v.y, b.y, fma(v.x, b.x, a.x));
                a.y = fma(v.y, b.x, fma(v.x, b.y, a.y));
            } else {
                bfly64(a, b, v);
            }
        }
    }
}

// The transform's runner: `sync` meets the TP threads of one transform.
template <int LOG2L, class Sync>
struct Fft64Run {
    using F = Fft64<LOG2L>;
    double2* z;                        // SLOTS
    const double2* __restrict__ tab;   // F::TABLE
    int t;                             // 0 .. TP - 1
    Sync sync;

    template <int SB>
    __device__ __forceinline__ int slot() const {
        return fpad64(((t >> SB) << (SB + 4)) + (t & ((1 << SB) - 1)));
    }
    template <int SB>
    __device__ __forceinline__ void load(double2 (&x)[16]) const {
        const double2* p = z + slot<SB>();
#pragma unroll
        for (int k = 0; k < 16; ++k) x[k] = p[(k << SB) + ((k << SB) >> 4)];
    }
    template <int SB>
    __device__ __forceinline__ void store(const double2 (&x)[16]) const {
        double2* p = z + slot<SB>();
#pragma unroll
        for (int k = 0; k < 16; ++k) p[(k << SB) + ((k << SB) >> 4)] = x[k];
    }
    template <int PASS>
    __device__ __forceinline__ void fwd_from(double2 (&x)[16]) const {
        if constexpr (PASS < F::PASSES) {
            constexpr int SB = F::sb(PASS), NB = 1 << (4 * PASS);
            double2 w[8];
#pragma unroll
            for (int s = 0; s < 8; ++s) w[s] = tab[F::fwd_off(PASS) + s * NB + (t >> SB)];
            sync();
            load<SB>(x);
            fft64_fwd_stage<3, false>(x, w);
            fft64_fwd_stage<2, false>(x, w);
            fft64_fwd_stage<1, false>(x, w);
            fft64_fwd_stage<0, false>(x, w);
            store<SB>(x);
            fwd_from<PASS + 1>(x);
        }
    }
    // Forward transform of the first L / 2 points (the rest are zero) into the middle pass's
    // registers: spectrum element 16 t + k in x[k].  z holds the points, every thread's written.
    __device__ __forceinline__ void forward(double2 (&x)[16]) const {
        constexpr int SB = F::sb(0);
        sync();
        {
            const double2* p = z + slot<SB>();
#pragma unroll
            for (int k = 0; k < 8; ++k) x[k + 8] = x[k] = p[(k << SB) + ((k << SB) >> 4)];
        }
        fft64_fwd_stage<2, true>(x, nullptr);
        fft64_fwd_stage<1, true>(x, nullptr);
        fft64_fwd_stage<0, true>(x, nullptr);
        store<SB>(x);
        fwd_from<1>(x);
        double2 w[8];
#pragma unroll
        for (int s = 0; s < 8; ++s)
            if (F::R == 4 || (F::R == 3 && s >= 1) || (F::R == 2 && s >= 2) || s >= 4)
                w[s] = tab[F::mid_off() + s * F::TP + t];
        sync();
        load<0>(x);
        if constexpr (F::R == 4) fft64_fwd_stage<3, false>(x, w);
        if constexpr (F::R >= 3) fft64_fwd_stage<2, false>(x, w);
        if constexpr (F::R >= 2) fft64_fwd_stage<1, false>(x, w);
        fft64_fwd_stage<0, false>(x, w);
    }
    template <int PASS>
    __device__ __forceinline__ void inv_from(double2 (&x)[16]) const {
        constexpr int SB = F::sb(PASS);
        double2 w[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) w[s] = tab[F::inv_off(PASS) + (s << SB) + (t & ((1 << SB) - 1))];
        sync();
        load<SB>(x);
        fft64_inv_stage<0, false, false>(x, w);
        fft64_inv_stage<1, false, false>(x, w);
        fft64_inv_stage<2, false, false>(x, w);
        fft64_inv_stage<3, false, PASS == 0>(x, w);
        if constexpr (PASS > 0) {
            store<SB>(x);
            inv_from<PASS - 1>(x);
        } else {
            double2* p = z + slot<SB>();
#pragma unroll
            for (int k = 0; k < 8; ++k) p[(k << SB) + ((k << SB) >> 4)] = x[k];
        }
    }
    // Backward transform from the middle pass's registers: the first L / 2 points into z
    __device__ __forceinline__ void backward(double2 (&x)[16]) const {
        fft64_inv_stage<0, true, false>(x, nullptr);
        if constexpr (F::R >= 2) fft64_inv_stage<1, true, false>(x, nullptr);
        if constexpr (F::R >= 3) fft64_inv_stage<2, true, false>(x, nullptr);
        if constexpr (F::R == 4) fft64_inv_stage<3, true, false>(x, nullptr);
        store<0>(x);
        inv_from<F::PASSES - 1>(x);
        sync();
    }
};

}  // namespace rb
