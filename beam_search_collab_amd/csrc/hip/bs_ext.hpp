// Arithmetic with a 64-bit significand, rounded to nearest even after every operation: what the
// reference's long double expressions compute on its x86 hosts (x87 extended precision, whose
// 15-bit exponent none of these products leaves).  Only the operations the RaBitQ factors need,
// in integers, for finite operands; callable on the host so that it can be compared with long
// double there.
#pragma once
#include <stdint.h>
#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define BSX_FN __host__ __device__ inline
#else
#define BSX_FN inline  // a plain host compiler (the comparison with long double)
#endif

namespace bsx {

// +-m * 2^e with the top bit of m set, or m = 0
struct Ext {
    uint64_t m;
    int32_t e;
    bool neg;
};

// a finite float as +-m * 2^e with 2^23 <= m < 2^24 (m = 0 for zero)
struct Parts {
    uint32_t m;
    int32_t e;
    bool neg;
};
BSX_FN Parts parts(float f) {
    const uint32_t b = __builtin_bit_cast(uint32_t, f);
    const uint32_t x = (b >> 23) & 0xFFu, f23 = b & 0x7FFFFFu;
    Parts p;
    p.neg = (b >> 31) != 0u;
    if (x != 0u) {
        p.m = f23 | 0x800000u;
        p.e = static_cast<int32_t>(x) - 150;
    } else if (f23 != 0u) {
        const int32_t s = __builtin_clz(f23) - 8;
        p.m = f23 << s;
        p.e = -149 - s;
    } else {
        p.m = 0u;
        p.e = 0;
    }
    return p;
}

// q (top bit set) plus one when `up`, the carry out of the top put into the exponent
BSX_FN Ext rounded(uint64_t q, bool up, int32_t e, bool neg) {
    Ext r = {q + (up ? 1u : 0u), e, neg};
    if (r.m == 0u) {
        r.m = 1ull << 63;
        r.e += 1;
    }
    return r;
}

// a / b, b != 0.  The 87- or 88-bit dividend is divided in two steps of 64-bit divisions; a
// quotient is never halfway between two 64-bit significands (it would have to divide exactly).
BSX_FN Ext div(float fa, float fb) {
    const Parts a = parts(fa), b = parts(fb);
    if (a.m == 0u) return Ext{0, 0, a.neg != b.neg};
    const int sh = a.m >= b.m ? 39 : 40;
    const uint64_t t = static_cast<uint64_t>(a.m) << sh;
    const uint64_t q1 = t / b.m, t2 = (t - q1 * b.m) << 24;
    const uint64_t q2 = t2 / b.m, rem = t2 - q2 * b.m;
    return rounded((q1 << 24) + q2, 2 * rem > b.m, a.e - b.e - (sh + 24), a.neg != b.neg);
}

// a * b
BSX_FN Ext mul(Ext a, float fb) {
    const Parts b = parts(fb);
    const bool neg = a.neg != b.neg;
    if (a.m == 0u || b.m == 0u) return Ext{0, 0, neg};
    const unsigned __int128 p = static_cast<unsigned __int128>(a.m) * b.m;  // 2^86 <= p < 2^88
    const int s = (p >> 87) != 0 ? 24 : 23;
    const uint64_t q = static_cast<uint64_t>(p >> s), rem = static_cast<uint64_t>(p) & ((1ull << s) - 1), half = 1ull << (s - 1);
    return rounded(q, rem > half || (rem == half && (q & 1u)), a.e + b.e + s, neg);
}

// a + b (an exact zero is +0)
BSX_FN Ext add(Ext a, Ext b) {
    if (a.m == 0u) return b;
    if (b.m == 0u) return a;
    if (b.e > a.e || (b.e == a.e && b.m > a.m)) {
        const Ext t = a;
        a = b;
        b = t;
    }
    const int32_t d = a.e - b.e;
    const unsigned __int128 A = static_cast<unsigned __int128>(a.m) << 63;
    unsigned __int128 B = static_cast<unsigned __int128>(b.m) << 63;
    if (d >= 127) {
        B = 1;  // far below: only that it is not zero matters
    } else if (d > 0) {
        const bool lost = (B & ((static_cast<unsigned __int128>(1) << d) - 1)) != 0;
        B = (B >> d) | (lost ? 1u : 0u);
    }
    const unsigned __int128 S = a.neg == b.neg ? A + B : A - B;
    if (S == 0) return Ext{0, 0, false};
    const uint64_t hi = static_cast<uint64_t>(S >> 64), lo = static_cast<uint64_t>(S);
    const int top = hi ? 127 - __builtin_clzll(hi) : 63 - __builtin_clzll(lo);
    const int s = top - 63;  // significand = bits top .. s
    if (s <= 0) return Ext{static_cast<uint64_t>(S) << -s, a.e - 63 + s, a.neg};
    const uint64_t q = static_cast<uint64_t>(S >> s);
    const unsigned __int128 one = 1, rem = S & ((one << s) - 1), half = one << (s - 1);
    return rounded(q, rem > half || (rem == half && (q & 1u)), a.e - 63 + s, a.neg);
}

// to the nearest float
BSX_FN float to_float(Ext x) {
    uint32_t bits = 0;
    if (x.m != 0u) {
        const int32_t E = x.e + 63;  // the leading bit's exponent
        if (E > 127) {
            bits = 0x7F800000u;
        } else {
            const int32_t s = E >= -126 ? 40 : 40 + (-126 - E);  // bits dropped
            if (s > 64) {
                bits = 0u;
            } else {
                const uint64_t q = s == 64 ? 0u : x.m >> s;
                const uint64_t rem = s == 64 ? x.m : x.m & ((1ull << s) - 1), half = 1ull << (s - 1);
                const uint64_t r = q + (rem > half || (rem == half && (q & 1u)) ? 1u : 0u);
                // a carry moves the sum into the next binade (or to infinity) by itself
                bits = E >= -126 ? (static_cast<uint32_t>(E + 126) << 23) + static_cast<uint32_t>(r) : static_cast<uint32_t>(r);
            }
        }
    }
    return __builtin_bit_cast(float, bits | (x.neg ? 0x80000000u : 0u));
}

// The factors of one edge (build_rabitq.cpp:250-256) from its finite float parts, r > 0:
//   x0 = (long double)r / fx0;  tx = r * r + 2 x0 fx1;  dq = -2 x0 fac_norm;  vq = dq * offset
// An infinity times zero is the x86 default NaN (sign bit set).
BSX_FN void rabitq_factors(float r, float fx0, float fx1, float fac_norm, float offset, float& tx,
                                               float& dq, float& vq) {
    const float nan = __builtin_bit_cast(float, 0xFFC00000u), inf = __builtin_inff();
    if (fx0 == 0.0f) {
        const bool neg = (__builtin_bit_cast(uint32_t, fx0) >> 31) != 0u;
        tx = fx1 == 0.0f ? nan : (fx1 < 0.0f) != neg ? -inf : inf;
        dq = neg ? inf : -inf;
    } else {
        Ext x2 = div(r, fx0);
        x2.e += 1;
        const Parts p = parts(r);
        const uint64_t sq = static_cast<uint64_t>(p.m) * p.m;  // 2^46 <= sq < 2^48: exact
        const int s = __builtin_clzll(sq);
        tx = to_float(add(Ext{sq << s, 2 * p.e - s, false}, mul(x2, fx1)));
        x2.neg = !x2.neg;
        dq = to_float(mul(x2, fac_norm));
    }
    vq = (dq == inf || dq == -inf) && offset == 0.0f ? nan : dq * offset;
}

}  // namespace bsx
