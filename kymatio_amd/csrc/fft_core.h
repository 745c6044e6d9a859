// Mixed-radix in-place FFT passes over data held in LDS.
//
// Length n = r_1 r_2 ... r_K (radices 2, 4, 8, 16, odd primes 3..31, and the
// products 9 and 15 where a plan asks for them).
// Two in-place Cooley-Tukey variants share one digit-reversal permutation
// `rev` (rev[p] = natural index of the element at storage position p):
//   * DIT, passes r_1 .. r_K: input stored digit-reversed, output natural.
//   * DIF, passes r_K .. r_1: input natural, output stored digit-reversed.
// So an inverse DIF, a point-wise op and a forward DIT chain with no
// permutation at all, and loads/stores from HBM fold the permutation into
// their index math.  Each butterfly reads and writes the same R slots, so a
// pass needs one barrier and no second buffer.
//
// Twiddles come from a per-length table tw[t] = exp(-2 pi i t / n) computed
// in double on the host; the inverse uses the conjugate.  Transforms are
// unnormalised in both directions.
#pragma once
#include "common.h"
#include "radix_consts.h"

#define KYM_MAX_RADICES 12

template <class T>
struct FftLen {
    int n;
    int nrad;
    int rad[KYM_MAX_RADICES];  // DIT order (r_1 first)
    const cpx<T>* tw;          // n entries
    const int* rev;            // n entries: storage position -> natural index
    const int* irev;           // n entries: natural index -> storage position (inverse of rev)
    // div_magic of n and, per pass q, of its butterflies n / rad[q] and of the
    // product rad[0] ... rad[q - 1]
    unsigned mn, mnb[KYM_MAX_RADICES], mlp[KYM_MAX_RADICES];
    // the twiddles in the order the passes read them from global memory: pass q
    // takes exp(-2 pi i j m / (Lp rad[q])) at ptw[poff[q] + (m - 1) Lp + j], so
    // neighbouring butterflies read neighbouring entries (from tw, element m of
    // a wave's butterflies lies m n / L entries apart: for the 8192-point
    // transform up to 60 cache lines a load)
    const cpx<T>* ptw;
    int poff[KYM_MAX_RADICES];
    KYM_HD KYM_INL FInt size() const { return {n, mn}; }
};

// ---------------------------------------------------------------- butterflies
template <bool INV, class T> KYM_HD KYM_INL void dft2(cpx<T>* v) {
    cpx<T> a = v[0], b = v[1];
    v[0] = a + b;
    v[1] = a - b;
}

template <bool INV, class T> KYM_HD KYM_INL void dft4(cpx<T>& x0, cpx<T>& x1, cpx<T>& x2, cpx<T>& x3) {
    cpx<T> a0 = x0 + x2, a1 = x0 - x2, a2 = x1 + x3, a3 = mul_mi<INV>(x1 - x3);
    x0 = a0 + a2;
    x2 = a0 - a2;
    x1 = a1 + a3;
    x3 = a1 - a3;
}

template <bool INV, class T> KYM_HD KYM_INL void dft4(cpx<T>* v) { dft4<INV>(v[0], v[1], v[2], v[3]); }

// multiply by exp(-/+ 2 pi i m / 16) with the trivial angles special-cased
template <int M, bool INV, class T> KYM_HD KYM_INL cpx<T> tw16(cpx<T> a) {
    constexpr int m = M % 16;
    if constexpr (m == 0) return a;
    else if constexpr (m == 4) return mul_mi<INV>(a);
    else if constexpr (m == 8) return {-a.re, -a.im};
    else if constexpr (m == 12) return mul_mi<!INV>(a);
    else {
        // cos/sin(2 pi m / 16) for m in 0..15
        constexpr double c1 = 0.92387953251128675613, s1 = 0.38268343236508977173, h = 0.70710678118654752440;
        constexpr double cs[16] = {1, c1, h, s1, 0, -s1, -h, -c1, -1, -c1, -h, -s1, 0, s1, h, c1};
        constexpr double sn[16] = {0, s1, h, c1, 1, c1, h, s1, 0, -s1, -h, -c1, -1, -c1, -h, -s1};
        const cpx<T> w = {T(cs[m]), T(INV ? sn[m] : -sn[m])};
        return cmul(a, w);
    }
}

template <bool INV, class T> KYM_HD KYM_INL void dft8(cpx<T>* v) {
    cpx<T> e0 = v[0], e1 = v[2], e2 = v[4], e3 = v[6];
    cpx<T> o0 = v[1], o1 = v[3], o2 = v[5], o3 = v[7];
    dft4<INV>(e0, e1, e2, e3);
    dft4<INV>(o0, o1, o2, o3);
    o1 = tw16<2, INV>(o1);
    o2 = tw16<4, INV>(o2);
    o3 = tw16<6, INV>(o3);
    v[0] = e0 + o0; v[4] = e0 - o0;
    v[1] = e1 + o1; v[5] = e1 - o1;
    v[2] = e2 + o2; v[6] = e2 - o2;
    v[3] = e3 + o3; v[7] = e3 - o3;
}

template <bool INV, class T> KYM_HD KYM_INL void dft16(cpx<T>* v) {
    // 4 x 4: inner DFTs over n1 for each n2, twiddle W16^(n2 k1), outer over n2
#pragma unroll
    for (int n2 = 0; n2 < 4; ++n2) dft4<INV>(v[n2], v[4 + n2], v[8 + n2], v[12 + n2]);
    // after this, v[4*k1 + n2] holds y[n2][k1]
    v[5] = tw16<1, INV>(v[5]);
    v[6] = tw16<2, INV>(v[6]);
    v[7] = tw16<3, INV>(v[7]);
    v[9] = tw16<2, INV>(v[9]);
    v[10] = tw16<4, INV>(v[10]);
    v[11] = tw16<6, INV>(v[11]);
    v[13] = tw16<3, INV>(v[13]);
    v[14] = tw16<6, INV>(v[14]);
    v[15] = tw16<9, INV>(v[15]);
    cpx<T> t[16];
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) {
        cpx<T> a = v[4 * k1], b = v[4 * k1 + 1], c = v[4 * k1 + 2], d = v[4 * k1 + 3];
        dft4<INV>(a, b, c, d);
        t[k1] = a;
        t[k1 + 4] = b;
        t[k1 + 8] = c;
        t[k1 + 12] = d;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = t[i];
}

// Odd prime P: pair inputs n and P-n, X_k and X_{P-k} share the cos/sin sums.
template <int P, bool INV, class T> KYM_HD KYM_INL void dft_odd(cpx<T>* v) {
    constexpr int H = (P - 1) / 2;
    cpx<T> a[H], b[H];
    cpx<T> x0 = v[0];
    cpx<T> s = x0;
#pragma unroll
    for (int n = 1; n <= H; ++n) {
        a[n - 1] = v[n] + v[P - n];
        b[n - 1] = v[n] - v[P - n];
        s = s + a[n - 1];
    }
    v[0] = s;
#pragma unroll
    for (int k = 1; k <= H; ++k) {
        T rc = x0.re, ic = x0.im, rs = T(0), is = T(0);
#pragma unroll
        for (int n = 1; n <= H; ++n) {
            const int m = (n * k) % P;
            const T c = T(KymCos<P>::v[m]);
            const T sn = T(KymSin<P>::v[m]);
            rc += a[n - 1].re * c;
            ic += a[n - 1].im * c;
            rs += b[n - 1].re * sn;
            is += b[n - 1].im * sn;
        }
        // forward: X_k = sum a cos - i b sin ; inverse flips the sin sign
        if (INV) {
            v[k] = {rc - is, ic + rs};
            v[P - k] = {rc + is, ic - rs};
        } else {
            v[k] = {rc + is, ic - rs};
            v[P - k] = {rc - is, ic + rs};
        }
    }
}

template <int R, bool INV, class T> KYM_HD KYM_INL void dft_r(cpx<T>* v);

// R = A B with A and B coprime: the prime-factor algorithm (Good 1958).  Inputs
// (B n1 + A n2) mod R, outputs k with k = k1 mod A and k = k2 mod B, and no
// twiddles between the two.
template <int A, int B, bool INV, class T> KYM_HD KYM_INL void dft_coprime(cpx<T>* v) {
    constexpr int R = A * B;
    constexpr int iB = [] { int i = 1; while (i * B % A != 1) ++i; return i; }();
    constexpr int iA = [] { int i = 1; while (i * A % B != 1) ++i; return i; }();
    cpx<T> t[R];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
        cpx<T> u[A];
#pragma unroll
        for (int n1 = 0; n1 < A; ++n1) u[n1] = v[(B * n1 + A * n2) % R];
        dft_r<A, INV>(u);
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) t[k1 * B + n2] = u[k1];
    }
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
        dft_r<B, INV>(t + k1 * B);
#pragma unroll
        for (int k2 = 0; k2 < B; ++k2) v[(k1 * B * iB + k2 * A * iA) % R] = t[k1 * B + k2];
    }
}

template <bool INV, class T> KYM_HD KYM_INL void dft9(cpx<T>* v) {
    // 3 x 3: inner over n1 for each n2, twiddle W9^(n2 k1), outer over n2
    // cos and sin of 2 pi m / 9, m = 1, 2, 4
    constexpr double cs[3] = {0.76604444311897803520, 0.17364817766693034885, -0.93969262078590838405};
    constexpr double sn[3] = {0.64278760968653932632, 0.98480775301220805937, 0.34202014332566873304};
    cpx<T> t[9];
#pragma unroll
    for (int n2 = 0; n2 < 3; ++n2) {
        cpx<T> u[3] = {v[n2], v[3 + n2], v[6 + n2]};
        dft_odd<3, INV>(u);
#pragma unroll
        for (int k1 = 0; k1 < 3; ++k1) {
            const int m = n2 * k1 == 4 ? 2 : n2 * k1 - 1;
            t[k1 * 3 + n2] = n2 * k1 == 0 ? u[k1] : cmul(u[k1], cpx<T>{T(cs[m]), T(INV ? sn[m] : -sn[m])});
        }
    }
#pragma unroll
    for (int k1 = 0; k1 < 3; ++k1) {
        dft_odd<3, INV>(t + 3 * k1);
#pragma unroll
        for (int k2 = 0; k2 < 3; ++k2) v[k1 + 3 * k2] = t[3 * k1 + k2];
    }
}

template <int R, bool INV, class T> KYM_HD KYM_INL void dft_r(cpx<T>* v) {
    if constexpr (R == 2) dft2<INV>(v);
    else if constexpr (R == 4) dft4<INV>(v);
    else if constexpr (R == 8) dft8<INV>(v);
    else if constexpr (R == 16) dft16<INV>(v);
    else if constexpr (R == 9) dft9<INV>(v);
    else if constexpr (R == 15) dft_coprime<5, 3, INV>(v);
    else dft_odd<R, INV>(v);
}

// ---------------------------------------------------------------- passes
// A batch of `ntr` transforms of length n; element e of transform t lives at
// buf[t * ts + e * es].  `tfast` selects which index varies fastest across
// threads: the transform (column batches, ts == 1) or the butterfly (rows).
struct Batch {
    int ntr, es, ts;
    bool tfast;
};

// q: the pass's index in fl.rad; mtr: div_magic(bt.ntr), used when bt.tfast.
template <int R, bool INV, bool TWL, class T>
KYM_HD KYM_INL void dit_pass(cpx<T>* buf, const FftLen<T>& fl, const cpx<T>* tw, int q, int Lp, const Batch& bt, unsigned mtr,
                     int tid, int nth) {
    const int n = fl.n, L = Lp * R, nb = div_by(n, div_magic(R)), tstep = nb / FInt{Lp, fl.mlp[q]};
    const int total = nb * bt.ntr, off = TWL ? 0 : fl.poff[q];
    const FInt dtr = bt.tfast ? FInt{bt.ntr, mtr} : FInt{nb, fl.mnb[q]}, dlp = {Lp, fl.mlp[q]};
    for (int f = tid; f < total; f += nth) {
        const int hi = f / dtr, lo = f - hi * dtr;
        const int t = bt.tfast ? lo : hi, u = bt.tfast ? hi : lo;
        const int b = u / dlp, j = u - b * Lp;
        cpx<T>* p = buf + (t * bt.ts + (b * L + j) * bt.es);
        const int st = Lp * bt.es;
        cpx<T> v[R];
#pragma unroll
        for (int m = 0; m < R; ++m) v[m] = p[m * st];
        if (j != 0) {
#pragma unroll
            for (int m = 1; m < R; ++m) {
                const cpx<T> w = TWL ? tw[j * m * tstep] : kym_ldg(tw + off + (m - 1) * Lp + j);
                v[m] = INV ? cmulc(v[m], w) : cmul(v[m], w);
            }
        }
        dft_r<R, INV>(v);
#pragma unroll
        for (int m = 0; m < R; ++m) p[m * st] = v[m];
    }
}

template <int R, bool INV, bool TWL, class T>
KYM_HD KYM_INL void dif_pass(cpx<T>* buf, const FftLen<T>& fl, const cpx<T>* tw, int q, int L, const Batch& bt, unsigned mtr,
                     int tid, int nth) {
    const int n = fl.n, Ls = div_by(L, div_magic(R)), nb = div_by(n, div_magic(R)), tstep = nb / FInt{Ls, fl.mlp[q]};
    const int total = nb * bt.ntr, off = TWL ? 0 : fl.poff[q];
    const FInt dtr = bt.tfast ? FInt{bt.ntr, mtr} : FInt{nb, fl.mnb[q]}, dls = {Ls, fl.mlp[q]};
    for (int f = tid; f < total; f += nth) {
        const int hi = f / dtr, lo = f - hi * dtr;
        const int t = bt.tfast ? lo : hi, u = bt.tfast ? hi : lo;
        const int b = u / dls, j = u - b * Ls;
        cpx<T>* p = buf + (t * bt.ts + (b * L + j) * bt.es);
        const int st = Ls * bt.es;
        cpx<T> v[R];
#pragma unroll
        for (int m = 0; m < R; ++m) v[m] = p[m * st];
        dft_r<R, INV>(v);
        if (j != 0) {
#pragma unroll
            for (int m = 1; m < R; ++m) {
                const cpx<T> w = TWL ? tw[j * m * tstep] : kym_ldg(tw + off + (m - 1) * Ls + j);
                v[m] = INV ? cmulc(v[m], w) : cmul(v[m], w);
            }
        }
#pragma unroll
        for (int m = 0; m < R; ++m) p[m * st] = v[m];
    }
}

// The primes a kernel is built for: every one up to MAXP, or (MAXP = 100 + p)
// those up to 7 and the prime p.
template <int MAXP>
KYM_HD constexpr bool kym_has_radix(int R) { return MAXP > 100 ? R <= 7 || R == MAXP - 100 : R <= MAXP; }

// Radices 9 and 15: in the kernels of the class 7 (kym_factor_list says why),
// and in the CPU harness, which runs every plan on the bodies of the class 31.
template <int MAXP> KYM_HD constexpr bool kym_has_products() {
#if defined(__HIP_DEVICE_COMPILE__)
    return MAXP == 7;
#else
    return true;
#endif
}

// MAXP of kernels with every radix up to 31 inline: the per-op transforms, low-
// passes and the frequency scatter, which hold each pass once or twice.  Inline
// and in functions: 512 x 14384 points 81 and 104 us, 64 x 124 x 116 48 and 72,
// FP64 64 x 58 x 62 23 and 55, low-passes of 4096 lines of 1984 points 74 and 109,
// frequency scatters to 92 points 33 and 45.
#define KYM_ALL_PRIMES 32

// The passes of large radices as functions, for the 2D kernels with every radix up to
// 31 (a node whose two lengths have different primes from 19 up), which would
// hold each of them four to six times (246 KB of code).
template <int R, bool INV, bool TWL, class T>
KYM_HD __attribute__((noinline)) void dit_pass_call(cpx<T>* buf, const FftLen<T>& fl, const cpx<T>* tw, int q, int Lp,
                                                    const Batch& bt, unsigned mtr, int tid, int nth) {
    dit_pass<R, INV, TWL, T>(buf, fl, tw, q, Lp, bt, mtr, tid, nth);
}
template <int R, bool INV, bool TWL, class T>
KYM_HD __attribute__((noinline)) void dif_pass_call(cpx<T>* buf, const FftLen<T>& fl, const cpx<T>* tw, int q, int L,
                                                    const Batch& bt, unsigned mtr, int tid, int nth) {
    dif_pass<R, INV, TWL, T>(buf, fl, tw, q, L, bt, mtr, tid, nth);
}

// Radix dispatch.  MAXP is the largest odd prime the kernel is built for, so a
// kernel only carries the butterflies its plan can use (large odd radices
// cost registers for every path through the kernel).
#define KYM_RADIX_SWITCH(R_, CALL)                                   \
    switch (R_) {                                                    \
        case 2: { CALL(2); } break;                                      \
        case 4: { CALL(4); } break;                                      \
        case 8: { CALL(8); } break;                                      \
        case 16: { CALL(16); } break;                                    \
        case 9: if constexpr (kym_has_products<MAXP>()) { CALL(9); } break;    \
        case 15: if constexpr (kym_has_products<MAXP>()) { CALL(15); } break;  \
        case 3: if constexpr (kym_has_radix<MAXP>(3)) { CALL(3); } break;    \
        case 5: if constexpr (kym_has_radix<MAXP>(5)) { CALL(5); } break;    \
        case 7: if constexpr (kym_has_radix<MAXP>(7)) { CALL(7); } break;    \
        case 11: if constexpr (kym_has_radix<MAXP>(11)) { CALL(11); } break;    \
        case 13: if constexpr (kym_has_radix<MAXP>(13)) { CALL(13); } break;    \
        case 17: if constexpr (kym_has_radix<MAXP>(17)) { CALL(17); } break;    \
        case 19: if constexpr (kym_has_radix<MAXP>(19)) { CALL(19); } break;    \
        case 23: if constexpr (kym_has_radix<MAXP>(23)) { CALL(23); } break;    \
        case 29: if constexpr (kym_has_radix<MAXP>(29)) { CALL(29); } break;    \
        case 31: if constexpr (kym_has_radix<MAXP>(31)) { CALL(31); } break;    \
        default: break;                                              \
    }

// Largest odd prime factor of n (1 if n is a power of two).
KYM_HD KYM_INL int kym_max_odd_prime(int n) {
    while (n % 2 == 0 && n > 1) n /= 2;
    int best = 1;
    for (int p = 3; p * p <= n; p += 2)
        while (n % p == 0) { best = p; n /= p; }
    if (n > 1) best = n > best ? n : best;
    return best;
}

// Kernel families by prime set: 2-only/3/5/7 -> 7, up to 17 -> 17, up to 31 -> 31.
KYM_HD KYM_INL int kym_prime_class(int maxp) { return maxp <= 7 ? 7 : maxp <= 17 ? 17 : 31; }

// The family of kernels for lengths 2^i a and 2^i b: also 100 + p where
// 19 <= p <= 31 is the only prime above 7 in them.  A kernel that holds the
// radix-19 to -31 butterflies together needs 246 KB of code and up to 250
// registers with spills; with one of them, 70 KB and the registers of that one.
// J=3, each before and after: 32 x 136^2 (19) 770 -> 361 us, 16 x 170^2 (23)
// 725 -> 318, 16 x 220^2 (29) 1149 -> 528, 16 x 235^2 (31) 1306 -> 616, FP64
// 4 x 141^2 676 -> 292; 16 x 136x170 (19 and 23, every radix, large ones in
// functions) 495 -> 353.
// KYM_GLOBAL_TW + 7, 17 or 31: the kernels that read their twiddles from global
// memory, for the few sizes whose data leaves no room in LDS.
#define KYM_GLOBAL_TW 200
inline int kym_plan_class(int a, int b) {
    int only = 0, maxp = 1;
    for (int v : {a, b})
        for (int p = 3; p <= 31; p += 2)
            while (v % p == 0) {
                v /= p;
                maxp = p > maxp ? p : maxp;
                if (p > 7) only = only == 0 || only == p ? p : -1;
            }
    return only >= 19 ? 100 + only : kym_prime_class(maxp);
}

// Full DIT transform (digit-reversed in, natural out); barrier after each pass.
// TWL: tw is fl's twiddle table copied to LDS (else fl.ptw is read).
template <bool INV, int MAXP, bool TWL = false, class T>
KYM_HD KYM_INL void fft_dit(cpx<T>* buf, const FftLen<T>& fl, const Batch& bt, int tid, int nth, const cpx<T>* tw = nullptr) {
    int Lp = 1;
    if (!TWL) tw = fl.ptw;
    const unsigned mtr = bt.tfast ? div_magic(bt.ntr) : 0;
    for (int q = 0; q < fl.nrad; ++q) {
        const int R = fl.rad[q];
#define KYM_DIT_CALL(RR)                                                                 \
    if constexpr (MAXP == 31 && RR >= 11) dit_pass_call<RR, INV, TWL, T>(buf, fl, tw, q, Lp, bt, mtr, tid, nth); \
    else dit_pass<RR, INV, TWL, T>(buf, fl, tw, q, Lp, bt, mtr, tid, nth)
        KYM_RADIX_SWITCH(R, KYM_DIT_CALL)
#undef KYM_DIT_CALL
        Lp *= R;
        wg_barrier();
    }
}

// Full DIF transform (natural in, digit-reversed out); barrier after each pass.
template <bool INV, int MAXP, bool TWL = false, class T>
KYM_HD KYM_INL void fft_dif(cpx<T>* buf, const FftLen<T>& fl, const Batch& bt, int tid, int nth, const cpx<T>* tw = nullptr) {
    int L = fl.n;
    if (!TWL) tw = fl.ptw;
    const unsigned mtr = bt.tfast ? div_magic(bt.ntr) : 0;
    for (int q = fl.nrad - 1; q >= 0; --q) {
        const int R = fl.rad[q];
#define KYM_DIF_CALL(RR)                                                                 \
    if constexpr (MAXP == 31 && RR >= 11) dif_pass_call<RR, INV, TWL, T>(buf, fl, tw, q, L, bt, mtr, tid, nth); \
    else dif_pass<RR, INV, TWL, T>(buf, fl, tw, q, L, bt, mtr, tid, nth);                 \
    L = div_by(L, div_magic(RR))
        KYM_RADIX_SWITCH(R, KYM_DIF_CALL)
#undef KYM_DIF_CALL
        wg_barrier();
    }
}

// Factor n into supported radices (DIT order): odd primes first (their
// butterflies then need no twiddles), then powers of two as 16/8/4/2.
// max_pow2 (16, 8, 4 or 2) caps the power-of-two radices (a tuning choice;
// 16 is the default every compile-time specialisation assumes).
// constexpr so compile-time specialisations use exactly the runtime order.
// products: 15 and 9 in one pass each from 48 points on (shorter lines would
// leave most of a workgroup's threads without a butterfly), for run-time-sized
// kernels of the class 7.  A pass over LDS less: 48 x 224^2, J=3 (15 x 16, 15 x
// 8) 1055 -> 961 us, 16 of them with the gradient 1157 -> 1064, 32 x 128^2 (9 x
// 16, 9 x 8) 322 -> 309.  Odd radices read a row's first pass without bank
// conflicts; 6, 10 and 14 were no faster than the passes they saved, and in
// the kernels up to 17 the added butterflies spilled (6 x 150x203 221 -> 417).
#define KYM_PRODUCT_MIN_N 48
struct RadList {
    int n = 0;
    int nrad = 0;
    int rad[KYM_MAX_RADICES] = {0};
    bool ok = false;
};

KYM_HD constexpr RadList kym_factor_list(int n, int max_pow2 = 16, bool products = false) {
    RadList rl;
    rl.n = n;
    int k = 0;
    int m = n;
    int a = 0;
    while (m % 2 == 0) { m /= 2; ++a; }
    const int product[2] = {15, 9};
    for (int i = 0; products && n >= KYM_PRODUCT_MIN_N && i < 2; ++i)
        while (m % product[i] == 0) {
            if (k >= KYM_MAX_RADICES) return rl;
            rl.rad[k++] = product[i];
            m /= product[i];
        }
    const int odd[10] = {3, 5, 7, 11, 13, 17, 19, 23, 29, 31};
    for (int i = 0; i < 10; ++i) {
        const int p = odd[i];
        while (m % p == 0) {
            if (k >= KYM_MAX_RADICES) return rl;
            rl.rad[k++] = p;
            m /= p;
        }
    }
    if (m != 1) return rl;
    const int dmax = max_pow2 >= 16 ? 4 : max_pow2 >= 8 ? 3 : max_pow2 >= 4 ? 2 : 1;
    while (a > 0) {
        int d = 1;
        if (dmax == 4) {
            if (a >= 8 || a == 4 || a == 7) d = 4;
            else if (a == 6 || a == 3 || a == 5) d = 3;
            else if (a == 2) d = 2;
        } else {
            d = a < dmax ? a : dmax;
            if (a - d == 1 && d > 2) d -= 1;  // 4 x 4 rather than 8 x 2
        }
        if (k >= KYM_MAX_RADICES) return rl;
        rl.rad[k++] = 1 << d;
        a -= d;
    }
    if (n == 1) rl.rad[k++] = 1;
    rl.nrad = k;
    rl.ok = true;
    return rl;
}

inline bool kym_factor(int n, int* rad, int* nrad, int max_pow2 = 16, bool products = false) {
    const RadList rl = kym_factor_list(n, max_pow2, products);
    if (!rl.ok) return false;
    for (int i = 0; i < rl.nrad; ++i) rad[i] = rl.rad[i];
    *nrad = rl.nrad;
    return true;
}

// Offset of pass Q's entries in FftLen::ptw (DIT order; a first pass has none).
KYM_HD constexpr int kym_ptw_off(const RadList& rl, int Q) {
    int off = 0, lp = 1;
    for (int q = 0; q < Q; ++q) {
        const int R = rl.rad[q] > 1 ? rl.rad[q] : 1;
        if (lp > 1) off += (R - 1) * lp;
        lp *= R;
    }
    return off;
}
