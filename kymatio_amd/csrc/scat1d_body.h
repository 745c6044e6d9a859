// Scattering1D: node tree, kernel arguments and workgroup bodies.
//
// Same tree as the 2D path, on the generator of
// kymatio/scattering1d/core/scattering1d.py:2-107:
//   root     U_0 = fft(pad(x))                                  length N_pad
//   order 1  U_1 = |ifft(P_2^k1(U_0 * psi1[n1].levels[0]))|        res k1
//   order 2  U_2 = |ifft(P_2^k2(fft(U_1) * psi2[n2].levels[k1]))|  res k1 + k2
// with k1 = min(j1, log2_stride) (j1 without local averaging) and
// k2 = max(min(j2, log2_stride) - k1, 0).  Each node emits one output path:
//   local average  S = Re(ifft(P_kl(fft(U) * phi.levels[res]))), kl = 2^max(log2_stride-res, 0),
//                  unpadded to [ind_start[log2_stride], ind_end[log2_stride])
//   no average     U itself, unpadded at [ind_start[r], ind_end[r]), r = max(j - oversampling, 0)
//   global         the sum of U over time (the DC bin of fft(U))
// written at out[signal * out_row + out_off + t].
#pragma once
#include "fft_static.h"

#define KYM_MAX_RES1 24

enum Avg1D { AVG1_LOCAL = 0, AVG1_NONE = 1, AVG1_GLOBAL = 2 };

struct Node1D {
    int order;       // 0 root, 1, 2
    int res;         // resolution index (length N_pad >> res)
    int parent;      // node index, -1 for the root
    int filt;        // packed-filter index of the wavelet at the parent's resolution
    int k;           // periodisation factor from the parent
    int leaf_filt;   // phi.levels[res] (local average)
    int leaf_k;      // low-pass periodisation factor (local average)
    int out_off;     // offset of this path in a signal's output row
    int unpad_res;   // border-index resolution of the unpad
    int need_fwd;    // forward FFT of |U| needed (children or local leaf or global sum)
    long long slot;  // spectrum slot in the per-signal workspace, -1 none
    // training
    int child_begin, child_end;  // node-index range of the children
    long long save;              // saved u (digit-reversed, unnormalised), read-only in the backward
    long long gsave;             // dL/dX (natural) written by the backward
    long long gpad;              // root: dL/dpad(x), real
};

template <class T>
struct Scat1DArgs {
    const Node1D* nodes;
    const FftLen<T>* lens;
    const long long* filt_off;
    const int* group;
    int ngroup;
    int len[KYM_MAX_RES1], n[KYM_MAX_RES1];
    int ind_start[KYM_MAX_RES1], ind_end[KYM_MAX_RES1];
    int mode, log2_stride;
    const T* x;
    int N, pad_left;
    const T* filt;
    cpx<T>* ws;
    long long ws_sig;
    T* out;
    long long out_row;
    int img0, ntask;
    // training
    int save;
    const T* dS;
    T* gx;
};

// FFT of a node's length: run-time (Dyn1D) or compile-time (Stat1D, length
// N and NT threads; the same factorisation and digit-reversed order).  at(i) is
// where element i of the transform sits in LDS, elems(n) the elements that n
// of them take.
template <class T, int MAXP>
struct Dyn1D {
    KYM_HD KYM_INL int at(int i) const { return i; }
    KYM_HD KYM_INL int elems(int n) const { return n; }
    KYM_HD KYM_INL void inv(cpx<T>* b, const FftLen<T>& fl, int tid, int nth) const {
        fft_dif<true, MAXP>(b, fl, Batch{1, 1, fl.n, false}, tid, nth);
    }
    KYM_HD KYM_INL void fwd(cpx<T>* b, const FftLen<T>& fl, int tid, int nth) const {
        fft_dit<false, MAXP>(b, fl, Batch{1, 1, fl.n, false}, tid, nth);
    }
};

template <class T, int N, int NT>
struct Stat1D {
    KYM_HD KYM_INL int at(int i) const { return pad16(i); }
    KYM_HD KYM_INL int elems(int n) const { return pad16(n); }
    KYM_HD KYM_INL void inv(cpx<T>* b, const FftLen<T>& fl, int tid, int) const {
        pad_dif<true, N, NT, T>(b, fl.ptw, tid);
    }
    KYM_HD KYM_INL void fwd(cpx<T>* b, const FftLen<T>& fl, int tid, int) const {
        pad_dit<false, N, NT, T>(b, fl.ptw, tid);
    }
};

// Threads of a node's workgroup by its length, and the threads per output
// point (powers of two) that share its low-pass sum: 64 aliases of 128 points
// kept 384 of 512 threads waiting otherwise.  The split follows the sizes
// alone, so that a node's sums do not depend on the launch it runs in.
KYM_HD KYM_INL constexpr int node1d_threads(int n) { return n / 16 < 64 ? 64 : n / 16 > 1024 ? 1024 : n / 16; }
KYM_HD KYM_INL constexpr int leaf1d_split(int n, int nl) {
    int S = 1;
    while (2 * S * nl <= node1d_threads(n) && 2 * S * nl <= n) S *= 2;
    return S;
}
// LDS elements after the node's line: the leaf's line of nl points as S partial sums.
KYM_HD KYM_INL constexpr int leaf1d_elems(int n, int nl) { return nl * leaf1d_split(n, nl); }

// Output of one path from the spectrum / modulus in LDS.  SPLIT = false: every
// sum by one thread, where the partial sums have no room (a compile-time choice:
// read from the node or the arguments, it cost 3 signals of 1000 J=5 1%).
template <class T, int MAXP, bool SPLIT, class F>
KYM_HD KYM_INL void leaf1d(const F& ff, const Scat1DArgs<T>& a, const Node1D& nd, const cpx<T>* U, int n, int img,
                           cpx<T>* B, int tid, int nth) {
    T* o = a.out + (long long)img * a.out_row + nd.out_off;
    if (a.mode == AVG1_GLOBAL) {
        if (tid == 0) o[0] = U[0].re;
        return;
    }
    const int kk = nd.leaf_k;
    // the low-passed path has length N_pad >> max(res, log2_stride) = nl
    const int lr = nd.res > a.log2_stride ? nd.res : a.log2_stride;
    const FftLen<T>& fB = a.lens[a.len[lr]];
    const FInt nl = fB.size();
    const T* phi = a.filt + a.filt_off[nd.leaf_filt];
    const T inv_k = T(1) / T(kk);
    const int S = SPLIT ? leaf1d_split(n, nl) : 1;
    for (int q = tid; q < S * nl; q += nth) {
        const int s = q / nl, i = q - s * nl;
        cpx<T> acc = {T(0), T(0)};
#pragma unroll 4
        for (int al = s; al < kk; al += S) {  // unrolled: several filter loads in flight
            const cpx<T> u = U[ff.at(i + al * nl)];
            const T f = kym_ldg(phi + i + al * nl);
            acc.re += u.re * f;
            acc.im += u.im * f;
        }
        B[q] = acc * inv_k;
    }
    wg_barrier();
    if (S > 1) {
        for (int i = tid; i < nl; i += nth) {
            cpx<T> acc = B[i];
            for (int s = 1; s < S; ++s) acc = acc + B[i + s * nl];
            B[i] = acc;
        }
        wg_barrier();
    }
    fft_dif<true, MAXP>(B, fB, Batch{1, 1, nl, false}, tid, nth);
    const int s = a.ind_start[a.log2_stride], e = a.ind_end[a.log2_stride];
    const T inv_n = T(1) / T(nl);
    for (int p = tid; p < nl; p += nth) {
        const int t = kym_ldg(fB.rev + p);
        if (t >= s && t < e) o[t - s] = B[p].re * inv_n;
    }
    wg_barrier();
}

template <class T, int MAXP, bool SPLIT = true, class F>
KYM_HD KYM_INL void node1d_body(const F& ff, const Scat1DArgs<T>& a, int task, cpx<T>* lds, int tid, int nth) {
    const int il = task / a.ngroup, gi = task - il * a.ngroup;
    const int img = a.img0 + il;
    const Node1D& nd = a.nodes[a.group[gi]];
    const int r = nd.res, n = a.n[r];
    const FftLen<T>& fl = a.lens[a.len[r]];
    cpx<T>* wsi = a.ws + il * a.ws_sig;
    T* o = a.out + (long long)img * a.out_row + nd.out_off;
    if (nd.order == 0) {
        const T* xin = a.x + (long long)img * a.N;
        copy_batched<8>(
            n, [&](int p) { return kym_ldg(xin + reflect_index(kym_ldg(fl.rev + p) - a.pad_left, a.N)); },
            [&](int p, T v) { lds[ff.at(p)] = {v, T(0)}; }, tid, nth);
        if (a.mode == AVG1_NONE) {
            // S_0 = U_0 unpadded = the input itself
            const int s = a.ind_start[0], e = a.ind_end[0];
            for (int t = s + tid; t < e; t += nth) o[t - s] = xin[reflect_index(t - a.pad_left, a.N)];
        }
        wg_barrier();
        ff.fwd(lds, fl, tid, nth);
    } else {
        const Node1D& pn = a.nodes[nd.parent];
        const cpx<T>* U = wsi + pn.slot;
        const T* f = a.filt + a.filt_off[nd.filt];
        const int k = nd.k;
        const T inv_k = T(1) / T(k);
        // mirror pairs: the parent is the spectrum of a real signal, so point
        // n - i reads the conjugates of point i's aliases in reverse order
        // (alias q of n - i is conj(U[i + (k-1-q) n])); one load serves both.
        // i = 0 and i = n/2 are their own mirrors.
        const int half = n / 2;
        for (int i = tid; i <= half; i += nth) {
            const int im = i == 0 ? 0 : n - i;
            cpx<T> d = {T(0), T(0)}, m = {T(0), T(0)};
            if (k == 1) {
                const cpx<T> u = kym_ldg(U + i);
                const T fd = kym_ldg(f + i), fm = kym_ldg(f + im);
                d = {u.re * fd, u.im * fd};
                m = {u.re * fm, -u.im * fm};
            } else {  // k is a power of two: alias pairs (q, k-1-q), several in flight
#pragma unroll 4
                for (int q = 0; q < k / 2; ++q) {
                    const int q2 = k - 1 - q;
                    const cpx<T> u = kym_ldg(U + i + q * n), u2 = kym_ldg(U + i + q2 * n);
                    const T fd = kym_ldg(f + i + q * n), fd2 = kym_ldg(f + i + q2 * n);
                    const T fm = kym_ldg(f + im + q * n), fm2 = kym_ldg(f + im + q2 * n);
                    d.re += u.re * fd;
                    d.im += u.im * fd;
                    d.re += u2.re * fd2;
                    d.im += u2.im * fd2;
                    m.re += u2.re * fm;  // alias q of the mirror is conj(u2)
                    m.im -= u2.im * fm;
                    m.re += u.re * fm2;
                    m.im -= u.im * fm2;
                }
            }
            lds[ff.at(i)] = d * inv_k;
            if (im != i) lds[ff.at(im)] = m * inv_k;
        }
        wg_barrier();
        ff.inv(lds, fl, tid, nth);
        const T inv_n = T(1) / T(n);
        const int s = a.ind_start[nd.unpad_res], e = a.ind_end[nd.unpad_res];
        cpx<T>* sv = (a.save && nd.save >= 0) ? wsi + nd.save : nullptr;
        for (int p = tid; p < n; p += nth) {
            cpx<T>& c = lds[ff.at(p)];
            const cpx<T> v = c;
            if (sv) sv[p] = v;
            const T m = kym_sqrt(v.re * v.re + v.im * v.im) * inv_n;
            c = {m, T(0)};
            if (a.mode == AVG1_NONE) {
                const int t = kym_ldg(fl.rev + p);
                if (t >= s && t < e) o[t - s] = m;
            }
        }
        wg_barrier();
        if (nd.need_fwd) ff.fwd(lds, fl, tid, nth);
    }
    if (nd.slot >= 0) {
        cpx<T>* dst = wsi + nd.slot;
        for (int i = tid; i < n; i += nth) dst[i] = lds[ff.at(i)];
    }
    if (a.mode != AVG1_NONE) leaf1d<T, MAXP, SPLIT>(ff, a, nd, lds, n, img, lds + ff.elems(n), tid, nth);
}

template <class T, int MAXP, bool SPLIT = true>
KYM_HD void body_node1d(const Scat1DArgs<T>& a, int task, cpx<T>* lds, int tid, int nth) {
    node1d_body<T, MAXP, SPLIT>(Dyn1D<T, MAXP>(), a, task, lds, tid, nth);
}

// Compile-time specialisations X(id, N, threads) of the nodes, forward and backward (FP32):
// a launch uses one when its nodes' length matches (threads follow the
// plan's rule max(64, min(1024, N / 16))).
#define KYM_NODE1D_SPECS(X) \
    X(0, 16384, 1024)       \
    X(1, 8192, 512)         \
    X(2, 4096, 256)         \
    X(3, 2048, 128)         \
    X(4, 1024, 64)          \
    X(5, 512, 64)           \
    X(6, 256, 64)           \
    X(7, 128, 64)

KYM_HD KYM_INL int node1d_spec_id(int n, int threads) {
#define KYM_N1_MATCH(id, nn, nt) \
    if (n == nn && threads == nt) return id;
    KYM_NODE1D_SPECS(KYM_N1_MATCH)
#undef KYM_N1_MATCH
    return -1;
}

// Body of specialisation SPEC; EMU = true: one thread (CPU harness).
template <class T, int SPEC, bool EMU>
KYM_HD KYM_INL void node1d_spec_body(const Scat1DArgs<T>& a, int task, cpx<T>* lds, int tid) {
#define KYM_N1_BODY(sid, nn, nt) \
    if constexpr (SPEC == sid) node1d_body<T, 2>(Stat1D<T, nn, (EMU ? 1 : nt)>(), a, task, lds, tid, EMU ? 1 : nt);
    KYM_NODE1D_SPECS(KYM_N1_BODY)
#undef KYM_N1_BODY
}

template <class T, bool EMU>
KYM_HD void dispatch_node1d_spec(int id, const Scat1DArgs<T>& a, int task, cpx<T>* lds, int tid) {
    switch (id) {
#define KYM_N1_CASE(sid, nn, nt) \
    case sid: node1d_spec_body<T, sid, EMU>(a, task, lds, tid); break;
        KYM_NODE1D_SPECS(KYM_N1_CASE)
#undef KYM_N1_CASE
        default: break;
    }
}

// ------------------------------------------------------------------ backward
// Adjoint of body_node1d (same conventions as the 2D backward):
//   local leaf  dL/dY = fft(unpad^T dS) / nl, dL/dU += phi * tile(dL/dY) / kl
//   children    dL/dU += f_c * tile(dL/dX_c) / kc
//   dL/dm = Re(n ifft(dL/dU)) (+ dS on the unpadded window without averaging,
//           + dS everywhere with global averaging)
//   dL/du = dL/dm u / |u|,  dL/dX = fft(dL/du) / n;  root: dL/dpad(x) = dL/dm.
template <class T, int MAXP, class F>
KYM_HD KYM_INL void bwd_node1d_body(const F& ff, const Scat1DArgs<T>& a, int task, cpx<T>* lds, int tid, int nth) {
    const int il = task / a.ngroup, gi = task - il * a.ngroup;
    const int img = a.img0 + il;
    const Node1D& nd = a.nodes[a.group[gi]];
    const int r = nd.res, n = a.n[r];
    const FftLen<T>& fl = a.lens[a.len[r]];
    cpx<T>* wsi = a.ws + il * a.ws_sig;
    const T* d = a.dS + (long long)img * a.out_row + nd.out_off;
    // leaf gradient (local average) into B
    cpx<T>* B = lds + ff.elems(n);
    int nl = 1, kk = 1;
    if (a.mode == AVG1_LOCAL) {
        kk = nd.leaf_k;
        nl = n / kk;
        const int lr = nd.res > a.log2_stride ? nd.res : a.log2_stride;
        const FftLen<T>& fB = a.lens[a.len[lr]];
        const int s = a.ind_start[a.log2_stride], e = a.ind_end[a.log2_stride];
        for (int p = tid; p < nl; p += nth) {
            const int t = kym_ldg(fB.rev + p);
            B[p] = {(t >= s && t < e) ? d[t - s] : T(0), T(0)};
        }
        wg_barrier();
        fft_dit<false, MAXP>(B, fB, Batch{1, 1, nl, false}, tid, nth);
    }
    const bool has_u_grad = (a.mode == AVG1_LOCAL) || (nd.child_end > nd.child_begin);
    const T* phi = a.mode == AVG1_LOCAL ? a.filt + a.filt_off[nd.leaf_filt] : nullptr;
    const T sc_leaf = T(1) / (T(nl) * T(kk));
    // E points per thread, two children at a time: 4 E loads in flight (the
    // root sums some sixty children in one workgroup per signal)
    constexpr int E = 4;
    for (int i0 = tid; i0 < n; i0 += E * nth) {
        int ix[E];
        cpx<T> acc[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            ix[e] = i0 + e * nth < n ? i0 + e * nth : i0;
            acc[e] = {T(0), T(0)};
            if (phi) {
                const cpx<T> gy = B[ix[e] & (nl - 1)];  // lengths are powers of two
                const T ph = kym_ldg(phi + ix[e]) * sc_leaf;
                acc[e] = {gy.re * ph, gy.im * ph};
            }
        }
#pragma unroll 2
        for (int c = nd.child_begin; c < nd.child_end; ++c) {
            const Node1D& cn = a.nodes[c];
            const int nm = a.n[cn.res] - 1;
            const T* f = a.filt + a.filt_off[cn.filt];
            const cpx<T>* g = wsi + cn.gsave;
            const T inv_k = T(1) / T(cn.k);  // a power of two: exact
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const T fv = kym_ldg(f + ix[e]) * inv_k;
                const cpx<T> gx = kym_ldg(g + (ix[e] & nm));
                acc[e].re += gx.re * fv;
                acc[e].im += gx.im * fv;
            }
        }
#pragma unroll
        for (int e = 0; e < E; ++e)
            if (i0 + e * nth < n) lds[ff.at(ix[e])] = acc[e];
    }
    wg_barrier();
    if (has_u_grad) ff.inv(lds, fl, tid, nth);
    // direct terms on dL/dm (positions p hold natural index rev[p])
    const int us = a.ind_start[nd.unpad_res], ue = a.ind_end[nd.unpad_res];
    for (int p = tid; p < n; p += nth) {
        cpx<T>& c = lds[ff.at(p)];
        T gm = has_u_grad ? c.re : T(0);
        const int t = kym_ldg(fl.rev + p);
        if (a.mode == AVG1_NONE && t >= us && t < ue) gm += d[t - us];
        if (a.mode == AVG1_GLOBAL) gm += d[0];
        if (nd.order == 0) {
            reinterpret_cast<T*>(wsi + nd.gpad)[t] = gm;
        } else {
            const cpx<T> u = kym_ldg(wsi + nd.save + p);
            const T mag = kym_sqrt(u.re * u.re + u.im * u.im);
            c = mag > T(0) ? cpx<T>{u.re * (gm / mag), u.im * (gm / mag)} : cpx<T>{T(0), T(0)};
        }
    }
    if (nd.order == 0) return;
    wg_barrier();
    ff.fwd(lds, fl, tid, nth);
    const T inv_n = T(1) / T(n);
    for (int i = tid; i < n; i += nth) wsi[nd.gsave + i] = lds[ff.at(i)] * inv_n;
}

template <class T, int MAXP>
KYM_HD void body_bwd_node1d(const Scat1DArgs<T>& a, int task, cpx<T>* lds, int tid, int nth) {
    bwd_node1d_body<T, MAXP>(Dyn1D<T, MAXP>(), a, task, lds, tid, nth);
}

template <class T, int SPEC, bool EMU>
KYM_HD KYM_INL void bwd_node1d_spec_body(const Scat1DArgs<T>& a, int task, cpx<T>* lds, int tid) {
#define KYM_B1_BODY(sid, nn, nt)                                                                         \
    if constexpr (SPEC == sid)                                                                           \
        bwd_node1d_body<T, 2>(Stat1D<T, nn, (EMU ? 1 : nt)>(), a, task, lds, tid, EMU ? 1 : nt);
    KYM_NODE1D_SPECS(KYM_B1_BODY)
#undef KYM_B1_BODY
}

template <class T, bool EMU>
KYM_HD void dispatch_bwd_node1d_spec(int id, const Scat1DArgs<T>& a, int task, cpx<T>* lds, int tid) {
    switch (id) {
#define KYM_B1_CASE(sid, nn, nt) \
    case sid: bwd_node1d_spec_body<T, sid, EMU>(a, task, lds, tid); break;
        KYM_NODE1D_SPECS(KYM_B1_CASE)
#undef KYM_B1_CASE
        default: break;
    }
}

// Reflect-pad adjoint (1D).  task -> signal.
template <class T>
KYM_HD void body_bwd_fold1d(const Scat1DArgs<T>& a, int task, int tid, int nth) {
    const int img = a.img0 + task;
    const T* gp = reinterpret_cast<const T*>(a.ws + task * a.ws_sig + a.nodes[0].gpad);
    T* gx = a.gx + (long long)img * a.N;
    const int P = a.n[0];
    for (int i = tid; i < a.N; i += nth) {
        T acc = T(0);
        if (a.N == 1) {
            for (int t = 0; t < P; ++t) acc += gp[t];
        } else {
            const int T_ = 2 * (a.N - 1);
            for (int t = (a.pad_left + i) % T_; t < P; t += T_) acc += gp[t];
            if (i != 0 && i != a.N - 1)
                for (int t = ((a.pad_left - i) % T_ + T_) % T_; t < P; t += T_) acc += gp[t];
        }
        gx[i] = acc;
    }
}

// A node of any length in one workgroup (FP32; launches that mix lengths):
// the compiled body of its length on the first node1d_threads(n) threads, the
// very code of a launch of that length alone, so that results do not depend on
// which launch a node ran in.  The other threads start beyond every loop and
// only meet the barriers.
#define KYM_N1_ANY 1000  // Launch1D::spec of such a launch
// Launch1D::spec of forward nodes whose partial sums do not fit a caller's LDS limit
#define KYM_N1_NOSPLIT 1001
template <class T, int KIND, bool EMU>
KYM_HD KYM_INL void node1d_any_body(const Scat1DArgs<T>& a, int task, cpx<T>* lds, int tid) {
    const Node1D& nd = a.nodes[a.group[task % a.ngroup]];
    const int n = a.n[nd.res], nt = EMU ? 1 : node1d_threads(n);
    if (tid >= nt) tid = 1 << 28;
    switch (node1d_spec_id(n, node1d_threads(n))) {
#define KYM_NA_CASE(sid, nn, nnt)                                                     \
    case sid:                                                                        \
        if constexpr (KIND == 0) node1d_spec_body<T, sid, EMU>(a, task, lds, tid);   \
        else bwd_node1d_spec_body<T, sid, EMU>(a, task, lds, tid);                   \
        break;
        KYM_NODE1D_SPECS(KYM_NA_CASE)
#undef KYM_NA_CASE
        default:
            if constexpr (KIND == 0) body_node1d<T, 2>(a, task, lds, tid, nt);
            else body_bwd_node1d<T, 2>(a, task, lds, tid, nt);
    }
}
