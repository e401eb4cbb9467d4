// tdw_rsfft.hpp -- in-place mixed-radix transforms of pencils held in LDS, of
// any length with factors 2 and 3, laid out at run time.
//
// Forward stages are decimation in frequency: R elements sub apart, DFT, times
// W_{R sub}^{j t}; the inverse stages undo them in reverse order, so the
// spectrum is used in the digit-reversed order it is left in, nothing is
// reordered, and one buffer suffices.  Consecutive lanes take consecutive
// pencils: with pencils one element or one padded row apart, a wave's LDS
// accesses fall in distinct banks.  Each stage is a function of the whole
// workgroup and ends behind a barrier.
#pragma once
#include "tdw_device.hpp"
#include "tdw_regfft.hpp"

#include <math.h>
#include <vector>

namespace tdw {

static constexpr int RS_MAXST = 6;    // stages per axis

// One radix-R stage of an axis: blocks of R * sub elements, tws = L / (R sub)
// the step of its twiddles in the table of exp(-2 pi i k / L).
struct RsStage {
    int R, sub, tws;
    unsigned msub;   // division by sub
};
// An axis of L points of P pencils.  Pencil q starts at q * qh (qd = 0) or at
// (q / qd) * qh + q % qd; its elements lie `is` apart; its twiddles start at
// tw of the kernel's table.
struct RsAxis {
    int L, nst, is, P, qd, qh, tw;
    unsigned mP, mqd;
    RsStage st[RS_MAXST];
};

// x / d for the small operands here (x d < 2^32), m = floor(2^32 / d) + 1
__device__ __forceinline__ unsigned rs_div(unsigned x, unsigned d, unsigned m) { return d == 1 ? x : __umulhi(x, m); }
inline unsigned rs_magic(int d) { return d > 1 ? (unsigned)((1ull << 32) / (unsigned)d) + 1u : 0u; }

// KIND 0: a forward stage; 1: an inverse stage; 2: the last forward stage,
// op(position, pencil, value) on the spectrum and the first inverse stage in
// registers.  pencil is q % qd (q for qd = 0).
template <int R, int KIND, typename C, typename OP>
__device__ __forceinline__ void rs_stage(C *A, const C *tw, const RsAxis &ax, const RsStage &st, OP &&op)
{
    const unsigned tot = ax.P * (ax.L / R);
    const unsigned is = ax.is;
    for (unsigned b = threadIdx.x; b < tot; b += blockDim.x) {
        const unsigned jj = rs_div(b, ax.P, ax.mP), q = b - jj * ax.P;
        const unsigned blk = rs_div(jj, st.sub, st.msub), j = jj - blk * st.sub;
        unsigned qi = q, base = q * ax.qh;
        if (ax.qd) {
            const unsigned hi = rs_div(q, ax.qd, ax.mqd);
            qi = q - hi * ax.qd;
            base = hi * ax.qh + qi;
        }
        const unsigned i0 = blk * (R * st.sub) + j, step = st.sub * is;
        C *p = A + base + i0 * is;
        C v[R];
#pragma unroll
        for (int t = 0; t < R; t++) v[t] = p[t * step];
        if constexpr (KIND == 1) {
            if (st.sub > 1) {
#pragma unroll
                for (int t = 1; t < R; t++) {
                    const C w = tw[j * t * st.tws];
                    v[t] = cmul(v[t], mk(w.x, -w.y));
                }
            }
            rf::dft_inplace<R, +1, C>(v);
        } else {
            rf::dft_inplace<R, -1, C>(v);
            if constexpr (KIND == 0) {
                if (st.sub > 1) {
#pragma unroll
                    for (int t = 1; t < R; t++) v[t] = cmul(v[t], tw[j * t * st.tws]);
                }
            } else {
#pragma unroll
                for (int t = 0; t < R; t++) op(i0 + t, qi, v[t]);
                rf::dft_inplace<R, +1, C>(v);
            }
        }
#pragma unroll
        for (int t = 0; t < R; t++) p[t * step] = v[t];
    }
    __syncthreads();
}

template <int KIND, typename C, typename OP>
__device__ __forceinline__ void rs_run(C *A, const C *tw, const RsAxis &ax, int s, OP &&op)
{
    const RsStage st = ax.st[s];
    switch (st.R) {
    case 2: rs_stage<2, KIND>(A, tw + ax.tw, ax, st, op); break;
    case 3: rs_stage<3, KIND>(A, tw + ax.tw, ax, st, op); break;
    case 4: rs_stage<4, KIND>(A, tw + ax.tw, ax, st, op); break;
    case 6: rs_stage<6, KIND>(A, tw + ax.tw, ax, st, op); break;
    case 8: rs_stage<8, KIND>(A, tw + ax.tw, ax, st, op); break;
    case 9: rs_stage<9, KIND>(A, tw + ax.tw, ax, st, op); break;
    default: rs_stage<12, KIND>(A, tw + ax.tw, ax, st, op); break;
    }
}
struct RsNop {
    template <typename C> __device__ void operator()(unsigned, unsigned, C &) const {}
};
// all forward / all inverse stages of an axis
template <typename C> __device__ __forceinline__ void rs_forward(C *A, const C *tw, const RsAxis &ax)
{
    for (int s = 0; s < ax.nst; s++) rs_run<0>(A, tw, ax, s, RsNop());
}
template <typename C> __device__ __forceinline__ void rs_inverse(C *A, const C *tw, const RsAxis &ax)
{
    for (int s = ax.nst - 1; s >= 0; s--) rs_run<1>(A, tw, ax, s, RsNop());
}
// F^-1 op F along the axis (nst >= 1)
template <typename C, typename OP>
__device__ __forceinline__ void rs_filter(C *A, const C *tw, const RsAxis &ax, OP &&op)
{
    for (int s = 0; s < ax.nst - 1; s++) rs_run<0>(A, tw, ax, s, RsNop());
    rs_run<2>(A, tw, ax, ax.nst - 1, op);
    for (int s = ax.nst - 2; s >= 0; s--) rs_run<1>(A, tw, ax, s, RsNop());
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
// The radices of an axis: the fewest stages, then the smallest largest radix
// (registers: the 12 values of a stage are 48 VGPRs in FP64).  -1: the length
// has another prime factor, or too many.
inline bool rs_split(int rem, int m, int top, int *R)
{
    if (m == 0) return rem == 1;
    for (int q : {12, 9, 8, 6, 4, 3, 2})
        if (q <= top && rem % q == 0) {
            R[0] = q;
            if (rs_split(rem / q, m - 1, top, R + 1)) return true;
        }
    return false;
}
inline int rs_radices(int L, int *R)
{
    for (int m = 0; m <= RS_MAXST; m++)
        for (int top : {2, 3, 4, 6, 8, 9, 12})
            if (rs_split(L, m, top, R)) return m;
    return -1;
}

// fills ax (geometry as given); false where the length has no plan
inline bool rs_axis(RsAxis &ax, int L, int is, int P, int qd, int qh, int tw)
{
    int R[RS_MAXST];
    ax.L = L;
    ax.is = is;
    ax.P = P;
    ax.qd = qd;
    ax.qh = qh;
    ax.tw = tw;
    ax.mP = rs_magic(P);
    ax.mqd = rs_magic(qd);
    ax.nst = rs_radices(L, R);
    if (ax.nst < 0) return false;
    int sub = L, mul = 1;
    for (int s = 0; s < ax.nst; s++) {
        RsStage &st = ax.st[s];
        st.tws = mul;
        sub /= R[s];
        mul *= R[s];
        st.R = R[s];
        st.sub = sub;
        st.msub = rs_magic(sub);
    }
    return true;
}
// index f of the frequency held at each position of the transformed axis
inline std::vector<int> rs_order(const RsAxis &ax)
{
    std::vector<int> o(ax.L);
    for (int p = 0; p < ax.L; p++) {
        int f = 0, w = 1, rem = p, blk = ax.L;
        for (int s = 0; s < ax.nst; s++) {
            blk /= ax.st[s].R;
            f += w * (rem / blk);
            rem %= blk;
            w *= ax.st[s].R;
        }
        o[p] = f;
    }
    return o;
}
// momentum of frequency index f on an axis of L points and length Lp, the
// convention of kval
inline double rs_k(int f, int L, double Lp) { return 2. * M_PI / Lp * (double)(f < L / 2 ? f : f - L); }

}  // namespace tdw
