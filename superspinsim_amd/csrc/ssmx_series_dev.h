// ssmx_series_dev.h - device code shared by the kernels of the series in the
// drive (ssmx_series.hip, ssmx_series_adjoint.hip): drive factors, broadcasts
// within lane rows, and one instance on a whole wavefront.
#pragma once

#include "ssmx_common.h"

namespace ssmx {

// Node times and weights of a run.
struct Clock {
    double t0, dt, h;
    int fine, n_node;
    const double *nodes, *w;
};

// Drive factors of a wavefront's members, lane-parallel: entry
// (b * members + member) * J + j of `fbuf` holds f_j of step b of the batch.
// The lane's waveform segment stays in registers between batches (node
// times only increase), and output and fine index come from the batch's
// first step by one 32-bit division: a batch of 16 steps is otherwise a tenth
// of the wavefront's instructions.
template <int J>
struct DriveFactors {
    int MJ, B, my_b, my_j, cursor, begin, count;
    double base;
    ssmx_segment seg;

    // `wv` is the waveform of the lane's entry (member (lane / J) % members)
    __device__ DriveFactors(const ssmx_wave *wv, const ssmx_segment *segs,
                            int gen, int members, int lane)
    {
        MJ = members * J;
        B = kWave / MJ;
        my_b = lane / MJ;
        my_j = lane % J;
        base = wv->base[gen];
        begin = wv->seg_begin[gen];
        count = wv->seg_count[gen];
        cursor = 0;
        if (count > 0)
            seg = segs[begin];
    }

    // wave_coef for times that only increase
    __device__ double coefficient(const ssmx_segment *segs, double t)
    {
#pragma clang fp contract(off)
        while (cursor < count && !(t < seg.t_end)) {
            ++cursor;
            if (cursor < count)
                seg = segs[begin + cursor];
        }
        double c = base;
        if (cursor < count && !(t < seg.t_start))
            c += seg.amp * cos(seg.omega * t + seg.phase);
        return c;
    }

    // The steps from output i, fine step k on, `left` at most.
    __device__ void fill(const Clock &c, const ssmx_segment *segs, long i,
                         int k, long left, int lane, double *fbuf)
    {
        const unsigned ahead = (unsigned)k + (unsigned)my_b;
        const unsigned di = ahead / (unsigned)c.fine;
        const int r = (int)(ahead - di * (unsigned)c.fine);
        const long out = i + di;
        const bool on = my_b < B && my_b < left;
        double f;
        if constexpr (J <= 2) {
            // schemes with as many nodes as exponentials: each lane
            // evaluates one node, pairs of lanes exchange theirs
            double v = 0.0;
            if (on)
                v = coefficient(segs, node_time(c.t0, c.dt, c.fine, r, out,
                                                c.nodes[my_j]));
            if constexpr (J == 2) {
                const double o = swap_pair(v);
                const double c0 = my_j == 0 ? v : o;
                const double c1 = my_j == 0 ? o : v;
                f = fma(c.w[my_j * 2 + 1], c1, fma(c.w[my_j * 2], c0, 0.0));
            } else {
                f = fma(c.w[0], v, 0.0);
            }
        } else {
            f = 0.0;
            if (on)
                for (int s = 0; s < c.n_node; ++s)
                    f = fma(c.w[my_j * c.n_node + s],
                            coefficient(segs, node_time(c.t0, c.dt, c.fine,
                                                        r, out,
                                                        c.nodes[s])),
                            f);
        }
        fbuf[lane] = c.h * f;
        wave_exchange();
    }
};

// a += wa[k] x(lane K0 + k), b += wb[k] x(lane K0 + k), k < N, for the lanes
// of each 16-lane row: x is broadcast within the row by the multiply-add's own
// DPP operand (row_newbcast).  One block per group of up to four: a DPP operand
// may be read two wait states after a VALU write, which the leading s_nop
// covers whatever the compiler places in front; nothing in the block writes
// x.
#define SSMX_BCAST(K, A, B)                                                 \
    "v_fmac_f64_dpp %0, %2, " A " row_newbcast:" K                          \
    " row_mask:0xf bank_mask:0xf\n\t"                                       \
    "v_fmac_f64_dpp %1, %2, " B " row_newbcast:" K                          \
    " row_mask:0xf bank_mask:0xf\n\t"

template <int K0, int N>
__device__ __forceinline__ void bcast_fma(double &a, double &b, double x,
                                          const double *wa, const double *wb)
{
    if constexpr (N >= 4) {
        asm("s_nop 1\n\t" SSMX_BCAST("%11", "%3", "%7")
                SSMX_BCAST("%12", "%4", "%8") SSMX_BCAST("%13", "%5", "%9")
                    SSMX_BCAST("%14", "%6", "%10")
            : "+v"(a), "+v"(b)
            : "v"(x), "v"(wa[0]), "v"(wa[1]), "v"(wa[2]), "v"(wa[3]),
              "v"(wb[0]), "v"(wb[1]), "v"(wb[2]), "v"(wb[3]), "n"(K0),
              "n"(K0 + 1), "n"(K0 + 2), "n"(K0 + 3));
        bcast_fma<K0 + 4, N - 4>(a, b, x, wa + 4, wb + 4);
    } else if constexpr (N >= 2) {
        asm("s_nop 1\n\t" SSMX_BCAST("%7", "%3", "%5")
                SSMX_BCAST("%8", "%4", "%6")
            : "+v"(a), "+v"(b)
            : "v"(x), "v"(wa[0]), "v"(wa[1]), "v"(wb[0]), "v"(wb[1]),
              "n"(K0), "n"(K0 + 1));
        bcast_fma<K0 + 2, N - 2>(a, b, x, wa + 2, wb + 2);
    } else if constexpr (N == 1) {
        asm("s_nop 1\n\t" SSMX_BCAST("%5", "%3", "%4")
            : "+v"(a), "+v"(b)
            : "v"(x), "v"(wa[0]), "v"(wb[0]), "n"(K0));
    }
}
#undef SSMX_BCAST

// a += w[k] x(lane K0 + k), k < N.
template <int K0, int N>
__device__ __forceinline__ void bcast_fma1(double &a, double x,
                                           const double *w)
{
    if constexpr (N >= 1) {
        asm("s_nop 1\n\tv_fmac_f64_dpp %0, %1, %2 row_newbcast:%3"
            " row_mask:0xf bank_mask:0xf"
            : "+v"(a)
            : "v"(x), "v"(w[0]), "n"(K0));
        bcast_fma1<K0 + 1, N - 1>(a, x, w + 1);
    }
}

// Coefficients of one exponential for one lane: P_s(u) = sum_o c[s][o] u^o.
template <int N, int D>
__device__ __forceinline__ void horner(double (&w)[N],
                                       const double (&c)[N][D + 1], double u)
{
#pragma unroll
    for (int s = 0; s < N; ++s) {
        w[s] = c[s][D];
#pragma unroll
        for (int o = D - 1; o >= 0; --o)
            w[s] = fma(u, w[s], c[s][o]);
    }
}

// v of the lane 16 further or back, i.e. of the other row of its pair.
__device__ __forceinline__ double swap_rows(double v, bool odd_row)
{
    const auto lo = __builtin_amdgcn_permlane16_swap(
        __double2loint(v), __double2loint(v), false, false);
    const auto hi = __builtin_amdgcn_permlane16_swap(
        __double2hiint(v), __double2hiint(v), false, false);
    // result 0 holds the even rows' values in both rows, result 1 the odd
    // rows'
    return odd_row ? __hiloint2double(hi[0], lo[0])
                   : __hiloint2double(hi[1], lo[1]);
}

// Sum of v over the wavefront's halves (lane, lane ^ 32), in every lane.
__device__ __forceinline__ double sum_halves(double v)
{
    const auto lo = __builtin_amdgcn_permlane32_swap(
        __double2loint(v), __double2loint(v), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(
        __double2hiint(v), __double2hiint(v), false, false);
    return __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
}

// One instance on the whole wavefront: both halves hold the state (rows as
// in series_row_kernel); the first half multiplies the first S = ceil(N / 2)
// components of its rows, the second half the others, which a rotation within
// the row brings to the same lanes.
template <int N>
struct Halves {
    static constexpr int S = (N + 1) / 2;

    // x in the first half, x of lane + S (of the row) in the second
    static __device__ __forceinline__ double shifted(double x)
    {
        constexpr int kRotate = 0x120 + 16 - S;     // row_ror
        const int lo = __double2loint(x), hi = __double2hiint(x);
        return __hiloint2double(
            __builtin_amdgcn_update_dpp(hi, hi, kRotate, 0xC, 0xF, false),
            __builtin_amdgcn_update_dpp(lo, lo, kRotate, 0xC, 0xF, false));
    }

    // x <- exp(A) x
    template <int DA, int DB>
    static __device__ __forceinline__ void exponential(
        double &x, double f, const double (&ca)[S][DA + 1],
        const double (&cb)[S][DB + 1], bool odd_row)
    {
        const double u = f * f;
        double wa[S], wb[S];
        horner<S, DA>(wa, ca, u);
        horner<S, DB>(wb, cb, u);
        double ya = 0.0, yb = 0.0;
        bcast_fma<0, S>(ya, yb, shifted(x), wa, wb);
        x += sum_halves(fma(f, swap_rows(yb, odd_row), ya));
    }

    // M x for a matrix within the sectors
    static __device__ __forceinline__ double within(double xs,
                                                    const double (&m)[S])
    {
        double y = 0.0;
        bcast_fma1<0, S>(y, xs, m);
        return sum_halves(y);
    }
};

}  // namespace ssmx
