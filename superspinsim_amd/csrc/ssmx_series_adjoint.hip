// ssmx_series_adjoint.hip - gradient of an integrated readout through the
// series in the drive.
//
// An exponential takes y to x = y + sum_k f^k E_k y with constant matrices
// E_k. In reverse, with the cotangent mu of x,
//     cotangent of y  = mu + sum_k f^k E_k^T mu,
//     dF/dE_k        += f^k mu y^T,      dF/df += mu^T (sum_k k f^(k-1) E_k) y.
// The derivative with respect to the parameters of the constant matrix is
// therefore a contraction of a few moments sum f^k mu y^T, summed over all
// steps in registers, with dE_k / dtheta, formed once on the host: no Frechet
// chain per exponential. Orders 0..4 are kept for entries within a sector, 0..3
// for those between the two (every order in both: parameters that break the
// model's parity enter E_k at the other parity), which the host allows only
// where the rest is below the adjoint's tolerance beside the first order that
// a parameter can act through.
//
// One instance per wavefront, both halves holding the cotangent (Halves): a
// lane owns a column s, i.e. component s of y and of the new cotangent, and
// multiplies half of the rows r, broadcast from the lanes that hold mu_r (the
// opposite sector's after one exchange of rows). The same broadcasts feed the
// product with E_k^T, the derivative in f and the moments.
//
// What bounds it: VALU issue, about 136 instructions per exponential of which
// 54 are moments and 24 the derivative in f. 512 points x 25,000 steps, 9
// parameters and 50 amplitudes: 33.6 ms after a forward run of 8.7; the Frechet
// chain of adjoint_kernel took 88 after a forward run of 51. (Without order 4
// within the sectors 32.9, and what a parameter does through the drive alone
// was off by up to 1e-9.)
#include "ssmx_series_dev.h"

namespace {

using ssmx::Clock;
using ssmx::Halves;
using ssmx::horner;
using ssmx::kWave;
using ssmx::node_time;
using ssmx::set_error;
using ssmx::swap_pair;
using ssmx::swap_rows;
using ssmx::wave_exchange;

// orders of the moments within a sector and between sectors
constexpr int kOwn = 5, kOpp = 4;

struct AParams {
    ssmx_series_desc d;
    const int32_t *lanes;
    const double *table;
    const double *dtable;
    const double *w;
    const double *nodes;
    const ssmx_wave *waves;
    const ssmx_segment *segs;
    const double *store;
    const double *obs;
    const double *seed;
    double *grad_theta;
    double *grad_seg;
    double *lambda_out;
    int32_t n_theta;
};

// a += wa[k] xa(lane k), b += wb[k] xb(lane k), k < N, broadcast within each
// 16-lane row as bcast_fma does.
template <int K0, int N>
__device__ __forceinline__ void bcast_two(double &a, double xa,
                                          const double *wa, double &b,
                                          double xb, const double *wb)
{
    if constexpr (N >= 2) {
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %0, %2, %4 row_newbcast:%8 row_mask:0xf "
            "bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %1, %3, %6 row_newbcast:%8 row_mask:0xf "
            "bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %0, %2, %5 row_newbcast:%9 row_mask:0xf "
            "bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %1, %3, %7 row_newbcast:%9 row_mask:0xf "
            "bank_mask:0xf"
            : "+v"(a), "+v"(b)
            : "v"(xa), "v"(xb), "v"(wa[0]), "v"(wa[1]), "v"(wb[0]),
              "v"(wb[1]), "n"(K0), "n"(K0 + 1));
        bcast_two<K0 + 2, N - 2>(a, xa, wa + 2, b, xb, wb + 2);
    } else if constexpr (N == 1) {
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %0, %2, %4 row_newbcast:%6 row_mask:0xf "
            "bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %1, %3, %5 row_newbcast:%6 row_mask:0xf "
            "bank_mask:0xf"
            : "+v"(a), "+v"(b)
            : "v"(xa), "v"(xb), "v"(wa[0]), "v"(wb[0]), "n"(K0));
    }
}

// m[s][k] += z[k] x(lane s), s < N.
template <int K0, int N, int O>
__device__ __forceinline__ void bcast_moments(double (*m)[O], double x,
                                              const double (&z)[kOwn])
{
    if constexpr (N >= 1 && O == 5) {
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %0, %5, %6 row_newbcast:%11 row_mask:0xf "
            "bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %1, %5, %7 row_newbcast:%11 row_mask:0xf "
            "bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %2, %5, %8 row_newbcast:%11 row_mask:0xf "
            "bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %3, %5, %9 row_newbcast:%11 row_mask:0xf "
            "bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %4, %5, %10 row_newbcast:%11 row_mask:0xf "
            "bank_mask:0xf"
            : "+v"(m[0][0]), "+v"(m[0][1]), "+v"(m[0][2]), "+v"(m[0][3]),
              "+v"(m[0][4])
            : "v"(x), "v"(z[0]), "v"(z[1]), "v"(z[2]), "v"(z[3]), "v"(z[4]),
              "n"(K0));
        bcast_moments<K0 + 1, N - 1>(m + 1, x, z);
    } else if constexpr (N >= 1) {
        static_assert(O == 4, "moments of four or five orders");
        asm("s_nop 1\n\t"
            "v_fmac_f64_dpp %0, %4, %5 row_newbcast:%9 row_mask:0xf "
            "bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %1, %4, %6 row_newbcast:%9 row_mask:0xf "
            "bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %2, %4, %7 row_newbcast:%9 row_mask:0xf "
            "bank_mask:0xf\n\t"
            "v_fmac_f64_dpp %3, %4, %8 row_newbcast:%9 row_mask:0xf "
            "bank_mask:0xf"
            : "+v"(m[0][0]), "+v"(m[0][1]), "+v"(m[0][2]), "+v"(m[0][3])
            : "v"(x), "v"(z[0]), "v"(z[1]), "v"(z[2]), "v"(z[3]), "n"(K0));
        bcast_moments<K0 + 1, N - 1>(m + 1, x, z);
    }
}

// Drive factors and amplitude weights of a batch of steps in reverse: entry
// (b, node) of the lane is step `top` - b. The lane's segment stays in
// registers; its times fall from call to call.
template <int J>
struct ReverseDrive {
    int b, node, cursor, begin, count;
    double base;
    ssmx_segment seg;

    __device__ ReverseDrive(const ssmx_wave *wv, const ssmx_segment *segs,
                            int gen, int lane)
    {
        b = lane / J;
        node = lane % J;
        base = wv->base[gen];
        begin = wv->seg_begin[gen];
        count = wv->seg_count[gen];
        cursor = count - 1;
        if (count > 0)
            seg = segs[begin + cursor];
    }

    // f[b * J + j], a[(b * J + j) * J + node] = h w[j, node] dc/d(amplitude)
    // and the segment record holding the node (or -1)
    __device__ void fill(const Clock &c, const ssmx_segment *segs, long top,
                         int lane, double *f, double *a, int *rec)
    {
        const long step = top - b;
        double v = base, damp = 0.0;
        int r = -1;
        if (step >= 0) {
            const long out = step / c.fine;
            const double t = node_time(c.t0, c.dt, c.fine,
                                       (int)(step - out * c.fine), out,
                                       c.nodes[node]);
            while (cursor > 0 && t < seg.t_start) {
                --cursor;
                seg = segs[begin + cursor];
            }
            if (count > 0 && !(t < seg.t_start) && t < seg.t_end) {
#pragma clang fp contract(off)
                damp = cos(seg.omega * t + seg.phase);
                v += seg.amp * damp;
                r = begin + cursor;
            }
        }
        double cw;
        if constexpr (J == 2) {
            const double o = swap_pair(v);
            const double c0 = node == 0 ? v : o;
            const double c1 = node == 0 ? o : v;
            cw = fma(c.w[node * 2 + 1], c1, fma(c.w[node * 2], c0, 0.0));
        } else {
            cw = fma(c.w[0], v, 0.0);
        }
        f[lane] = c.h * cw;
#pragma unroll
        for (int j = 0; j < J; ++j)
            a[(b * J + j) * J + node] = c.h * c.w[j * J + node] * damp;
        rec[lane] = r;
        wave_exchange();
    }
};

template <int DA, int DB, int J>
__global__ __launch_bounds__(kWave)
__attribute__((amdgpu_waves_per_eu(1))) void series_adjoint_kernel(AParams p)
{
    constexpr int N = 11, S = Halves<N>::S, B = kWave / J;
    // steps of stored inputs in flight: the loads are issued this far ahead
    constexpr int kAhead = 8;
    __shared__ double fbuf[kWave], abuf[kWave * J];
    __shared__ int rbuf[kWave];
    const ssmx_series_desc &d = p.d;
    const int lane = threadIdx.x;
    const bool odd_row = (lane & 16) != 0;
    const int state = p.lanes[lane];
    const bool has = state >= 0;
    const long inst = blockIdx.x;
    double ca[S][DA + 1], cb[S][DB + 1];
#pragma unroll
    for (int s = 0; s < S; ++s) {
#pragma unroll
        for (int o = 0; o <= DA; ++o)
            ca[s][o] = p.table[(s * (DA + 1) + o) * kWave + lane];
#pragma unroll
        for (int o = 0; o <= DB; ++o)
            cb[s][o] =
                p.table[(S * (DA + 1) + s * (DB + 1) + o) * kWave + lane];
    }
    double mown[S][kOwn], mopp[S][kOpp];
#pragma unroll
    for (int s = 0; s < S; ++s) {
#pragma unroll
        for (int k = 0; k < kOwn; ++k)
            mown[s][k] = 0.0;
#pragma unroll
        for (int k = 0; k < kOpp; ++k)
            mopp[s][k] = 0.0;
    }
    double source = 0.0;
    if (has)
        for (int o = 0; o < d.n_obs; ++o)
            source = fma(p.seed[inst * d.n_obs + o], p.obs[o * d.n + state],
                         source);
    const Clock clk{d.t0, d.dt, d.h, d.fine, d.n_node, p.nodes, p.w};
    ReverseDrive<J> drive(p.waves + inst, p.segs, d.gen, lane);
    const long total = (long)d.n_out * d.fine;
    const double *store = p.store + (size_t)inst * total * 32 * J;
    const int at = J == 2 ? lane : lane % 32;
    const double half_h = 0.5 * d.h;
    double lambda = half_h * source;
    const bool grad = p.grad_seg != nullptr;
    int current = -1;
    double acc = 0.0;
    auto flush = [&](int next) {
        if (current >= 0) {
            double v = acc;
#pragma unroll
            for (int off = 32; off > 0; off >>= 1)
                v += __shfl_xor(v, off, kWave);
            if (lane == 0)
                p.grad_seg[current] += v;
        }
        current = next;
        acc = 0.0;
    };

    double ahead[kAhead];
#pragma unroll
    for (int k = 0; k < kAhead; ++k)
        ahead[k] = total - 1 - k >= 0
                       ? store[(size_t)(total - 1 - k) * 32 * J + at]
                       : 0.0;
    int b = B;
    long top = total - 1;                    // step of ahead[0]
    while (top >= 0) {
        // (B is a multiple of kAhead, so a batch ends with a group)
        if (b == B) {
            b = 0;
            drive.fill(clk, p.segs, top, lane, fbuf, abuf, rbuf);
        }
#pragma unroll
        for (int g = 0; g < kAhead; ++g) {
            const long step = top - g;
            if (step < 0)
                break;
            const double both = ahead[g];
            const long load = step - kAhead;
            if (load >= 0)
                ahead[g] = store[(size_t)load * 32 * J + at];
            // both exponentials' inputs in every lane
            double y[J];
            if constexpr (J == 2) {
                const auto lo = __builtin_amdgcn_permlane32_swap(
                    __double2loint(both), __double2loint(both), false,
                    false);
                const auto hi = __builtin_amdgcn_permlane32_swap(
                    __double2hiint(both), __double2hiint(both), false,
                    false);
                y[1] = __hiloint2double(hi[0], lo[0]);
                y[0] = __hiloint2double(hi[1], lo[1]);
            } else {
                y[0] = both;
            }
            const int e = b + g;
            int r0 = -1, r1 = -1;
            if (grad) {
                r0 = __builtin_amdgcn_readfirstlane(rbuf[e * J]);
                r1 = J == 2 ? __builtin_amdgcn_readfirstlane(rbuf[e * J + 1])
                            : r0;
                if (r1 != current)
                    flush(r1);
            }
            double early = 0.0;              // node 0's record where it differs
#pragma unroll
            for (int j = 0; j < J; ++j) {
                const double f = fbuf[e * J + j], u = f * f;
                const double ms = Halves<N>::shifted(lambda);
                const double mo =
                    Halves<N>::shifted(swap_rows(lambda, odd_row));
                double wa[S], wb[S];
                horner<S, DA>(wa, ca, u);
                horner<S, DB>(wb, cb, u);
                double ya = 0.0, yb = 0.0;
                bcast_two<0, S>(ya, ms, wa, yb, mo, wb);
                if (grad) {
                    ssmx::keep_branch();
                    // d/df: 2 f (E_2 + 2 u E_4) and E_1 + 3 u (E_3 + ..)
                    double da[S], db[S];
#pragma unroll
                    for (int s = 0; s < S; ++s) {
                        if constexpr (DA == 2)
                            da[s] = fma(2.0 * u, ca[s][2], ca[s][1]);
                        else
                            da[s] = ca[s][1];
                        if constexpr (DB == 2)
                            db[s] = fma(3.0 * u,
                                        fma((5.0 / 3.0) * u, cb[s][2],
                                            cb[s][1]),
                                        cb[s][0]);
                        else
                            db[s] = fma(3.0 * u, cb[s][1], cb[s][0]);
                    }
                    double ga = 0.0, gb = 0.0;
                    bcast_two<0, S>(ga, ms, da, gb, mo, db);
                    const double g1 = y[j] * fma(2.0 * f, ga, gb);
                    if constexpr (J == 2) {
                        const double a0 = abuf[(e * 2 + j) * 2];
                        const double a1 = abuf[(e * 2 + j) * 2 + 1];
                        acc = fma(a1, g1, acc);
                        if (r0 == r1)
                            acc = fma(a0, g1, acc);
                        else
                            early = fma(a0, g1, early);
                    } else {
                        acc = fma(abuf[e], g1, acc);
                    }
                }
                double z[kOwn];
                z[0] = y[j];
                z[1] = f * y[j];
                z[2] = u * y[j];
                z[3] = u * z[1];
                z[4] = u * z[2];
                bcast_moments<0, S>(mown, ms, z);
                bcast_moments<0, S>(mopp, mo, z);
                lambda += ssmx::sum_halves(fma(f, yb, ya));
            }
            if (grad && r0 != r1) {
                flush(r0);
                acc = early;
            }
            lambda = fma(step == 0 ? half_h : d.h, source, lambda);
        }
        b += kAhead;
        top -= kAhead;
        wave_exchange();
    }
    if (grad)
        flush(-1);
    for (int i = 0; i < p.n_theta; ++i) {
        const double *t =
            p.dtable + (size_t)i * S * (kOwn + kOpp) * kWave + lane;
        double v = 0.0;
#pragma unroll
        for (int s = 0; s < S; ++s) {
#pragma unroll
            for (int k = 0; k < kOwn; ++k)
                v = fma(mown[s][k], t[(s * kOwn + k) * kWave], v);
#pragma unroll
            for (int k = 0; k < kOpp; ++k)
                v = fma(mopp[s][k], t[(S * kOwn + s * kOpp + k) * kWave], v);
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1)
            v += __shfl_xor(v, off, kWave);
        if (lane == 0)
            p.grad_theta[(size_t)inst * p.n_theta + i] = v;
    }
    if (p.lambda_out && has && lane < 32)
        p.lambda_out[(size_t)inst * d.n + state] = lambda;
}

template <int DA, int DB>
int launch(const AParams &p, hipStream_t stream)
{
    if (p.d.n_exp == 1)
        hipLaunchKernelGGL((series_adjoint_kernel<DA, DB, 1>),
                           dim3(p.d.n_inst), dim3(kWave), 0, stream, p);
    else
        hipLaunchKernelGGL((series_adjoint_kernel<DA, DB, 2>),
                           dim3(p.d.n_inst), dim3(kWave), 0, stream, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return set_error(SSMX_ELAUNCH, "series adjoint launch: %s",
                         hipGetErrorString(e));
    return SSMX_OK;
}

}  // namespace

extern "C" int ssmx_series_adjoint(
    const ssmx_series_desc *desc, const int32_t *lanes, const double *table,
    const double *dtable, int32_t n_theta, const double *cf_weights,
    const double *cf_nodes, const ssmx_wave *waves,
    const ssmx_segment *segments, const double *store, const double *obs,
    const double *seed, double *grad_theta, double *grad_seg,
    double *lambda_out, void *stream)
{
    ssmx::error_buffer()[0] = '\0';
    if (!desc)
        return set_error(SSMX_EINVAL, "null descriptor");
    const ssmx_series_desc &d = *desc;
    if (d.n < 1 || d.n_inst < 1 || (d.n_exp != 1 && d.n_exp != 2) ||
        d.n_node != d.n_exp || d.fine < 1 || d.n_out < 1 || d.n_obs < 1 ||
        d.n_obs > SSMX_MAX_OBS || d.gen < 0 || d.gen >= SSMX_MAX_GEN ||
        d.na != 11 || d.nb != 11 || d.wave_group != 1 || d.members != 1 ||
        n_theta < 0 || !(d.h > 0.0) || !(d.dt > 0.0))
        return set_error(SSMX_EINVAL, "series adjoint: n=%d, n_inst=%d, "
                         "n_exp=%d, n_node=%d, n_out=%d, n_obs=%d, gen=%d, "
                         "n_theta=%d", d.n, d.n_inst, d.n_exp, d.n_node,
                         d.n_out, d.n_obs, d.gen, n_theta);
    if (!lanes || !table || !cf_weights || !cf_nodes || !waves ||
        !segments || !store || !obs || !seed ||
        (n_theta > 0 && (!dtable || !grad_theta)))
        return set_error(SSMX_EINVAL, "null required pointer");
    AParams p;
    p.d = d;
    p.lanes = lanes;
    p.table = table;
    p.dtable = dtable;
    p.w = cf_weights;
    p.nodes = cf_nodes;
    p.waves = waves;
    p.segs = segments;
    p.store = store;
    p.obs = obs;
    p.seed = seed;
    p.grad_theta = grad_theta;
    p.grad_seg = grad_seg;
    p.lambda_out = lambda_out;
    p.n_theta = n_theta;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (d.da == 1 && d.db == 1)
        return launch<1, 1>(p, s);
    if (d.da == 2 && d.db == 1)
        return launch<2, 1>(p, s);
    if (d.da == 2 && d.db == 2)
        return launch<2, 2>(p, s);
    return set_error(SSMX_EINVAL, "no series kernel for orders da=%d, db=%d",
                     d.da, d.db);
}
