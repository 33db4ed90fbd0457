// ssmx_series.hip - propagation by the exponential's series in the drive.
//
// Exponents A = h w C + f G hold one constant matrix C (precession, static
// couplings, damping: 1-norm about 0.2 at 20 ps steps) and one driven matrix
// G whose share f G is small (about 1e-3).  A Taylor chain in A needs 11
// dependent products to 1e-16.  Expanded in f alone, with every order of C
// summed into constant matrices E_k on the host,
//     exp(A) x = x + E_0 x + f E_1 x + f^2 E_2 x + ..,
// four or five orders reach the same accuracy, and all of them read the same
// x: one LDS exchange per exponential instead of eleven.
//
// Split.  C is block diagonal over sectors and G couples each sector with
// its opposite one (populations and double-quantum coherences against
// single-quantum coherences: 11 + 8 of the 7-level model's 19 reachable
// states, 5 + 4 of the 3-level one's 9), so even orders stay in the row's own
// sector and odd orders come from the opposite one.  Lane r holds row r's
// coefficients of every order in registers (at most 11 (da + 1) + 11 (db + 1)
// doubles), forms its row of the exponential by Horner in f^2, and
// multiplies it by the two sectors read from LDS in 16-byte reads, which all
// lanes of a sector read at one address.
#include "ssmx_common.h"

namespace {

using ssmx::kWave;
using ssmx::node_time;
using ssmx::set_error;
using ssmx::swap_pair;
using ssmx::wave_coef;
using ssmx::wave_exchange;

struct SParams {
    ssmx_series_desc d;
    const int32_t *layout;
    const int32_t *state_pos;
    const double *table;
    const double *w;
    const double *nodes;
    const ssmx_wave *waves;
    const ssmx_segment *segs;
    const double *rho0;
    const double *obs;
    double *out;
};

// Table set of exponential j: the weight rows of the symmetric schemes
// repeat from both ends.
template <int J>
constexpr int set_of(int j)
{
    return j < J - 1 - j ? j : J - 1 - j;
}

// One instance per `rows` lanes.  J = n_exp.
template <int NA, int DA, int NB, int DB, int J>
__global__ __launch_bounds__(kWave)
__attribute__((amdgpu_waves_per_eu(NA > 6 || J > 2 ? 2 : 3))) void series_kernel(
    SParams p)
{
    constexpr int SETS = (J + 1) / 2 == 1 || J == 2 ? 1 : (J + 1) / 2;
    constexpr int PA = (NA + 1) / 2, PB = (NB + 1) / 2;
    extern __shared__ __attribute__((aligned(16))) double lds[];
    const ssmx_series_desc &d = p.d;
    const int lane = threadIdx.x;
    const int rows = d.rows;
    const int used = d.members * rows;
    const int q = lane < used ? lane / rows : 0;
    const int r = lane < used ? lane - q * rows : 0;
    const int stride = d.sectors * d.sector;  // LDS doubles per member
    double *xbuf = lds;                       // [members][stride], scratch
    double *fbuf = lds + d.members * stride + 2;
    double *red = fbuf + kWave;
    // every sector is padded with zeros up to `sector`, so the fixed-length
    // reads beyond a short sector meet zeros only
    for (int e = lane; e < d.members * stride + 2; e += kWave)
        xbuf[e] = 0.0;

    // idle lanes write to the scratch double behind the members
    const int pos = lane < used ? q * stride + p.layout[4 * r]
                                : d.members * stride;
    const double2 *own = reinterpret_cast<const double2 *>(
        xbuf + q * stride + p.layout[4 * r + 1]);
    const double2 *opp = reinterpret_cast<const double2 *>(
        xbuf + q * stride + p.layout[4 * r + 2]);
    const int state = p.layout[4 * r + 3];

    double ca[SETS][NA][DA + 1], cb[SETS][NB][DB + 1];
#pragma unroll
    for (int set = 0; set < SETS; ++set) {
        const double *t =
            p.table + (size_t)set * (NA * (DA + 1) + NB * (DB + 1)) * rows;
#pragma unroll
        for (int e = 0; e < NA * (DA + 1); ++e)
            ca[set][e / (DA + 1)][e % (DA + 1)] =
                lane < used ? t[(size_t)e * rows + r] : 0.0;
#pragma unroll
        for (int e = 0; e < NB * (DB + 1); ++e)
            cb[set][e / (DB + 1)][e % (DB + 1)] =
                lane < used
                    ? t[(size_t)(NA * (DA + 1) + e) * rows + r]
                    : 0.0;
    }

    const long sys = blockIdx.x;
    const long inst = sys * d.members + q;
    const bool live = lane < used && inst < d.n_inst;
    double x = live ? p.rho0[(size_t)inst * d.n + state] : 0.0;
    const bool read_full = (d.flags & SSMX_READ_FULL) != 0;
    const bool read_int = (d.flags & SSMX_READ_INTEGRAL) != 0;
    double ob0 = 0.0, ob1 = 0.0;
    if (!read_full && live) {
        ob0 = p.obs[state];
        if (d.n_obs > 1)
            ob1 = p.obs[d.n + state];
    }
    // sum of v over the member's rows, written for readout o of output i
    auto observe = [&](double v, long index) {
        red[lane] = v;
        wave_exchange();
        if (live && r == 0) {
            double s = 0.0;
            for (int k = 0; k < rows; ++k)
                s += red[lane + k];
            p.out[index] = s;
        }
        wave_exchange();
    };

    // drive factors, lane-parallel: entry (b * members + member) * J + j
    // holds f_j of step b of the batch
    const int MJ = d.members * J;
    const int B = kWave / MJ;
    const int my_b = lane / MJ;
    const int my_j = lane % J;
    const long total = (long)d.n_out * d.fine;
    const ssmx_wave *wv;
    {
        long wi = sys * d.members + (lane / J) % d.members;
        if (wi >= d.n_inst)
            wi = d.n_inst - 1;
        wv = p.waves + wi / d.wave_group;
    }
    int cursor = 0;
    auto fill = [&](long first) {
        const long mine = first + my_b;
        const bool on = my_b < B && mine < total;
        const long i = on ? mine / d.fine : 0;
        const int rr = on ? (int)(mine - i * d.fine) : 0;
        double f;
        if constexpr (J <= 2) {
            // schemes with as many nodes as exponentials: each lane
            // evaluates one node, pairs of lanes exchange theirs
            double c = 0.0;
            if (on)
                c = wave_coef(wv, p.segs, d.gen,
                              node_time(d.t0, d.dt, d.fine, rr, i,
                                        p.nodes[my_j]),
                              cursor);
            if constexpr (J == 2) {
                const double o = swap_pair(c);
                const double c0 = my_j == 0 ? c : o;
                const double c1 = my_j == 0 ? o : c;
                f = fma(p.w[my_j * 2 + 1], c1, fma(p.w[my_j * 2], c0, 0.0));
            } else {
                f = fma(p.w[0], c, 0.0);
            }
        } else {
            f = 0.0;
            if (on)
                for (int s = 0; s < d.n_node; ++s)
                    f = fma(p.w[my_j * d.n_node + s],
                            wave_coef(wv, p.segs, d.gen,
                                      node_time(d.t0, d.dt, d.fine, rr, i,
                                                p.nodes[s]),
                                      cursor),
                            f);
        }
        fbuf[lane] = d.h * f;
        wave_exchange();
    };

    double xint = 0.0;
    const double half_h = 0.5 * d.h;
    double fc[J];
#pragma unroll
    for (int j = 0; j < J; ++j)
        fc[j] = 0.0;
    wave_exchange();
    long step = 0;
    int b = B;
    for (int i = 0; i < d.n_out; ++i) {
        for (int k = 0; k < d.fine; ++k, ++step) {
            if (b == B) {
                b = 0;
                fill(step);
#pragma unroll
                for (int j = 0; j < J; ++j)
                    fc[j] = fbuf[q * J + j];
            }
            // the next step's factors, read while this step runs
            double fn[J];
            const int nb = b + 1 < B ? b + 1 : b;
#pragma unroll
            for (int j = 0; j < J; ++j)
                fn[j] = fbuf[nb * MJ + q * J + j];
            const double before = x;
#pragma unroll
            for (int j = J - 1; j >= 0; --j) {
                constexpr int kSets = SETS;
                const int set = kSets == 1 ? 0 : set_of<J>(j);
                xbuf[pos] = x;
                __builtin_amdgcn_sched_barrier(0);
                wave_exchange();
                double va[2 * PA], vb[2 * PB];
#pragma unroll
                for (int s = 0; s < PA; ++s) {
                    const double2 v = own[s];
                    va[2 * s] = v.x;
                    va[2 * s + 1] = v.y;
                }
#pragma unroll
                for (int s = 0; s < PB; ++s) {
                    const double2 v = opp[s];
                    vb[2 * s] = v.x;
                    vb[2 * s + 1] = v.y;
                }
                __builtin_amdgcn_sched_barrier(0);
                // the row of exp(A), formed behind the reads
                const double f = fc[j], u = f * f;
                double ra[NA], rb[NB];
#pragma unroll
                for (int s = 0; s < NA; ++s) {
                    ra[s] = ca[set][s][DA];
#pragma unroll
                    for (int o = DA - 1; o >= 0; --o)
                        ra[s] = fma(u, ra[s], ca[set][s][o]);
                }
#pragma unroll
                for (int s = 0; s < NB; ++s) {
                    rb[s] = cb[set][s][DB];
#pragma unroll
                    for (int o = DB - 1; o >= 0; --o)
                        rb[s] = fma(u, rb[s], cb[set][s][o]);
                }
                wave_exchange();
                double ya = ra[0] * va[0], yb = rb[0] * vb[0];
#pragma unroll
                for (int s = 1; s < NA; ++s)
                    ya = fma(ra[s], va[s], ya);
#pragma unroll
                for (int s = 1; s < NB; ++s)
                    yb = fma(rb[s], vb[s], yb);
                x += fma(f, yb, ya);
            }
            if (read_int) {
                ssmx::keep_branch();
                xint = fma(half_h, before + x, xint);
            }
#pragma unroll
            for (int j = 0; j < J; ++j)
                fc[j] = fn[j];
            ++b;
        }
        if (read_full) {
            xbuf[pos] = x;
            wave_exchange();
            // the members' states in standard order, one per lane
            for (int e = lane; e < d.members * d.n; e += kWave) {
                const int m = e / d.n, s = e - m * d.n;
                const long to = sys * d.members + m;
                const int sp = p.state_pos[s];
                if (to < d.n_inst)
                    p.out[((size_t)to * d.n_out + i) * d.n + s] =
                        sp >= 0 ? xbuf[m * stride + sp] : 0.0;
            }
            wave_exchange();
        } else if (!read_int) {
            observe(ob0 * x, ((size_t)inst * d.n_out + i) * d.n_obs);
            if (d.n_obs > 1)
                observe(ob1 * x, ((size_t)inst * d.n_out + i) * d.n_obs + 1);
        }
    }
    if (read_int) {
        observe(ob0 * xint, (size_t)inst * d.n_obs);
        if (d.n_obs > 1)
            observe(ob1 * xint, (size_t)inst * d.n_obs + 1);
    }
}

template <int NA, int DA, int NB, int DB, int J>
int launch(const SParams &p, hipStream_t stream)
{
    const ssmx_series_desc &d = p.d;
    const size_t lds = ((size_t)d.members * d.sectors * d.sector + 2 +
                        2 * kWave) * sizeof(double);
    const int systems = (d.n_inst + d.members - 1) / d.members;
    hipLaunchKernelGGL((series_kernel<NA, DA, NB, DB, J>), dim3(systems),
                       dim3(kWave), lds, stream, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return set_error(SSMX_ELAUNCH, "series launch: %s",
                         hipGetErrorString(e));
    return SSMX_OK;
}

template <int N, int DA, int DB>
int launch_scheme(const SParams &p, hipStream_t stream)
{
    if (p.d.n_exp == 1)
        return launch<N, DA, N, DB, 1>(p, stream);
    if (p.d.n_exp == 2)
        return launch<N, DA, N, DB, 2>(p, stream);
    if constexpr (N <= 5)
        if (p.d.n_exp == 5)
            return launch<N, DA, N, DB, 5>(p, stream);
    return set_error(SSMX_EINVAL, "no series kernel for %d exponentials and "
                                  "%d components", p.d.n_exp, N);
}

template <int N>
int launch_orders(const SParams &p, hipStream_t stream)
{
    const int da = p.d.da, db = p.d.db;
    if (da == 1 && db == 1)
        return launch_scheme<N, 1, 1>(p, stream);
    if (da == 2 && db == 1)
        return launch_scheme<N, 2, 1>(p, stream);
    if (da == 2 && db == 2)
        return launch_scheme<N, 2, 2>(p, stream);
    return set_error(SSMX_EINVAL, "no series kernel for orders da=%d, db=%d",
                     da, db);
}

int validate(const ssmx_series_desc *d)
{
    if (!d)
        return set_error(SSMX_EINVAL, "null descriptor");
    if (d->n < 1 || d->n > SSMX_MAX_N_WIDE || d->rows < 1 ||
        d->rows > kWave || d->rows > d->n)
        return set_error(SSMX_EINVAL, "n=%d, rows=%d", d->n, d->rows);
    if (d->n_inst < 1 || d->members < 1 ||
        d->members * (long)d->rows > kWave)
        return set_error(SSMX_EINVAL, "n_inst=%d, members=%d of %d rows",
                         d->n_inst, d->members, d->rows);
    if ((d->n_exp != 1 && d->n_exp != 2 && d->n_exp != 5) ||
        d->n_node < 1 || d->n_node > SSMX_MAX_NODE ||
        (d->n_exp <= 2 && d->n_node != d->n_exp) ||
        d->members * d->n_exp > kWave)
        return set_error(SSMX_EINVAL, "n_exp=%d, n_node=%d, members=%d",
                         d->n_exp, d->n_node, d->members);
    if (d->fine < 1 || d->n_out < 0 || d->wave_group < 1 || d->gen < 0 ||
        d->gen >= SSMX_MAX_GEN)
        return set_error(SSMX_EINVAL, "fine=%d, n_out=%d, wave_group=%d, "
                         "gen=%d", d->fine, d->n_out, d->wave_group, d->gen);
    const bool full = (d->flags & SSMX_READ_FULL) != 0;
    if ((d->flags & ~(SSMX_READ_FULL | SSMX_READ_INTEGRAL)) != 0 ||
        (full && (d->flags & SSMX_READ_INTEGRAL)))
        return set_error(SSMX_EINVAL, "flags=%d", d->flags);
    if (!full && (d->n_obs < 1 || d->n_obs > SSMX_MAX_OBS))
        return set_error(SSMX_EINVAL, "n_obs=%d outside 1..2", d->n_obs);
    if (d->na != d->nb || (d->na != 5 && d->na != 11) || d->sector < d->na + 1 ||
        (d->sector & 1) || d->sectors < 1 || d->sectors > 2 * d->rows)
        return set_error(SSMX_EINVAL, "na=%d, nb=%d, %d sectors of %d",
                         d->na, d->nb, d->sectors, d->sector);
    if (!(d->h > 0.0) || !(d->dt > 0.0))
        return set_error(SSMX_EINVAL, "h and dt must be positive");
    if ((size_t)d->members * d->sectors * d->sector * 8 > 48 * 1024)
        return set_error(SSMX_EINVAL, "%d members of %d sectors exceed the "
                         "LDS buffer", d->members, d->sectors);
    return SSMX_OK;
}

}  // namespace

extern "C" int ssmx_propagate_series(
    const ssmx_series_desc *desc, const int32_t *layout,
    const int32_t *state_pos, const double *table, const double *cf_weights,
    const double *cf_nodes, const ssmx_wave *waves,
    const ssmx_segment *segments, const double *rho0, const double *obs,
    double *out, void *stream)
{
    ssmx::error_buffer()[0] = '\0';
    const int rc = validate(desc);
    if (rc)
        return rc;
    if (!layout || !state_pos || !table || !cf_weights || !cf_nodes ||
        !waves || !segments || !rho0 || !out ||
        (!(desc->flags & SSMX_READ_FULL) && !obs))
        return set_error(SSMX_EINVAL, "null required pointer");
    SParams p;
    p.d = *desc;
    p.layout = layout;
    p.state_pos = state_pos;
    p.table = table;
    p.w = cf_weights;
    p.nodes = cf_nodes;
    p.waves = waves;
    p.segs = segments;
    p.rho0 = rho0;
    p.obs = obs;
    p.out = out;
    hipStream_t s = static_cast<hipStream_t>(stream);
    return desc->na == 5 ? launch_orders<5>(p, s) : launch_orders<11>(p, s);
}
