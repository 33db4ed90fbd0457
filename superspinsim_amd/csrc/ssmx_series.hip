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
//
// What bounds it (4096 points of the 7-level sweep, n = 19, two instances per
// wavefront, two wavefronts per SIMD, 99,900 steps): the Taylor kernel took
// 260 ms on all 49 states. With the exchange through LDS the sweep takes 68
// ms, bound by LDS (24 16-byte reads per wavefront and step at 8 CU-cycles);
// with the broadcast exchange of series_row_kernel 57-61 ms, bound by VALU
// issue (135 VALU instructions per wavefront and step, 110 of them the
// multiply-adds). A wavefront alone on its SIMD issues a 64-bit multiply-add
// every 8 cycles, two together one every 4.
#include "ssmx_series_dev.h"

namespace {

using ssmx::bcast_fma;
using ssmx::Clock;
using ssmx::DriveFactors;
using ssmx::Halves;
using ssmx::horner;
using ssmx::kWave;
using ssmx::set_error;
using ssmx::swap_rows;
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

// Waveform of a lane's drive-factor entry in a sweep.
template <int J>
__device__ const ssmx_wave *entry_wave(const SParams &p, long sys, int lane)
{
    long wi = sys * p.d.members + (lane / J) % p.d.members;
    if (wi >= p.d.n_inst)
        wi = p.d.n_inst - 1;
    return p.waves + wi / p.d.wave_group;
}

__device__ __forceinline__ Clock clock_of(const SParams &p)
{
    return Clock{p.d.t0, p.d.dt, p.d.h, p.d.fine, p.d.n_node, p.nodes, p.w};
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

    const Clock clk = clock_of(p);
    DriveFactors<J> drive(entry_wave<J>(p, sys, lane), p.segs, d.gen,
                          d.members, lane);
    const long total = (long)d.n_out * d.fine;
    const int MJ = drive.MJ, B = drive.B;

    double xint = 0.0;
    const double half_h = 0.5 * d.h;
    double fc[J];
#pragma unroll
    for (int j = 0; j < J; ++j)
        fc[j] = 0.0;
    wave_exchange();
    int b = B;
    for (int i = 0; i < d.n_out; ++i) {
        for (int k = 0; k < d.fine; ++k) {
            if (b == B) {
                b = 0;
                drive.fill(clk, p.segs, i, k,
                           total - ((long)i * d.fine + k), lane, fbuf);
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

// The same exponentials for models of one sector pair, without LDS in the
// exchange: a pair of 16-lane rows holds an instance, each row one sector.
// A lane multiplies its row's broadcast components into two sums, its own
// component's (own-sector coefficients) and that of the opposite sector's
// component with its index, and the rows exchange the second sums.  Two
// instances per wavefront.
template <int N, int DA, int DB, int J>
__global__ __launch_bounds__(kWave)
__attribute__((amdgpu_waves_per_eu(2))) void series_row_kernel(SParams p)
{
    __shared__ double fbuf[kWave], red[kWave];
    const ssmx_series_desc &d = p.d;
    const int lane = threadIdx.x;
    const int q = lane / 32, i16 = lane % 16;
    const bool odd_row = (lane & 16) != 0;
    const int rows = d.rows;
    const int first = d.sectors > 1 ? d.sector_rows : rows;
    const int own_rows = odd_row ? rows - first : first;
    const int row0 = odd_row ? first : 0;
    const int other_rows = rows - own_rows, other0 = odd_row ? 0 : first;
    const bool has = q < d.members && i16 < own_rows;
    const bool other = q < d.members && i16 < other_rows;

    double ca[N][DA + 1], cb[N][DB + 1];
#pragma unroll
    for (int e = 0; e < N * (DA + 1); ++e)
        ca[e / (DA + 1)][e % (DA + 1)] =
            has ? p.table[(size_t)e * rows + row0 + i16] : 0.0;
#pragma unroll
    for (int e = 0; e < N * (DB + 1); ++e)
        cb[e / (DB + 1)][e % (DB + 1)] =
            other ? p.table[(size_t)(N * (DA + 1) + e) * rows + other0 + i16]
                  : 0.0;

    const long sys = blockIdx.x;
    const long inst = sys * d.members + q;
    const bool live = has && inst < d.n_inst;
    const int state = has ? p.layout[4 * (row0 + i16) + 3] : 0;
    double x = live ? p.rho0[(size_t)inst * d.n + state] : 0.0;
    const bool read_full = (d.flags & SSMX_READ_FULL) != 0;
    const bool read_int = (d.flags & SSMX_READ_INTEGRAL) != 0;
    double ob0 = 0.0, ob1 = 0.0;
    if (!read_full && live) {
        ob0 = p.obs[state];
        if (d.n_obs > 1)
            ob1 = p.obs[d.n + state];
    }
    // sum over the member's 32 lanes (idle ones hold 0)
    auto observe = [&](double v, long index) {
#pragma unroll
        for (int off = 16; off > 0; off >>= 1)
            v += __shfl_xor(v, off, kWave);
        if (live && lane % 32 == 0)
            p.out[index] = v;
    };

    const Clock clk = clock_of(p);
    DriveFactors<J> drive(entry_wave<J>(p, sys, lane), p.segs, d.gen,
                          d.members, lane);
    const long total = (long)d.n_out * d.fine;
    const int MJ = drive.MJ, B = drive.B;
    const int qf = q < d.members ? q : 0;
    double xint = 0.0;
    const double half_h = 0.5 * d.h;
    double fc[J];
#pragma unroll
    for (int j = 0; j < J; ++j)
        fc[j] = 0.0;
    int b = B;
    for (int i = 0; i < d.n_out; ++i) {
        for (int k = 0; k < d.fine; ++k) {
            if (b == B) {
                b = 0;
                drive.fill(clk, p.segs, i, k,
                           total - ((long)i * d.fine + k), lane, fbuf);
#pragma unroll
                for (int j = 0; j < J; ++j)
                    fc[j] = fbuf[qf * J + j];
            }
            double fn[J];
            const int nb = b + 1 < B ? b + 1 : b;
#pragma unroll
            for (int j = 0; j < J; ++j)
                fn[j] = fbuf[nb * MJ + qf * J + j];
            const double before = x;
#pragma unroll
            for (int j = J - 1; j >= 0; --j) {
                const double f = fc[j], u = f * f;
                double wa[N], wb[N];
                horner<N, DA>(wa, ca, u);
                horner<N, DB>(wb, cb, u);
                double ya = 0.0, yb = 0.0;
                bcast_fma<0, N>(ya, yb, x, wa, wb);
                x += fma(f, swap_rows(yb, odd_row), ya);
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
            // components to LDS, then states in standard order
            red[lane] = x;
            wave_exchange();
            for (int e = lane; e < d.members * d.n; e += kWave) {
                const int m = e / d.n, s = e - m * d.n;
                const long to = sys * d.members + m;
                const int sp = p.state_pos[s];
                if (to < d.n_inst)
                    p.out[((size_t)to * d.n_out + i) * d.n + s] =
                        sp < 0 ? 0.0
                               : red[32 * m + 16 * (sp / d.sector) +
                                     sp % d.sector];
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

// Sweeps of one instance per wavefront (Halves): fewer instructions per
// step than two instances on a wavefront, for launches that do not fill the
// SIMDs (64 points of the 7-level sweep: 300 ns a step, 344 in
// series_row_kernel).
// With p.store every exponential's input is kept for the adjoint: at J = 2
// half 0 of the wavefront's 64 doubles per step holds the input of
// exponential 1 and half 1 that of exponential 0, one coalesced store.
struct HParams {
    ssmx_series_desc d;
    const int32_t *lanes;
    const double *table;
    const double *w;
    const double *nodes;
    const ssmx_wave *waves;
    const ssmx_segment *segs;
    const double *rho0;
    const double *obs;
    double *out;
    double *store;
};

template <int N, int DA, int DB, int J, bool STORE>
__global__ __launch_bounds__(kWave)
__attribute__((amdgpu_waves_per_eu(2))) void series_half_kernel(HParams p)
{
    constexpr int S = Halves<N>::S;
    __shared__ double fbuf[kWave];
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
    double x = has ? p.rho0[(size_t)inst * d.n + state] : 0.0;
    const bool read_full = (d.flags & SSMX_READ_FULL) != 0;
    const bool read_int = (d.flags & SSMX_READ_INTEGRAL) != 0;
    const double ob0 = !read_full && has ? p.obs[state] : 0.0;
    const double ob1 =
        !read_full && has && d.n_obs > 1 ? p.obs[d.n + state] : 0.0;
    // sum over the first half's lanes (idle ones hold 0)
    auto observe = [&](double v, long index) {
#pragma unroll
        for (int off = 16; off > 0; off >>= 1)
            v += __shfl_xor(v, off, kWave);
        if (lane == 0)
            p.out[index] = v;
    };
    const Clock clk{d.t0, d.dt, d.h, d.fine, d.n_node, p.nodes, p.w};
    DriveFactors<J> drive(p.waves + inst / d.wave_group, p.segs, d.gen, 1,
                          lane);
    const int B = drive.B;
    const long total = (long)d.n_out * d.fine;
    double *store = STORE ? p.store + (size_t)inst * total * 32 * J : nullptr;
    double xint = 0.0;
    const double half_h = 0.5 * d.h;
    double fc[J];
#pragma unroll
    for (int j = 0; j < J; ++j)
        fc[j] = 0.0;
    int b = B;
    long step = 0;
    for (int i = 0; i < d.n_out; ++i) {
        for (int k = 0; k < d.fine; ++k, ++step) {
            if (b == B) {
                b = 0;
                drive.fill(clk, p.segs, i, k, total - step, lane, fbuf);
#pragma unroll
                for (int j = 0; j < J; ++j)
                    fc[j] = fbuf[j];
            }
            double fn[J];
            const int nb = b + 1 < B ? b + 1 : b;
#pragma unroll
            for (int j = 0; j < J; ++j)
                fn[j] = fbuf[nb * J + j];
            const double before = x;
#pragma unroll
            for (int j = J - 1; j >= 0; --j) {
                if constexpr (STORE && J == 2) {
                    if (j == 0)
                        store[(size_t)step * 64 + lane] =
                            lane < 32 ? before : x;
                }
                if constexpr (STORE && J == 1) {
                    if (lane < 32)
                        store[(size_t)step * 32 + lane] = x;
                }
                Halves<N>::template exponential<DA, DB>(x, fc[j], ca, cb,
                                                        odd_row);
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
            // (the host clears the states without a lane)
            if (has && lane < 32)
                p.out[((size_t)inst * d.n_out + i) * d.n + state] = x;
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

struct QSParams {
    ssmx_series_desc d;
    const int32_t *lanes;
    const double *table;
    const double *powers;
    const double *w;
    const double *nodes;
    const ssmx_wave *waves;
    const ssmx_segment *segs;
    const double *rho0;
    const double *obs;
    const ssmx_run *runs;
    const int32_t *run_begin;
    const int32_t *order;
    int32_t *counter;
    double *out;
    int32_t levels;
    int32_t n_waves;
};

// Uneven protocols, one per wavefront at a time (ssmx_series_queue).
//
// A protocol is a list of runs.  Driven runs go step by step.  In a free run
// every step is the same matrix, so its 2^b-th powers (formed on the host) take
// the state through it in one product per set bit of the step count, and the
// readout integral over 2^b steps is a matrix as well: the 100,000s of steps
// of free precession and the readout window become some twenty products.
// 2,048 protocols of 58k-742k steps (at most 200k of them driven) took 1046 ms
// step by step with the Taylor action, 68 ms so: the driven steps at two
// wavefronts per SIMD, 105 VALU instructions each.
template <int N, int DA, int DB, int J>
__global__ __launch_bounds__(kWave * 8) __attribute__((
    amdgpu_waves_per_eu(2))) void series_queue_kernel(QSParams p)
{
    constexpr int S = Halves<N>::S;
    constexpr int kEntries = S * (DA + 1) + S * (DB + 1);
    __shared__ double fbufs[8][kWave];
    const ssmx_series_desc &d = p.d;
    const int lane = threadIdx.x % kWave;
    double *fbuf = fbufs[threadIdx.x / kWave];
    const bool odd_row = (lane & 16) != 0;
    const int state = p.lanes[lane];
    const bool has = state >= 0;
    const double ob0 = has ? p.obs[state] : 0.0;
    const double ob1 = has && d.n_obs > 1 ? p.obs[d.n + state] : 0.0;
    const Clock clk{d.t0, d.dt, d.h, 1, d.n_node, p.nodes, p.w};
    const double half_h = 0.5 * d.h;

    // The opaque lane offset keeps the table addresses out of the run loop's
    // registers (they would be hoisted and spill).
    double ca[S][DA + 1], cb[S][DB + 1];
    auto load_set = [&](int set) {
        int at = lane;
        asm volatile("" : "+v"(at));
        const double *t = p.table + (size_t)set * kEntries * kWave;
#pragma unroll
        for (int s = 0; s < S; ++s) {
#pragma unroll
            for (int o = 0; o <= DA; ++o)
                ca[s][o] = t[(s * (DA + 1) + o) * kWave + at];
#pragma unroll
            for (int o = 0; o <= DB; ++o)
                cb[s][o] = t[(S * (DA + 1) + s * (DB + 1) + o) * kWave + at];
        }
    };
    auto load_power = [&](double (&m)[S], int set, int level, int which) {
        int at = lane;
        asm volatile("" : "+v"(at));
        const double *t =
            p.powers +
            (((size_t)set * p.levels + level) * 2 + which) * S * kWave;
#pragma unroll
        for (int s = 0; s < S; ++s)
            m[s] = t[s * kWave + at];
    };

    int entry = (int)(blockIdx.x * (blockDim.x / kWave) +
                      threadIdx.x / kWave);
    if (entry >= p.n_waves)
        return;
    for (;;) {
        if (p.counter)
            entry = ssmx::next_entry(p.counter, lane);
        if (entry >= d.n_inst)
            return;
        const int inst = __builtin_amdgcn_readfirstlane(p.order[entry]);
        DriveFactors<J> drive(p.waves + inst, p.segs, d.gen, 1, lane);
        const int B = drive.B;
        double x = has ? p.rho0[(size_t)inst * d.n + state] : 0.0;
        double xint = 0.0;
        int loaded = -1;
        const int end = p.run_begin[inst + 1];
        for (int ri = p.run_begin[inst]; ri < end; ++ri) {
            const ssmx_run run = p.runs[ri];
            const bool reads = run.read != 0;
            if (run.kind == SSMX_RUN_FREE) {
                long left = run.count;
                for (int level = 0; left > 0; ++level, left >>= 1) {
                    if (!(left & 1))
                        continue;
                    double m[S];
                    const double xs = Halves<N>::shifted(x);
                    if (reads) {
                        load_power(m, run.set0, level, 1);
                        xint += Halves<N>::within(xs, m);
                    }
                    load_power(m, run.set0, level, 0);
                    x += Halves<N>::within(xs, m);
                }
                continue;
            }
            for (long done = 0; done < run.count;) {
                const long left = run.count - done;
                drive.fill(clk, p.segs, run.first + done, 0, left, lane,
                           fbuf);
                const int steps = left < B ? (int)left : B;
                double fc[J];
#pragma unroll
                for (int j = 0; j < J; ++j)
                    fc[j] = fbuf[j];
                for (int b = 0; b < steps; ++b) {
                    // the next step's factors, read while this runs
                    const int nb = b + 1 < B ? b + 1 : b;
                    double fn[J];
#pragma unroll
                    for (int j = 0; j < J; ++j)
                        fn[j] = fbuf[nb * J + j];
                    const double before = x;
#pragma unroll
                    for (int j = J - 1; j >= 0; --j) {
                        // (set1 differs from set0 in split runs only)
                        const int set = j == 0 ? run.set0 : run.set1;
                        if (set != loaded) {
                            load_set(set);
                            loaded = set;
                        }
                        Halves<N>::template exponential<DA, DB>(
                            x, fc[j], ca, cb, odd_row);
                    }
                    if (reads) {
                        ssmx::keep_branch();
                        xint = fma(half_h, before + x, xint);
                    }
#pragma unroll
                    for (int j = 0; j < J; ++j)
                        fc[j] = fn[j];
                }
                wave_exchange();
                done += steps;
            }
        }
        // (the first half's lanes; lane o writes readout o)
        double v0 = ob0 * xint, v1 = ob1 * xint;
#pragma unroll
        for (int off = 16; off > 0; off >>= 1) {
            v0 += __shfl_xor(v0, off, kWave);
            v1 += __shfl_xor(v1, off, kWave);
        }
        if (lane < d.n_obs)
            p.out[(size_t)inst * d.n_obs + lane] = lane == 0 ? v0 : v1;
        if (!p.counter)
            entry += p.n_waves;
    }
}

template <int NA, int DA, int NB, int DB, int J>
int launch(const SParams &p, hipStream_t stream)
{
    const ssmx_series_desc &d = p.d;
    const size_t lds = ((size_t)d.members * d.sectors * d.sector + 2 +
                        2 * kWave) * sizeof(double);
    const int systems = (d.n_inst + d.members - 1) / d.members;
    if constexpr (NA == 11 && J <= 2) {
        if (d.sector_rows > 0 && d.members <= 2) {
            hipLaunchKernelGGL((series_row_kernel<NA, DA, DB, J>),
                               dim3(systems), dim3(kWave), 0, stream, p);
            const hipError_t e = hipGetLastError();
            if (e != hipSuccess)
                return set_error(SSMX_ELAUNCH, "series launch: %s",
                                 hipGetErrorString(e));
            return SSMX_OK;
        }
    }
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
    if (d->sector_rows < 0 || d->sector_rows > d->na ||
        (d->sector_rows > 0 &&
         (d->sectors > 2 || d->rows - d->sector_rows > d->na ||
          d->rows < d->sector_rows ||
          (d->sectors == 1 && d->rows != d->sector_rows))))
        return set_error(SSMX_EINVAL, "sector_rows=%d of %d rows, %d sectors",
                         d->sector_rows, d->rows, d->sectors);
    if (!(d->h > 0.0) || !(d->dt > 0.0))
        return set_error(SSMX_EINVAL, "h and dt must be positive");
    if ((size_t)d->members * d->sectors * d->sector * 8 > 48 * 1024)
        return set_error(SSMX_EINVAL, "%d members of %d sectors exceed the "
                         "LDS buffer", d->members, d->sectors);
    return SSMX_OK;
}

}  // namespace

namespace {

template <int DA, int DB, int J>
int launch_queue(const QSParams &p, int waves_per_block, hipStream_t stream)
{
    const int blocks = (p.n_waves + waves_per_block - 1) / waves_per_block;
    hipLaunchKernelGGL((series_queue_kernel<11, DA, DB, J>), dim3(blocks),
                       dim3(kWave * waves_per_block), 0, stream, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return set_error(SSMX_ELAUNCH, "series queue launch: %s",
                         hipGetErrorString(e));
    return SSMX_OK;
}

template <int DA, int DB>
int launch_queue_scheme(const QSParams &p, int waves_per_block,
                        hipStream_t stream)
{
    return p.d.n_exp == 1 ? launch_queue<DA, DB, 1>(p, waves_per_block, stream)
                          : launch_queue<DA, DB, 2>(p, waves_per_block,
                                                    stream);
}

}  // namespace

extern "C" int ssmx_series_queue(
    const ssmx_series_desc *desc, const int32_t *lanes, const double *table,
    const double *powers, int32_t levels, const double *cf_weights,
    const double *cf_nodes, const ssmx_wave *waves,
    const ssmx_segment *segments, const double *rho0, const double *obs,
    const ssmx_run *runs, const int32_t *run_begin, const int32_t *order,
    int32_t *counter, int32_t n_waves, int32_t waves_per_block, double *out,
    void *stream)
{
    ssmx::error_buffer()[0] = '\0';
    const int rc = validate(desc);
    if (rc)
        return rc;
    if (desc->flags != SSMX_READ_INTEGRAL || desc->na != 11 ||
        desc->n_exp > 2 || desc->sector_rows < 1 || desc->members != 1 ||
        desc->wave_group != 1 || desc->fine != 1)
        return set_error(SSMX_EINVAL, "series queue: flags=%d, na=%d, "
                         "n_exp=%d, sector_rows=%d, members=%d",
                         desc->flags, desc->na, desc->n_exp,
                         desc->sector_rows, desc->members);
    if (n_waves < 1 || waves_per_block < 1 || waves_per_block > 8 ||
        levels < 0 || levels > 62)
        return set_error(SSMX_EINVAL, "n_waves=%d, waves_per_block=%d, "
                         "levels=%d", n_waves, waves_per_block, levels);
    if (!lanes || !table || !powers || !cf_weights || !cf_nodes || !waves ||
        !segments || !rho0 || !obs || !runs || !run_begin || !order || !out)
        return set_error(SSMX_EINVAL, "null required pointer");
    QSParams p;
    p.d = *desc;
    p.lanes = lanes;
    p.table = table;
    p.powers = powers;
    p.w = cf_weights;
    p.nodes = cf_nodes;
    p.waves = waves;
    p.segs = segments;
    p.rho0 = rho0;
    p.obs = obs;
    p.runs = runs;
    p.run_begin = run_begin;
    p.order = order;
    p.counter = counter;
    p.out = out;
    p.levels = levels;
    p.n_waves = n_waves;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int da = desc->da, db = desc->db;
    if (da == 1 && db == 1)
        return launch_queue_scheme<1, 1>(p, waves_per_block, s);
    if (da == 2 && db == 1)
        return launch_queue_scheme<2, 1>(p, waves_per_block, s);
    if (da == 2 && db == 2)
        return launch_queue_scheme<2, 2>(p, waves_per_block, s);
    return set_error(SSMX_EINVAL, "no series kernel for orders da=%d, db=%d",
                     da, db);
}

namespace {

template <int DA, int DB, int J>
int launch_half(const HParams &p, hipStream_t stream)
{
    if (p.store)
        hipLaunchKernelGGL((series_half_kernel<11, DA, DB, J, true>),
                           dim3(p.d.n_inst), dim3(kWave), 0, stream, p);
    else
        hipLaunchKernelGGL((series_half_kernel<11, DA, DB, J, false>),
                           dim3(p.d.n_inst), dim3(kWave), 0, stream, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return set_error(SSMX_ELAUNCH, "series launch: %s",
                         hipGetErrorString(e));
    return SSMX_OK;
}

template <int DA, int DB>
int launch_half_scheme(const HParams &p, hipStream_t stream)
{
    return p.d.n_exp == 1 ? launch_half<DA, DB, 1>(p, stream)
                          : launch_half<DA, DB, 2>(p, stream);
}

}  // namespace

extern "C" int ssmx_propagate_series_wave(
    const ssmx_series_desc *desc, const int32_t *lanes, const double *table,
    const double *cf_weights, const double *cf_nodes, const ssmx_wave *waves,
    const ssmx_segment *segments, const double *rho0, const double *obs,
    double *out, double *store, void *stream)
{
    ssmx::error_buffer()[0] = '\0';
    const int rc = validate(desc);
    if (rc)
        return rc;
    if (desc->na != 11 || desc->n_exp > 2 || desc->sector_rows < 1 ||
        desc->members != 1)
        return set_error(SSMX_EINVAL, "one instance per wavefront: na=%d, "
                         "n_exp=%d, sector_rows=%d, members=%d", desc->na,
                         desc->n_exp, desc->sector_rows, desc->members);
    if (!lanes || !table || !cf_weights || !cf_nodes || !waves ||
        !segments || !rho0 || !out ||
        (!(desc->flags & SSMX_READ_FULL) && !obs))
        return set_error(SSMX_EINVAL, "null required pointer");
    HParams p;
    p.d = *desc;
    p.lanes = lanes;
    p.table = table;
    p.w = cf_weights;
    p.nodes = cf_nodes;
    p.waves = waves;
    p.segs = segments;
    p.rho0 = rho0;
    p.obs = obs;
    p.out = out;
    p.store = store;
    hipStream_t s = static_cast<hipStream_t>(stream);
    const int da = desc->da, db = desc->db;
    if (da == 1 && db == 1)
        return launch_half_scheme<1, 1>(p, s);
    if (da == 2 && db == 1)
        return launch_half_scheme<2, 1>(p, s);
    if (da == 2 && db == 2)
        return launch_half_scheme<2, 2>(p, s);
    return set_error(SSMX_EINVAL, "no series kernel for orders da=%d, db=%d",
                     da, db);
}

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
