// ssmx_series_wide.hip - the series in the drive for models of more rows than
// a wavefront (the 21-level NV + 14N model, 171 involved states).
//
// The Taylor kernel for such models (ssmx_wide.hip) pays 11 exchanges across
// the workgroup's wavefronts per exponential, each about 430 cycles of LDS
// round trip and barrier for some 10 multiply-adds a row. The series reads
// every component that a row depends on once: about 70 a row here (the E_k
// fill in, entries far below the tolerance are left out), one barrier per
// exponential.
//
// Split. Two rows with nearly the same columns share 8 lanes (16 for the widest
// pairs), half of them in either half of the wavefront: a lane gathers each of
// its columns once for both rows, a swap of the halves leaves each half one
// row to add up by DPP. Pairs are sorted by width, and each wavefront runs
// code for its own entries per lane (C own-sector and C opposite-sector
// columns, coefficients and LDS addresses in registers). 171 rows take 12
// wavefronts, three per SIMD. One wavefront, the last and narrowest,
// evaluates the drive for all; the first one adds up readouts.
//
// What bounds it: VALU issue, about 700 of 1,130 cycles per exponential (134
// gathers with four multiply-adds each over the workgroup); the rest is the
// latency from the barrier to the first gathers and that of the sum. Measured,
// us per step of 256 points (512): orders (1, 1) 1.15 (2.1), Taylor 4.4 (4.7);
// orders (2, 1) 1.45 to 1.7. 1.3 with rows in pair order in LDS (2.4 ways of
// bank conflict a gather instead of 1.8) and pairs on consecutive lanes
// (selects and a DPP step where the half swap is). Coefficients evaluated ahead
// of the gathers gained 1% and spilled.
//
// Orders 4 and 5 do not fit the registers: their coefficients are read from
// LDS, as are all of an eighth column per lane.
//
// Gradients store the inputs of all exponentials forward and the cotangents of
// their results in reverse (kStore, kBack); ssmx_series_moments.hip contracts
// the two. 128 points x 5,000 steps, 12 parameters: 5.9 + 5.9 + 4.9 ms; Taylor
// forward 22 and Frechet adjoint 77.
#include "ssmx_series_dev.h"

namespace {

using ssmx::Clock;
using ssmx::DriveFactors;
using ssmx::kWave;
using ssmx::quad_perm;
using ssmx::set_error;

constexpr int kMaxWaves = 12;
constexpr int kMaxRows = 16 * kMaxWaves;    // eight pairs a wavefront
// LDS for the coefficients that registers don't hold, and for one column of them
constexpr int kHighBytes = 150 * 1024;
constexpr int kColumnBytes = kWave * sizeof(double2);
constexpr int kRegSlots = 7, kMaxSlots = 8;
enum { kRun, kStore, kBack };

typedef __attribute__((address_space(3))) double lds_double;

struct WSParams {
    ssmx_series_desc d;
    const ssmx_series_block *blocks;
    const int32_t *states;
    const int32_t *columns;
    const double *table;
    const double *w;
    const double *nodes;
    const ssmx_wave *waves;
    const ssmx_segment *segs;
    const double *rho0;
    const double *obs;
    double *out;
    // gradients (null otherwise): every exponential's input (forward) or its
    // result's cotangent (reverse), [instance][step][j][pad]; its factor
    double *store;
    double *factors;
    const double *seed;
    int pad;
};

// The sum of a pair's rows over its lanes: that of row a in the lanes of the
// wavefront's lower half, of row b in those of its upper half.
__device__ __forceinline__ double sum_pair(double a, double b, bool sixteen)
{
    // the upper half of a for the lower one of b
    const auto lo = __builtin_amdgcn_permlane32_swap(
        __double2loint(a), __double2loint(b), false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap(
        __double2hiint(a), __double2hiint(b), false, false);
    double v = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);
    if (sixteen)
        v += quad_perm<0x141>(v);               // row_half_mirror
    v += quad_perm<0xB1>(v);                    // lane ^ 1
    v += quad_perm<0x4E>(v);                    // lane ^ 2
    return v;
}

// Readouts of the components in `x` (LDS) by one wavefront.
__device__ __forceinline__ void observe(const WSParams &p, const double *x,
                                        const double *obs, long index,
                                        int lane)
{
    double v[kMaxRows / kWave];
#pragma unroll
    for (int k = 0; k < kMaxRows / kWave; ++k)
        v[k] = x[k * kWave + lane];
    for (int o = 0; o < p.d.n_obs; ++o) {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < kMaxRows / kWave; ++k)
            s = fma(obs[o * kMaxRows + k * kWave + lane], v[k], s);
        s = ssmx::wave_sum(s);
        if (lane == 0)
            p.out[index * p.d.n_obs + o] = s;
    }
}

extern __shared__ double2 high_orders[];

// Columns of `slots` slots in LDS: of the orders above 3, and four for each slot
// beyond the registers'.
__host__ __device__ constexpr int high_columns(int slots, int hi)
{
    return hi * slots + 4 * (slots > kRegSlots ? slots - kRegSlots : 0);
}

// What an exponential of factor f adds to the lane's row, from the components
// at `from` in LDS. Registers hold orders 0..3 of up to kRegSlots columns;
// coefficients of E_4 (HI >= 1), E_5 (HI 2) and of the columns beyond come from
// `high` in LDS, for both rows.
template <int C, int HI, int R>
__device__ __forceinline__ double
exponential(const double (&ca)[R][2][2], const double (&cb)[R][2][2],
            lds_double *const (&xa)[C], lds_double *const (&xb)[C], int from,
            const double2 *high, double f, bool sixteen)
{
    double va[C], vb[C];
#pragma unroll
    for (int s = 0; s < C; ++s)
        va[s] = xa[s][from];
#pragma unroll
    for (int s = 0; s < C; ++s)
        vb[s] = xb[s][from];
    const double u = f * f;
    double a0 = 0.0, a1 = 0.0, b0 = 0.0, b1 = 0.0;
#pragma unroll
    for (int s = 0; s < C; ++s) {
        double w0, w1, v0, v1;
        if (s < R) {
            w0 = ca[s < R ? s : 0][1][0];
            w1 = ca[s < R ? s : 0][1][1];
            v0 = ca[s < R ? s : 0][0][0];
            v1 = ca[s < R ? s : 0][0][1];
        } else {
            const double2 *more = high + (HI * C + (s - R) * 4) * kWave;
            w0 = more[kWave].x;
            w1 = more[kWave].y;
            v0 = more[0].x;
            v1 = more[0].y;
        }
        if constexpr (HI >= 1) {
            const double2 c = high[s * kWave];
            w0 = fma(u, c.x, w0);
            w1 = fma(u, c.y, w1);
        }
        a0 = fma(fma(u, w0, v0), va[s], a0);
        a1 = fma(fma(u, w1, v1), va[s], a1);
    }
#pragma unroll
    for (int s = 0; s < C; ++s) {
        double w0, w1, v0, v1;
        if (s < R) {
            w0 = cb[s < R ? s : 0][1][0];
            w1 = cb[s < R ? s : 0][1][1];
            v0 = cb[s < R ? s : 0][0][0];
            v1 = cb[s < R ? s : 0][0][1];
        } else {
            const double2 *more = high + (HI * C + (s - R) * 4 + 2) * kWave;
            w0 = more[kWave].x;
            w1 = more[kWave].y;
            v0 = more[0].x;
            v1 = more[0].y;
        }
        if constexpr (HI >= 2) {
            const double2 c = high[(C + s) * kWave];
            w0 = fma(u, c.x, w0);
            w1 = fma(u, c.y, w1);
        }
        b0 = fma(fma(u, w0, v0), vb[s], b0);
        b1 = fma(fma(u, w1, v1), vb[s], b1);
    }
    return sum_pair(fma(f, b0, a0), fma(f, b1, a1), sixteen);
}

// One wavefront's part of its workgroup's instance: C own-sector and C
// opposite-sector columns per lane. FILL: this wavefront evaluates the drive.
// M is kRun, kStore (a run that keeps every exponential's input and factor) or
// kBack: the cotangents of an integrated readout in reverse, with transposed
// matrices and the factors that kStore left.
template <int C, bool FILL, int M, int HI>
__device__ __forceinline__ void run_wave(const WSParams &p, double *xbuf,
                                         double *fbuf, const double *obs,
                                         const ssmx_series_block &blk,
                                         int wave, int lane, long inst)
{
    constexpr int J = 2, B = kWave / J;
    const ssmx_series_desc &d = p.d;
    const int row = p.states[2 * (wave * kWave + lane)];
    const int state = p.states[2 * (wave * kWave + lane) + 1];
    const bool sixteen = blk.lanes == 16;
    const bool leader = row >= 0 && lane % (blk.lanes / 2) == 0;
    const double *t = p.table + blk.table + lane;
    const int32_t *col = p.columns + blk.columns + lane;
    // [column][order][row of the pair]
    constexpr int R = C < kRegSlots ? C : kRegSlots;
    double ca[R][2][2], cb[R][2][2];
    lds_double *xa[C], *xb[C];
#pragma unroll
    for (int s = 0; s < R; ++s)
#pragma unroll
        for (int o = 0; o < 4; ++o) {
            ca[s][o / 2][o % 2] = t[(s * 4 + o) * kWave];
            cb[s][o / 2][o % 2] = t[((R + s) * 4 + o) * kWave];
        }
#pragma unroll
    for (int s = 0; s < C; ++s) {
        xa[s] = (lds_double *)xbuf + col[s * kWave];
        xb[s] = (lds_double *)xbuf + col[(C + s) * kWave];
    }
    // the wavefront's own part of LDS, behind those of the ones before
    constexpr int kHigh = HI * C + 4 * (C - R);
    int before_me = 0;
    if constexpr (HI > 0 || kRegSlots < kMaxSlots)
        for (int k = 0; k < wave; ++k)
            before_me += high_columns(p.blocks[k].slots, HI);
    double2 *high = high_orders + before_me * kWave + lane;
    const double2 *from = (const double2 *)(t - lane + R * 8 * kWave) + lane;
#pragma unroll
    for (int s = 0; s < kHigh; ++s)
        high[s * kWave] = from[s * kWave];
    const double half_h = 0.5 * d.h;
    double x = 0.0, source = 0.0;
    if constexpr (M == kBack) {
        if (row >= 0)
            for (int o = 0; o < d.n_obs; ++o)
                source = fma(p.seed[inst * d.n_obs + o],
                             p.obs[o * d.n + state], source);
        x = half_h * source;
    } else if (row >= 0) {
        x = p.rho0[(size_t)inst * d.n + state];
    }
    if (leader)
        xbuf[row] = x;
    const bool read_full = (d.flags & SSMX_READ_FULL) != 0;
    const bool read_int = (d.flags & SSMX_READ_INTEGRAL) != 0;
    const long total = (long)d.n_out * d.fine;
    double *store = nullptr;
    if (M != kRun && leader)
        store = p.store + (size_t)inst * total * J * p.pad + row;
    if constexpr (M == kBack) {
        const double *factors = p.factors + (size_t)inst * total * J;
        __syncthreads();
        double n0 = factors[(total - 1) * J], n1 = factors[total * J - 1];
        for (long step = total - 1; step >= 0; --step) {
            const double fc[J] = {n0, n1};
            const long next = step > 0 ? step - 1 : 0;
            n0 = factors[next * J];
            n1 = factors[next * J + 1];
#pragma unroll
            for (int j = 0; j < J; ++j) {
                if (leader)
                    store[(step * J + j) * p.pad] = x;
                x += exponential<C, HI>(ca, cb, xa, xb, j == 0 ? 0 : kMaxRows,
                                        high, fc[j], sixteen);
                // readouts after the step before and before this one
                if (j == J - 1)
                    x = fma(step == 0 ? half_h : d.h, source, x);
                if (leader)
                    xbuf[(j == 0 ? kMaxRows : 0) + row] = x;
                __syncthreads();
            }
        }
        if (p.out && leader)
            p.out[(size_t)inst * d.n + state] = x;
        return;
    }
    const Clock clk{d.t0, d.dt, d.h, d.fine, d.n_node, p.nodes, p.w};
    DriveFactors<J> drive(p.waves + inst / d.wave_group, p.segs, d.gen, 1,
                          lane);
    // the drive factors from output i, step k on
    auto fill = [&](long i, int k, long step, double *f) {
        drive.fill(clk, p.segs, i, k, total - step, lane, f);
        if (M == kStore && step * J + lane < total * J)
            p.factors[(inst * total + step) * J + lane] = f[lane];
    };
    if constexpr (FILL)
        fill(0, 0, 0, fbuf);
    double xint = 0.0;
    __syncthreads();
    int b = 0;
    long step = 0;
    double *fcur = fbuf;
    for (int i = 0; i < d.n_out; ++i) {
        for (int k = 0; k < d.fine; ++k, ++step) {
            const double fc[J] = {fcur[b * J], fcur[b * J + 1]};
            if (++b == B) {
                // the next batch: read from the next step on, two barriers
                // from here; its buffer was last read a batch ago
                fcur = fcur == fbuf ? fbuf + kWave : fbuf;
                b = 0;
                if constexpr (FILL)
                    fill(i, k + 1, step + 1, fcur);
            }
            const double before = x;
#pragma unroll
            for (int j = J - 1; j >= 0; --j) {
                // the first exponential reads buffer 0 and writes buffer 1,
                // the second goes back: a wavefront that still reads a buffer
                // is one barrier ahead of any that writes it
                const int from = j == 1 ? 0 : kMaxRows;
                const int to = j == 1 ? kMaxRows : 0;
                if (M == kStore && leader)
                    store[(step * J + j) * p.pad] = x;
                x += exponential<C, HI>(ca, cb, xa, xb, from, high, fc[j],
                                        sixteen);
                if (leader)
                    xbuf[to + row] = x;
                __syncthreads();
            }
            if (read_int) {
                ssmx::keep_branch();
                xint = fma(half_h, before + x, xint);
            }
        }
        if (read_full) {
            if (leader)
                p.out[((size_t)inst * d.n_out + i) * d.n + state] = x;
        } else if (!read_int && wave == 0) {
            observe(p, xbuf, obs, inst * d.n_out + i, lane);
        }
    }
    if (read_int) {
        // (buffer 1 was last read before the last barrier)
        if (leader)
            xbuf[kMaxRows + row] = xint;
        __syncthreads();
        if (wave == 0)
            observe(p, xbuf + kMaxRows, obs, inst, lane);
    }
}

template <int C, int M, int HI>
__device__ __forceinline__ void run_class(const WSParams &p, double *xbuf,
                                          double *fbuf, const double *obs,
                                          const ssmx_series_block &blk,
                                          int wave, int lane, long inst,
                                          bool fill)
{
    if constexpr (M == kBack)
        run_wave<C, false, M, HI>(p, xbuf, fbuf, obs, blk, wave, lane, inst);
    else if (fill)
        run_wave<C, true, M, HI>(p, xbuf, fbuf, obs, blk, wave, lane, inst);
    else
        run_wave<C, false, M, HI>(p, xbuf, fbuf, obs, blk, wave, lane, inst);
}

template <int M, int HI>
__global__ __launch_bounds__(kWave *kMaxWaves)
__attribute__((amdgpu_waves_per_eu(3))) void series_wide_kernel(WSParams p)
{
    __shared__ double xbuf[2 * kMaxRows];
    __shared__ double fbuf[2 * kWave];
    __shared__ double obs[SSMX_MAX_OBS * kMaxRows];
    const int lane = threadIdx.x % kWave;
    const int wave =
        __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    const ssmx_series_block blk = p.blocks[wave];
    const long inst = blockIdx.x;
    const bool fill = wave == (int)(blockDim.x / kWave) - 1;
    for (int k = threadIdx.x; k < 2 * kMaxRows; k += blockDim.x)
        xbuf[k] = 0.0;
    for (int k = threadIdx.x; k < p.d.n_obs * kMaxRows; k += blockDim.x)
        obs[k] = 0.0;
    __syncthreads();
    const int row = p.states[2 * (wave * kWave + lane)];
    if (M != kBack && row >= 0)
        for (int o = 0; o < p.d.n_obs; ++o)
            obs[o * kMaxRows + row] =
                p.obs[o * p.d.n + p.states[2 * (wave * kWave + lane) + 1]];
    // every wavefront meets the same barriers whatever its class
    switch (blk.slots) {
    case 4:
        run_class<4, M, HI>(p, xbuf, fbuf, obs, blk, wave, lane, inst, fill);
        break;
    case 5:
        run_class<5, M, HI>(p, xbuf, fbuf, obs, blk, wave, lane, inst, fill);
        break;
    case 6:
        run_class<6, M, HI>(p, xbuf, fbuf, obs, blk, wave, lane, inst, fill);
        break;
    case 7:
        run_class<7, M, HI>(p, xbuf, fbuf, obs, blk, wave, lane, inst, fill);
        break;
    default:
        run_class<8, M, HI>(p, xbuf, fbuf, obs, blk, wave, lane, inst, fill);
    }
}

int check(const ssmx_series_desc &d, int32_t n_blocks, const char *what)
{
    const bool full = (d.flags & SSMX_READ_FULL) != 0;
    if (d.n < 1 || d.n > SSMX_MAX_N_WIDE || d.rows < 1 ||
        d.rows > kMaxRows || d.n_inst < 1 || d.n_exp != 2 ||
        d.n_node != 2 || d.da < 1 || d.da > 2 || d.db < 1 || d.db > d.da ||
        d.fine < 1 ||
        d.n_out < 0 || d.wave_group < 1 || d.gen < 0 ||
        d.gen >= SSMX_MAX_GEN || !(d.h > 0.0) || !(d.dt > 0.0) ||
        (d.flags & ~(SSMX_READ_FULL | SSMX_READ_INTEGRAL)) != 0 ||
        (full && (d.flags & SSMX_READ_INTEGRAL)) ||
        (!full && (d.n_obs < 1 || d.n_obs > SSMX_MAX_OBS)))
        return set_error(SSMX_EINVAL, "%s: n=%d, rows=%d, n_inst=%d, "
                         "n_exp=%d, da=%d, db=%d, fine=%d, n_out=%d, "
                         "n_obs=%d, flags=%d", what, d.n, d.rows, d.n_inst,
                         d.n_exp, d.da, d.db, d.fine, d.n_out, d.n_obs,
                         d.flags);
    if (n_blocks < 1 || n_blocks > kMaxWaves)
        return set_error(SSMX_EINVAL, "%d wavefronts outside 1..%d",
                         n_blocks, kMaxWaves);
    if (d.lds_columns < 0 || d.lds_columns * kColumnBytes > kHighBytes)
        return set_error(SSMX_EINVAL, "%d columns of coefficients exceed the "
                         "LDS", d.lds_columns);
    return SSMX_OK;
}

template <int M, int HI>
int launch(const WSParams &p, int n_blocks, void *stream, const char *what)
{
    const size_t bytes = (size_t)p.d.lds_columns * kColumnBytes;
    hipError_t e = hipSuccess;
    // (one limit for every launch: another thread may launch with more)
    if (bytes > 0)
        e = hipFuncSetAttribute(
            reinterpret_cast<const void *>(series_wide_kernel<M, HI>),
            hipFuncAttributeMaxDynamicSharedMemorySize, kHighBytes);
    if (e == hipSuccess) {
        hipLaunchKernelGGL((series_wide_kernel<M, HI>), dim3(p.d.n_inst),
                           dim3(kWave * n_blocks), bytes,
                           static_cast<hipStream_t>(stream), p);
        e = hipGetLastError();
    }
    if (e != hipSuccess)
        return set_error(SSMX_ELAUNCH, "%s launch: %s", what,
                         hipGetErrorString(e));
    return SSMX_OK;
}

template <int M>
int launch_orders(const WSParams &p, int n_blocks, void *stream,
                  const char *what)
{
    switch (p.d.da - 1 + p.d.db - 1) {
    case 0:
        return launch<M, 0>(p, n_blocks, stream, what);
    case 1:
        return launch<M, 1>(p, n_blocks, stream, what);
    default:
        return launch<M, 2>(p, n_blocks, stream, what);
    }
}

}  // namespace

extern "C" int ssmx_propagate_series_wide(
    const ssmx_series_desc *desc, const ssmx_series_block *blocks,
    int32_t n_blocks, const int32_t *states, const int32_t *columns,
    const double *table, const double *cf_weights, const double *cf_nodes,
    const ssmx_wave *waves, const ssmx_segment *segments, const double *rho0,
    const double *obs, double *out, double *store, double *factors,
    void *stream)
{
    ssmx::error_buffer()[0] = '\0';
    if (!desc)
        return set_error(SSMX_EINVAL, "null descriptor");
    const int rc = check(*desc, n_blocks, "wide series");
    if (rc != SSMX_OK)
        return rc;
    if (!blocks || !states || !columns || !table || !cf_weights ||
        !cf_nodes || !waves || !segments || !rho0 || !out ||
        (!(desc->flags & SSMX_READ_FULL) && !obs) || !store != !factors)
        return set_error(SSMX_EINVAL, "null required pointer");
    WSParams p{};
    p.d = *desc;
    if (desc->flags & SSMX_READ_FULL)
        p.d.n_obs = 0;          // no readout rows to stage
    p.blocks = blocks;
    p.states = states;
    p.columns = columns;
    p.table = table;
    p.w = cf_weights;
    p.nodes = cf_nodes;
    p.waves = waves;
    p.segs = segments;
    p.rho0 = rho0;
    p.obs = obs;
    p.out = out;
    p.store = store;
    p.factors = factors;
    p.pad = (desc->rows + 15) / 16 * 16;
    return store ? launch_orders<kStore>(p, n_blocks, stream, "wide series")
                 : launch_orders<kRun>(p, n_blocks, stream, "wide series");
}

extern "C" int ssmx_series_wide_adjoint(
    const ssmx_series_desc *desc, const ssmx_series_block *blocks,
    int32_t n_blocks, const int32_t *states, const int32_t *columns,
    const double *table, const double *factors, const double *obs,
    const double *seed, double *store, double *lambda_out, void *stream)
{
    ssmx::error_buffer()[0] = '\0';
    if (!desc)
        return set_error(SSMX_EINVAL, "null descriptor");
    const int rc = check(*desc, n_blocks, "wide series adjoint");
    if (rc != SSMX_OK)
        return rc;
    if (desc->n_out < 1 || desc->n_obs < 1 || desc->n_obs > SSMX_MAX_OBS)
        return set_error(SSMX_EINVAL, "wide series adjoint: n_out=%d, "
                         "n_obs=%d", desc->n_out, desc->n_obs);
    if (!blocks || !states || !columns || !table || !factors || !obs ||
        !seed || !store)
        return set_error(SSMX_EINVAL, "null required pointer");
    WSParams p{};
    p.d = *desc;
    p.blocks = blocks;
    p.states = states;
    p.columns = columns;
    p.table = table;
    p.factors = const_cast<double *>(factors);
    p.obs = obs;
    p.seed = seed;
    p.out = lambda_out;
    p.store = store;
    p.pad = (desc->rows + 15) / 16 * 16;
    return launch_orders<kBack>(p, n_blocks, stream, "wide series adjoint");
}
