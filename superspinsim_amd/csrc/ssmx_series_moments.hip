// ssmx_series_moments.hip - parameter gradients of the wide series: d E_k /
// d theta, and their contraction with the moments of a run.
//
// An exponential takes y to y + sum_k f^k E_k y; with the cotangent mu of its
// result, dF/dtheta = sum over exponentials and k of f^k mu^T (dE_k/dtheta) y,
// i.e. the contraction of dE_k/dtheta with the moments
// M_k = sum f^k mu y^T. Both factors of a moment are stored by the runs
// (ssmx_propagate_series_wide, ssmx_series_wide_adjoint), so that the moments of
// one instance are a matrix product over its exponentials.
#include <type_traits>

#include "ssmx_series_dev.h"

namespace {

using ssmx::kWave;
using ssmx::set_error;

constexpr int kOrders = 4;
constexpr int kTile = 16;       // v_mfma_f64_16x16x4
constexpr int kRows = 2;        // tiles per wavefront: 2 x 3 or 2 x 2
constexpr int kWaves = 4;
constexpr int kXcds = 8;
constexpr int kMaxN = 192;

typedef double double4_t __attribute__((ext_vector_type(4)));

struct MParams {
    int n, npad, tiles, n_inst, n_theta, exps, groups;
    const double *y, *mu, *factors, *dtable;
    double *work;
};

// Columns of tiles a wavefront holds: as many as leave two wavefronts to a
// SIMD.
__host__ __device__ constexpr int tile_cols(int orders)
{
    return orders == 3 ? 3 : 2;
}

// One wavefront holds 2 x 3 (2 x 2) tiles of all three (four) moments of one
// instance, 144 (128) registers, and runs over the instance's exponentials, four
// per matrix instruction. Operands come straight from memory, 16 neighbours per
// exponential and tile. All workgroups of an instance go to one XCD (workgroups
// are dealt to the eight in turn), whose L2 then serves its 27 MB of rows to
// the wavefronts that pass over them at the same time.
//
// Bound by the matrix pipe: 128 instances of 171 rows x 10,000 exponentials,
// three orders, 4.9 ms = 283 GFLOP (with the padding) at 58 TFLOP/s (the
// card's large product: 73); 11.5 with four orders, workgroups over all XCDs
// and loads waited for ahead of the products instead of behind them.
template <int ORDERS>
__global__ __launch_bounds__(kWave *kWaves)
__attribute__((amdgpu_waves_per_eu(2))) void moments_kernel(MParams p)
{
    constexpr int kCols = tile_cols(ORDERS);
    const int lane = threadIdx.x % kWave;
    const int blocks = (p.groups + kWaves - 1) / kWaves;
    const int turn = blockIdx.x / kXcds;
    const long inst = (long)(turn / blocks) * kXcds + blockIdx.x % kXcds;
    const int group = turn % blocks * kWaves +
        __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    if (inst >= p.n_inst || group >= p.groups)
        return;
    const int col_groups = (p.tiles + kCols - 1) / kCols;
    const int tr = group / col_groups * kRows, tc = group % col_groups * kCols;
    const int within = lane % kTile, k = lane / kTile;
    const double *mu = p.mu + (size_t)inst * p.exps * p.npad + within;
    const double *y = p.y + (size_t)inst * p.exps * p.npad + within;
    const double *factors = p.factors + (size_t)inst * p.exps;
    // tiles past the last repeat it; their sums are not used
    int ra[kRows], cb[kCols];
#pragma unroll
    for (int i = 0; i < kRows; ++i)
        ra[i] = min(tr + i, p.tiles - 1) * kTile;
#pragma unroll
    for (int i = 0; i < kCols; ++i)
        cb[i] = min(tc + i, p.tiles - 1) * kTile;
    double4_t acc[kRows][kCols][ORDERS];
#pragma unroll
    for (int i = 0; i < kRows; ++i)
#pragma unroll
        for (int j = 0; j < kCols; ++j)
#pragma unroll
            for (int o = 0; o < ORDERS; ++o)
                acc[i][j][o] = {0.0, 0.0, 0.0, 0.0};
    double a[kRows], b[kCols], f;
    // operands of the exponentials e .. e + 3, past the last one its own
    auto load = [&](int e) {
        const size_t at = (size_t)min(e + k, p.exps - 1);
        f = factors[at];
#pragma unroll
        for (int i = 0; i < kRows; ++i)
            a[i] = mu[at * p.npad + ra[i]];
#pragma unroll
        for (int i = 0; i < kCols; ++i)
            b[i] = y[at * p.npad + cb[i]];
    };
    load(0);
    // (as plain loads these and the loop's are merged into one at its head)
    asm volatile("" : "+v"(f));
#pragma unroll
    for (int i = 0; i < kRows; ++i)
        asm volatile("" : "+v"(a[i]));
#pragma unroll
    for (int i = 0; i < kCols; ++i)
        asm volatile("" : "+v"(b[i]));
    for (int e = 0; e < p.exps; e += 4) {
        // zeros past the last exponential and in the padding of the rows,
        // which the runs leave as it was; chosen here, not in load, so that
        // the loads stay in flight over an iteration's products
        const bool on = e + k < p.exps;
        double ca[kRows], z[kCols];
        const double cf = f;
#pragma unroll
        for (int i = 0; i < kRows; ++i)
            ca[i] = on && ra[i] + within < p.n ? a[i] : 0.0;
#pragma unroll
        for (int i = 0; i < kCols; ++i)
            z[i] = on && cb[i] + within < p.n ? b[i] : 0.0;
        load(e + 4);
#pragma unroll
        for (int o = 0; o < ORDERS; ++o) {
#pragma unroll
            for (int i = 0; i < kRows; ++i)
#pragma unroll
                for (int j = 0; j < kCols; ++j)
                    acc[i][j][o] = __builtin_amdgcn_mfma_f64_16x16x4f64(
                        ca[i], z[j], acc[i][j][o], 0, 0, 0);
#pragma unroll
            for (int j = 0; j < kCols; ++j)
                z[j] *= cf;
        }
    }
    // element q of a lane: row 4 q + lane / 16, column lane % 16
    for (int t = 0; t < p.n_theta; ++t) {
        double s = 0.0;
        for (int o = 0; o < ORDERS; ++o) {
            const double *d = p.dtable + ((size_t)t * ORDERS + o) * p.npad *
                p.npad + (size_t)k * p.npad + within;
            // the moment of this order, by constant indexes
            auto part = [&](auto order) {
#pragma unroll
                for (int i = 0; i < kRows; ++i)
#pragma unroll
                    for (int q = 0; q < 4; ++q)
#pragma unroll
                        for (int j = 0; j < kCols; ++j)
                            if (tr + i < p.tiles && tc + j < p.tiles)
                                s = fma(d[(size_t)((tr + i) * kTile + 4 * q) *
                                          p.npad + (tc + j) * kTile],
                                        acc[i][j][order()][q], s);
            };
            if (o == 0)
                part(std::integral_constant<int, 0>{});
            else if (o == 1)
                part(std::integral_constant<int, 1>{});
            else if (o == 2)
                part(std::integral_constant<int, 2>{});
            else
                part(std::integral_constant<int, ORDERS - 1>{});
        }
        s = ssmx::wave_sum(s);
        if (lane == 0)
            p.work[((size_t)inst * p.groups + group) * p.n_theta + t] = s;
    }
}

// grad[inst][theta] = sum over the wavefronts' parts, in their order.
__global__ void moments_sum_kernel(const double *work, double *grad,
                                   long count, int groups, int n_theta)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count)
        return;
    const long inst = i / n_theta;
    double s = 0.0;
    for (int g = 0; g < groups; ++g)
        s += work[(inst * groups + g) * n_theta + i % n_theta];
    grad[i] = s;
}

struct DParams {
    int n, npad, terms, orders;
    double fold;
    int slots_a, slots_g, slots_d;
    const int32_t *col_a, *col_g, *col_d;
    const double *val_a, *val_g, *val_d;
    double *out;
};

// Column blockIdx.x of dE_0..3 in direction blockIdx.y, by the Taylor
// recurrence of exp(A + f G) and its derivative; a thread holds one row. A few
// tens of microseconds for 12 directions of 171 rows.
__global__ __launch_bounds__(kMaxN) void derivative_kernel(DParams p)
{
    __shared__ double buf[2][2 * kOrders][kMaxN];
    const int row = threadIdx.x, n = p.n;
    const int column = blockIdx.x, dir = blockIdx.y;
    double total[kOrders];
#pragma unroll
    for (int o = 0; o < kOrders; ++o) {
        total[o] = 0.0;
        buf[0][o][row] =
            o == 0 && row == column && row < n ? 1.0 : 0.0;
        buf[0][kOrders + o][row] = 0.0;
    }
    __syncthreads();
    const int32_t *cd = p.col_d + (size_t)dir * p.slots_d * n;
    const double *vd = p.val_d + (size_t)dir * p.slots_d * n;
    for (int t = 1; t <= p.terms; ++t) {
        const double (*from)[kMaxN] = buf[(t - 1) & 1];
        double (*to)[kMaxN] = buf[t & 1];
        double v[2 * kOrders];
#pragma unroll
        for (int o = 0; o < 2 * kOrders; ++o)
            v[o] = 0.0;
        if (row < n) {
            for (int s = 0; s < p.slots_a; ++s) {
                const int c = p.col_a[s * n + row];
                const double w = p.val_a[s * n + row];
#pragma unroll
                for (int o = 0; o < 2 * kOrders; ++o)
                    v[o] = fma(w, from[o][c], v[o]);
            }
            for (int s = 0; s < p.slots_g; ++s) {
                const int c = p.col_g[s * n + row];
                const double w = p.val_g[s * n + row];
#pragma unroll
                for (int o = 1; o < kOrders; ++o) {
                    v[o] = fma(w, from[o - 1][c], v[o]);
                    v[kOrders + o] = fma(w, from[kOrders + o - 1][c],
                                         v[kOrders + o]);
                }
            }
            for (int s = 0; s < p.slots_d; ++s) {
                const int c = cd[s * n + row];
                const double w = vd[s * n + row];
#pragma unroll
                for (int o = 0; o < kOrders; ++o)
                    v[kOrders + o] = fma(w, from[o][c], v[kOrders + o]);
            }
        }
        const double scale = 1.0 / t;
#pragma unroll
        for (int o = 0; o < 2 * kOrders; ++o)
            to[o][row] = v[o] * scale;
#pragma unroll
        for (int o = 0; o < kOrders; ++o)
            total[o] += v[kOrders + o] * scale;
        __syncthreads();
    }
    // order 3 without its Chebyshev polynomial is a part of order 1
    if (p.orders == 3)
        total[1] = fma(p.fold, total[3], total[1]);
    // (rows and columns of the padding: zeros)
    if (row < p.npad)
#pragma unroll
        for (int o = 0; o < kOrders; ++o)
            if (o < p.orders)
                p.out[(((size_t)dir * p.orders + o) * p.npad + row) * p.npad +
                      column] = total[o];
}

int launched(const char *what)
{
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess)
        return set_error(SSMX_ELAUNCH, "%s launch: %s", what,
                         hipGetErrorString(e));
    return SSMX_OK;
}

int tile_count(int n) { return (n + kTile - 1) / kTile; }

int group_count(int n, int orders)
{
    const int t = tile_count(n), cols = tile_cols(orders);
    return (t + kRows - 1) / kRows * ((t + cols - 1) / cols);
}

}  // namespace

extern "C" int ssmx_series_derivatives(
    int32_t n, int32_t n_theta, int32_t terms, int32_t orders,
    double drive_max, int32_t slots_a,
    const int32_t *col_a, const double *val_a, int32_t slots_g,
    const int32_t *col_g, const double *val_g, int32_t slots_d,
    const int32_t *col_d, const double *val_d, double *out, void *stream)
{
    ssmx::error_buffer()[0] = '\0';
    if (n < 1 || n > kMaxN || n_theta < 1 || n_theta > 65535 || terms < 1 ||
        (orders != 3 && orders != 4) || !(drive_max >= 0.0) || slots_a < 0 || slots_g < 0 || slots_d < 0)
        return set_error(SSMX_EINVAL, "series derivatives: n=%d, n_theta=%d, "
                         "terms=%d, slots=%d/%d/%d", n, n_theta, terms,
                         slots_a, slots_g, slots_d);
    if ((slots_a && (!col_a || !val_a)) || (slots_g && (!col_g || !val_g)) ||
        (slots_d && (!col_d || !val_d)) || !out)
        return set_error(SSMX_EINVAL, "null required pointer");
    const int npad = tile_count(n) * kTile;
    // f^3 = F^3 / 4 T_3(f / F) + 3 / 4 F^2 f
    const DParams p{n, npad, terms, orders, 0.75 * drive_max * drive_max,
                    slots_a, slots_g, slots_d, col_a, col_g, col_d,
                    val_a, val_g, val_d, out};
    hipLaunchKernelGGL(derivative_kernel, dim3(npad, n_theta), dim3(kMaxN), 0,
                       static_cast<hipStream_t>(stream), p);
    return launched("series derivatives");
}

extern "C" int ssmx_series_moments(
    int32_t n, int32_t n_inst, int32_t exps, int32_t orders, int32_t n_theta,
    const double *y, const double *mu, const double *factors,
    const double *dtable, double *work, double *grad_theta, void *stream)
{
    ssmx::error_buffer()[0] = '\0';
    if (n < 1 || n > kMaxN || n_inst < 1 || exps < 1 || n_theta < 1 ||
        (orders != 3 && orders != 4))
        return set_error(SSMX_EINVAL, "series moments: n=%d, n_inst=%d, "
                         "exps=%d, orders=%d, n_theta=%d", n, n_inst, exps,
                         orders, n_theta);
    if (!y || !mu || !factors || !dtable || !work || !grad_theta)
        return set_error(SSMX_EINVAL, "null required pointer");
    MParams p;
    p.n = n;
    p.tiles = tile_count(n);
    p.npad = p.tiles * kTile;
    p.n_inst = n_inst;
    p.n_theta = n_theta;
    p.exps = exps;
    p.groups = group_count(n, orders);
    p.y = y;
    p.mu = mu;
    p.factors = factors;
    p.dtable = dtable;
    p.work = work;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const long blocks = (long)(n_inst + kXcds - 1) / kXcds * kXcds *
        ((p.groups + kWaves - 1) / kWaves);
    if (blocks > 0x7fffffffL)
        return set_error(SSMX_EINVAL, "series moments: %d instances", n_inst);
    if (orders == 3)
        hipLaunchKernelGGL(moments_kernel<3>, dim3((unsigned)blocks),
                           dim3(kWave * kWaves), 0, s, p);
    else
        hipLaunchKernelGGL(moments_kernel<4>, dim3((unsigned)blocks),
                           dim3(kWave * kWaves), 0, s, p);
    const int rc = launched("series moments");
    if (rc != SSMX_OK)
        return rc;
    const long count = (long)n_inst * n_theta;
    hipLaunchKernelGGL(moments_sum_kernel, dim3((count + 255) / 256),
                       dim3(256), 0, s, work, grad_theta, count, p.groups,
                       n_theta);
    return launched("series moment sum");
}

extern "C" int ssmx_series_moment_groups(int32_t n, int32_t orders)
{
    return n < 1 || n > kMaxN || (orders != 3 && orders != 4)
               ? 0
               : group_count(n, orders);
}
