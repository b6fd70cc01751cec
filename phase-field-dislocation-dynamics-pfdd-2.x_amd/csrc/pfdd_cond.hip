// pfdd_cond.hip -- kernels of the conductivity sub-problem (solve_style GLCond,
// solve_GL+cond.cpp:70-150): divcurrent and backwardcond with
// update_conduct_order_param around the line passes.
//
// Where the x (z) length has register transforms (pfdd_reg.hpp) the x passes
// with divcurrent between them (the inverse z passes, the update and the next
// iteration's forward z pass) are one kernel: per iteration 14 trips of a field
// over memory instead of 29.  128^3, us per iteration: x passes and divcurrent
// 59 -> 23, inverse z pass, update and forward z pass 60 -> 30.
#include "pfdd_reg.hpp"

namespace pfdd {

// divcurrent at one k-point (fft_fftw_slab.cpp:1704-1741): a = i c f_y / f^2
// and b = c f_y^2 / f^2, zero at f = 0.
__device__ __forceinline__ void cond_point(double2 c, const double *f, double2 &a, double2 &b)
{
    const double f2 = f[0] * f[0] + f[1] * f[1] + f[2] * f[2];
    const double r = f2 > 0.0 ? f[1] / f2 : 0.0;
    a = make_double2(-(c.y * r), c.x * r);
    b = make_double2(c.x * r * f[1], c.y * r * f[1]);
}

// Raises *done where a total of the update before (nu partials per slot, 0 at the
// start of a run) is not finite; called by one block of a kernel that runs
// between two updates.  From there on the updates and the line passes return at
// once, so c stays as that iteration left it.  The kernels that call this do not
// read the flag themselves: their blocks run while it is raised.
template <int W>
__device__ __forceinline__ void cond_check(const double *part, long long pstride, int nu, int *done, double *red,
                                           int tid)
{
    double v[3] = {0.0, 0.0, 0.0};
    const int slot[3] = {0, 2, 3};
#pragma unroll
    for (int q = 0; q < 3; ++q)
#pragma unroll 4
        for (int b = tid; b < nu; b += W) v[q] += part[slot[q] * pstride + b];
    block_sum<3, W>(v, red, tid);
    if (tid == 0 && !(isfinite(v[0]) && isfinite(v[1]) && isfinite(v[2]))) *done = 1;
}

// divcurrent on the transformed field in the [k][j][i] layout, written as
// [2][k][j][i].  The block also sums sig[(ny - j) mod ny] Re a over its
// k-points: backwardcond called a second time on its own output (the trailing
// call of SolveGLCond::iterate) transforms a back once more, and two
// unnormalised inverse transforms give N a(-r).
__global__ void __launch_bounds__(NTHR)
    k_cond_div(const double2 *__restrict__ ch, double2 *__restrict__ ab, const double *__restrict__ sig, CondParams P,
               long long N, double *__restrict__ part, long long pstride, int nu, int *done)
{
    __shared__ double red[3 * (NTHR / 64)];
    const int tid = threadIdx.x;
    if (blockIdx.x == 0) cond_check<NTHR>(part, pstride, nu, done, red, tid);
    double v[1] = {0.0};
    for (long long idx = (long long)blockIdx.x * NTHR + tid; idx < N; idx += (long long)gridDim.x * NTHR) {
        const int i = (int)(idx % P.nx);
        const int j = (int)((idx / P.nx) % P.ny);
        const int k = (int)(idx / ((long long)P.nx * P.ny));
        const double kx = frac_freq(i, P.nx), ky = frac_freq(j, P.ny), kz = frac_freq(k, P.nz);
        double f[3];
        for (int c = 0; c < 3; ++c) f[c] = kx * P.four[c] + ky * P.four[3 + c] + kz * P.four[6 + c];
        double2 a, b;
        cond_point(ch[idx], f, a, b);
        ab[idx] = a;
        ab[N + idx] = b;
        v[0] += sig[(P.ny - j) % P.ny] * a.x;
    }
    block_sum<1, NTHR>(v, red, tid);
    if (tid == 0) part[4 * pstride + blockIdx.x] = v[0];
}

// The same between the forward x transform and the two inverse ones: a block
// of 128 threads holds its lines in registers as k_mid_r does, contracts each
// value where it lies, and transforms a, then b, back.  Bound by the three
// trips over memory.
template <int N> struct CondX {
    static constexpr int VPT = N <= 64 ? 8 : 16, D = N / VPT, W = 128, NL = W / D;
};
template <int N>
__global__ void __launch_bounds__((CondX<N>::W)) __attribute__((amdgpu_waves_per_eu(2, 8)))
    k_cond_x(const double2 *__restrict__ ch, double2 *__restrict__ ab, const double *__restrict__ sig, CondParams P,
             long long ntot, const double2 *__restrict__ tw, double *__restrict__ part, long long pstride, int nu,
             int *done)
{
    typedef CondX<N> X;
    constexpr int VPT = X::VPT, D = X::D, W = X::W, NL = X::NL;
    typedef RegSwzX<N> L;
    __shared__ __align__(16) char mem[N * NL * RegLds<double2>::bytes];
    __shared__ double2 tws[N];
    __shared__ double red[3 * (W / 64)];
    RegLds<double2> lds{(double *)mem};
    const int t = threadIdx.x, l = t / D, p0 = t % D;
    if (blockIdx.x == 0) cond_check<W>(part, pstride, nu, done, red, t);
    const long long line = (long long)blockIdx.x * NL + l;
    const long long at = line * N + p0;
    double2 v[VPT], w[VPT];
#pragma unroll
    for (int m = 0; m < VPT; ++m) v[m] = ld_stream(ch + at + D * m);
    reg_twiddles<N, W>(tws, tw, t);
    reg_fft<N, 1, 1, NL, VPT, false, true, true, true, L>(v, lds, tws, t);
    const int j = (int)(line % P.ny), k = (int)(line / P.ny);
    const double ky = frac_freq(j, P.ny), kz = frac_freq(k, P.nz);
    double s = 0.0;
#pragma unroll
    for (int m = 0; m < VPT; ++m) {
        const double kx = frac_freq(p0 + D * m, P.nx);
        double f[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) f[c] = kx * P.four[c] + ky * P.four[3 + c] + kz * P.four[6 + c];
        double2 b;
        cond_point(v[m], f, w[m], b);
        v[m] = b;
        s += w[m].x;
    }
    double sum[1] = {sig[j ? P.ny - j : 0] * s};
    block_sum<1, W>(sum, red, t);
    if (t == 0) part[4 * pstride + blockIdx.x] = sum[0];
    int t2 = t;
    __asm__ volatile("" : "+v"(t2)); // addresses formed again, as in k_update_r
    reg_fft<N, 1, 1, NL, VPT, true, true, true, false, L>(w, lds, tws, t2);
#pragma unroll
    for (int m = 0; m < VPT; ++m) ab[at + D * m] = w[m];
    reg_fft<N, 1, 1, NL, VPT, true, true, true, false, L>(v, lds, tws, t2);
#pragma unroll
    for (int m = 0; m < VPT; ++m) ab[ntot + at + D * m] = v[m];
}

// backwardcond's per-cell assembly on the (unnormalised) inverse transforms a,
// b, then update_conduct_order_param:
//   j     = sig (El - Re a / eps0) - i sig Im a / eps0
//   rhs   = (sig / eps0) b + (a / eps0 - El) dsig      (El on the real part)
//   c    -= rate * rhs / N
// sums: Re j, Im j, |dc|^2, Re c_new.
struct CondCell {
    double s, ds, se; // sig, dsig, sig / eps0 of the row
    // a's part of rhs
    __device__ __forceinline__ double2 from_a(double2 a, const CondParams &P, double *v) const
    {
        const double ax = a.x / P.eps0, ay = a.y / P.eps0;
        v[0] += s * (P.El - ax);
        v[1] += -s * a.y / P.eps0;
        return make_double2((ax - P.El) * ds, ay * ds);
    }
    __device__ __forceinline__ double2 update(double2 ra, double2 b, double2 c0, const CondParams &P, double *v) const
    {
        const double rr = ab_c(se, b.x, ra.x), ri = ab_c(se, b.y, ra.y);
        const double2 c1 = make_double2(c0.x - P.rate * (rr * P.invN), c0.y - P.rate * (ri * P.invN));
        const double dr = c1.x - c0.x, di = c1.y - c0.y;
        v[2] += dr * dr + di * di;
        v[3] += c1.x;
        return c1;
    }
};

__global__ void __launch_bounds__(NTHR)
    k_cond_update(const double2 *__restrict__ ab, double2 *__restrict__ c, const double *__restrict__ sig,
                  const double *__restrict__ dsig, CondParams P, long long N, double *__restrict__ part,
                  long long pstride, const int *__restrict__ done)
{
    if (*done) return;
    __shared__ double red[4 * (NTHR / 64)];
    const int tid = threadIdx.x;
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    for (long long idx = (long long)blockIdx.x * NTHR + tid; idx < N; idx += (long long)gridDim.x * NTHR) {
        const int j = (int)((idx / P.nz) % P.ny);
        const CondCell cell{sig[j], dsig[j], sig[j] / P.eps0};
        c[idx] = cell.update(cell.from_a(ab[idx], P, v), ab[N + idx], c[idx], P, v);
    }
    block_sum<4, NTHR>(v, red, tid);
    if (tid == 0)
        for (int q = 0; q < 4; ++q) part[q * pstride + blockIdx.x] = v[q];
}

// The same after the two inverse z transforms (a, b in the [2][i][k][j] layout,
// read line-fastest, in registers from there on) and, with FW, before the
// forward z transform of the new c into T ([i][k][j]).  a's part of rhs waits in
// registers for b's transform: two waves per SIMD.  Bound by the five trips
// over memory.
template <int N, bool FW>
__global__ void __launch_bounds__((RegTile<double, N>::W)) __attribute__((amdgpu_waves_per_eu(2, 8)))
    k_cond_update_r(const double2 *__restrict__ ab, double2 *__restrict__ c, double2 *__restrict__ T,
                    const double *__restrict__ sig, const double *__restrict__ dsig, CondParams P, long long ntot,
                    const double2 *__restrict__ tw, double *__restrict__ part, long long pstride,
                    const int *__restrict__ done)
{
    typedef RegTile<double, N> G;
    constexpr int NL = G::NL, VPT = G::VPT, D = G::D, W = G::W;
    if (*done) return;
    __shared__ __align__(16) char mem[N * NL * RegLds<double2>::bytes];
    __shared__ double2 tws[N];
    __shared__ double red[4 * (W / 64)];
    RegLds<double2> lds{(double *)mem};
    const int t = threadIdx.x;
    // lines L = i ny + j; a tile may cross rows of j
    const unsigned ny = P.ny, L0 = blockIdx.x * NL, r0 = L0 / ny;
    unsigned o1; // element offset of this thread's first value from the tile's row of T
    {
        const unsigned l = t % NL, p0 = t / NL, j = L0 - r0 * ny + l, row = j / ny;
        o1 = row * ny * N + (j - row * ny) + p0 * ny;
    }
    const long long row0 = (long long)r0 * ny * N;
    double2 a[VPT], b[VPT];
#pragma unroll
    for (int m = 0; m < VPT; ++m) a[m] = ld_stream(ab + row0 + (size_t)(D * m) * ny + o1);
#pragma unroll
    for (int m = 0; m < VPT; ++m) b[m] = ld_stream(ab + ntot + row0 + (size_t)(D * m) * ny + o1);
    reg_twiddles<N, W>(tws, tw, t);
    const unsigned l = t / D, p0 = t % D, j = (L0 + l) % ny;
    const CondCell cell{sig[j], dsig[j], sig[j] / P.eps0};
    double2 *const own = c + (long long)(L0 + l) * N + p0;
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    reg_fft<N, 1, 1, NL, VPT, true, false, true, true>(a, lds, tws, t);
#pragma unroll
    for (int m = 0; m < VPT; ++m) a[m] = cell.from_a(a[m], P, v);
    __asm__ volatile("" : "+v"(v[0]), "+v"(v[1]));
    reg_fft<N, 1, 1, NL, VPT, true, false, true, false>(b, lds, tws, t);
#pragma unroll
    for (int m = 0; m < VPT; ++m) {
        a[m] = cell.update(a[m], b[m], own[D * m], P, v);
        own[D * m] = a[m];
    }
    __asm__ volatile("" : "+v"(v[2]), "+v"(v[3]));
    if constexpr (FW) {
        int t2 = t;
        __asm__ volatile("" : "+v"(t2)); // addresses formed again, as in k_update_r
        reg_fft<N, 1, 1, NL, VPT, false, true, false, false>(a, lds, tws, t2);
#pragma unroll
        for (int m = 0; m < VPT; ++m) T[row0 + (size_t)(D * m) * ny + o1] = a[m];
    }
    block_sum_comp<4, W>(v, red, t);
    if (t == 0)
        for (int q = 0; q < 4; ++q) part[q * pstride + blockIdx.x] = v[q];
}

// The sums of a run's last iteration: nu partials of the update (slots 0-3), nd
// of divcurrent (slot 4), to pinned host memory with the stop flag, which is
// cleared.
__global__ void __launch_bounds__(NTHR)
    k_cond_sums(const double *__restrict__ part, long long pstride, int nu, int nd, CondStat *stat, int *done)
{
    __shared__ double red[5 * (NTHR / 64)];
    const int tid = threadIdx.x;
    double v[5];
#pragma unroll
    for (int q = 0; q < 5; ++q) {
        const int n = q == 4 ? nd : nu;
        double sum = 0.0, c = 0.0;
        for (int b = tid; b < n; b += NTHR) {
            const double y = part[q * pstride + b] - c;
            const double t = sum + y;
            c = (t - sum) - y;
            sum = t;
        }
        v[q] = sum;
    }
    block_sum<5, NTHR>(v, red, tid);
    if (tid == 0) {
        for (int q = 0; q < 5; ++q) stat->s[q] = v[q];
        stat->done = *done;
        *done = 0;
    }
}

// ---------------------------------------------------------------- launchers
// Blocks of the kernels that go cell by cell: 8 to a CU.  One block adds their
// partials up (cond_check, k_cond_sums); one block per 256 cells made that 650 of
// 1950 us an iteration at 512 x 256 x 160.
static int cell_blocks(long long N)
{
    const long long nb = (N + NTHR - 1) / NTHR;
    return (int)(nb < 2048 ? nb : 2048);
}

hipError_t launch_cond_div(const double2 *ch, double2 *ab, const double *sig, const CondParams &P, double *part,
                           long long pstride, int nu, int *nparts, int *done, hipStream_t st)
{
    const long long N = (long long)P.nx * P.ny * P.nz;
    *nparts = cell_blocks(N);
    hipLaunchKernelGGL(k_cond_div, dim3((unsigned)*nparts), dim3(NTHR), 0, st, ch, ab, sig, P, N, part, pstride,
                       nu, done);
    return hipGetLastError();
}

hipError_t launch_cond_x(const double2 *ch, double2 *ab, const double *sig, const CondParams &P, const void *tw,
                         double *part, long long pstride, int nu, int *nparts, int *done, hipStream_t st)
{
    const long long lines = (long long)P.ny * P.nz;
#define PFDD_CASE(n_)                                                                                           \
    if (P.nx == n_) {                                                                                           \
        if constexpr (reg_length<n_>()) {                                                                       \
            typedef CondX<n_> X;                                                                                \
            if (lines % X::NL) return hipErrorInvalidValue;                                                     \
            *nparts = (int)(lines / X::NL);                                                                     \
            hipLaunchKernelGGL((k_cond_x<n_>), dim3((unsigned)*nparts), dim3(X::W), 0, st, ch, ab, sig, P,      \
                               lines * n_, (const double2 *)tw, part, pstride, nu, done);                       \
            return hipGetLastError();                                                                           \
        }                                                                                                       \
    }
    PFDD_SIZES(PFDD_CASE)
#undef PFDD_CASE
    return hipErrorInvalidValue;
}

hipError_t launch_cond_update(const double2 *ab, double2 *c, const double *sig, const double *dsig,
                              const CondParams &P, double *part, long long pstride, int *nparts, const int *done,
                              hipStream_t st)
{
    const long long N = (long long)P.nx * P.ny * P.nz;
    *nparts = cell_blocks(N);
    hipLaunchKernelGGL(k_cond_update, dim3((unsigned)*nparts), dim3(NTHR), 0, st, ab, c, sig, dsig, P, N, part,
                       pstride, done);
    return hipGetLastError();
}

hipError_t launch_cond_update_r(bool fw, const double2 *ab, double2 *c, double2 *T, const double *sig,
                                const double *dsig, const CondParams &P, const void *tw, double *part,
                                long long pstride, int *nparts, const int *done, hipStream_t st)
{
    const long long lines = (long long)P.nx * P.ny;
#define PFDD_UPD(FW_)                                                                                           \
    hipLaunchKernelGGL((k_cond_update_r<N, FW_>), dim3((unsigned)*nparts), dim3(RegTile<double, N>::W), 0, st,  \
                       ab, c, T, sig, dsig, P, lines * N, (const double2 *)tw, part, pstride, done)
#define PFDD_CASE(n_)                                                                                           \
    if (P.nz == n_) {                                                                                           \
        if constexpr (reg_length<n_>()) {                                                                       \
            constexpr int N = n_;                                                                               \
            if (lines % RegTile<double, N>::NL) return hipErrorInvalidValue;                                    \
            *nparts = (int)(lines / RegTile<double, N>::NL);                                                    \
            if (fw) PFDD_UPD(true);                                                                             \
            else PFDD_UPD(false);                                                                               \
            return hipGetLastError();                                                                           \
        }                                                                                                       \
    }
    PFDD_SIZES(PFDD_CASE)
#undef PFDD_CASE
#undef PFDD_UPD
    return hipErrorInvalidValue;
}

hipError_t launch_cond_sums(const double *part, long long pstride, int nu, int nd, CondStat *stat, int *done,
                            hipStream_t st)
{
    hipLaunchKernelGGL(k_cond_sums, dim3(1), dim3(NTHR), 0, st, part, pstride, nu, nd, stat, done);
    return hipGetLastError();
}

} // namespace pfdd
