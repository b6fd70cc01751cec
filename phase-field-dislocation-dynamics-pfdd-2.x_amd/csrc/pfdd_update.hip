// pfdd_update.hip -- the last inverse pass fused with the GL update, and its
// reverse-mode counterpart, with their launchers.
#include "pfdd_kern.hpp"
#include "pfdd_reg.hpp"

namespace pfdd {

// ------------------------------------- pass 5: inverse z FFT + fused update
// update_order_parameter (fft_fftw_slab.cpp:1746-1790) with the core-energy
// derivative of core_energy_* evaluated on the old field, as the reference
// does (it reads data_fftw = xi before the update).  Masked cells keep their
// value; their xinorm term uses the previous unmasked cell's old value in
// (a, i, j, k) order (prev[] precomputed on the host, -1 = the initial 0).
// The FP64 sine-series update on its smallest tile at 40-96 points (19-20 KB
// of LDS: 8 blocks per CU) asks for 8 waves per SIMD (64 instead of 68 VGPRs;
// the same hint made the FP32 one 9 % slower).
//
// FW: 0 the update alone (last iteration of a run); 1, 2 the update followed
// by the forward z transform of the new field, written back over the block's
// own lines of T1: pass 1 of the next iteration, with radix plan FW - 1.  The
// lines are complete in the tile after the update, so the next iteration
// needs no pass that reads the field again: 4 S N e bytes instead of 5 in two
// kernels.
template <typename R, int N, int TQ, bool GEN, int FW> constexpr int update_waves()
{
    return (sizeof(R) == 8 && TQ == 0 && !GEN && FW < 2 && N >= 40 && N <= 96) ? 8 : 1;
}

template <typename R, int N, int TQ, bool GEN, int FW>
__global__ void __launch_bounds__(NTHR) __attribute__((amdgpu_waves_per_eu(update_waves<R, N, TQ, GEN, FW>(), 8)))
    k_update(typename cvec<R>::type *T1, const typename cvec<R>::type *__restrict__ xo,
             typename cvec<R>::type *__restrict__ xn, const uint8_t *__restrict__ mask,
             const long long *__restrict__ prev, const R *__restrict__ amp, LineMap mi, LineMap mo,
             long long nlines, long long lines_per_sys, StepParams P,
             const typename cvec<R>::type *__restrict__ tw, bool keep, double *__restrict__ partial,
             long long pstride, const int *__restrict__ done)
{
    typedef typename cvec<R>::type V;
    if (*done) return;
    constexpr int NL = tile_lines_u<R, N, TQ>(), LDP = NL + 1, TOT = N * NL;
    PFDD_TILE(V, lds, N * LDP);
    __shared__ long long bin[NL], bout[NL];
    // per-line tau and core coefficients: read once per block here, since
    // kernel-argument arrays indexed per lane compile to per-lane memory loads
    __shared__ R ltau[NL], lcoef[MAXM * NL];
    __shared__ int lsub[NL]; // position of the line's system in its plane triple (coupled model)
    __shared__ double red[4 * (NTHR / 64)];
    const int tid = threadIdx.x;
    const bool ext = GEN && P.model == PFDD_CORE_EXTENDED;
    unsigned tile = blockIdx.x;
    if constexpr (GEN) {
        // The coupled model reads Re xi of all three systems of a plane: the
        // same lines of the three are 8 blocks apart, that is on the same XCD
        // and close in time, so two of the three reads find them in its L2.
        const unsigned per = (unsigned)(lines_per_sys / NL); // tiles of a system
        if (ext && per % 8 == 0 && per * (unsigned)NL == lines_per_sys) {
            const unsigned plane = tile / (3 * per), r = tile - plane * 3 * per, w = r % 24;
            tile = (plane * 3 + w / 8) * per + r / 24 * 8 + w % 8;
        }
    }
    const long long L0 = (long long)tile * NL;
    for (int l = tid; l < NL; l += NTHR) {
        const long long L = L0 + l;
        const bool ok = L < nlines;
        bin[l] = ok ? line_base(mi, L) : -1;
        bout[l] = ok ? line_base(mo, L) : -1;
        const int a = ok ? (int)(L / lines_per_sys) : 0; // system in the batch
        const int as = a % P.S;                           // system within its member
        ltau[l] = (R)(P.taud ? P.taud[a] : P.tau[a]);
        for (int m = 0; m < MAXM; ++m) lcoef[m * NL + l] = (R)P.coef[as * MAXM + m];
        lsub[l] = as % 3;
    }
    __syncthreads();
    tile_load<N, NL, NTHR>(lds, T1, bin, mi.SP, tid);
    // the old field of this thread's output cells, all loads in flight at
    // once: 8-byte elements while the FFT runs, 16-byte elements right after
    // it (holding them in registers across the FFT measured slower)
    constexpr int PER = (TOT + NTHR - 1) / NTHR;
    constexpr bool PREF = sizeof(V) < 16;
    V xold[PER];
    R others[GEN ? 2 * PER : 2] = {}; // coupled model: of the other two systems
    auto load_old = [&] {
#pragma unroll
        for (int t = 0; t < PER; ++t) {
            const int e = tid + t * NTHR;
            const long long b = (TOT % NTHR == 0 || e < TOT) ? bout[e / N] : -1;
            const V *const at = xo + (b >= 0 ? b + e % N : 0);
            xold[t] = GEN ? *at : ld_stream(at); // plain: the other systems' blocks read it, too
            if constexpr (GEN) {
                if (ext) {
                    const int j = e < TOT ? lsub[e / N] : 0;
                    others[2 * t] = at[j == 2 ? -2 * P.ncell : P.ncell].x;
                    others[2 * t + 1] = at[j == 0 ? 2 * P.ncell : -P.ncell].x;
                }
            }
        }
    };
    if constexpr (PREF) load_old();
    __syncthreads();
    fft_stages<N, 1, NL, NTHR, true>(lds, tw, tid);
    if constexpr (!PREF) load_old();

    const R cddt = (R)P.cddt, invN = (R)P.invN;
    const int nm = P.ncoef;
    // each thread sums at most 16 cells in FP64 (relative error below 16 u);
    // the block level is a pairwise tree with a compensated wave combine
    // (block_sum_comp), the grid level a Kahan sum (k_sums)
    double s_norm = 0.0, s_ave = 0.0, s_core = 0.0, s_str = 0.0;
#pragma unroll
    for (int t = 0; t < PER; ++t) {
        const int e = tid + t * NTHR;
        if (TOT % NTHR != 0 && e >= TOT) continue;
        const int l = e / N, p = e % N; // mo.SP == 1: rows of xi are contiguous
        const long long b = bout[l];
        if (b < 0) continue;
        const long long idx = b + p;
        const V g = lds.ld(p * LDP + l);
        const V x = xold[t];
        const R tau = ltau[l];
        R dens;
        double dn;
        const V y = gl_update_cell<R, GEN>(g, x, others + (GEN ? 2 * t : 0), idx, tau, [&](int m) { return lcoef[m * NL + l]; }, P, nm,
                                           cddt, invN, mask, prev, xo, amp, dn, dens);
        st_stream(&xn[idx], y);
        if constexpr (FW != 0) lds.st(p * LDP + l, y); // this thread's own cell, read above
        s_norm += dn;
        s_ave += (double)y.x;
        s_core += (double)dens;
        s_str += (double)tau * (double)x.x;
    }
    double v[4] = {s_norm, s_ave, s_core, s_str};
    block_sum_comp<4, NTHR>(v, red, tid); // its barriers also order the tile writes above
    if (tid == 0) {
        partial[0 * pstride + blockIdx.x] = v[0];
        partial[1 * pstride + blockIdx.x] = v[1];
        partial[2 * pstride + blockIdx.x] = v[2];
        partial[3 * pstride + blockIdx.x] = v[3];
    }
    if constexpr (FW != 0) {
        // a thread index the compiler cannot trace: the addresses of the second
        // transform are formed again instead of held in registers through the
        // update
        int t2 = tid;
        __asm__ volatile("" : "+v"(t2));
        if constexpr (FW == 2) fft_stages_x<N, 1, NL, NTHR, false>(lds, tw, t2);
        else fft_stages<N, 1, NL, NTHR, false>(lds, tw, t2);
        tile_store<N, NL, NTHR>(T1, lds, bin, mi.SP, t2, keep);
    }
}

// Pass 5 with the transforms held in registers (pfdd_reg.hpp), for the lengths
// that have them: a thread reads its values of T1 (line-fastest: runs of NL
// lines), transforms them back, holds after the last stage VPT cells of one
// row of xi (position-fastest: runs of D cells), updates them in place and,
// with FW, transforms them forward from the same registers and writes T1.  Two
// LDS accesses per value and transform are left (six in k_update at 128
// points) and no barrier at all where a tile is one wave (FP64 at 32 points).
// The twiddles sit in LDS: loads from memory would wait, in order,
// for the streams in flight.
//
// NM: terms of the core's sine series, padded to 2, 4 or 8; MA: with an
// obstacle mask or a per-cell amplitude (whichever is absent is read from one
// constant element: mstep, astep 0).
template <typename R, int N, int PL, bool FW, int NM, bool MA>
__global__ void __launch_bounds__((RegTile<R, N>::W)) __attribute__((amdgpu_waves_per_eu(sizeof(R) == 8 ? 3 : 4, 8)))
    k_update_r(typename cvec<R>::type *T1, const typename cvec<R>::type *__restrict__ xo,
               typename cvec<R>::type *__restrict__ xn, const uint8_t *__restrict__ mask,
               const long long *__restrict__ prev, const R *__restrict__ amp, unsigned mstep, unsigned astep,
               unsigned ny, unsigned lines_per_sys, StepParams P, const typename cvec<R>::type *__restrict__ tw,
               bool keep, double *__restrict__ partial, long long pstride, const int *__restrict__ done)
{
    typedef typename cvec<R>::type V;
    typedef RegTile<R, N> G;
    constexpr int NL = G::NL, VPT = G::VPT, D = G::D, W = G::W, NW = (W + 63) / 64;
    if (*done) return;
    __shared__ __align__(16) char mem[N * NL * RegLds<V>::bytes];
    __shared__ V tws[N];
    __shared__ double red[4 * NW];
    RegLds<V> lds{(decltype(RegLds<V>::p))mem};
    const int t = threadIdx.x;
    // lines L = (a nx + i) ny + j; a tile may cross rows of j
    const unsigned L0 = blockIdx.x * NL, r0 = L0 / ny;
    V v[VPT];
    unsigned o1; // byte offset of this thread's first value from the tile's T1 row
    V *const T1b = T1 + (long long)r0 * ny * N;
    {
        const unsigned l = t % NL, p0 = t / NL;
        const unsigned j = L0 - r0 * ny + l, row = j / ny;
        o1 = (row * ny * N + (j - row * ny) + p0 * ny) * (unsigned)sizeof(V);
#pragma unroll
        for (int m = 0; m < VPT; ++m)
            v[m] = ld_stream((const V *)((const char *)(T1b + (size_t)(D * m) * ny) + o1));
    }
    reg_twiddles<N, W>(tws, tw, t);
    const unsigned l = t / D, p0 = t % D;
    const unsigned a = (L0 + l) / lines_per_sys; // system in the batch
    // this thread's line: its stress and core coefficients
    const R tau = (R)(P.taud ? P.taud[a] : P.tau[a]);
    const double *const cf = P.coef + (a % P.S) * MAXM;
    R lc[NM], ldp[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m) {
        lc[m] = (R)cf[m];
        ldp[m] = lc[m] * ((R)(m + 1) * (R)M_PI);
    }
    const long long base = (long long)L0 * N;
    const unsigned o2 = l * N + p0;
    // the old field comes in chunks of CH cells, AHEAD chunks before the update
    // (the first one during the transform): enough bytes in flight with 3-4
    // waves per SIMD, where holding all of it costs the registers of one
    constexpr int CH = 2, AHEAD = 1, NCK = VPT / CH;
    V x[AHEAD + 1][CH];
    auto fetch = [&](int ck) {
#pragma unroll
        for (int c = 0; c < CH; ++c) x[ck % (AHEAD + 1)][c] = ld_stream(xo + base + o2 + D * (ck * CH + c));
    };
#pragma unroll
    for (int ck = 0; ck < AHEAD; ++ck) fetch(ck);
    reg_fft<N, 1, PL, NL, VPT, true, false, true, true>(v, lds, tws, t);

    const R cddt = (R)P.cddt, invN = (R)P.invN;
    // a thread sums its VPT cells in FP64; block and grid levels as in k_update
    double s_norm = 0.0, s_ave = 0.0, s_core = 0.0, s_str = 0.0;
    unsigned frozen = 0; // this thread's masked cells
#pragma unroll
    for (int ck = 0; ck < NCK; ++ck) {
        // one chunk's temporaries at a time
        __builtin_amdgcn_sched_barrier(0);
        if (ck + AHEAD < NCK) fetch(ck + AHEAD);
        const V *xc = x[ck % (AHEAD + 1)];
        unsigned fz = 0;
        R A[CH];
        if constexpr (MA) {
#pragma unroll
            for (int c = 0; c < CH; ++c) {
                const long long at = base + D * (ck * CH + c); // uniform; o2 is the lane's offset
                fz |= (unsigned)(mask + at * mstep)[o2 * mstep] << c; // 0 or 1
                A[c] = (amp + at * astep)[o2 * astep];
            }
            frozen |= fz << (ck * CH);
        }
        V y[CH];
        R dens[CH];
        double dn[CH];
        gl_update_chunk<R, NM, MA, CH>(&v[ck * CH], xc, A, fz, tau, lc, ldp, cddt, invN, y, dn, dens);
#pragma unroll
        for (int c = 0; c < CH; ++c) {
            st_stream(&xn[base + o2 + D * (ck * CH + c)], y[c]);
            v[ck * CH + c] = y[c];
            s_norm += dn[c];
            s_ave += (double)y[c].x;
            s_core += (double)dens[c];
            s_str += (double)tau * (double)xc[c].x;
        }
        // the sums are formed here: sunk to their use behind the next branch
        // they would keep every cell's values in registers until then
        __asm__ volatile("" : "+v"(s_norm), "+v"(s_ave), "+v"(s_core), "+v"(s_str));
    }
    __builtin_amdgcn_sched_barrier(0);
    // quirk Q3: a masked cell's xinorm term takes the previous unmasked cell
    while (MA && frozen) {
        const unsigned m = __builtin_ctz(frozen);
        frozen &= frozen - 1;
        const long long idx = base + o2 + D * m, pi = prev[idx];
        const V xm = xo[idx], pv = pi >= 0 ? xo[pi] : mk<V>((R)0, (R)0);
        const double dr = (double)xm.x - (double)pv.x, di = (double)xm.y - (double)pv.y;
        s_norm += dr * dr + di * di;
    }
    if constexpr (FW) {
        // a thread index the compiler cannot trace: addresses are formed again
        // instead of held in registers through the update
        int t2 = t;
        __asm__ volatile("" : "+v"(t2));
        reg_fft<N, 1, PL, NL, VPT, false, true, false, false>(v, lds, tws, t2);
#pragma unroll
        for (int m = 0; m < VPT; ++m) st_work((V *)((char *)(T1b + (size_t)(D * m) * ny) + o1), v[m], keep);
    }
    double sum[4] = {s_norm, s_ave, s_core, s_str};
    block_sum_comp<4, W>(sum, red, t);
    if (t == 0) {
#pragma unroll
        for (int q = 0; q < 4; ++q) partial[q * pstride + blockIdx.x] = sum[q];
    }
}

// ------------------------------------------ adjoint of pass 5 (reverse mode)
// One GL iteration (k_update) maps xi to
//   xi' = xi - cddt U (g/N - tau + dE(Re xi))      (Re part; Im: xi' = xi - cddt U g/N)
// with U = 1 on unmasked cells and g = IFFT(B FFT xi).  The elastic operator
// is self-adjoint (B(k) real, symmetric in (a, b) and even in k), so for
// lam' = dL/dxi' (Re and Im taken as independent real variables)
//   mu  = U lam'
//   lam = lam' - cddt (IFFT(B FFT mu)/N + dE'(Re xi) Re mu)   (dE' acts on Re only)
//   dL/dtau_a   += cddt sum_r Re mu_a
//   dL/dc_{a,m} += -cddt sum_r Re mu_a A m pi sin(2 m pi Re xi_a)
// with dE = A sum_m c_m m pi sin(2 m pi x), dE' = A sum_m c_m 2 m^2 pi^2 cos(2 m pi x).
// The extended model couples the three systems of a plane: there dE'(Re xi)
// Re mu becomes the Hessian of the plane density applied to the triple's
// Re mu (core_extended_adj).
// T1 holds mu after passes 1-4; this kernel applies the last inverse pass and
// the update above, and leaves per-block sums of Re mu (slot 0) and of
// Re mu A m pi sin(2 m pi x) (slot m) in gpart.  Every block covers lines of
// one system (the host checks nx*ny % NL == 0).
template <typename R, int N, int TQ>
__global__ void __launch_bounds__(NTHR)
    k_adj_update(const typename cvec<R>::type *__restrict__ T1, const typename cvec<R>::type *__restrict__ lam,
                 const typename cvec<R>::type *__restrict__ xs, typename cvec<R>::type *__restrict__ lam_out,
                 const uint8_t *__restrict__ mask, const R *__restrict__ amp, LineMap mi, LineMap mo,
                 long long nlines, long long lines_per_sys, StepParams P,
                 const typename cvec<R>::type *__restrict__ tw, double *__restrict__ gpart, long long gstride,
                 const int *__restrict__ done)
{
    typedef typename cvec<R>::type V;
    if (*done) return;
    constexpr int NL = tile_lines_u<R, N, TQ>(), LDP = NL + 1, TOT = N * NL;
    constexpr int PER = (TOT + NTHR - 1) / NTHR;
    constexpr int NG = 1 + MAXM;
    PFDD_TILE(V, lds, N * LDP);
    __shared__ long long bin[NL], bout[NL];
    __shared__ double red[NG * (NTHR / 64)];
    const int tid = threadIdx.x;
    const long long L0 = (long long)blockIdx.x * NL;
    for (int l = tid; l < NL; l += NTHR) {
        const long long L = L0 + l;
        const bool ok = L < nlines;
        bin[l] = ok ? line_base(mi, L) : -1;
        bout[l] = ok ? line_base(mo, L) : -1;
    }
    __syncthreads();
    tile_load<N, NL, NTHR>(lds, T1, bin, mi.SP, tid);
    __syncthreads();
    fft_stages<N, 1, NL, NTHR, true>(lds, tw, tid);

    const int a = (int)(L0 / lines_per_sys) % P.S;
    const R cddt = (R)P.cddt, invN = (R)P.invN;
    const int nm = P.ncoef;
    double acc[NG];
#pragma unroll
    for (int q = 0; q < NG; ++q) acc[q] = 0.0;
#pragma unroll 2
    for (int t = 0; t < PER; ++t) {
        const int e = tid + t * NTHR;
        if (TOT % NTHR != 0 && e >= TOT) continue;
        const int l = e / N, p = e % N;
        const long long b = bout[l];
        if (b < 0) continue;
        const long long idx = b + p;
        const V g = lds.ld(p * LDP + l);
        const V lm = lam[idx];
        const V x = xs[idx];
        const R mr = (mask && mask[idx]) ? (R)0 : lm.x;
        const R A = amp ? (R)amp[idx] : (R)1;
        // sin, cos of 2 pi m x by the angle-addition recurrence from m = 1
        R sp, cp;
        sincospi_poly(x.x, sp, cp);
        const R s1 = (R)2 * sp * cp, c1 = cp * cp - sp * sp;
        R sm = s1, cm = c1, d2 = (R)0, hv = (R)0;
        if (P.model == PFDD_CORE_EXTENDED) {
            // the triple of systems of this plane at the same cell (no amp[])
            const int j = a % 3;
            const long long b0 = idx - (long long)j * P.ncell;
            R y[3], m3[3], cc[7];
#pragma unroll
            for (int q = 0; q < 3; ++q) {
                const long long iq = b0 + q * P.ncell;
                y[q] = q == j ? x.x : xs[iq].x;
                m3[q] = q == j ? mr : ((mask && mask[iq]) ? (R)0 : lam[iq].x);
            }
#pragma unroll
            for (int q = 0; q < 7; ++q) cc[q] = (R)P.coef[a * MAXM + q];
            double gc[7];
            core_extended_adj<R>(y, m3, j, cc, hv, gc);
#pragma unroll
            for (int q = 0; q < 7; ++q) acc[1 + q] += gc[q];
        } else if (P.model == PFDD_CORE_FOURIER || P.model == PFDD_CORE_PYRII) {
            // Fourier density a0 + sum_m a_m cos(w x) + b_m sin(w x), w = 2 pi m:
            //   dE = sum_m w (b_m cos - a_m sin),  dE' = -sum_m w^2 (a_m cos + b_m sin)
            //   d(dE)/d a_m = -w sin(w x),  d(dE)/d b_m = w cos(w x)   (slots m, 4 + m)
            // pyrII as executed: only the last cell of each system carries dE
            if (P.model == PFDD_CORE_FOURIER || (idx % P.ncell) == P.ncell - 1) {
#pragma unroll
                for (int m = 1; m <= 4; ++m) {
                    const R am = (R)P.coef[a * MAXM + m - 1], bm = (R)P.coef[a * MAXM + m + 3];
                    const double w = 2.0 * M_PI * m;
                    d2 -= (R)(w * w) * (am * cm + bm * sm);
                    acc[m] += (double)mr * (double)A * (-w * (double)sm);
                    acc[4 + m] += (double)mr * (double)A * (w * (double)cm);
                    const R sn = sm * c1 + cm * s1, cn = cm * c1 - sm * s1;
                    sm = sn;
                    cm = cn;
                }
            }
        } else {
#pragma unroll
            for (int m = 1; m <= MAXM; ++m) {
                if (m <= nm) {
                    const R c = (R)P.coef[a * MAXM + m - 1];
                    d2 += c * ((R)(2 * m * m) * (R)(M_PI * M_PI)) * cm;
                    acc[m] += (double)mr * (double)A * (double)m * M_PI * (double)sm;
                    const R sn = sm * c1 + cm * s1, cn = cm * c1 - sm * s1;
                    sm = sn;
                    cm = cn;
                }
            }
        }
        V y;
        y.x = lm.x - cddt * (g.x * invN + A * d2 * mr + hv);
        y.y = lm.y - cddt * (g.y * invN);
        lam_out[idx] = y;
        acc[0] += (double)mr;
    }
    block_sum<NG, NTHR>(acc, red, tid);
    if (tid == 0) {
#pragma unroll
        for (int q = 0; q < NG; ++q) gpart[q * gstride + blockIdx.x] = acc[q];
    }
}


template <typename R> int update_blocks_max(int n, long long nlines)
{
    // the smallest tiles: shape 0, and on short lines the register update's
    int nl = tile_lines_rt<R>(n, 0);
#define PFDD_CASE(n_)                                                                          \
    if (n == n_) {                                                                             \
        if constexpr (reg_length<n_>()) nl = RegTile<R, n_>::NL < nl ? RegTile<R, n_>::NL : nl; \
    }
    PFDD_SIZES(PFDD_CASE)
#undef PFDD_CASE
    return (int)((nlines + nl - 1) / nl);
}

template <typename R>
hipError_t launch_update(int n, int tq, int plan, bool fw, void *T1, const void *xo, void *xn, const uint8_t *mask,
                         const long long *prev, const void *amp, LineMap mi, LineMap mo, long long nlines,
                         long long lps, const StepParams &P, const void *tw, const UpdNone *none, bool keep,
                         double *partial, long long pstride, const int *done, hipStream_t st, int *nblocks)
{
    typedef typename cvec<R>::type V;
    const uint8_t *no_mask = &none->zero;
    const R *no_amp = sizeof(R) == 8 ? (const R *)&none->one64 : (const R *)&none->one32;
    (void)no_mask;
    (void)no_amp;
    // the coupled and Fourier core models get their own instantiation (one
    // tile shape) so that the common sine-series kernel carries none of
    // their registers
    const bool gen = P.model == PFDD_CORE_EXTENDED || P.model == PFDD_CORE_PYRII || P.model == PFDD_CORE_FOURIER;
    // plan 1 falls back to plan 0 where the two coincide
#define PFDD_UPR_(PL_, FW_, NM_, MA_)                                                                \
    PFDD_LAUNCH((k_update_r<R, N, (PL_ && radix16_plan_differs<N>()), FW_, NM_, MA_>),               \
                dim3((unsigned)*nblocks), dim3(RegTile<R, N>::W), st, (V *)T1,                       \
                (const V *)xo, (V *)xn, mask ? mask : no_mask, prev,                                 \
                amp ? (const R *)amp : no_amp, mask ? 1u : 0u, amp ? 1u : 0u, (unsigned)mi.D,        \
                (unsigned)lps, P, (const V *)tw, keep, partial, pstride, done)
#define PFDD_UPR(PL_, FW_)                                                                           \
    do {                                                                                             \
        if (mask || amp) {                                                                           \
            if (P.ncoef <= 2) PFDD_UPR_(PL_, FW_, 2, true);                                          \
            else if (P.ncoef <= 4) PFDD_UPR_(PL_, FW_, 4, true);                                     \
            else PFDD_UPR_(PL_, FW_, 8, true);                                                       \
        } else {                                                                                     \
            if (P.ncoef <= 2) PFDD_UPR_(PL_, FW_, 2, false);                                         \
            else if (P.ncoef <= 4) PFDD_UPR_(PL_, FW_, 4, false);                                    \
            else PFDD_UPR_(PL_, FW_, 8, false);                                                      \
        }                                                                                            \
    } while (0)
#define PFDD_UPD(TQ_, GEN_, FW_)                                                                     \
    *nblocks = (int)((nlines + tile_lines_u<R, N, TQ_>() - 1) / tile_lines_u<R, N, TQ_>());          \
    PFDD_LAUNCH((k_update<R, N, TQ_, GEN_, FW_>), dim3((unsigned)*nblocks), dim3(NTHR), st,         \
                (V *)T1, (const V *)xo, (V *)xn, mask, prev, (const R *)amp, mi, mo, \
                nlines, lps, P, (const V *)tw, keep, partial, pstride, done)
#define PFDD_UPD_FW(TQ_, GEN_)                                                                       \
    if (!fw) { PFDD_UPD(TQ_, GEN_, 0); }                                                             \
    else if (plan == 1 && radix16_plan_differs<N>()) { PFDD_UPD(TQ_, GEN_, (radix16_plan_differs<N>() ? 2 : 1)); } \
    else { PFDD_UPD(TQ_, GEN_, 1); }
#define PFDD_CASE(n_)                                                                                \
    if (n == n_) {                                                                                   \
        constexpr int N = n_;                                                                        \
        if constexpr (reg_length<N>()) {                                                             \
            if (!gen) {                                                                              \
                const bool p1 = plan == 1 && radix16_plan_differs<N>();                              \
                *nblocks = (int)(nlines / RegTile<R, N>::NL);                                        \
                if (p1 && fw) PFDD_UPR(1, true);                                                     \
                else if (p1) PFDD_UPR(1, false);                                                     \
                else if (fw) PFDD_UPR(0, true);                                                      \
                else PFDD_UPR(0, false);                                                             \
                return hipGetLastError();                                                            \
            }                                                                                        \
        }                                                                                            \
        if (gen) {                                                                                   \
            PFDD_UPD_FW(0, true);                                                                    \
            return hipGetLastError();                                                                \
        }                                                                                            \
        if constexpr (!reg_length<N>()) {                                                            \
            PFDD_TQ_DISPATCH(tq, { PFDD_UPD_FW(TQ, false); })                                        \
        }                                                                                            \
        return hipGetLastError();                                                                    \
    }
    PFDD_SIZES(PFDD_CASE)
#undef PFDD_CASE
#undef PFDD_UPD_FW
#undef PFDD_UPD
#undef PFDD_UPR
#undef PFDD_UPR_
    return hipErrorInvalidValue;
}

template <typename R>
hipError_t launch_adj_update(int n, int tq, const void *T1, const void *lam, const void *xs, void *lam_out,
                             const uint8_t *mask, const void *amp, LineMap mi, LineMap mo, long long nlines,
                             long long lps, const StepParams &P, const void *tw, double *gpart,
                             long long gstride, const int *done, hipStream_t st)
{
    typedef typename cvec<R>::type V;
#define PFDD_CASE(n_)                                                                                  \
    if (n == n_) {                                                                                     \
        PFDD_TQ_DISPATCH(tq, {                                                                         \
            constexpr int NL = tile_lines_u<R, n_, TQ>();                                              \
            const unsigned nb = (unsigned)((nlines + NL - 1) / NL);                                    \
            hipLaunchKernelGGL((k_adj_update<R, n_, TQ>), dim3(nb), dim3(NTHR), 0, st, (const V *)T1,  \
                               (const V *)lam, (const V *)xs, (V *)lam_out, mask, (const R *)amp, mi, mo, \
                               nlines, lps, P, (const V *)tw, gpart, gstride, done);                   \
        })                                                                                             \
        return hipGetLastError();                                                                      \
    }
    PFDD_SIZES(PFDD_CASE)
#undef PFDD_CASE
    return hipErrorInvalidValue;
}

#define PFDD_INST(R)                                                                                          \
    template int update_blocks_max<R>(int, long long);                                                                \
    template hipError_t launch_update<R>(int, int, int, bool, void *, const void *, void *, const uint8_t *,           \
                                         const long long *, const void *, LineMap, LineMap, long long, long long, \
                                         const StepParams &, const void *, const UpdNone *, bool, double *, long long, \
                                         const int *, hipStream_t, int *);                                        \
    template hipError_t launch_adj_update<R>(int, int, const void *, const void *, const void *, void *,         \
                                             const uint8_t *, const void *, LineMap, LineMap, long long,          \
                                             long long, const StepParams &, const void *, double *, long long,    \
                                             const int *, hipStream_t);
PFDD_INST(double)
PFDD_INST(float)
#undef PFDD_INST

} // namespace pfdd
