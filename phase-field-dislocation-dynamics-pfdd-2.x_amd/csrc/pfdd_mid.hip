// pfdd_mid.hip -- the x pass: FFT along x, Green's-function contraction,
// inverse FFT along x (stored-B and on-the-fly variants), and launchers.
#include "pfdd_kern.hpp"
#include "pfdd_reg.hpp"

namespace pfdd {

// Load the S lines of NP consecutive columns (T2[a][c0+q][0..N)) into the
// tile, lines ordered (a, q); column-contiguous runs of N elements.  Every
// load of a thread is issued before its first LDS write, in both precisions
// (for the 16-byte elements of the FP64 x pass at 128^3 x 12 this measured
// 191 -> 184 us against a strided loop of 4 loads in flight).
template <int N, int NL, int NP, int NTHR, typename XA, typename V>
__device__ __forceinline__ void tile_load_cols(const Tile<V> lds, const V *__restrict__ T2, long long c0, long long ncol,
                                               long long ntot, int tid)
{
    constexpr int TOT = NL * N, PER = (TOT + NTHR - 1) / NTHR;
    {
        V r[PER];
#pragma unroll
        for (int t = 0; t < PER; ++t) {
            const int e = tid + t * NTHR;
            const int l = e / N, p = e % N;
            const int a = l / NP, q = l % NP;
            if ((TOT % NTHR == 0 || e < TOT) && c0 + q < ncol) r[t] = ld_stream(&T2[(long long)a * ntot + (c0 + q) * N + p]);
        }
#pragma unroll
        for (int t = 0; t < PER; ++t) {
            const int e = tid + t * NTHR;
            if (TOT % NTHR == 0 || e < TOT) lds.st(XA::at(e % N, e / N), r[t]);
        }
    }
}

// --------------------------------------------- pass 3: x FFT + contraction
// Columns per x-pass tile with the stages in LDS (any length with stored B, the
// plane layout, and lengths without register transforms): the largest power of
// two whose S*NP lines of N elements stay within `target` elements.  FP64 with 12 systems takes twice
// the tile of the other FP64 cases: at 128^3 x 12 two columns per block (one
// thread per k-point, no duplicated contraction work, 3 blocks per CU) ran
// the pass 12 % faster than one column (two threads per k-point, 5 blocks).
// So do 512-point FP64 lines (two columns of 3 systems instead of one:
// 512 x 512 x 256 x 3, 2.52 -> 2.27 ms; in FP32 four columns instead of two
// were slower).
template <typename R, int N, int S> constexpr int mid_pairs()
{
    constexpr int target = sizeof(R) == 8 ? ((S == 12 || N >= 512) ? 4096 : 2048) : 4096;
    int np = 1;
    while (np * 2 * S * N <= target) np *= 2;
    // the padded tile stays within 60 KB of LDS (the constants and the
    // reduction scratch of the pass come on top)
    while (np > 1 && (long long)N * (S * np + 1) * 2 * (int)sizeof(R) > 61440) np /= 2;
    return np;
}

// Tile addressing of the on-the-fly x pass where its stages are in LDS: Swz8 for
// 24-line FP64 tiles (12 systems x 2 columns, at 96 points and, in the plane
// layout, 128); RowPad otherwise.
template <typename R, int N, int S> struct XLay {
    static constexpr int NL = S * mid_pairs<R, N, S>();
    typedef typename std::conditional<(sizeof(R) == 8 && NL == 24 && N % 16 == 0), Swz8<NL>, RowPad<NL>>::type type;
};

template <typename R, typename RB, int N, int S>
__global__ void __launch_bounds__(NTHR)
    k_mid(typename cvec<R>::type *__restrict__ T2, const RB *__restrict__ B, long long ncol,
          long long ntot, int bpm, const typename cvec<R>::type *__restrict__ tw, double *__restrict__ part_el,
          const int *__restrict__ done)
{
    typedef typename cvec<R>::type V;
    if (*done) return;
    constexpr int NP = mid_pairs<R, N, S>();
    constexpr int NL = S * NP, LDP = NL + 1, TOT = NL * N;
    constexpr int NPAIR = S * (S + 1) / 2;
    PFDD_TILE(V, lds, N * LDP);
    __shared__ double red[NTHR / 64];
    const int tid = threadIdx.x;
    // member of a batch (bpm blocks per member), first column of the block
    const int mem = blockIdx.x / bpm;
    const long long c0 = (long long)(blockIdx.x - mem * bpm) * NP;
    T2 += (long long)mem * S * ntot;
    // load: lines (a, q) -> T2[a][c0+q][0..N)
#pragma unroll 4
    for (int e = tid; e < TOT; e += NTHR) {
        const int l = e / N, p = e % N;
        const int a = l / NP, q = l % NP;
        if (c0 + q < ncol) lds.st(p * LDP + l, ld_stream(&T2[(long long)a * ntot + (c0 + q) * N + p]));
    }
    __syncthreads();
    fft_stages<N, 1, NL, NTHR, false>(lds, tw, tid);
    double el = 0.0; // few k-points per thread; the block and grid sums are compensated
    for (int e = tid; e < NP * N; e += NTHR) {
        const int q = e / N, p = e % N;
        if (c0 + q >= ncol) continue;
        const long long kp = (c0 + q) * N + p;
        V x[S];
#pragma unroll
        for (int b = 0; b < S; ++b) x[b] = lds.ld(p * LDP + b * NP + q);
        R g[S][2];
#pragma unroll
        for (int a = 0; a < S; ++a) g[a][0] = g[a][1] = (R)0;
        int slot = 0;
#pragma unroll
        for (int a = 0; a < S; ++a) {
#pragma unroll
            for (int b = a; b < S; ++b, ++slot) {
                const R bab = (R)B[(long long)slot * ntot + kp];
                g[a][0] += bab * x[b].x;
                g[a][1] += bab * x[b].y;
                if (b != a) {
                    g[b][0] += bab * x[a].x;
                    g[b][1] += bab * x[a].y;
                }
            }
        }
        (void)NPAIR;
#pragma unroll
        for (int a = 0; a < S; ++a) {
            el += (double)x[a].x * (double)g[a][0] + (double)x[a].y * (double)g[a][1];
            lds.st(p * LDP + a * NP + q, mk<V>(g[a][0], g[a][1]));
        }
    }
    __syncthreads();
    fft_stages<N, 1, NL, NTHR, true>(lds, tw, tid);
#pragma unroll 4
    for (int e = tid; e < TOT; e += NTHR) {
        const int l = e / N, p = e % N;
        const int a = l / NP, q = l % NP;
        if (c0 + q < ncol) st_work(&T2[(long long)a * ntot + (c0 + q) * N + p], lds.ld(p * LDP + l), false);
    }
    double v[1] = {el};
    block_sum_comp<1, NTHR>(v, red, tid);
    if (tid == 0) part_el[blockIdx.x] = v[0];
}


// x pass with B(k) evaluated on the fly in FP64 instead of streamed from HBM.
// Bmatrix's kernel (fft_fftw_slab.cpp:577-634) is mu B_ab = eps_a:A:eps_b with
// A = C - (C f) G (f C), G = (2 I/f^2 - f f/((1-nu) f^4))/(2 C44).  Applied as
// internal_energy does (:1670-1695) to all systems at once:
//   Sig = sum_b xihat_b sigma_b        (sigma_b = C:eps_b)
//   w = Sig f,  V = f.w
//   Q = [2 sym(w f)/f^2 - V f f/((1-nu) f^4)] / (2 C44)
//   P = Sig - C:Q = Sig - 2 C44 Q - C12 tr(Q) I
//     = Sig - D - c5 tr(D) I,  D = u f + f u,  u = c2 w - c4 V f,
//       c2 = 1/f^2, c4 = 1/(2 (1-nu) f^4), c5 = C12 / (2 C44)
//   ghat_a = eps_a : P / mu
// (80 instead of 110 instructions a point for P from Sig; FP32 error of P over
// the k-points of planar fields on 48 to 160 points, rms: 2.1e-7 to 3.9e-7 ->
// 1.8e-7 to 2.7e-7.  sigma_a:Q = eps_a:(C:Q) for the isotropic C), and ghat = 0 at f = 0
// (B(0) = 0).  TPP threads share one k-point (wave-uniform split of the
// systems), each producing S/TPP of the outputs.
template <typename R, int N, int S> constexpr int otf_tpp()
{
    constexpr int pts = mid_pairs<R, N, S>() * N;
    return (2 * pts == NTHR && S % 2 == 0) ? 2 : 1;
}

// A k-point: f and the scalars of P and ghat (above) in the arithmetic type T of
// the x pass; nz: f != 0.  In FP64 the constants eps_a hold 1/mu.  In FP32 it is
// a factor of ghat: the components of eps_a are mostly exact, those of eps_a /
// mu are not, and with them the energy at 128^3 x 12 moved by 1.5e-7 of itself.
template <typename T> struct KPoint {
    T f[3], c2, c4, c5, invmu;
    bool nz;
};

// Sig -> P at one k-point (real and imaginary part; symmetric components xx,
// yy, zz, xy, xz, yz).  The order of every sum of products is written out, so
// that all x-pass variants round alike.
template <typename T> __device__ __forceinline__ void otf_green(T Pr[6], T Pi[6], const KPoint<T> &K)
{
    const T *const f = K.f;
    auto half = [&](T *p) { // one of the two parts
        auto dot3 = [](T a0, T a1, T a2, const T *b) { return ab_c(a2, b[2], ab_cd(a1, b[1], a0, b[0])); };
        const T w[3] = {dot3(p[0], p[3], p[4], f), dot3(p[3], p[1], p[5], f), dot3(p[4], p[5], p[2], f)};
        const T V = dot3(w[0], w[1], w[2], f), v = K.c4 * V;
        T u[3], d[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) u[i] = ab_cd(K.c2, w[i], -v, f[i]);
#pragma unroll
        for (int i = 0; i < 3; ++i) d[i] = u[i] * ((T)2 * f[i]);
        const T tr = K.c5 * (d[0] + d[1] + d[2]);
#pragma unroll
        for (int i = 0; i < 3; ++i) p[i] -= d[i] + tr;
        const int ci[3] = {0, 0, 1}, cj[3] = {1, 2, 2};
#pragma unroll
        for (int c = 0; c < 3; ++c) p[3 + c] = ab_c(-u[ci[c]], f[cj[c]], ab_c(-u[cj[c]], f[ci[c]], p[3 + c]));
    };
    half(Pr);
    half(Pi);
}

// P at f = 0, where B vanishes.
template <typename T> __device__ __forceinline__ void otf_zero(T Pr[6], T Pi[6])
{
#pragma unroll
    for (int c = 0; c < 6; ++c) Pr[c] = Pi[c] = (T)0;
}

// Hands ghat_a for a = H*SA .. H*SA+SA-1 of one k-point to sink(aa, re, im,
// xihat_a), computed in T (double in the FP64 path, float in the FP32 mode).
// xihat_a is the value read for the contraction, kept in registers so that
// the sink does not read the tile again (FP64 x pass at 128^3 x 12: 189 ->
// 186 us).
template <typename T, int S, int SA, int H, int NP, typename XA, typename V, typename Sink>
__device__ __forceinline__ void otf_point(const Tile<V> lds, int p, int q, const KPoint<T> &K,
                                          const T *__restrict__ cst, Sink sink)
{
    // compiler-only barriers keep the (LDS-broadcast) constants from being
    // hoisted and held in registers across points and systems
    __asm__ volatile("" ::: "memory");
    T Pr[6], Pi[6]; // Sig, then P
    V xk[SA];
#pragma unroll
    for (int b = 0; b < S; ++b) {
        const V v = lds.ld(XA::at(p, b * NP + q));
        if (b >= H * SA && b < H * SA + SA) xk[b - H * SA] = v;
        const T xr = (T)v.x, xi = (T)v.y;
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            Pr[c] = b ? ab_c(cst[b * 12 + c], xr, Pr[c]) : cst[c] * xr;
            Pi[c] = b ? ab_c(cst[b * 12 + c], xi, Pi[c]) : cst[c] * xi;
        }
    }
    if (K.nz) otf_green(Pr, Pi, K);
    else otf_zero(Pr, Pi);
#pragma unroll
    for (int aa = 0; aa < SA; ++aa) {
        __asm__ volatile("" ::: "memory");
        const int a = H * SA + aa;
        const T *ep = cst + a * 12 + 6;
        T gr = Pr[0] * ep[0], gi = Pi[0] * ep[0];
#pragma unroll
        for (int c = 1; c < 6; ++c) {
            gr = ab_c(Pr[c], ep[c], gr);
            gi = ab_c(Pi[c], ep[c], gi);
        }
        if constexpr (sizeof(T) == 4) {
            gr *= K.invmu;
            gi *= K.invmu;
        }
        sink(aa, gr, gi, xk[aa]);
    }
}

// f = four^T k~ (frec, fft_fftw_slab.cpp:280-367) in two parts: that of a
// column, (k, j) = (col / ny, col % ny) in the line layout of the five-kernel
// iteration and (j, k) = (col / nz, col % nz) in the plane layout, and that of
// position p.  f is formed in FP64 and rounded to T, its square and the scalars of
// B(k) are formed in FP64 from what it was rounded to and rounded once: in the
// FP32 mode only the contraction with xihat runs in FP32.
// frec's k/n with the reciprocal of n (one rounding more than the division for
// sizes that are not powers of two): the x pass evaluates it for every k-point
// of every step.
__device__ __forceinline__ double otf_frac(int kk, int n, double inv)
{
    return (double)(kk >= n / 2 ? kk - n : kk) * inv;
}
template <bool PL = false> __device__ __forceinline__ void otf_col(const GParams &G, long long col, double *fc)
{
    const int c = (int)col; // column of one member: ny * nz < 2^31
    int j, k;
    if constexpr (PL) {
        j = c / G.nz;
        k = c - j * G.nz;
    } else {
        k = c / G.ny;
        j = c - k * G.ny;
    }
    const double ky = otf_frac(j, G.ny, G.inv_n[1]), kz = otf_frac(k, G.nz, G.inv_n[2]);
#pragma unroll
    for (int c = 0; c < 3; ++c) fc[c] = ab_cd(kz, G.four[6 + c], ky, G.four[3 + c]);
}
template <typename T> __device__ __forceinline__ KPoint<T> otf_freq(const GParams &G, const double *fc, int p)
{
    // f rounded first, f^2 from what it was rounded to: c2 f f is then a
    // projector to one rounding, and P of f parallel to the slip plane's normal,
    // where it vanishes, keeps less of Sig.  FP32 elastic energy against FP64 over
    // 18 grids of 16 to 512 points, rms, f^2 from the unrounded f -> so: loops of
    // 1, 3, 6 and 12 systems 8.1e-8 -> 7.2e-8, 1.20e-7 -> 1.07e-7, 6.6e-8 -> 6.5e-8,
    // 6.6e-8 -> 6.4e-8, of 3 in a skewed cell 1.61e-7 -> 1.53e-7, straight edges
    // 2.8e-7 -> 2.3e-7 (the forward FFT's bias, -4e-8 to -1.4e-7, is in all of them)
    const double kx = otf_frac(p, G.nx, G.inv_n[0]);
    double f[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) f[c] = (double)(T)ab_c(kx, G.four[c], fc[c]);
    const double f2 = ab_c(f[2], f[2], ab_cd(f[1], f[1], f[0], f[0]));
    const double if2 = 1.0 / f2;
    return KPoint<T>{{(T)f[0], (T)f[1], (T)f[2]}, (T)if2, (T)(G.c4f * if2 * if2), (T)G.c5, (T)G.invmu, f2 > 0};
}

// Minimum waves per SIMD asked of the x pass (one wave per SIMD per resident
// block of 256 threads).  The 12- and 3-system FP64 passes ask for 3, 168
// VGPRs instead of 172-190 (96 points x 12 at 96 x 80 x 48: 55.5 -> 48.5 us;
// 3-system batches at 48^3: 80 -> 67 us).  Other system counts and FP32 are not
// constrained: at 48-96 points 5 or 6 waves (96 or 80 VGPRs, with spills) were
// slower than the compiler's 4.
template <typename R, int N, int S> constexpr int otf_waves()
{
    if (S == 12 && sizeof(R) == 8) return 3;
    if (S == 3 && sizeof(R) == 8) return 3;
    return 1;
}

// The transform of one x-pass tile held in LDS (NP columns x S systems):
// forward FFT along x, on-the-fly contraction ghat_a = sum_b B_ab xihat_b,
// inverse FFT.  Returns this thread's share of sum Re(conj(xihat_a) ghat_a).
template <typename R, int N, int S, bool PL = false>
__device__ __forceinline__ double otf_tile(const Tile<typename cvec<R>::type> lds,
                                           const typename cvec<R>::type *__restrict__ tw, const GParams &G,
                                           const R *cst, long long c0, long long ncol, int tid)
{
    typedef typename cvec<R>::type V;
    typedef R T;
    constexpr int NP = mid_pairs<R, N, S>();
    constexpr int NL = S * NP;
    typedef typename XLay<R, N, S>::type XA;
    constexpr int TPP = otf_tpp<R, N, S>();
    constexpr int SA = S / TPP;
    constexpr int NPT = NP * N; // k-points per tile
    fft_stages_x<N, 1, NL, NTHR, false, XA>(lds, tw, tid);
    // the elastic-energy term Re(conj(xihat_a) ghat_a) is taken as each ghat_a
    // replaces xihat_a in the tile
    double el = 0.0; // a thread handles one or two k-points; the block and grid sums are compensated
    if constexpr (TPP == 1) {
        // one thread per k-point: it reads all xihat_b of the point, then
        // overwrites them with ghat_a
        for (int pt = tid; pt < NPT; pt += NTHR) {
            const int q = pt / N, p = pt % N;
            if (c0 + q >= ncol) continue;
            double fc[3];
            otf_col<PL>(G, c0 + q, fc);
            const KPoint<T> K = otf_freq<T>(G, fc, p);
            otf_point<T, S, SA, 0, NP, XA>(lds, p, q, K, cst, [&](int a, T gr, T gi, V x) {
                const int idx = XA::at(p, a * NP + q);
                el += (double)x.x * gr + (double)x.y * gi;
                lds.st(idx, mk<V>((R)gr, (R)gi));
            });
        }
    } else {
        // two waves per set of k-points, each producing half of the systems;
        // all reads of the tile finish (barrier) before any thread writes
        const int h = tid / NPT, pt = tid % NPT;
        const int q = pt / N, p = pt % N;
        const bool ok = c0 + q < ncol;
        double fc[3];
        otf_col<PL>(G, c0 + q, fc);
        const KPoint<T> K = otf_freq<T>(G, fc, p);
        T g[SA][2];
        auto keep = [&](int aa, T gr, T gi, V) {
            g[aa][0] = gr;
            g[aa][1] = gi;
        };
        if (ok) {
            if (__builtin_amdgcn_readfirstlane(h) == 0)
                otf_point<T, S, SA, 0, NP, XA>(lds, p, q, K, cst, keep);
            else
                otf_point<T, S, SA, 1, NP, XA>(lds, p, q, K, cst, keep);
        }
        __syncthreads();
        if (ok) {
#pragma unroll
            for (int aa = 0; aa < SA; ++aa) {
                const int idx = XA::at(p, (h * SA + aa) * NP + q);
                const V x = lds.ld(idx);
                el += (double)x.x * g[aa][0] + (double)x.y * g[aa][1];
                lds.st(idx, mk<V>((R)g[aa][0], (R)g[aa][1]));
            }
        }
    }
    __syncthreads();
    fft_stages_x<N, 1, NL, NTHR, true, XA>(lds, tw, tid);
    return el;
}

template <typename R, int S>
__device__ __forceinline__ void otf_consts(R *cst, const GParams &G, int tid)
{
    for (int c = tid; c < S * 12; c += NTHR) cst[c] = (R)((c % 12) < 6 ? G.sig6[(c / 12) * 6 + c % 12]
                                                                       : G.eps6[(c / 12) * 6 + c % 12 - 6] *
                                                                             (sizeof(R) == 8 ? G.invmu : 1.0));
}

// x pass, one tile per block.
template <typename R, int N, int S>
__global__ void __launch_bounds__(NTHR) __attribute__((amdgpu_waves_per_eu(otf_waves<R, N, S>(), 8)))
    k_mid_otf(typename cvec<R>::type *__restrict__ T2, GParams G, long long ncol, long long ntot, int bpm,
              const typename cvec<R>::type *__restrict__ tw, double *__restrict__ part_el,
              const int *__restrict__ done)
{
    typedef typename cvec<R>::type V;
    if (*done) return;
    constexpr int NP = mid_pairs<R, N, S>();
    constexpr int NL = S * NP, TOT = NL * N;
    typedef typename XLay<R, N, S>::type XA;
    PFDD_TILE(V, lds, XA::size(N));
    __shared__ R cst[S * 12];
    __shared__ double red[NTHR / 64];
    const int tid = threadIdx.x;
    // member of a batch (bpm blocks per member), first column of the block
    const int mem = blockIdx.x / bpm;
    const long long c0 = (long long)(blockIdx.x - mem * bpm) * NP;
    T2 += (long long)mem * S * ntot;
    otf_consts<R, S>(cst, G, tid);
    tile_load_cols<N, NL, NP, NTHR, XA>(lds, T2, c0, ncol, ntot, tid);
    __syncthreads();
    double v[1] = {otf_tile<R, N, S>(lds, tw, G, cst, c0, ncol, tid)};
#pragma unroll 4
    for (int e = tid; e < TOT; e += NTHR) {
        const int l = e / N, p = e % N;
        const int a = l / NP, q = l % NP;
        if (c0 + q < ncol) st_work(&T2[(long long)a * ntot + (c0 + q) * N + p], lds.ld(XA::at(p, l)), G.keep);
    }
    block_sum_comp<1, NTHR>(v, red, tid);
    if (tid == 0) part_el[blockIdx.x] = v[0];
}

// x pass over the plane layout T[a][i][j][k] of the two-pass iteration
// (pfdd_plane.hip).  Column c = j * nz + k is strided by ny * nz along i and
// the NP columns of a tile are consecutive in k, so each (a, i) of a tile is
// a run of NP elements, often shorter than a 128-byte line.  The other tiles
// of the line are put on the same XCD at about the same time: blocks are
// dispatched to the 8 XCDs round-robin (block b to XCD b % 8), and block b
// takes tile 64 (b / 64) + 8 (b % 8) + (b / 8) % 8, so the 8 consecutive tiles
// 8 r .. 8 r + 7 of a group of 64 run on one XCD and share each line through
// its L2.  The grid is a multiple of 64 blocks; blocks past the last tile
// contribute a zero partial.
template <typename R, int N, int S>
__global__ void __launch_bounds__(NTHR) __attribute__((amdgpu_waves_per_eu(otf_waves<R, N, S>(), 8)))
    k_mid_otf_pl(typename cvec<R>::type *__restrict__ T, GParams G, long long ncol, long long ntot, int bpm,
                 long long ntiles, const typename cvec<R>::type *__restrict__ tw, double *__restrict__ part_el,
                 const int *__restrict__ done)
{
    typedef typename cvec<R>::type V;
    if (*done) return;
    constexpr int NP = mid_pairs<R, N, S>();
    constexpr int NL = S * NP, TOT = NL * N, PER = (TOT + NTHR - 1) / NTHR;
    typedef typename XLay<R, N, S>::type XA;
    PFDD_TILE(V, lds, XA::size(N));
    __shared__ R cst[S * 12];
    __shared__ double red[NTHR / 64];
    const int tid = threadIdx.x;
    const int b = blockIdx.x;
    const long long t = ((long long)(b >> 6) << 6) + ((b & 7) << 3) + ((b >> 3) & 7);
    if (t >= ntiles) {
        if (tid == 0) part_el[b] = 0.0;
        return;
    }
    const int mem = (int)(t / bpm);
    const long long c0 = (t - (long long)mem * bpm) * NP;
    T += (long long)mem * S * ntot;
    otf_consts<R, S>(cst, G, tid);
    // element e of the tile: column q fastest, then position p (= i), then
    // system a; every load of a thread is in flight before its LDS writes.
    // Plain (temporal) accesses: the lines are shared with the other tiles.
    V r[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int e = tid + k * NTHR;
        const int q = e % NP, p = (e / NP) % N, a = e / (NP * N);
        if ((TOT % NTHR == 0 || e < TOT) && c0 + q < ncol) r[k] = T[(long long)a * ntot + (long long)p * ncol + c0 + q];
    }
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int e = tid + k * NTHR;
        const int q = e % NP, p = (e / NP) % N, a = e / (NP * N);
        if (TOT % NTHR == 0 || e < TOT) lds.st(XA::at(p, a * NP + q), r[k]);
    }
    __syncthreads();
    double v[1] = {otf_tile<R, N, S, true>(lds, tw, G, cst, c0, ncol, tid)};
#pragma unroll
    for (int k = 0; k < PER; ++k) {
        const int e = tid + k * NTHR;
        const int q = e % NP, p = (e / NP) % N, a = e / (NP * N);
        if ((TOT % NTHR == 0 || e < TOT) && c0 + q < ncol)
            T[(long long)a * ntot + (long long)p * ncol + c0 + q] = lds.ld(XA::at(p, a * NP + q));
    }
    block_sum_comp<1, NTHR>(v, red, tid);
    if (tid == 0) part_el[b] = v[0];
}

// x pass, persistent and software-pipelined: each block walks the tiles
// t = blockIdx.x, + gridDim.x, ... and keeps the next tile's input in
// registers, loaded while the current tile is transformed, so that memory
// traffic and the FFT/contraction arithmetic of the resident blocks overlap
// instead of running in lock-step phases.  Tile t is member t / bpm, columns
// (t % bpm) * NP ...; part_el gets one partial per block.
template <int N, int NL, int NP, int NTHR, typename V>
__device__ __forceinline__ void cols_fetch(V *r, const V *__restrict__ T2, long long c0, long long ncol,
                                           long long ntot, int tid)
{
    constexpr int TOT = NL * N, PER = (TOT + NTHR - 1) / NTHR;
#pragma unroll
    for (int t = 0; t < PER; ++t) {
        const int e = tid + t * NTHR;
        const int l = e / N, p = e % N;
        const int a = l / NP, q = l % NP;
        if ((TOT % NTHR == 0 || e < TOT) && c0 + q < ncol) r[t] = ld_stream(&T2[(long long)a * ntot + (c0 + q) * N + p]);
    }
}

template <typename R, int N, int S>
__global__ void __launch_bounds__(NTHR)
    k_mid_otf_pipe(typename cvec<R>::type *__restrict__ T2, GParams G, long long ncol, long long ntot, int bpm,
                   int ntiles, const typename cvec<R>::type *__restrict__ tw, double *__restrict__ part_el,
                   const int *__restrict__ done)
{
    typedef typename cvec<R>::type V;
    if (*done) return;
    constexpr int NP = mid_pairs<R, N, S>();
    constexpr int NL = S * NP, TOT = NL * N, PER = (TOT + NTHR - 1) / NTHR;
    typedef typename XLay<R, N, S>::type XA;
    PFDD_TILE(V, lds, XA::size(N));
    __shared__ R cst[S * 12];
    __shared__ double red[NTHR / 64];
    otf_consts<R, S>(cst, G, threadIdx.x);
    int t = blockIdx.x;
    V r[PER];
    {
        const int mem = t / bpm;
        cols_fetch<N, NL, NP, NTHR>(r, T2 + (long long)mem * S * ntot, (long long)(t - mem * bpm) * NP, ncol, ntot,
                                    threadIdx.x);
    }
    double el = 0.0;
    for (; t < ntiles; t += gridDim.x) {
        // the thread index is re-read per tile so that per-element addresses
        // are recomputed rather than held in registers across the loop
        int tid = threadIdx.x;
        __asm__ volatile("" : "+v"(tid));
        const int mem = t / bpm;
        const long long c0 = (long long)(t - mem * bpm) * NP;
        V *T2m = T2 + (long long)mem * S * ntot;
#pragma unroll
        for (int k = 0; k < PER; ++k) {
            const int e = tid + k * NTHR;
            if (TOT % NTHR == 0 || e < TOT) lds.st(XA::at(e % N, e / N), r[k]);
        }
        __syncthreads();
        const int tn = t + gridDim.x;
        if (tn < ntiles) {
            const int mn = tn / bpm;
            cols_fetch<N, NL, NP, NTHR>(r, T2 + (long long)mn * S * ntot, (long long)(tn - mn * bpm) * NP, ncol,
                                        ntot, tid);
        }
        el += otf_tile<R, N, S>(lds, tw, G, cst, c0, ncol, tid);
#pragma unroll 4
        for (int e = tid; e < TOT; e += NTHR) {
            const int l = e / N, p = e % N;
            const int a = l / NP, q = l % NP;
            if (c0 + q < ncol) T2m[(long long)a * ntot + (c0 + q) * N + p] = lds.ld(XA::at(p, l));
        }
        __syncthreads();
    }
    double v[1] = {el};
    block_sum_comp<1, NTHR>(v, red, threadIdx.x);
    if (threadIdx.x == 0) part_el[blockIdx.x] = v[0];
}


// Tile of the register x pass: NP columns of S systems, W = S NP D threads of
// VPT values, 192 threads for 3, 6 and 12 systems (384 for 12 systems of 512
// points) and 128 for 1, 2 and 4.
template <int N, int S> struct XTile {
    static constexpr int VPT = N <= 64 ? 8 : 16, D = N / VPT;
    static constexpr int pairs()
    {
        int np = 1;
        while (2 * np * S * D <= 192) np *= 2;
        return np;
    }
    static constexpr int NP = pairs(), NL = S * NP, W = NL * D;
    static constexpr int PTS = (NP * N + W - 1) / W; // k-points per thread of the contraction
};

// x pass with the transforms in registers (pfdd_reg.hpp): natural ownership,
// position-fastest, straight from memory into the first stage and from the last
// stage back; through LDS go the exchanges between stages and the turn from
// lines to k-points and back (every thread contracts whole k-points): 8 LDS
// accesses per value at 128 and 256 points, 12 with the stages in LDS.  The
// FP64 tile is one plane of doubles (real parts, then imaginary parts), half
// the LDS of k_mid_otf for the same columns.
// Bound by instructions as much as by memory (162 VALU instructions per value at
// 3 systems before the following, 134 after): the constants of the contraction
// come by scalar loads instead of LDS broadcasts, which were a third of all LDS
// accesses; a column's part of f is formed once; P as above.  Measured, us:
// 512 x 512 x 256 x 3 FP64 1613 -> 1410, FP32 893 -> 787; 128^3 x 12 192 -> 182,
// 87 -> 81.
template <typename R, int N, int S>
__global__ void __launch_bounds__((XTile<N, S>::W)) __attribute__((amdgpu_waves_per_eu(sizeof(R) == 8 ? 3 : 4, 8)))
    k_mid_r(typename cvec<R>::type *__restrict__ T2, GParams G, long long ncol, long long ntot, int bpm,
            const typename cvec<R>::type *__restrict__ tw, double *__restrict__ part_el, const int *__restrict__ done)
{
    typedef typename cvec<R>::type V;
    typedef XTile<N, S> X;
    constexpr int NP = X::NP, NL = X::NL, VPT = X::VPT, D = X::D, W = X::W, PTS = X::PTS, NW = (W + 63) / 64;
    typedef RegSwzX<N> L;
    typedef RegNat<N, NL, VPT, true, L> Nat;
    if (*done) return;
    __shared__ __align__(16) char mem[N * NL * RegLds<V>::bytes];
    __shared__ V tws[N];
    __shared__ double red[NW], fcol[3 * NP];
    RegLds<V> lds{(decltype(RegLds<V>::p))mem};
    const int t = threadIdx.x;
    // member of a batch (bpm blocks per member), first column of the block
    const int mem_b = blockIdx.x / bpm;
    const long long c0 = (long long)(blockIdx.x - mem_b * bpm) * NP;
    T2 += (long long)mem_b * S * ntot + c0 * N; // the NP columns of a system are contiguous
    const int l = t / D;                        // line (a, q)
    V *const own = T2 + (long long)(l / NP) * ntot + (l % NP) * N + t % D;
    V v[VPT];
#pragma unroll
    for (int m = 0; m < VPT; ++m) v[m] = ld_stream(own + D * m);
    reg_twiddles<N, W>(tws, tw, t);
    if (t < NP) otf_col(G, c0 + t, fcol + 3 * t);
    reg_fft<N, 1, 1, NL, VPT, false, true, true, true, L>(v, lds, tws, t);
    // lines -> k-points: slot i S + a of a thread is system a of point t + W i
    V x[PTS * S];
    int at[PTS];
    bool ok[PTS];
#pragma unroll
    for (int i = 0; i < PTS; ++i) {
        const int pt = t + W * i;
        ok[i] = (NP * N) % W == 0 || pt < NP * N;
        at[i] = ok[i] ? L::at(pt % N, 0, pt / N) : 0;
    }
    constexpr int AS = NP * N; // from one system to the next
    const Nat nat(t);
    __syncthreads();
    if constexpr (sizeof(V) == 8) {
#pragma unroll
        for (int m = 0; m < VPT; ++m) lds.p[nat(m)] = v[m];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < PTS; ++i)
#pragma unroll
            for (int a = 0; a < S; ++a) x[i * S + a] = lds.p[at[i] + a * AS];
    } else {
#pragma unroll
        for (int m = 0; m < VPT; ++m) lds.p[nat(m)] = v[m].x;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < PTS; ++i)
#pragma unroll
            for (int a = 0; a < S; ++a) x[i * S + a].x = lds.p[at[i] + a * AS];
        __syncthreads();
#pragma unroll
        for (int m = 0; m < VPT; ++m) lds.p[nat(m)] = v[m].y;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < PTS; ++i)
#pragma unroll
            for (int a = 0; a < S; ++a) x[i * S + a].y = lds.p[at[i] + a * AS];
    }
    // the contraction of each point in place; the elastic-energy term
    // Re(conj(xihat_a) ghat_a) is taken as each ghat_a replaces xihat_a
    double el = 0.0;
#pragma unroll
    for (int i = 0; i < PTS; ++i) {
        if (ok[i]) {
            const int pt = t + W * i;
            const KPoint<R> K = otf_freq<R>(G, fcol + 3 * (pt / N), pt % N);
            // the constants come by scalar loads, a few systems' at a time: each
            // group through a pointer of its own
            typedef const R __attribute__((address_space(4))) CR;
            CR *cst = (CR *)G.cst;
            R Pr[6], Pi[6];
#pragma unroll
            for (int b = 0; b < S; ++b) {
                if (b % (sizeof(R) == 8 ? 2 : 3) == 0) __asm__ volatile("" : "+s"(cst));
#pragma unroll
                for (int c = 0; c < 6; ++c) {
                    Pr[c] = b ? ab_c(cst[b * 6 + c], x[i * S + b].x, Pr[c]) : cst[c] * x[i * S].x;
                    Pi[c] = b ? ab_c(cst[b * 6 + c], x[i * S + b].y, Pi[c]) : cst[c] * x[i * S].y;
                }
            }
            if (K.nz) otf_green(Pr, Pi, K);
            else otf_zero(Pr, Pi);
#pragma unroll
            for (int a = 0; a < S; ++a) {
                if (a % (sizeof(R) == 8 ? 2 : 3) == 0) __asm__ volatile("" : "+s"(cst));
                CR *const ep = cst + S * 6 + a * 6;
                R gr = Pr[0] * ep[0], gi = Pi[0] * ep[0];
#pragma unroll
                for (int c = 1; c < 6; ++c) {
                    gr = ab_c(Pr[c], ep[c], gr);
                    gi = ab_c(Pi[c], ep[c], gi);
                }
                if constexpr (sizeof(R) == 4) {
                    gr *= K.invmu;
                    gi *= K.invmu;
                }
                el += (double)x[i * S + a].x * gr + (double)x[i * S + a].y * gi;
                x[i * S + a] = mk<V>(gr, gi);
            }
        }
        // formed here, not sunk past the next branch with every point alive
        __asm__ volatile("" : "+v"(el));
    }
    __syncthreads();
    if constexpr (sizeof(V) == 8) {
#pragma unroll
        for (int i = 0; i < PTS; ++i)
#pragma unroll
            for (int a = 0; a < S; ++a)
                if (ok[i]) lds.p[at[i] + a * AS] = x[i * S + a];
        __syncthreads();
#pragma unroll
        for (int m = 0; m < VPT; ++m) v[m] = lds.p[nat(m)];
    } else {
#pragma unroll
        for (int i = 0; i < PTS; ++i)
#pragma unroll
            for (int a = 0; a < S; ++a)
                if (ok[i]) lds.p[at[i] + a * AS] = x[i * S + a].x;
        __syncthreads();
#pragma unroll
        for (int m = 0; m < VPT; ++m) v[m].x = lds.p[nat(m)];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < PTS; ++i)
#pragma unroll
            for (int a = 0; a < S; ++a)
                if (ok[i]) lds.p[at[i] + a * AS] = x[i * S + a].y;
        __syncthreads();
#pragma unroll
        for (int m = 0; m < VPT; ++m) v[m].y = lds.p[nat(m)];
    }
    int t2 = t;
    __asm__ volatile("" : "+v"(t2)); // addresses formed again, as in k_update_r
    reg_fft<N, 1, 1, NL, VPT, true, true, true, false, L>(v, lds, tws, t2);
#pragma unroll
    for (int m = 0; m < VPT; ++m) st_work(own + D * m, v[m], G.keep);
    double sum[1] = {el};
    block_sum_comp<1, W>(sum, red, t);
    if (t == 0) part_el[blockIdx.x] = sum[0];
}

template <typename R, int S>
int mid_blocks_rt(int n, long long ncol)
{
    // the most blocks of any x-pass kernel of this length: sizes the partials
#define PFDD_CASE(n_)                                                                           \
    if (n == n_) {                                                                              \
        const int nb = (int)((ncol + mid_pairs<R, n_, S>() - 1) / mid_pairs<R, n_, S>());       \
        if constexpr (reg_length<n_>()) {                                                       \
            const int nr = (int)(ncol / XTile<n_, S>::NP);                                      \
            return nb > nr ? nb : nr;                                                           \
        }                                                                                       \
        return nb;                                                                              \
    }
    PFDD_SIZES(PFDD_CASE)
#undef PFDD_CASE
    return 0;
}

template <typename R>
int mid_blocks(int n, int S, long long ncol)
{
    switch (S) {
    case 1: return mid_blocks_rt<R, 1>(n, ncol);
    case 2: return mid_blocks_rt<R, 2>(n, ncol);
    case 3: return mid_blocks_rt<R, 3>(n, ncol);
    case 4: return mid_blocks_rt<R, 4>(n, ncol);
    case 6: return mid_blocks_rt<R, 6>(n, ncol);
    case 12: return mid_blocks_rt<R, 12>(n, ncol);
    }
    return 0;
}

template <typename R, int N, int S> constexpr bool mid_fits()
{
    return (long long)N * (S * mid_pairs<R, N, S>() + 1) * 2 * sizeof(R) <= 61440;
}

template <typename R, int S>
hipError_t launch_mid_s(int n, int M, void *T2, const void *B, long long ncol, long long ntot, const void *tw,
                        double *part_el, const int *done, hipStream_t st, int *nblocks)
{
    typedef typename cvec<R>::type V;
#define PFDD_CASE(n_)                                                                             \
    if (n == n_) {                                                                                \
        if constexpr (mid_fits<R, n_, S>()) {                                                     \
            constexpr int NP = mid_pairs<R, n_, S>();                                             \
            const int bpm = (int)((ncol + NP - 1) / NP);                                          \
            *nblocks = M * bpm;                                                                   \
            PFDD_LAUNCH((k_mid<R, R, n_, S>), dim3((unsigned)(M * bpm)), dim3(NTHR), st,          \
                               (V *)T2, (const R *)B, ncol, ntot, bpm, (const V *)tw, part_el, done); \
            return hipGetLastError();                                                             \
        } else {                                                                                  \
            return hipErrorInvalidValue;                                                          \
        }                                                                                         \
    }
    PFDD_SIZES(PFDD_CASE)
#undef PFDD_CASE
    return hipErrorInvalidValue;
}

template <typename R>
bool mid_supported(int n, int S)
{
    auto chk = [&](auto sconst) -> bool {
        constexpr int SS = decltype(sconst)::value;
#define PFDD_CASE(n_) if (n == n_) return mid_fits<R, n_, SS>();
        PFDD_SIZES(PFDD_CASE)
#undef PFDD_CASE
        return false;
    };
    switch (S) {
    case 1: return chk(std::integral_constant<int, 1>());
    case 2: return chk(std::integral_constant<int, 2>());
    case 3: return chk(std::integral_constant<int, 3>());
    case 4: return chk(std::integral_constant<int, 4>());
    case 6: return chk(std::integral_constant<int, 6>());
    case 12: return chk(std::integral_constant<int, 12>());
    }
    return false;
}

template <typename R>
hipError_t launch_mid(int n, int S, int M, void *T2, const void *B, long long ncol, long long ntot, const void *tw,
                      double *part_el, const int *done, hipStream_t st, int *nblocks)
{
    switch (S) {
    case 1: return launch_mid_s<R, 1>(n, M, T2, B, ncol, ntot, tw, part_el, done, st, nblocks);
    case 2: return launch_mid_s<R, 2>(n, M, T2, B, ncol, ntot, tw, part_el, done, st, nblocks);
    case 3: return launch_mid_s<R, 3>(n, M, T2, B, ncol, ntot, tw, part_el, done, st, nblocks);
    case 4: return launch_mid_s<R, 4>(n, M, T2, B, ncol, ntot, tw, part_el, done, st, nblocks);
    case 6: return launch_mid_s<R, 6>(n, M, T2, B, ncol, ntot, tw, part_el, done, st, nblocks);
    case 12: return launch_mid_s<R, 12>(n, M, T2, B, ncol, ntot, tw, part_el, done, st, nblocks);
    }
    return hipErrorInvalidValue;
}

template <typename R, int S>
hipError_t launch_mid_otf_s(int n, int M, void *T2, const GParams &G, long long ncol, long long ntot,
                            const void *tw, double *part_el, const int *done, hipStream_t st, int pipe, int ncu,
                            int *nblocks)
{
    typedef typename cvec<R>::type V;
#define PFDD_CASE(n_)                                                                             \
    if (n == n_) {                                                                                \
        if constexpr (mid_fits<R, n_, S>() && reg_length<n_>()) {                                 \
            typedef XTile<n_, S> X;                                                               \
            if (ncol % X::NP) return hipErrorInvalidValue;                                        \
            const int bpm = (int)(ncol / X::NP);                                                  \
            *nblocks = M * bpm;                                                                   \
            PFDD_LAUNCH((k_mid_r<R, n_, S>), dim3((unsigned)*nblocks), dim3(X::W), st, (V *)T2, G, \
                        ncol, ntot, bpm, (const V *)tw, part_el, done);                           \
            return hipGetLastError();                                                             \
        } else if constexpr (mid_fits<R, n_, S>()) {                                              \
            constexpr int NP = mid_pairs<R, n_, S>();                                             \
            const int bpm = (int)((ncol + NP - 1) / NP);                                          \
            if (!pipe) {                                                                          \
                *nblocks = M * bpm;                                                               \
                PFDD_LAUNCH((k_mid_otf<R, n_, S>), dim3((unsigned)(M * bpm)), dim3(NTHR), st,      \
                            (V *)T2, G, ncol, ntot, bpm, (const V *)tw, part_el, done);           \
            } else {                                                                              \
                /* as many blocks as fit on the device at once */                                 \
                static const int occ = [] {                                                       \
                    int o = 0;                                                                    \
                    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(                             \
                            &o, (const void *)k_mid_otf_pipe<R, n_, S>, NTHR, 0) != hipSuccess)   \
                        o = 1;                                                                    \
                    return o > 0 ? o : 1;                                                         \
                }();                                                                              \
                const long long nt = (long long)M * bpm, cap = (long long)ncu * occ;             \
                *nblocks = (int)(nt < cap ? nt : cap);                                            \
                PFDD_LAUNCH((k_mid_otf_pipe<R, n_, S>), dim3((unsigned)*nblocks), dim3(NTHR), st,  \
                            (V *)T2, G, ncol, ntot, bpm, (int)nt, (const V *)tw, part_el, done);  \
            }                                                                                     \
            return hipGetLastError();                                                             \
        } else {                                                                                  \
            return hipErrorInvalidValue;                                                          \
        }                                                                                         \
    }
    PFDD_SIZES(PFDD_CASE)
#undef PFDD_CASE
    return hipErrorInvalidValue;
}

template <typename R>
hipError_t launch_mid_otf(int n, int S, int M, void *T2, const GParams &G, long long ncol, long long ntot,
                          const void *tw, double *part_el, const int *done, hipStream_t st, int pipe, int ncu,
                          int *nblocks)
{
    switch (S) {
    case 1: return launch_mid_otf_s<R, 1>(n, M, T2, G, ncol, ntot, tw, part_el, done, st, pipe, ncu, nblocks);
    case 2: return launch_mid_otf_s<R, 2>(n, M, T2, G, ncol, ntot, tw, part_el, done, st, pipe, ncu, nblocks);
    case 3: return launch_mid_otf_s<R, 3>(n, M, T2, G, ncol, ntot, tw, part_el, done, st, pipe, ncu, nblocks);
    case 4: return launch_mid_otf_s<R, 4>(n, M, T2, G, ncol, ntot, tw, part_el, done, st, pipe, ncu, nblocks);
    case 6: return launch_mid_otf_s<R, 6>(n, M, T2, G, ncol, ntot, tw, part_el, done, st, pipe, ncu, nblocks);
    case 12: return launch_mid_otf_s<R, 12>(n, M, T2, G, ncol, ntot, tw, part_el, done, st, pipe, ncu, nblocks);
    }
    return hipErrorInvalidValue;
}


// x pass of the plane layout: the grid sizes of the plane iteration.
#define PFDD_PL_SIZES(X) X(16) X(32) X(48) X(64) X(80) X(96) X(128)

template <typename R, int S>
hipError_t launch_mid_pl_s(int n, int M, void *T, const GParams &G, long long ncol, long long ntot, const void *tw,
                           double *part_el, const int *done, hipStream_t st, int *nblocks)
{
    typedef typename cvec<R>::type V;
#define PFDD_CASE(n_)                                                                                  \
    if (n == n_) {                                                                                     \
        if constexpr (mid_fits<R, n_, S>()) {                                                          \
            constexpr int NP = mid_pairs<R, n_, S>();                                                  \
            const int bpm = (int)((ncol + NP - 1) / NP);                                               \
            const long long nt = (long long)M * bpm;                                                   \
            *nblocks = (int)((nt + 63) / 64 * 64);                                                     \
            PFDD_LAUNCH((k_mid_otf_pl<R, n_, S>), dim3((unsigned)*nblocks), dim3(NTHR), st, (V *)T, G,  \
                        ncol, ntot, bpm, nt, (const V *)tw, part_el, done);                            \
            return hipGetLastError();                                                                  \
        }                                                                                              \
        return hipErrorInvalidValue;                                                                   \
    }
    PFDD_PL_SIZES(PFDD_CASE)
#undef PFDD_CASE
    return hipErrorInvalidValue;
}

template <typename R>
hipError_t launch_mid_pl(int n, int S, int M, void *T, const GParams &G, long long ncol, long long ntot,
                         const void *tw, double *part_el, const int *done, hipStream_t st, int *nblocks)
{
    switch (S) {
    case 1: return launch_mid_pl_s<R, 1>(n, M, T, G, ncol, ntot, tw, part_el, done, st, nblocks);
    case 2: return launch_mid_pl_s<R, 2>(n, M, T, G, ncol, ntot, tw, part_el, done, st, nblocks);
    case 3: return launch_mid_pl_s<R, 3>(n, M, T, G, ncol, ntot, tw, part_el, done, st, nblocks);
    case 4: return launch_mid_pl_s<R, 4>(n, M, T, G, ncol, ntot, tw, part_el, done, st, nblocks);
    case 6: return launch_mid_pl_s<R, 6>(n, M, T, G, ncol, ntot, tw, part_el, done, st, nblocks);
    case 12: return launch_mid_pl_s<R, 12>(n, M, T, G, ncol, ntot, tw, part_el, done, st, nblocks);
    }
    return hipErrorInvalidValue;
}

// Blocks of the plane-layout x pass (a multiple of 64), 0 if unsupported.
template <typename R>
int mid_pl_blocks(int n, int S, int M, long long ncol)
{
    bool ok = false;
#define PFDD_CASE(n_) if (n == n_) ok = true;
    PFDD_PL_SIZES(PFDD_CASE)
#undef PFDD_CASE
    if (!ok || !mid_supported<R>(n, S)) return 0;
    const long long nt = (long long)M * mid_blocks<R>(n, S, ncol);
    return (int)((nt + 63) / 64 * 64);
}

#define PFDD_INST(R)                                                                                              \
    template int mid_blocks<R>(int, int, long long);                                                              \
    template bool mid_supported<R>(int, int);                                                                     \
    template hipError_t launch_mid<R>(int, int, int, void *, const void *, long long, long long, const void *,     \
                                      double *, const int *, hipStream_t, int *);                                        \
    template hipError_t launch_mid_otf<R>(int, int, int, void *, const GParams &, long long, long long,            \
                                          const void *, double *, const int *, hipStream_t, int, int, int *);      \
    template hipError_t launch_mid_pl<R>(int, int, int, void *, const GParams &, long long, long long,             \
                                         const void *, double *, const int *, hipStream_t, int *);                  \
    template int mid_pl_blocks<R>(int, int, int, long long);
PFDD_INST(double)
PFDD_INST(float)
#undef PFDD_INST

} // namespace pfdd
