// pfdd_pass.hip -- the line-pass kernel (FFT along one axis of every line of
// a batch, transposed write through LDS) and its launcher.
#include "pfdd_kern.hpp"
#include "pfdd_reg.hpp"

namespace pfdd {

// ------------------------------------------------- generic FFT pass (1, 2, 4)
// TQ: tile shape (tile_lines_q); PL: radix plan (0 radix 8 first, 1 radix 16
// where it saves a stage).
template <typename R, int N, bool INV, int TQ, int PL>
__global__ void __launch_bounds__(NTHR)
    k_fft_pass(const typename cvec<R>::type *__restrict__ in, typename cvec<R>::type *__restrict__ out,
               LineMap mi, LineMap mo, long long nlines, const typename cvec<R>::type *__restrict__ tw,
               const int *__restrict__ done, const uint8_t *__restrict__ zmask, Order order)
{
    typedef typename cvec<R>::type V;
    if (*done) return;
    constexpr int NL = tile_lines_q<R, N, TQ>(), LDP = NL + 1, TOT = N * NL;
    PFDD_TILE(V, lds, N * LDP);
    __shared__ long long bin[NL], bout[NL];
    const int tid = threadIdx.x;
    const long long L0 = (long long)(order.rev ? gridDim.x - 1 - blockIdx.x : blockIdx.x) * NL;
    for (int l = tid; l < NL; l += NTHR) {
        const long long L = L0 + l;
        const bool ok = L < nlines;
        bin[l] = ok ? line_base(mi, L) : -1;
        bout[l] = ok ? line_base(mo, L) : -1;
    }
    __syncthreads();
    tile_load<N, NL, NTHR>(lds, in, bin, mi.SP, tid);
    __syncthreads();
    if (zmask) {
        // input elements whose zmask byte is set enter the transform as 0
        for (int e = tid; e < TOT; e += NTHR) {
            const int l = e / N, p = e % N;
            const long long b = bin[l];
            if (b >= 0 && zmask[b + p * mi.SP]) lds.st(p * LDP + l, mk<V>((R)0, (R)0));
        }
        __syncthreads();
    }
    if constexpr (PL == 1) fft_stages_x<N, 1, NL, NTHR, INV>(lds, tw, tid);
    else fft_stages<N, 1, NL, NTHR, INV>(lds, tw, tid);
    tile_store<N, NL, NTHR>(out, lds, bout, mo.SP, tid, order.keep);
}


// The same pass with the transform in registers (pfdd_reg.hpp), for the
// lengths that have it.  CI, CO: the input / output lines are contiguous in
// memory; otherwise neighbouring lines are (line-fastest natural ownership).
// Contiguous lines are read and written in linear ownership, at the price of
// one more exchange: in natural ownership a wave's accesses are pieces of 128
// bytes of 8 lines, and the FP64 forward passes at 128^3 x 12 took 145 us
// against 129-135 with whole runs.
//
// Offsets within a tile are 32-bit byte offsets from the block's first line
// group: they stay below twice a system's bytes where the tile crosses into
// the next system and below one system's otherwise, and tiles cross only on
// grids whose line count is no multiple of the tile's, far below 4 GiB.
struct RegBase {
    unsigned D, B, sa, sb, sd, d0, ob;
    long long ref; // element index of (first line group, line 0)
    __device__ __forceinline__ RegBase(const LineMap &m, unsigned L0)
        : D((unsigned)m.D), B((unsigned)m.B), sa((unsigned)m.SA), sb((unsigned)m.SB), sd((unsigned)m.SD)
    {
        const unsigned t0 = L0 / D, oa = t0 / B;
        d0 = L0 - t0 * D;
        ob = t0 - oa * B;
        ref = oa * m.SA + ob * m.SB;
    }
    // elements from ref to the start of the tile's line l
    __device__ __forceinline__ unsigned line(unsigned l) const
    {
        const unsigned dl = d0 + l, tl = dl / D, bl = ob + tl, al = bl / B;
        return al * sa + (bl - al * B) * sb - ob * sb + (dl - tl * D) * sd;
    }
};

template <typename R, int N, int PL, bool INV, bool CI, bool CO>
__global__ void __launch_bounds__((RegTile<R, N>::W))
    k_pass_r(const typename cvec<R>::type *__restrict__ in, typename cvec<R>::type *__restrict__ out, LineMap mi,
             LineMap mo, const typename cvec<R>::type *__restrict__ tw, const int *__restrict__ done,
             const uint8_t *__restrict__ zmask, Order order)
{
    typedef typename cvec<R>::type V;
    typedef RegTile<R, N> G;
    constexpr int NL = G::NL, VPT = G::VPT, D = G::D, W = G::W;
    typedef RegLin<N, NL, VPT> Lin;
    if (*done) return;
    __shared__ __align__(16) char mem[N * NL * RegLds<V>::bytes];
    __shared__ V tws[N];
    // starts of the tile's lines where a thread's linear elements span several
    __shared__ unsigned li[CI ? NL : 1], lo[CO ? NL : 1];
    RegLds<V> lds{(decltype(RegLds<V>::p))mem};
    const int t = threadIdx.x;
    const unsigned L0 = (order.rev ? gridDim.x - 1 - blockIdx.x : blockIdx.x) * NL;
    const RegBase bi(mi, L0), bo(mo, L0);
    constexpr int PW = W < N ? W : N; // positions that W threads cover in linear ownership
    if constexpr (CI || CO) {
        if (t < NL) {
            if constexpr (CI) li[t] = bi.line(t);
            if constexpr (CO) lo[t] = bo.line(t);
        }
        __syncthreads();
    }
    V v[VPT];
    if constexpr (CI) {
#pragma unroll
        for (int m = 0; m < VPT; ++m) {
            const unsigned e = li[Lin::line(t, m)] + Lin::pos_s(m) + t % PW;
            v[m] = ld_stream((const V *)((const char *)(in + bi.ref) + e * (unsigned)sizeof(V)));
            if (zmask && (zmask + bi.ref)[e]) v[m] = mk<V>((R)0, (R)0); // masked elements enter as 0
        }
    } else {
        const unsigned e = bi.line(t % NL) + (t / NL) * (unsigned)mi.SP;
#pragma unroll
        for (int m = 0; m < VPT; ++m)
            v[m] = ld_stream((const V *)((const char *)(in + bi.ref + D * m * mi.SP) + e * (unsigned)sizeof(V)));
    }
    reg_twiddles<N, W>(tws, tw, t);
    if constexpr (CI) reg_shuffle<VPT, true>(v, lds, Lin(t), RegNat<N, NL, VPT, false>(t));
    reg_fft<N, 1, PL, NL, VPT, INV, false, false, !CI>(v, lds, tws, t);
    if constexpr (CO) {
        reg_shuffle<VPT, false>(v, lds, RegNat<N, NL, VPT, false>(t), Lin(t));
#pragma unroll
        for (int m = 0; m < VPT; ++m) {
            const unsigned e = lo[Lin::line(t, m)] + Lin::pos_s(m) + t % PW;
            st_work((V *)((char *)(out + bo.ref) + e * (unsigned)sizeof(V)), v[m], order.keep);
        }
    } else {
        const unsigned e = bo.line(t % NL) + (t / NL) * (unsigned)mo.SP;
#pragma unroll
        for (int m = 0; m < VPT; ++m)
            st_work((V *)((char *)(out + bo.ref + D * m * mo.SP) + e * (unsigned)sizeof(V)), v[m], order.keep);
    }
}

template <typename R, bool INV>
hipError_t launch_pass(int n, const void *in, void *out, LineMap mi, LineMap mo, long long nlines,
                       const void *tw, const int *done, hipStream_t st, const uint8_t *zmask,
                       int tq, Order order)
{
    typedef typename cvec<R>::type V;
    // tq = shape + 3 * plan; plan 1 falls back to plan 0 where they coincide
    const int shape = tq % 3, plan = tq / 3;
#define PFDD_PASS_R(PL_, PFI_, PFO_)                                                                \
    PFDD_LAUNCH((k_pass_r<R, N, (PL_ && radix16_plan_differs<N>()), INV, PFI_, PFO_>),              \
                dim3((unsigned)(nlines / RegTile<R, N>::NL)), dim3(RegTile<R, N>::W), st,           \
                (const V *)in, (V *)out, mi, mo, (const V *)tw, done, zmask, order)
#define PFDD_CASE(n_)                                                                               \
    if (n == n_) {                                                                                  \
        constexpr int N = n_;                                                                       \
        if constexpr (reg_length<N>()) {                                                            \
            /* forward passes go from contiguous lines to neighbouring ones, inverse passes */      \
            /* back; x lines are contiguous on both sides */                                        \
            const bool pfi = mi.SP == 1, pfo = mo.SP == 1, p1 = plan == 1 && radix16_plan_differs<N>(); \
            if (nlines % RegTile<R, N>::NL || !(pfi && pfo) && pfi != !INV || !pfi && !pfo)         \
                return hipErrorInvalidValue;                                                        \
            if (pfi && pfo) { if (p1) PFDD_PASS_R(1, true, true); else PFDD_PASS_R(0, true, true); } \
            else { if (p1) PFDD_PASS_R(1, !INV, INV); else PFDD_PASS_R(0, !INV, INV); }             \
            return hipGetLastError();                                                               \
        } else {                                                                                    \
        PFDD_TQ_DISPATCH(shape, {                                                                   \
            constexpr int NL = tile_lines_q<R, n_, TQ>();                                           \
            const unsigned nb = (unsigned)((nlines + NL - 1) / NL);                                 \
            if (plan == 1 && radix16_plan_differs<n_>())                                            \
                PFDD_LAUNCH((k_fft_pass<R, n_, INV, TQ, radix16_plan_differs<n_>() ? 1 : 0>),      \
                            dim3(nb), dim3(NTHR), st, (const V *)in, (V *)out, mi, mo, nlines,      \
                            (const V *)tw, done, zmask, order);                                       \
            else                                                                                    \
                PFDD_LAUNCH((k_fft_pass<R, n_, INV, TQ, 0>), dim3(nb), dim3(NTHR), st,              \
                            (const V *)in, (V *)out, mi, mo, nlines, (const V *)tw, done, zmask, order); \
        })                                                                                          \
        return hipGetLastError();                                                                   \
        }                                                                                           \
    }
    PFDD_SIZES(PFDD_CASE)
#undef PFDD_CASE
#undef PFDD_PASS_R
    return hipErrorInvalidValue;
}

template hipError_t launch_pass<double, false>(int, const void *, void *, LineMap, LineMap, long long, const void *,
                                               const int *, hipStream_t, const uint8_t *, int, Order);
template hipError_t launch_pass<double, true>(int, const void *, void *, LineMap, LineMap, long long, const void *,
                                              const int *, hipStream_t, const uint8_t *, int, Order);
template hipError_t launch_pass<float, false>(int, const void *, void *, LineMap, LineMap, long long, const void *,
                                              const int *, hipStream_t, const uint8_t *, int, Order);
template hipError_t launch_pass<float, true>(int, const void *, void *, LineMap, LineMap, long long, const void *,
                                             const int *, hipStream_t, const uint8_t *, int, Order);

} // namespace pfdd
