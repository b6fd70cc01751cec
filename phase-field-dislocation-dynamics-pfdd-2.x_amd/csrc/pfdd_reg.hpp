// pfdd_reg.hpp -- line transforms held in registers.
//
// A block of W threads transforms a tile of NL lines of N points; every thread
// holds VPT values of one line, W = NL * N / VPT.  In its natural ownership
// thread (l, p0), p0 < D = N / VPT, holds the positions p0 + D m, m < VPT, of
// line l.  These are the inputs of VPT / RAD butterflies of any radix RAD that
// divides VPT, of a first stage as of a last one (a last stage's outputs
// j + r N / RAD are its inputs' positions), so that
//
//   * the first stage reads its inputs straight from memory and the last one
//     writes its outputs straight to memory: only the exchanges between stages
//     go through LDS (128 = 16 x 8: one exchange, 2 LDS accesses per value,
//     where stages that work in place in LDS take 6);
//   * an inverse transform's results can be updated in place and transformed
//     forward again without leaving the registers.
//
// The mapping of threads to (l, p0) is line-fastest or position-fastest and
// may change at an exchange: a wave reads and writes runs of consecutive lines
// on an axis where lines are neighbours in memory, and runs of consecutive
// positions where the line is contiguous.
//
// Stages, radix order, twiddles and butterflies are those of fft_stages
// (plan 0) and fft_stages_x (plan 1) of pfdd_fft.hpp, so a line transformed
// here is bit for bit the line transformed there.
#pragma once
#include "pfdd_kern.hpp"

namespace pfdd {

template <int PL> constexpr int plan_radix(int m) { return PL == 1 ? pick_radix_x(m) : pick_radix(m); }

// Exchange tile of NL lines: value (p, l) at an address whose low four bits
// (the 8-byte slot within 128 bytes of LDS, which serves 16 lanes at a time)
// are a linear function of the bits of p and l.  It has full rank on these
// groups of 16 lanes: 16 lines of a row, 16 consecutive positions of a line, 8
// consecutive positions of two lines; there are no conflicts there and no
// padding.  It has not on the first exchange of a transform that starts
// position-fastest, as the one after an update does: neighbouring lanes write
// rows RAD apart, f knows two values on multiples of 8, and 8 lanes share a slot
// (16 where RAD is 16 and a line has 16 threads, at 256 points).  Counted at 128^3
// x 12: 2.25e7 (FP64) and 1.1e7 (FP32) conflict cycles a launch of the update
// with that transform, 4.9e5 and 0 without; the forward line passes 0, the
// inverse ones 1.6e6 and 7.9e5.  The position comes as pv | ps with disjoint
// bits, ps known at compile time: the ps part folds into constants.
template <int NL> struct RegSwz {
    static_assert(NL % 16 == 0, "tiles of a multiple of 16 lines");
    __device__ __forceinline__ static constexpr int f(int p) { return ((p & 7) << 1) | ((p >> 3) & 1); }
    __device__ __forceinline__ static int at(int pv, int ps, int l)
    {
        return pv * NL + ((l ^ f(pv)) ^ f(ps)) + ps * NL;
    }
};

// Exchange tile of the x pass, whose lines are all contiguous: line by line,
// the low four bits of the position XORed so that 16 lanes of any of its
// accesses (consecutive positions of one line, or of neighbouring lines where
// a line has fewer than 16 threads; stage outputs RAD apart) hit 16 slots.
template <int N> struct RegSwzX {
    __device__ __forceinline__ static constexpr int f(int p) // of position bits 4 and up
    {
        const int p4 = (p >> 4) & 1, p5 = (p >> 5) & 1, p6 = (p >> 6) & 1, p7 = (p >> 7) & 1;
        if constexpr (N >= 256) return p4 | (p5 << 1) | (p6 * 12) ^ (p7 << 2);
        else return p4 | (p5 << 1) | (p6 << 2);
    }
    __device__ __forceinline__ static constexpr int g(int l) // of the line
    {
        if constexpr (N >= 256) return 0;
        else if constexpr (N == 128) return (l & 1) << 3;
        else if constexpr (N == 64) return (l & 1) * 12;
        else return ((l & 1) << 2) | ((l & 2) * 5); // N == 32: bit 0 -> 4, bit 1 -> 8 + 2
    }
    __device__ __forceinline__ static int at(int pv, int ps, int l)
    {
        return l * N + (((pv ^ f(pv)) ^ g(l)) ^ ((ps & 15) ^ f(ps))) + (ps & ~15);
    }
};

// Position written by butterfly j = p0 + D q, output r, of a stage (NS, RAD):
// (j / NS) NS RAD + j % NS + r NS, split into its thread part and its static
// part (NS, D powers of two).
template <int D, int NS, int RAD> struct RegWr {
    __device__ __forceinline__ static int pv(int p0)
    {
        if constexpr (NS <= D) return (p0 / NS) * (NS * RAD) + p0 % NS;
        else return p0;
    }
    __device__ __forceinline__ static constexpr int ps(int q, int r)
    {
        if constexpr (NS <= D) return D * RAD * q + r * NS;
        else return (q / (NS / D)) * (NS * RAD) + D * (q % (NS / D)) + r * NS;
    }
};

// LDS of an exchange: FP32 values interleaved (8-byte accesses); FP64 values
// one component at a time through a single plane of doubles, the real parts
// first: as many LDS accesses as with two planes (each is 8 bytes wide), half
// the LDS, two more barriers (none in one-wave blocks).
template <typename V> struct RegLds;
template <> struct RegLds<float2> {
    static constexpr int bytes = 8;
    float2 *p;
};
template <> struct RegLds<double2> {
    static constexpr int bytes = 8;
    double *p;
};

// All values of the block through LDS: slot m goes to address wr(m) and comes
// back from address rd(m).  FIRST: nothing of the tile's LDS is being read.
template <int VPT, bool FIRST, typename V, typename WrA, typename RdA>
__device__ __forceinline__ void reg_shuffle(V (&v)[VPT], RegLds<V> lds, WrA wr, RdA rd)
{
    if constexpr (!FIRST) __syncthreads(); // the last exchange's reads are done
    if constexpr (sizeof(V) == 8) {
#pragma unroll
        for (int m = 0; m < VPT; ++m) lds.p[wr(m)] = v[m];
        __syncthreads();
#pragma unroll
        for (int m = 0; m < VPT; ++m) v[m] = lds.p[rd(m)];
    } else {
#pragma unroll
        for (int m = 0; m < VPT; ++m) lds.p[wr(m)] = v[m].x;
        __syncthreads();
#pragma unroll
        for (int m = 0; m < VPT; ++m) v[m].x = lds.p[rd(m)];
        __syncthreads();
#pragma unroll
        for (int m = 0; m < VPT; ++m) lds.p[wr(m)] = v[m].y;
        __syncthreads();
#pragma unroll
        for (int m = 0; m < VPT; ++m) v[m].y = lds.p[rd(m)];
    }
}

// LDS address of slot m in natural ownership; S the tile's layout.
template <int N, int NL, int VPT, bool PF, typename S = RegSwz<NL>> struct RegNat {
    static constexpr int D = N / VPT;
    int l, p0;
    __device__ __forceinline__ RegNat(int t) : l(PF ? t / D : t % NL), p0(PF ? t % D : t / NL) {}
    __device__ __forceinline__ int operator()(int m) const { return S::at(p0, D * m, l); }
};
// ... after stage (NS, RAD): slot q + NB r holds output r of butterfly q.
template <int NS, int RAD, int N, int NL, int VPT, bool PF, typename S = RegSwz<NL>> struct RegOut {
    static constexpr int D = N / VPT, NB = VPT / RAD;
    int l, pv;
    __device__ __forceinline__ RegOut(int t)
        : l(PF ? t / D : t % NL), pv(RegWr<D, NS, RAD>::pv(PF ? t % D : t / NL))
    {
    }
    __device__ __forceinline__ int operator()(int m) const
    {
        return S::at(pv, RegWr<D, NS, RAD>::ps(m % NB, m / NB), l);
    }
};
// ... in linear ownership: slot m holds element t + W m of the tile's NL lines
// in memory order (line by line), so that a wave reads or writes runs of 64
// positions of contiguous lines.
template <int N, int NL, int VPT> struct RegLin {
    static constexpr int W = NL * N / VPT;
    int t;
    __device__ __forceinline__ RegLin(int t_) : t(t_) {}
    __device__ __forceinline__ static int line(int t, int m)
    {
        if constexpr (W >= N) return t / N + (W / N) * m;
        else return m / (N / W);
    }
    __device__ __forceinline__ static int pos_s(int m) // the static part of the position; the rest is t % min(N, W)
    {
        if constexpr (W >= N) return 0;
        else return W * (m % (N / W));
    }
    __device__ __forceinline__ int operator()(int m) const
    {
        return RegSwz<NL>::at(t % (W < N ? W : N), pos_s(m), line(t, m));
    }
};

// The transform of a tile from its natural ownership with mapping PFI
// (position-fastest or not) to that with mapping PFO.  tws: twiddles of N in
// LDS, complete before the first exchange's barrier.  FIRST: nothing of the
// tile's LDS is still being read.
template <int N, int NS, int PL, int NL, int VPT, bool INV, bool PFI, bool PFO, bool FIRST,
          typename S = RegSwz<NL>, typename V>
__device__ __forceinline__ void reg_fft(V (&v)[VPT], RegLds<V> lds, const V *tws, int t)
{
    constexpr int RAD = plan_radix<PL>(N / NS), NB = VPT / RAD, D = N / VPT;
    static_assert(VPT % RAD == 0, "a thread holds whole butterflies");
    const int p0 = PFI ? t % D : t / NL;
#pragma unroll
    for (int q = 0; q < NB; ++q) {
        V x[RAD];
#pragma unroll
        for (int r = 0; r < RAD; ++r) x[r] = v[q + NB * r];
        if constexpr (NS > 1) {
            const int k = NS <= D ? p0 % NS : p0 + D * (q % (NS > D ? NS / D : 1));
#pragma unroll
            for (int r = 1; r < RAD; ++r) x[r] = cmulw<INV>(x[r], tws[r * k * (N / (NS * RAD))]);
        }
        dft<RAD, INV>(x);
#pragma unroll
        for (int r = 0; r < RAD; ++r) v[q + NB * r] = x[r];
    }
    if constexpr (NS * RAD < N) {
        reg_shuffle<VPT, FIRST>(v, lds, RegOut<NS, RAD, N, NL, VPT, PFI, S>(t), RegNat<N, NL, VPT, PFO, S>(t));
        reg_fft<N, NS * RAD, PL, NL, VPT, INV, PFO, PFO, false, S>(v, lds, tws, t);
    }
}

// Twiddles of length N into LDS (complete at the block's next barrier).
template <int N, int W, typename V>
__device__ __forceinline__ void reg_twiddles(V *tws, const V *__restrict__ tw, int t)
{
#pragma unroll
    for (int m = 0; m < (N + W - 1) / W; ++m)
        if (N % W == 0 || t + m * W < N) tws[t + m * W] = tw[t + m * W];
}

// Values per thread and lines per tile of the line passes and the update: 256
// bytes of neighbouring lines (16 FP64, 32 FP32 lines), and the 128 bytes of 16
// FP32 lines from 256 points up: exchange tiles of 4 to 32 KB, and of 64 KB at 512
// points.  Half of that
// cost the FP64 update at 512 x 512 x 256 x 3 2317 -> 2545 us; twice the LDS
// cost the FP32 one 1245 -> 1459 us.
template <typename R, int N> struct RegTile {
    static constexpr int VPT = N <= 64 ? 8 : 16;
    static constexpr int NL = sizeof(R) == 8 ? 16 : (N >= 256 ? 16 : 32);
    static constexpr int D = N / VPT, W = NL * D;
};

} // namespace pfdd
