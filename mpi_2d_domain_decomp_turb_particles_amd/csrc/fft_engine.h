// fft_engine.h -- batched complex FFT of TC columns held in LDS, for gfx950.
//
// A tile holds TC independent columns of N complex points, point-major
// (lds[n * LDR + c], LDR >= TC; an odd LDR avoids bank conflicts).  All NT threads
// of the work-group run a self-sorting Stockham FFT through the radix plan of N:
// each pass loads R points per work item from LDS into registers, applies the
// twiddles, runs a radix-R butterfly in registers and writes the R outputs back in
// Stockham order.  Output is in natural order; transforms are unnormalised with
// forward sign -1, inverse +1.  Twiddles come from a table tw[m] = exp(-2 pi i m/N).
#pragma once
#include "ddns_internal.h"

namespace ddns {

// ---------------------------------------------------------------- tile transfers
// A tile is R rows of W adjacent complex values in HBM (row r at src + r * rstride)
// and R * LDR values in LDS (row-major, or transposed when TRANS: lds[c * LDR + r]).
// Every lane moves 16 bytes per access and the trip count is a compile-time
// constant, so a lane issues all of its loads before the first wait.
template <typename C> struct vec16;
template <> struct vec16<float2> {
    using V = float4;
    static constexpr int VW = 2;
    __device__ static void split(const V& v, float2* o) { o[0] = make_float2(v.x, v.y); o[1] = make_float2(v.z, v.w); }
};
template <> struct vec16<double2> {
    using V = double2;
    static constexpr int VW = 1;
    __device__ static void split(const V& v, double2* o) { o[0] = v; }
};

// the registers one lane holds for a tile in flight
template <typename C, int R, int W, int NT>
struct TileRegs {
    using VT = vec16<C>;
    static constexpr int VW = VT::VW, PER_ROW = W / VW, TOT = R * PER_ROW, Q = TOT / NT;
    static_assert(W % VW == 0 && TOT % NT == 0, "tile must split evenly over the work-group");
    typename VT::V v[Q];
};

// issue the loads of a tile into registers (returns without waiting)
template <typename C, int R, int W, int NT>
__device__ __forceinline__ void tile_fetch(TileRegs<C, R, W, NT>& t, const C* __restrict__ src, size_t rstride, int tid)
{
    using TR = TileRegs<C, R, W, NT>;
#pragma unroll
    for (int q = 0; q < TR::Q; ++q) {
        const int e = tid + q * NT, r = e / TR::PER_ROW, c = (e % TR::PER_ROW) * TR::VW;
        t.v[q] = *(const typename TR::VT::V*)(src + (size_t)r * rstride + c);
    }
}

// write a fetched tile to LDS
template <typename C, int R, int W, int LDR, int NT, bool TRANS = false>
__device__ __forceinline__ void tile_put(C* __restrict__ lds, const TileRegs<C, R, W, NT>& t, int tid)
{
    using TR = TileRegs<C, R, W, NT>;
#pragma unroll
    for (int q = 0; q < TR::Q; ++q) {
        const int e = tid + q * NT, r = e / TR::PER_ROW, c = (e % TR::PER_ROW) * TR::VW;
        C v[TR::VW];
        TR::VT::split(t.v[q], v);
#pragma unroll
        for (int k = 0; k < TR::VW; ++k) lds[TRANS ? (c + k) * LDR + r : r * LDR + c + k] = v[k];
    }
}

template <typename C, int R, int W, int LDR, int NT, bool TRANS = false>
__device__ __forceinline__ void tile_load(C* __restrict__ lds, const C* __restrict__ src, size_t rstride, int tid)
{
    TileRegs<C, R, W, NT> t;
    tile_fetch<C, R, W, NT>(t, src, rstride, tid);
    tile_put<C, R, W, LDR, NT, TRANS>(lds, t, tid);
}

// ---------------------------------------------------------------- register DFTs
template <typename C, bool INV>
__device__ __forceinline__ void dft2(C* v)
{
    C a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
}

template <typename C, bool INV>
__device__ __forceinline__ void dft4(C* v)
{
    C t0 = cadd(v[0], v[2]), t1 = csub(v[0], v[2]);
    C t2 = cadd(v[1], v[3]), t3 = cmul_mi<C, INV>(csub(v[1], v[3]));
    v[0] = cadd(t0, t2);
    v[2] = csub(t0, t2);
    v[1] = cadd(t1, t3);
    v[3] = csub(t1, t3);
}

template <typename C, bool INV>
__device__ __forceinline__ void dft8(C* v)
{
    using T = decltype(C{}.x);
    const T h = (T)0.70710678118654752440;
    C e[4] = {v[0], v[2], v[4], v[6]};
    C o[4] = {v[1], v[3], v[5], v[7]};
    dft4<C, INV>(e);
    dft4<C, INV>(o);
    // v[k] = e[k] +- exp(-+ 2 pi i k / 8) o[k], the products fused into the sums
    const C w1 = mk<C>(h, INV ? h : -h), w3 = mk<C>(-h, INV ? h : -h);
    o[2] = cmul_mi<C, INV>(o[2]);
    v[0] = cadd(e[0], o[0]);
    v[4] = csub(e[0], o[0]);
    v[1] = cmadd(e[1], o[1], w1);
    v[5] = cmsub(e[1], o[1], w1);
    v[2] = cadd(e[2], o[2]);
    v[6] = csub(e[2], o[2]);
    v[3] = cmadd(e[3], o[3], w3);
    v[7] = cmsub(e[3], o[3], w3);
}

template <typename C, bool INV>
__device__ __forceinline__ void dft16(C* v)
{
    using T = decltype(C{}.x);
    C e[8], o[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) { e[k] = v[2 * k]; o[k] = v[2 * k + 1]; }
    dft8<C, INV>(e);
    dft8<C, INV>(o);
    const T c1 = (T)0.92387953251128675613, s1 = (T)0.38268343236508977173;
    const T h = (T)0.70710678118654752440;
    const T sg = INV ? (T)1 : (T)-1;
    // w_k = cos(2 pi k/16) + sg i sin(2 pi k/16); v[k] = e[k] +- w_k o[k], fused
    const C w[8] = {mk<C>((T)1, (T)0), mk<C>(c1, sg * s1), mk<C>(h, sg * h), mk<C>(s1, sg * c1),
                    mk<C>((T)0, sg), mk<C>(-s1, sg * c1), mk<C>(-h, sg * h), mk<C>(-c1, sg * s1)};
    o[4] = cmul_mi<C, INV>(o[4]);
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        if (k == 0 || k == 4) {
            v[k] = cadd(e[k], o[k]);
            v[k + 8] = csub(e[k], o[k]);
        } else {
            v[k] = cmadd(e[k], o[k], w[k]);
            v[k + 8] = cmsub(e[k], o[k], w[k]);
        }
    }
}

template <int R, typename C, bool INV>
__device__ __forceinline__ void dft(C* v)
{
    if constexpr (R == 2) dft2<C, INV>(v);
    else if constexpr (R == 4) dft4<C, INV>(v);
    else if constexpr (R == 8) dft8<C, INV>(v);
    else if constexpr (R == 16) dft16<C, INV>(v);
}

// ---------------------------------------------------------------- radix plans
// of the x stage's half-length lines, N / 2 points
template <int N> struct Plan;
template <> struct Plan<16>   { static constexpr int P = 1, R0 = 16, R1 = 1,  R2 = 1; };
template <> struct Plan<32>   { static constexpr int P = 2, R0 = 8,  R1 = 4,  R2 = 1; };
template <> struct Plan<64>   { static constexpr int P = 2, R0 = 8,  R1 = 8,  R2 = 1; };
template <> struct Plan<128>  { static constexpr int P = 2, R0 = 16, R1 = 8,  R2 = 1; };
template <> struct Plan<256>  { static constexpr int P = 2, R0 = 16, R1 = 16, R2 = 1; };
template <> struct Plan<512>  { static constexpr int P = 3, R0 = 8,  R1 = 8,  R2 = 8; };

// One Stockham pass of stride NS (product of the radices already applied) over K
// tiles at once (tile k at lds + k * TS): each work item runs one radix-R butterfly
// per tile, so a lane has K independent butterflies in flight.  Caller guarantees the
// tiles are complete (barrier) before the call; the pass ends with a barrier.  tw may
// point to LDS or to global memory.
template <typename T, int N, int R, int NS, bool INV, int TC, int LDR, int NT, int K = 1, int TS = 0>
__device__ __forceinline__ void fft_pass(cpx<T>* __restrict__ lds, const cpx<T>* __restrict__ tw, int tid)
{
    using C = cpx<T>;
    constexpr int NJ = N / R;
    constexpr int ITEMS = TC * NJ;
    constexpr int Q = (ITEMS + NT - 1) / NT;
    C v[K][Q][R];
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int it = tid + NT * q;
        if (ITEMS % NT == 0 || it < ITEMS) {
            const int c = it % TC, j = it / TC;
#pragma unroll
            for (int k = 0; k < K; ++k)
#pragma unroll
                for (int r = 0; r < R; ++r) v[k][q][r] = lds[k * TS + (j + r * NJ) * LDR + c];
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        const int it = tid + NT * q;
        if (ITEMS % NT == 0 || it < ITEMS) {
            const int c = it % TC, j = it / TC;
            const int m = j % NS;
            if constexpr (NS > 1) {
                constexpr int STEP = N / (NS * R);
#pragma unroll
                for (int r = 1; r < R; ++r) {
                    C w = tw[(m * r * STEP) & (N - 1)];
                    if (INV) w.y = -w.y;
#pragma unroll
                    for (int k = 0; k < K; ++k) v[k][q][r] = cmul(v[k][q][r], w);
                }
            }
            const int base = (j / NS) * NS * R + m;
#pragma unroll
            for (int k = 0; k < K; ++k) {
                dft<R, C, INV>(v[k][q]);
#pragma unroll
                for (int r = 0; r < R; ++r) lds[k * TS + (base + r * NS) * LDR + c] = v[k][q][r];
            }
        }
    }
    __syncthreads();
}

// FFT of every column of K tiles (tile k at lds + k * TS) through the plan of N.
template <typename T, int N, bool INV, int TC, int LDR, int NT, int K = 1, int TS = 0>
__device__ __forceinline__ void fft_tile(cpx<T>* __restrict__ lds, const cpx<T>* __restrict__ tw, int tid)
{
    using P = Plan<N>;
    fft_pass<T, N, P::R0, 1, INV, TC, LDR, NT, K, TS>(lds, tw, tid);
    if constexpr (P::P > 1) fft_pass<T, N, P::R1, P::R0, INV, TC, LDR, NT, K, TS>(lds, tw, tid);
    if constexpr (P::P > 2) fft_pass<T, N, P::R2, P::R0 * P::R1, INV, TC, LDR, NT, K, TS>(lds, tw, tid);
}

// ---------------------------------------------------------------- columns in registers
// The y and z stages hold a column in the registers of N / E threads: thread t of column c
// has points t + (N / E) q, q < E, in v[q].  A Stockham pass of radix R takes points
// j + r N / R, which are v[i + r E / R] of the thread with j = t + (N / E) i, so every pass
// works on registers, the last pass leaves its output (points j + r N / R again) where the
// input was, and LDS serves only the exchange between two passes: one write and one read
// per value and exchange, where tiles kept in LDS cost a write and a read per pass and two
// more for the transfers to HBM.  Rows go straight between HBM and the registers (TC
// adjacent kx of one row: 128 bytes at the default widths).
template <int N, int E> struct RPlan;
template <> struct RPlan<32, 4>    { static constexpr int R0 = 4,  R1 = 4,  R2 = 2, R3 = 1; };
template <> struct RPlan<64, 4>    { static constexpr int R0 = 4,  R1 = 4,  R2 = 4, R3 = 1; };
template <> struct RPlan<32, 8>    { static constexpr int R0 = 8,  R1 = 4,  R2 = 1, R3 = 1; };
template <> struct RPlan<64, 8>    { static constexpr int R0 = 8,  R1 = 8,  R2 = 1, R3 = 1; };
template <> struct RPlan<128, 8>   { static constexpr int R0 = 8,  R1 = 4,  R2 = 4, R3 = 1; };
template <> struct RPlan<128, 16>  { static constexpr int R0 = 16, R1 = 8,  R2 = 1, R3 = 1; };
template <> struct RPlan<256, 8>   { static constexpr int R0 = 8,  R1 = 8,  R2 = 4, R3 = 1; };
template <> struct RPlan<256, 16>  { static constexpr int R0 = 16, R1 = 16, R2 = 1, R3 = 1; };
template <> struct RPlan<512, 8>   { static constexpr int R0 = 8,  R1 = 8,  R2 = 8, R3 = 1; };
template <> struct RPlan<512, 16>  { static constexpr int R0 = 8,  R1 = 8,  R2 = 8, R3 = 1; };
template <> struct RPlan<1024, 8>  { static constexpr int R0 = 8,  R1 = 8,  R2 = 4, R3 = 4; };
template <> struct RPlan<1024, 16> { static constexpr int R0 = 16, R1 = 16, R2 = 4, R3 = 1; };

// One pass of radix R and stride NS on a thread's E points; LAST leaves the result in v, the
// other passes exchange it through lds (N rows of LDR, this column at lds[n * LDR]).  All
// threads of the work-group call it; lds may be reused when it returns.
template <typename T, int N, int E, int R, int NS, bool INV, int LDR, bool LAST>
__device__ __forceinline__ void col_pass(cpx<T> (&v)[E], cpx<T>* __restrict__ lds, const cpx<T>* __restrict__ tw, int t)
{
    using C = cpx<T>;
    constexpr int TT = N / E, B = E / R;
#pragma unroll
    for (int i = 0; i < B; ++i) {
        const int j = t + TT * i;
        const int m = j % NS;
        C a[R];
#pragma unroll
        for (int r = 0; r < R; ++r) a[r] = v[i + r * B];
        if constexpr (NS > 1) {
            constexpr int STEP = N / (NS * R);
#pragma unroll
            for (int r = 1; r < R; ++r) {
                C w = tw[(m * r * STEP) & (N - 1)];
                if (INV) w.y = -w.y;
                a[r] = cmul(a[r], w);
            }
        }
        dft<R, C, INV>(a);
        if constexpr (LAST) {
#pragma unroll
            for (int r = 0; r < R; ++r) v[i + r * B] = a[r];
        } else {
            const int base = (j / NS) * NS * R + m;
#pragma unroll
            for (int r = 0; r < R; ++r) lds[(base + r * NS) * LDR] = a[r];
        }
    }
    if constexpr (!LAST) {
        __syncthreads();
#pragma unroll
        for (int q = 0; q < E; ++q) v[q] = lds[(t + TT * q) * LDR];
        __syncthreads();
    }
}

// The transform of one column: in and out as v[q] = point t + (N / E) q.
template <typename T, int N, int E, bool INV, int LDR>
__device__ __forceinline__ void col_fft(cpx<T> (&v)[E], cpx<T>* __restrict__ lds, const cpx<T>* __restrict__ tw, int t)
{
    using P = RPlan<N, E>;
    col_pass<T, N, E, P::R0, 1, INV, LDR, P::R1 == 1>(v, lds, tw, t);
    if constexpr (P::R1 > 1) col_pass<T, N, E, P::R1, P::R0, INV, LDR, P::R2 == 1>(v, lds, tw, t);
    if constexpr (P::R2 > 1) col_pass<T, N, E, P::R2, P::R0 * P::R1, INV, LDR, P::R3 == 1>(v, lds, tw, t);
    if constexpr (P::R3 > 1) col_pass<T, N, E, P::R3, P::R0 * P::R1 * P::R2, INV, LDR, true>(v, lds, tw, t);
}

// the twiddle table exp(-2 pi i m / N), m < N, copied to LDS by the whole work-group
template <typename C, int N, int NT>
__device__ __forceinline__ void stage_twiddles(C* __restrict__ tws, const C* __restrict__ tw, int tid)
{
#pragma unroll
    for (int m = tid; m < N; m += NT) tws[m] = tw[m];
}

}  // namespace ddns
