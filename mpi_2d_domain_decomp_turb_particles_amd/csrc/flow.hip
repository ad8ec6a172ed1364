// flow.hip -- spectral Navier-Stokes step on one MI355X.
//
// Reference: turb.f90:506-691 (curl, inverse FFTs, u x w, forward FFTs, dealiasing,
// AB2/Crank-Nicolson update, projection, forcing, symmetrize), mpifft.f90:81-198
// (the 3-D real FFT as x / y / z line transforms with a 1/N scale after each
// forward stage), flowlib.f90:180-562 (dealiasing, supforDET, symmetrize,
// supforSTH).
//
// Layout: ddns_internal.h (rows of 128 bytes of kx, z columns of the state contiguous).  The
// step runs as:
//   Ky(inverse, 6 fields, kx = 0 column symmetrised)  ->  Kx(6 C2R, u x w, 3 R2C,
//   physical u for the droplets)  ->  Ky(forward, 3 fields)  ->  Kpre (one block:
//   deterministic-forcing shell energies or the OU forcing table)  ->  Kz(forward z
//   FFT, update, curl, inverse z FFT of u and w)  ->  Ksym (kx = 0 plane of u-hat).
// The z stage therefore closes step n and opens step n + 1 in one pass over HBM.
#include "fft_engine.h"

#include <algorithm>
#include <cstdlib>
#include <cmath>
#include <cstring>
#include <map>
#include <mutex>

namespace ddns {

constexpr int NT = 256;

enum { KZ_FULL = 0, KZ_CURL_INV = 1, KZ_PLAIN_FWD = 2, KZ_PLAIN_INV = 3 };

// Points per thread of a column (fft_engine.h).  The plain transforms hold one value set per
// column (16 points: at most one exchange up to N = 256).  The z stage holds three and a
// fourth in flight: 16 points in single precision from N = 256 on (8 points cost a
// second exchange: 300 against 258 us at 256^3), 8 where that leaves a second wavefront per
// SIMD its registers (27 against 32 us at 128^3; all of double: 16 would need 512), 4 on the
// grids that do not fill the chip (12 against 15 us at 32^3).
template <typename T, int N> constexpr int col_e() { return N == 32 || N == 64 || (sizeof(T) == 8 && N == 512) ? 8 : 16; }
template <typename T, int N> constexpr int kz_e() { return N <= 64 ? 4 : (sizeof(T) == 4 && N >= 256 ? 16 : 8); }
// wavefronts per SIMD that the z stage's registers leave room for (double at 256^3: one, its
// values spill at two: 484 against 542 us)
template <typename T, int N> constexpr int kz_waves() { return sizeof(T) == 8 && N >= 256 ? 1 : 2; }
template <int TC> constexpr int ldr_of() { return (TC >= 8) ? TC + 1 : TC; }

// tile width (kx columns per work-group) of the y stage: rows of 128 bytes below N = 1024,
// 64 there (two work-groups per CU); at least a wavefront of threads (N = 32)
template <typename T, int N> constexpr int ky_tc() { return (sizeof(T) == 4) ? (N >= 1024 ? 8 : 16) : (N >= 1024 ? 4 : (N == 32 ? 16 : 8)); }
// The y stage runs at one of three tile widths, chosen per grid and precision by timing
// (flow_tune): half, once and twice the default, where a work-group has 64 to 1024 threads
// and its exchange buffer fits LDS with the twiddles.  The width changes only which columns a
// work-group transforms together, never the arithmetic of a column, so every choice gives
// the same bits.
template <typename T, int N, int TC> constexpr bool ky_fits()
{
    constexpr int nt = TC * (N / col_e<T, N>());
    return TC >= 1 && TC <= N / 2 && nt >= 64 && nt <= 1024 && (N * ldr_of<TC>() + N) * (int)sizeof(cpx<T>) <= 160 * 1024;
}
template <typename T, int N> constexpr int ky_cand(int k) { return k == 0 ? ky_tc<T, N>() / 2 : (k == 1 ? ky_tc<T, N>() : 2 * ky_tc<T, N>()); }
// tile width of the fused z stage: rows of 128 bytes, half that where the threads that would
// take could have no more than 128 registers each (N = 1024); at least a wavefront (N = 32)
template <typename T, int N> constexpr int kz_tc()
{
    if constexpr (sizeof(T) == 4) return N >= 1024 ? 8 : 16;
    else return N >= 1024 ? 4 : (N == 32 ? 16 : 8);
}
template <typename T, int N, int TC> constexpr int kz_threads() { return TC * (N / kz_e<T, N>()); }

// Work-groups are dispatched to the 8 XCDs round-robin by linear id, and each XCD has
// its own L2.  When a tile row is narrower than a 128-byte line, the P tiles that share
// a line get linear ids L, L+8, ..., so they land on the same XCD and meet in its L2.
// Returns the tile index of linear work-group id L (total a multiple of 8 P).
template <int P>
__device__ __forceinline__ int xcd_tile(int L)
{
    if constexpr (P <= 1) {
        return L;
    } else {
        const int g = L / (8 * P), r = L % (8 * P);
        return g * (8 * P) + (r % 8) * P + r / 8;
    }
}
// tile width of the plain z transforms (the diagnostics, the stand-alone transforms): rows of 128 bytes
template <typename T, int N> constexpr int kz_tc_plain() { return sizeof(T) == 4 || N == 32 ? 16 : 8; }
template <typename T, int N> constexpr int kz_plain_threads() { return kz_tc_plain<T, N>() * (N / col_e<T, N>()); }
__device__ __forceinline__ int wave_index(int i, int N) { return i <= N / 2 ? i : i - N; }

// Is mode (kx, ky, kz) inside the dealiasing sphere, shell int(|k| + 1/2) <= nek (turb.f90:405,
// 648-650)?  |k| < nek + 1/2 is k^2 <= nek (nek + 1) in whole numbers; the reference's rounded
// square root gives the same (the two k^2 next to the limit are 1e-4 of a shell away from
// it at N = 1024).  Outside it the update sets both the new u-hat and the stored nonlinear term
// to zero (the mean mode counts as inside: its u-hat is zero but its nonlinear term is kept).
__device__ __forceinline__ bool mode_in_sphere(int kx, int ky, int kz, int N, int nek)
{
    const int kyw = wave_index(ky, N), kzw = wave_index(kz, N);
    return kx * kx + kyw * kyw + kzw * kzw <= nek * (nek + 1);
}

// Batched realisations: realisation r of a field starts r * rstride complex values after
// realisation 0 (rstride = 0 for one realisation), its low-mode table r * LOW_STRIDE
// doubles after, and the physical velocity r * pstride reals after.  With forcing < 0
// every realisation takes its forcing kind and amplitudes from its own low-mode table
// (LOW_PAR onwards).
constexpr int LOW_STRIDE = 1024;
constexpr int LOW_PAR = 1000;       // [0] forcing kind, [1..2] force(1:2), [3] OU time scale, [4] OU variance
// [LOW_ZOUT] = 1 once a step has written the state's modes beyond the dealiasing sphere,
// which every update sets to zero.  The z stage never loads them and stores the zeros only
// while the flag is clear; the inverse y stage takes the columns beyond the sphere as zero once
// it is set.  Cleared by every upload of the state; set by the step's k_sym, which runs after
// the z stage.
constexpr int LOW_ZOUT = LOW_PAR + 5;
constexpr int STH_STATE_STRIDE = 64;
constexpr int STH_B_STRIDE = 512;

__device__ __forceinline__ int real_forcing(int forcing, const double* lowr)
{
    return forcing >= 0 ? forcing : (int)lowr[LOW_PAR];
}

struct KzArgs {
    const void* B[3];  // N-hat: A[0..2] themselves, each point read and written by one thread
    void* U[3];
    void* O[3];
    void* A[6];
    const void* tw;
    const double* low;
    double dt, rnu;
    int nek, forcing;
    double scale;      // plain modes: output scale
    size_t rstride;    // complex values between realisations of one field
};

// A field as plain rows, row (z, y) of realisations in a row at p + (z N + y) rs.
struct PlainRows {
    void* p[6];
    int rs[6];         // complex values from row to row
};

struct KyArgs {
    void* F[6];        // the fields in the intermediate layout
    PlainRows L;       // and as plain rows
    const void* tw;
    double scale;
    size_t rstride;
    const double* low; // the step's stages (null: every row is read and written)
    int nek;
};

struct KxArgs {
    void* B[3];        // u in, u x w out
    void* uphys;       // w in (three rows per line), the physical velocity out
    const void* tw;    // N entries (post/pre-processing twiddles)
    const void* twh;   // N/2 entries (half-length FFT)
};

// ------------------------------------------------------------------ spectral update
// One mode of turb.f90:662-687 for the three components held in n[3] (forward FFT
// output, already scaled) and the state u[3], o[3]; returns the new u-hat in v[3]
// and the dealiased nonlinear term in nd[3].  ff: supforDET factors; fa: the
// supforSTH table a(6,5,5) per component.
template <typename T>
__device__ __forceinline__ void update_mode(int kx, int ky, int kz, int N, int nek, int forcing,
                                            T dt, T rnu, const double* __restrict__ low,
                                            const cpx<T>* n, const cpx<T>* u, const cpx<T>* o,
                                            cpx<T>* v, cpx<T>* nd)
{
    using C = cpx<T>;
    const int kyw = wave_index(ky, N), kzw = wave_index(kz, N);
    const T fx = (T)kx, fy = (T)kyw, fz = (T)kzw;
    // the shells of turb.f90:405 in whole numbers (mode_in_sphere): shell 1 holds k^2 = 1, 2,
    // shell 2 k^2 = 3 .. 6
    const int ki2 = kx * kx + kyw * kyw + kzw * kzw;
    const bool zero_mode = ki2 == 0;
    const T k2 = zero_mode ? (T)1.e-5 : (T)ki2;                     // flowlib.f90:36-38
    const bool inside = ki2 <= nek * (nek + 1);
    const bool keep = inside && !zero_mode;
    const T dt_h = (T)0.5 * dt, dtr = (T)1.5 * dt;                   // turb.f90:483-484
    const T ac = rnu * dt_h * k2;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        nd[c] = inside ? n[c] : mk<C>((T)0, (T)0);             // dealiasing, 648-650
        v[c] = csmadd(csmadd(cscale(u[c], (T)1 - ac), nd[c], dtr), o[c], -dt_h);
    }
    if (forcing == 2 && kx < 3) {                                    // supforSTH add, flowlib.f90:529-559
        const int js = ky <= 2 ? ky : (ky >= N - 2 ? ky - (N - 5) : -1);
        const int ks = kz <= 2 ? kz : (kz >= N - 2 ? kz - (N - 5) : -1);
        if (js >= 0 && ks >= 0) {
            const double* fa = low + 8;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                const int o0 = 2 * kx + 6 * (js + 5 * ks);
                v[c].x = v[c].x + dt * (T)fa[150 * c + o0];
                v[c].y = v[c].y + dt * (T)fa[150 * c + o0 + 1];
            }
        }
    }
    // projection, 669-672
    const C t = cscale(csmadd(csmadd(cscale(v[0], fx), v[1], fy), v[2], fz), (T)1 / k2);
    v[0] = csmadd(v[0], t, -fx);
    v[1] = csmadd(v[1], t, -fy);
    v[2] = csmadd(v[2], t, -fz);
    const T den = (T)1 + ac;                                         // 674-676
    T f = (T)1 / den;
    if (forcing == 1 && ki2 >= 1 && ki2 <= 6) f = f * (T)low[ki2 <= 2 ? 0 : 1];   // supforDET
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        v[c] = keep ? cscale(v[c], f) : mk<C>((T)0, (T)0);
    }
}

// ------------------------------------------------------------------ z stage
// How far plane t + TT q of an intermediate field lies behind plane t (t < TT, TT a divisor or
// a multiple of the planes per block)
template <typename T, int N, int TT>
__device__ __forceinline__ constexpr size_t plane_step(int q)
{
    static_assert(TT % LZB == 0 || LZB % TT == 0, "a thread's planes must step through the blocks evenly");
    constexpr size_t block = (size_t)N * (N / 2) * LZB;
    return q * TT / LZB * block + q * TT % LZB * lay_w<T>();
}

// A plain forward / inverse z transform of one field.
template <typename T, int N, bool INV>
__global__ void __launch_bounds__((kz_plain_threads<T, N>())) k_z(KzArgs a)
{
    using C = cpx<T>;
    constexpr int M = N / 2, E = col_e<T, N>(), TT = N / E;
    constexpr int TC = kz_tc_plain<T, N>(), LDR = ldr_of<TC>(), NTK = kz_plain_threads<T, N>();
    __shared__ C lds[N * LDR];
    __shared__ C tws[N];
    const int tid = threadIdx.x, c = tid % TC, t = tid / TC;
    constexpr int NBX = M / TC;
    const int kx0 = (blockIdx.x % NBX) * TC, ky = blockIdx.x / NBX;
    stage_twiddles<C, N, NTK>(tws, (const C*)a.tw, tid);
    // inverse: spectral to intermediate layout; forward: back
    const size_t sb = spec_index<T>(N, t, ky, kx0 + c), pb = pipe_index<T>(N, t, ky, kx0 + c);
    constexpr int SS = TT * lay_w<T>();
    const C* src = (const C*)a.B[0] + (INV ? sb : pb);
    C* dst = (C*)a.U[0] + (INV ? pb : sb);
    C v[E];
#pragma unroll
    for (int q = 0; q < E; ++q) v[q] = src[INV ? q * SS : plane_step<T, N, TT>(q)];
    __syncthreads();
    col_fft<T, N, E, INV, LDR>(v, lds + c, tws, t);
    const T sc = (T)a.scale;
#pragma unroll
    for (int q = 0; q < E; ++q) dst[INV ? plane_step<T, N, TT>(q) : q * SS] = cscale(v[q], sc);
}

// The whole z stage of a column tile in registers.  FULL: forward z transforms of N-hat, the
// update, the curl of the new u-hat, inverse z transforms of u-hat and w-hat.  Otherwise (a
// new state) the curl and the inverse transforms of the stored u-hat alone.
//   - A thread holds points kz = t + (N / E) q of its column for all three components: the
//     forward transforms end with the modes where the update and the curl need them and the
//     inverse ones start, so the stage has no pointwise pass over LDS and only the exchange
//     buffer of one field in it (36 KB at 256^3 FP32, four tiles took 141 KB).
//   - It is bound by HBM: at 256^3 FP32 it moves 9C x 0.77 + 12C x 0.51 (0.87 GB).
//   - Beyond the dealiasing sphere nothing is moved: a column with kx^2 + ky^2 beyond it
//     (23 % of them) is neither read from B nor written to A (the y stages leave it out too),
//     a tile of such columns ends at once, and the state's modes beyond the sphere are only
//     written while they may still be nonzero (LOW_ZOUT).
// The tile width (and with it the work-group's size) is timed at set-up; it changes no
// column's arithmetic.
template <typename T, int N, int TC> constexpr bool kz_fits()
{
    constexpr int nt = kz_threads<T, N, TC>();
    return TC <= N / 2 && nt >= 64 && nt <= 512 && (N * ldr_of<TC>() + N) * (int)sizeof(cpx<T>) <= 160 * 1024;
}
template <typename T, int N> constexpr int kz_cand(int k) { return kz_tc<T, N>() << k; }

template <typename T, int N, int TC, bool FULL>
__global__ void __launch_bounds__((kz_threads<T, N, TC>()), (kz_waves<T, N>())) k_z_full(KzArgs a)
{
    using C = cpx<T>;
    constexpr int M = N / 2, E = kz_e<T, N>(), TT = N / E, NBX = M / TC, TPR = NBX * N;
    constexpr int LDR = ldr_of<TC>();
    constexpr int P = (TC * (int)sizeof(C) >= 128) ? 1 : 128 / (TC * (int)sizeof(C));
    __shared__ C lds[N * LDR];
    __shared__ C tws[N];
    const int tid = threadIdx.x, c = tid % TC, t = tid / TC;
    // tile = realisation * TPR + local tile (tiles that share a 128-byte line on one XCD)
    const int tile = xcd_tile<(NBX % P == 0 && TPR % (8 * P) == 0) ? P : 1>(blockIdx.x);
    const int rr = tile / TPR, lt = tile - rr * TPR;
    const int kx = (lt % NBX) * TC + c, ky = lt / NBX;
    const size_t roff = (size_t)rr * a.rstride;
    // point t of the column in the state (steps of SS) and between the transforms
    const size_t sbase = roff + spec_index<T>(N, t, ky, kx), pbase = roff + pipe_index<T>(N, t, ky, kx);
    constexpr int SS = TT * lay_w<T>();
    const double* lowr = a.low + (size_t)rr * LOW_STRIDE;
    // beyond the dealiasing sphere the state is zero once a step has written it
    const bool zout = lowr[LOW_ZOUT] != 0.0;
    C u[3][E];
    bool colin = true;
    if constexpr (FULL) {
        colin = mode_in_sphere(kx, ky, 0, N, a.nek);
        if (!mode_in_sphere(kx - c, ky, 0, N, a.nek)) {          // the whole tile is beyond the sphere
            if (!zout) {
#pragma unroll
                for (int q = 0; q < E; ++q)
#pragma unroll
                    for (int k = 0; k < 3; ++k) {
                        ((C*)a.U[k])[sbase + q * SS] = mk<C>((T)0, (T)0);
                        ((C*)a.O[k])[sbase + q * SS] = mk<C>((T)0, (T)0);
                    }
            }
            return;
        }
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
            for (int q = 0; q < E; ++q)
                u[k][q] = colin ? ((const C*)a.B[k])[pbase + plane_step<T, N, TT>(q)] : mk<C>((T)0, (T)0);
    } else {
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
            for (int q = 0; q < E; ++q) u[k][q] = ((const C*)a.U[k])[sbase + q * SS];
    }
    stage_twiddles<C, N, kz_threads<T, N, TC>()>(tws, (const C*)a.tw, tid);
    __syncthreads();
    C* col = lds + c;
    if constexpr (FULL) {
#pragma unroll
        for (int k = 0; k < 3; ++k) col_fft<T, N, E, false, LDR>(u[k], col, tws, t);
        const int forcing = real_forcing(a.forcing, lowr);
        const T inv_n = (T)1 / (T)N;
#pragma unroll
        for (int q = 0; q < E; ++q) {
            const int n = t + TT * q;
            const size_t g = sbase + q * SS;
            if (mode_in_sphere(kx, ky, n, N, a.nek)) {
                C nn[3], u3[3], o3[3], vv[3], nd[3];
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    nn[k] = cscale(u[k][q], inv_n);
                    u3[k] = ((const C*)a.U[k])[g];
                    o3[k] = ((const C*)a.O[k])[g];
                }
                update_mode<T>(kx, ky, n, N, a.nek, forcing, (T)a.dt, (T)a.rnu, lowr, nn, u3, o3, vv, nd);
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    ((C*)a.U[k])[g] = vv[k];
                    ((C*)a.O[k])[g] = nd[k];
                    u[k][q] = vv[k];
                }
            } else {
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    u[k][q] = mk<C>((T)0, (T)0);
                    if (!zout) {
                        ((C*)a.U[k])[g] = u[k][q];
                        ((C*)a.O[k])[g] = u[k][q];
                    }
                }
            }
        }
    }
    // vorticity w = i k x u (turb.f90:506-517), one component at a time
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        C w[E];
#pragma unroll
        for (int q = 0; q < E; ++q) {
            const T fx = (T)kx, fy = (T)wave_index(ky, N), fz = (T)wave_index(t + TT * q, N);
            C x;
            if (k == 0) x = csmadd(cscale(u[2][q], fy), u[1][q], -fz);
            else if (k == 1) x = csmadd(cscale(u[0][q], fz), u[2][q], -fx);
            else x = csmadd(cscale(u[1][q], fx), u[0][q], -fy);
            w[q] = mk<C>(-x.y, x.x);
        }
        col_fft<T, N, E, true, LDR>(w, col, tws, t);
        if (colin) {
#pragma unroll
            for (int q = 0; q < E; ++q) ((C*)a.A[3 + k])[pbase + plane_step<T, N, TT>(q)] = w[q];
        }
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        col_fft<T, N, E, true, LDR>(u[k], col, tws, t);
        if (colin) {
#pragma unroll
            for (int q = 0; q < E; ++q) ((C*)a.A[k])[pbase + plane_step<T, N, TT>(q)] = u[k][q];
        }
    }
}

// ------------------------------------------------------------------ y stage
// Columns in registers as in the z stage; bound by memory.  The inverse stage takes a plane
// from the intermediate layout to plain [y][kx] rows, where the x stage finds its lines; the
// forward stage goes the other way.  In a step (a.low given) the rows beyond the circle
// kx^2 + ky^2 of the dealiasing sphere (23 % of them) are left out: the inverse stage takes
// them as zero (unless the state was set since the last step, when the z transforms of that
// state fill them), the forward stage does not store them.
template <typename T, int N, bool INV, bool SYM, int TC>
__global__ void __launch_bounds__((TC * (N / col_e<T, N>()))) k_y(KyArgs a)
{
    using C = cpx<T>;
    constexpr int M = N / 2, E = col_e<T, N>(), TT = N / E, NTK = TC * TT;
    constexpr int LDR = ldr_of<TC>();
    __shared__ C lds[N * LDR];
    __shared__ C tws[N];
    const int tid = threadIdx.x, c = tid % TC, t = tid / TC;
    // tiles whose rows share a 128-byte line (P of them, side by side in kx) go to linear
    // ids L, L+8, ..., i.e. to one XCD, where the second finds the line in L2
    constexpr int P = (TC * (int)sizeof(C) >= 128) ? 1 : 128 / (TC * (int)sizeof(C));
    int kxb = blockIdx.x, lp = blockIdx.y, fi = blockIdx.z;
    if constexpr (P > 1) {
        if ((M / TC) % P == 0 && (gridDim.y * gridDim.z) % 8 == 0) {
            const int l = xcd_tile<P>(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z));
            kxb = l % gridDim.x;
            lp = (l / gridDim.x) % gridDim.y;
            fi = l / (gridDim.x * gridDim.y);
        }
    }
    const int kx = kxb * TC + c;
    const int rr = lp / N, z = lp % N;
    // row n of this plane's column: n * PS behind pf in the intermediate layout, n * ls behind lf
    // as plain rows
    C* pf = (C*)a.F[fi] + (size_t)rr * a.rstride + pipe_index<T>(N, z, 0, kx);
    const int ls = a.L.rs[fi];
    C* lf = (C*)a.L.p[fi] + (size_t)lp * N * ls + kx;
    constexpr int PS = LZB * lay_w<T>();
    const bool all = !a.low || (INV && a.low[(size_t)rr * LOW_STRIDE + LOW_ZOUT] == 0.0);
    C v[E];
#pragma unroll
    for (int q = 0; q < E; ++q) {
        const int n = t + TT * q;
        v[q] = !INV || all || mode_in_sphere(kx, n, 0, N, a.nek) ? (INV ? pf[(size_t)n * PS] : lf[(size_t)n * ls]) : mk<C>((T)0, (T)0);
    }
    stage_twiddles<C, N, NTK>(tws, (const C*)a.tw, tid);
    if constexpr (SYM) {
        // kx = 0 column: (c(ky) + conj c(-ky)) / 2, the z-transformed form of the
        // kx = 0 plane symmetrisation of flowlib.f90:264-329
        if (kxb == 0) {
            if (c == 0) {
#pragma unroll
                for (int q = 0; q < E; ++q) lds[t + TT * q] = v[q];
            }
            __syncthreads();
            if (c == 0) {
#pragma unroll
                for (int q = 0; q < E; ++q) {
                    const C m = lds[(N - (t + TT * q)) & (N - 1)];
                    v[q] = mk<C>((T)0.5 * (v[q].x + m.x), (T)0.5 * (v[q].y - m.y));
                }
            }
        }
    }
    __syncthreads();
    col_fft<T, N, E, INV, LDR>(v, lds + c, tws, t);
    const T sc = (T)a.scale;
#pragma unroll
    for (int q = 0; q < E; ++q) {
        const int n = t + TT * q;
        if (INV) lf[(size_t)n * ls] = v[q];
        else if (all || mode_in_sphere(kx, n, 0, N, a.nek)) pf[(size_t)n * PS] = cscale(v[q], sc);
    }
}

// ------------------------------------------------------------------ x stage
// Half-length packing of a real line of N points as N/2 complex points.
template <int N> constexpr int kx_lines() { return 2048 / N; }   // 4 complex points per thread
// lines of one k_x_fused work-group: 4 complex points per thread and field, and the least that
// 16-byte accesses allow (1 in FP64, 2 in FP32) up to 64^3, where 4 left 16 or 128 work-groups
// for 256 CUs, each with four times the serial work: 32^3 FP64 18.8 -> 13.1 us, FP32 16.1 -> 13.9;
// 64^3 20.5 -> 15.1, 16.7 -> 13.6; at 128^3 the small tile is the slower one (FP32 28.9 -> 34.5)
template <typename T, int N> constexpr int kxf_lines()
{
    return (N <= 64 ? 8192 / (int)sizeof(cpx<T>) : 2048) / N;
}

// C2R pre-processing of the tile (in place, pairs k and M-k of every line).
template <typename T, int N, int TL, int LDR>
__device__ __forceinline__ void c2r_pack(cpx<T>* lds, const cpx<T>* tw, int tid)
{
    using C = cpx<T>;
    constexpr int M = N / 2;
    for (int e = tid; e < TL * (M / 2 + 1); e += NT) {
        const int line = e / (M / 2 + 1), k = e % (M / 2 + 1);
        if (k == 0) {
            const C x0 = lds[line];
            lds[line] = mk<C>(x0.x, x0.x);               // X(N/2) = 0, Im X(0) ignored
        } else {
            const int k2 = M - k;
            const C xa = lds[k * LDR + line], xb = lds[k2 * LDR + line];
            C w = tw[k];                                  // exp(-2 pi i k / N)
            w.y = -w.y;                                   // exp(+2 pi i k / N)
            const C sa = cadd(xa, cconj(xb)), da = csub(xa, cconj(xb));
            const C za = cmadd(sa, mk<C>(-w.y, w.x), da);            // + i w (xa - conj xb)
            if (k2 != k) {
                const C wb = mk<C>(-w.x, w.y);            // exp(+2 pi i (M-k)/N) = -conj(w)
                const C sb = cadd(xb, cconj(xa)), db = csub(xb, cconj(xa));
                const C zb = cmadd(sb, mk<C>(-wb.y, wb.x), db);
                lds[k2 * LDR + line] = zb;
            }
            lds[k * LDR + line] = za;
        }
    }
}

// R2C post-processing: from Z = FFT_{N/2}(x even + i x odd) to X(k), k < N/2, scaled.
template <typename T, int N, int TL, int LDR>
__device__ __forceinline__ void r2c_unpack_store(const cpx<T>* lds, const cpx<T>* tw, cpx<T>* dst,
                                                 size_t line0, T scale, int tid)
{
    using C = cpx<T>;
    constexpr int M = N / 2;
    for (int e = tid; e < TL * (M / 2 + 1); e += NT) {
        const int line = e / (M / 2 + 1), k = e % (M / 2 + 1);
        C* out = dst + (line0 + line) * M;
        if (k == 0) {
            const C z0 = lds[line];
            out[0] = mk<C>((z0.x + z0.y) * scale, (T)0);
        } else {
            const int k2 = M - k;
            const C za = lds[k * LDR + line], zb = lds[k2 * LDR + line];
            const C w = tw[k];                            // exp(-2 pi i k / N)
            const C e1 = cadd(za, cconj(zb)), d1 = csub(za, cconj(zb));
            // X = e1/2 - (i/2) w d1
            const C xa = cscale(cmadd(e1, mk<C>(w.y, -w.x), d1), (T)0.5);
            out[k] = cscale(xa, scale);
            if (k2 != k) {
                const C wb = mk<C>(-w.x, w.y);            // exp(-2 pi i (M-k)/N) = -conj(w)
                const C e2 = cadd(zb, cconj(za)), d2 = csub(zb, cconj(za));
                const C xb = cscale(cmadd(e2, mk<C>(wb.y, -wb.x), d2), (T)0.5);
                out[k2] = cscale(xb, scale);
            }
        }
    }
}

// two neighbouring nodes (x = 2m, 2m + 1) of the physical velocity, three components
// each, 6 values in a row: three 2-vector stores (p is 2-vector aligned)
__device__ __forceinline__ void store_node_pair(float* p, float a0, float b0, float c0, float a1, float b1, float c1)
{
    ((float2*)p)[0] = make_float2(a0, b0);
    ((float2*)p)[1] = make_float2(c0, a1);
    ((float2*)p)[2] = make_float2(b1, c1);
}
__device__ __forceinline__ void store_node_pair(double* p, double a0, double b0, double c0, double a1, double b1,
                                                double c1)
{
    ((double2*)p)[0] = make_double2(a0, b0);
    ((double2*)p)[1] = make_double2(c0, a1);
    ((double2*)p)[2] = make_double2(b1, c1);
}

// Stand-alone x transforms of one field (kernel-level parity of mpifft3DRC/CR).
template <typename T, int N, bool INV>
__global__ void __launch_bounds__(NT) k_x_plain(const void* src, void* dst, const void* tw_, const void* twh_)
{
    using C = cpx<T>;
    constexpr int M = N / 2;
    constexpr int TL = kx_lines<N>();
    constexpr int LDR = TL + 1;
    __shared__ C lds[M * LDR];
    const int tid = threadIdx.x;
    const size_t line0 = (size_t)blockIdx.x * TL;
    const C* tw = (const C*)tw_;
    const C* twh = (const C*)twh_;
    // both directions see the line as M complex values (real pairs for the C2R output / R2C input)
    tile_load<C, TL, M, LDR, NT, true>(lds, (const C*)src + line0 * M, M, tid);
    __syncthreads();
    if constexpr (INV) {
        c2r_pack<T, N, TL, LDR>(lds, tw, tid);
        __syncthreads();
        fft_tile<T, M, true, TL, LDR, NT>(lds, twh, tid);
        C* d = (C*)dst + line0 * M;
        for (int e = tid; e < TL * M; e += NT) {
            const int line = e / M, m = e % M;
            d[(size_t)line * M + m] = lds[m * LDR + line];
        }
    } else {
        fft_tile<T, M, false, TL, LDR, NT>(lds, twh, tid);
        r2c_unpack_store<T, N, TL, LDR>(lds, tw, (C*)dst, line0, (T)1 / (T)N, tid);
    }
}

// ------------------------------------------------------------------ low-mode pre-kernel
// DET (forcing = 1): the new value of every mode with |k| < 2.5 is computed from a
// direct z-DFT of the y-transformed nonlinear term, then the shell-1 and shell-2
// energies (kx = 0 halved, flowlib.f90:207-217) give ff = sqrt(force/E); low[0..1].
// STH (forcing = 2): ranff white noise, OU step, projection and Hermitian fix-up
// (flowlib.f90:399-510) into low[8 .. 8+450).
constexpr int LOW_DFT = 512;   // offset of the supforDET z-DFT sums in FlowBuffers::low

struct PreArgs {
    const void* B[3];
    const void* U[3];
    const void* O[3];
    const void* tw;
    double* low;
    int* sth_state;
    double* sth_b;
    double dt, rnu, force0, force1, ou_tf, ou_var, pi2;
    int nek, forcing;  // forcing < 0: each realisation's kind and amplitudes from its table
    size_t rstride;    // complex values between realisations of one field
};

// ranff (accesories.f90:38-68) for one wavefront: n draws of the stream in state st
// (idum, iy, iv(32)), each left in seq as the integer that ranff scales by 1/IM.  The
// generator's two parts cost one lane 240 us for the 450 draws of a step; here
//   - the linear congruence x -> 16807 x mod (2^31 - 1) jumps ahead: lane i multiplies by
//     16807^(i+1), so 64 values come at once (exact in 64 bits, the values of the
//     reference's Schrage steps);
//   - the Bays-Durham shuffle is serial in iy, so its table lives in the lanes of one
//     register (lane i holds iv(i+1)) and a draw is one readlane and one writelane.
__device__ __forceinline__ unsigned ranff_mul(unsigned a, unsigned b)
{
    const unsigned long long p = (unsigned long long)a * b;
    unsigned r = (unsigned)(p & 0x7fffffffu) + (unsigned)(p >> 31);
    return r >= 0x7fffffffu ? r - 0x7fffffffu : r;      // a <= 2^31 - 1, b < 2^31 - 1: one fold is enough
}

__device__ __forceinline__ void ranff_draws(int* st, int n, int* seq)
{
    const int lane = threadIdx.x & 63;
    const int IM = 2147483647;
    // 16807^(lane + 1) mod IM by squaring
    unsigned pw = 1, sq = 16807u;
    for (int e = lane + 1; e; e >>= 1) {
        if (e & 1) pw = ranff_mul(pw, sq);
        sq = ranff_mul(sq, sq);
    }
    int idum = __builtin_amdgcn_readfirstlane(st[0]), iy = __builtin_amdgcn_readfirstlane(st[1]);
    int iv = lane < 32 ? st[2 + lane] : 0;
    auto seed = [&]() {
        idum = (-idum > 1) ? -idum : 1;
        // 8 warm-up values, then the table from iv(32) down to iv(1): value 9 + q of the
        // stream is iv(32 - q)
        const unsigned x = ranff_mul((unsigned)(idum % IM), pw);
        iv = __shfl((int)x, 39 - (lane & 31), 64);
        idum = __builtin_amdgcn_readlane((int)x, 39);
        iy = __builtin_amdgcn_readlane(iv, 0);
    };
    if (idum <= 0 || iy == 0) seed();
    // draws [n0, n0 + m), m <= 64
    auto draws = [&](int n0, int m) {
        const int x = (int)ranff_mul((unsigned)idum, pw);
        int out = 0;
        for (int q = 0; q < m; ++q) {
            const int j = iy >> 26;                     // iy / NDIV, NDIV = 1 + (IM - 1) / 32 = 2^26
            iy = __builtin_amdgcn_readlane(iv, j);
            iv = lane == j ? __builtin_amdgcn_readlane(x, q) : iv;
            out = lane == q ? iy : out;
        }
        idum = __builtin_amdgcn_readlane(x, m - 1);
        if (lane < m) seq[n0 + lane] = out;
    };
    if (idum % IM != 0 && !__any(lane < 32 && iv == 0)) {
        for (int n0 = 0; n0 < n; n0 += 64) draws(n0, min(64, n - n0));
    } else {
        // A seed that IM divides gives zeros only, and a table that holds a zero can hand it to
        // iy: the next draw then seeds the generator again.  From any other state no zero comes.
        for (int q = 0; q < n; ++q) {
            if (q > 0 && (idum <= 0 || iy == 0)) seed();
            draws(q, 1);
        }
    }
    if (lane == 0) { st[0] = idum; st[1] = iy; }
    if (lane < 32) st[2 + lane] = iv;
}

// Index of mode (i, j, k) (1-based j, k; i = 0 real part) in a forcing table a(6,5,5)
__device__ __forceinline__ int sth_at(int j, int k) { return 6 * ((j - 1) + 5 * (k - 1)); }

// The Hermitian fix-up of the kx = 0 modes of a table (flowlib.f90:424-440, 481-510): pair q
// of 12, whose target is never another pair's source; then the mean mode is zero
__device__ __forceinline__ void sth_hermitian(double* t, int q)
{
    int src, dst;
    if (q < 10) {
        const int k = q / 2 + 1, j = q % 2 + 2;
        src = sth_at(j, k);
        dst = sth_at(7 - j, k == 1 ? 1 : 7 - k);
    } else {
        const int k = q - 8;                            // 2, 3
        src = sth_at(1, k);
        dst = sth_at(1, 7 - k);
    }
    t[dst] = t[src];
    t[dst + 1] = -t[src + 1];
    if (q == 0) { t[0] = 0.0; t[1] = 0.0; }
}

// supforSTH by the whole work-group: the draws by one wavefront, then one mode per thread (225
// modes of white noise, 150 table entries per component).  The loops over the tables run once per
// step on one work-group, so latency is all they cost (24 us, half of them the chain of draws).
// It reads no field of the step: where a whole step is queued at once, a work-group of the x
// stage does it beside the lines (a step at 64^3 FP32 64 -> 55 us, at 32^3 FP64 63 -> 44, at 128^3
// FP32 107 -> 88).
constexpr int OU_SCRATCH = 900 + 225;          // doubles of LDS
__device__ __forceinline__ void ou_step(const PreArgs& a, int rr, double* scratch)
{
    const int tid = threadIdx.x;
    double* low = a.low + (size_t)rr * LOW_STRIDE;
    const bool own = a.forcing < 0;
    int* st = a.sth_state + (size_t)rr * STH_STATE_STRIDE;
    double (*fr)[150] = (double (*)[150])scratch, (*fo)[150] = fr + 3;
    int* seq = (int*)(scratch + 900);
    const double dt = a.dt, tf = own ? low[LOW_PAR + 3] : a.ou_tf, var = own ? low[LOW_PAR + 4] : a.ou_var;
    const double pi2 = a.pi2;
    if (tid < 64) ranff_draws(st, 450, seq);
    __syncthreads();
    if (tid < 225) {                                                 // flowlib.f90:405-419
        const double AM = 1.0 / 2147483647, RNMX = 1.0 - 1.2e-7;
        double cont1 = AM * (double)seq[2 * tid], rph = AM * (double)seq[2 * tid + 1];
        cont1 = cont1 < RNMX ? cont1 : RNMX;
        rph = rph < RNMX ? rph : RNMX;
        if (cont1 < 1.e-6) cont1 = 1.e-6;
        const double rmag = sqrt(-4.0 * var * dt * log(cont1) / tf);
        const int mc = tid / 75, o = 2 * (tid % 75);
        fr[mc][o] = rmag * cos(pi2 * rph);
        fr[mc][o + 1] = rmag * sin(pi2 * rph);
    }
    __syncthreads();
    if (tid < 36) sth_hermitian(fr[tid / 12], tid % 12);             // 424-440
    __syncthreads();
    double* b = a.sth_b + (size_t)rr * STH_B_STRIDE;
    double* fa = low + 8;
    if (tid < 150) {                                                 // 447-478
        const double smallx = 1.0e-18, xkf = sqrt(8.0);
        const int o = tid, i = o % 6, j = (o / 6) % 5, k = o / 30;
        const double kx_ = (double)(i / 2);
        const double ky_ = (double)(j <= 2 ? j : j - 5);
        const double kz_ = (double)(k <= 2 ? k : k - 5);
        const double radm = sqrt(kx_ * kx_ + ky_ * ky_ + kz_ * kz_);
        double f0 = 0.0, f1 = 0.0, f2 = 0.0;
        if (radm < xkf) {
            const double b0 = b[o] * (1.0 - dt / tf) + fr[0][o];
            const double b1 = b[150 + o] * (1.0 - dt / tf) + fr[1][o];
            const double b2 = b[300 + o] * (1.0 - dt / tf) + fr[2][o];
            b[o] = b0; b[150 + o] = b1; b[300 + o] = b2;
            const double t1 = kx_ * b0, t2 = ky_ * b1, t3 = kz_ * b2;
            double divb = (t1 + t2 + t3) / ((radm + smallx) * (radm + smallx));
            if (radm == 0.) divb = 0.0;
            f0 = b0 - kx_ * divb;
            f1 = b1 - ky_ * divb;
            f2 = b2 - kz_ * divb;
        }
        fo[0][o] = f0; fo[1][o] = f1; fo[2][o] = f2;
    }
    __syncthreads();
    if (tid < 36) sth_hermitian(fo[tid / 12], tid % 12);             // 481-510
    __syncthreads();
    for (int e = tid; e < 450; e += NT) fa[e] = fo[e / 150][e % 150];
}

// Fused x stage: six C2R (u, w), physical u for the droplets, u x w, three R2C.
// The C2R transforms run two fields at a time and the R2C transforms three at a time
// through the same FFT passes, so every pass has two or three butterflies per lane;
// the next pair's loads are in flight while the current pair is transformed.
// OU: the first nou work-groups do the step's stochastic forcing (ou_step), one a realisation.
template <typename T, int N, bool OU>
__global__ void __launch_bounds__(NT) k_x_fused(KxArgs a, PreArgs pre, int nou)
{
    using C = cpx<T>;
    constexpr int M = N / 2;
    constexpr int TL = kxf_lines<T, N>();
    constexpr int LDR = TL + 1;
    constexpr int TS = M * LDR;
    constexpr int QP = TL * M / NT;
    static_assert((TL * M) % NT == 0, "the lines must split evenly over the work-group");
    constexpr size_t LDS = 3 * TS * sizeof(C), NEED = OU && LDS < OU_SCRATCH * sizeof(double) ? OU_SCRATCH * sizeof(double) : LDS;
    __shared__ __align__(16) char ldsb[NEED];
    C* const lds = (C*)ldsb;
    __shared__ C tws[N], twhs[M];
    const int tid = threadIdx.x;
    if (OU && (int)blockIdx.x < nou) {
        ou_step(pre, blockIdx.x, (double*)ldsb);
        return;
    }
    const size_t line0 = (size_t)(blockIdx.x - (OU ? nou : 0)) * TL;
    stage_twiddles<C, N, NT>(tws, (const C*)a.tw, tid);
    stage_twiddles<C, M, NT>(twhs, (const C*)a.twh, tid);
    const C* tw = tws;
    const C* twh = twhs;
    C ph[6][QP];
    TileRegs<C, TL, M, NT> next0, next1;
    // field f of this work-group's lines; every line is read before it is written
    auto fetch = [&](TileRegs<C, TL, M, NT>& r, int f) {
        if (f < 3) tile_fetch<C, TL, M, NT>(r, (const C*)a.B[f] + line0 * M, M, tid);
        else tile_fetch<C, TL, M, NT>(r, (const C*)a.uphys + (3 * line0 + f - 3) * M, 3 * M, tid);
    };
    fetch(next0, 0);
    fetch(next1, 1);
#pragma unroll
    for (int f = 0; f < 6; f += 2) {
        tile_put<C, TL, M, LDR, NT, true>(lds, next0, tid);
        tile_put<C, TL, M, LDR, NT, true>(lds + TS, next1, tid);
        if (f < 4) {
            fetch(next0, f + 2);
            fetch(next1, f + 3);
        }
        __syncthreads();
        c2r_pack<T, N, TL, LDR>(lds, tw, tid);
        c2r_pack<T, N, TL, LDR>(lds + TS, tw, tid);
        __syncthreads();
        fft_tile<T, M, true, TL, LDR, NT, 2, TS>(lds, twh, tid);
#pragma unroll
        for (int q = 0; q < QP; ++q) {
            const int e = tid + NT * q;
            const int line = e / M, m = e % M;
            ph[f][q] = lds[m * LDR + line];
            ph[f + 1][q] = lds[TS + m * LDR + line];
        }
        __syncthreads();
    }
    // physical velocity for the droplet gather: [line][x][3], the two nodes of a complex
    // value in three vector stores
    {
        T* up = (T*)a.uphys + line0 * (size_t)N * 3;
#pragma unroll
        for (int q = 0; q < QP; ++q) {
            const int e = tid + NT * q;
            const int line = e / M, m = e % M;
            T* p = up + ((size_t)line * N + 2 * m) * 3;
            store_node_pair(p, ph[0][q].x, ph[1][q].x, ph[2][q].x, ph[0][q].y, ph[1][q].y, ph[2][q].y);
        }
    }
    // nonlinear term u x w (turb.f90:634-637) in natural component order, into the
    // three tiles
#pragma unroll
    for (int q = 0; q < QP; ++q) {
        const int e = tid + NT * q;
        const int line = e / M, m = e % M;
        const C ux = ph[0][q], uy = ph[1][q], uz = ph[2][q];
        const C wx = ph[3][q], wy = ph[4][q], wz = ph[5][q];
        lds[m * LDR + line] = mk<C>(uy.x * wz.x - uz.x * wy.x, uy.y * wz.y - uz.y * wy.y);
        lds[TS + m * LDR + line] = mk<C>(uz.x * wx.x - ux.x * wz.x, uz.y * wx.y - ux.y * wz.y);
        lds[2 * TS + m * LDR + line] = mk<C>(ux.x * wy.x - uy.x * wx.x, ux.y * wy.y - uy.y * wx.y);
    }
    __syncthreads();
    fft_tile<T, M, false, TL, LDR, NT, 3, TS>(lds, twh, tid);
    const T scale = (T)1 / (T)N;
#pragma unroll
    for (int c = 0; c < 3; ++c) r2c_unpack_store<T, N, TL, LDR>(lds + c * TS, tw, (C*)a.B[c], line0, scale, tid);
}

// supforDET's 225 low-mode sums (75 modes kx in 0..2, ky, kz in -2..2, times 3
// components) of the forward z transform of N-hat, by direct DFT: one work-group per
// sum, lanes over z, a fixed-order reduction; the result, scaled by 1/N like the
// forward FFT, goes to low[LOW_DFT ...] for k_pre.
template <typename T, int N>
__global__ void __launch_bounds__(NT) k_pre_dft(PreArgs a)
{
    using C = cpx<T>;
    constexpr int M = N / 2;
    const int id = blockIdx.x, comp = id / 75, mi = id % 75;
    const int kx = mi % 3, kyw = (mi / 3) % 5 - 2, kzw = mi / 15 - 2;
    const int ky = (kyw + N) % N, kzi = (kzw + N) % N;
    double* low = a.low + (size_t)blockIdx.y * LOW_STRIDE;     // realisation blockIdx.y
    if (real_forcing(a.forcing, low) != 1) return;
    const C* b = (const C*)a.B[comp] + (size_t)blockIdx.y * a.rstride;
    const C* tw = (const C*)a.tw;
    double sr = 0.0, si = 0.0;
    for (int z = threadIdx.x; z < N; z += NT) {
        const C v = b[pipe_index<T>(N, z, ky, kx)];
        const C w = tw[(kzi * z) & (N - 1)];
        sr += (double)v.x * (double)w.x - (double)v.y * (double)w.y;
        si += (double)v.x * (double)w.y + (double)v.y * (double)w.x;
    }
    __shared__ double wr[NT / 64], wi[NT / 64];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        sr += __shfl_xor(sr, o, 64);
        si += __shfl_xor(si, o, 64);
    }
    if ((threadIdx.x & 63) == 0) { wr[threadIdx.x >> 6] = sr; wi[threadIdx.x >> 6] = si; }
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = 0.0, i = 0.0;
#pragma unroll
        for (int w = 0; w < NT / 64; ++w) { r += wr[w]; i += wi[w]; }
        low[LOW_DFT + id] = r / N;
        low[LOW_DFT + 225 + id] = i / N;
    }
}

template <typename T, int N>
__global__ void __launch_bounds__(NT) k_pre(PreArgs a)
{
    using C = cpx<T>;
    constexpr int M = N / 2;
    const int tid = threadIdx.x;
    const int rr = blockIdx.x;                                       // realisation
    double* low = a.low + (size_t)rr * LOW_STRIDE;
    const int forcing = real_forcing(a.forcing, low);
    const bool own = a.forcing < 0;
    if (forcing == 2) {
        __shared__ double scratch[OU_SCRATCH];
        ou_step(a, rr, scratch);
        return;
    }
    if (forcing != 1) return;
    // 75 low modes: kx in 0..2, ky, kz in -2..2; 225 (mode, component) DFT sums
    __shared__ double nre[225], nim[225];
    __shared__ double emode[75];
    if (tid < 225) {                      // the z-DFT sums of k_pre_dft
        nre[tid] = low[LOW_DFT + tid];
        nim[tid] = low[LOW_DFT + 225 + tid];
    }
    __syncthreads();
    if (tid < 75) {
        const int kx = tid % 3, kyw = (tid / 3) % 5 - 2, kzw = tid / 15 - 2;
        const int ky = (kyw + N) % N, kz = (kzw + N) % N;
        const size_t g = spec_index<T>(N, kz, ky, kx);
        C nn[3], uu[3], oo[3], vv[3], nd[3];
        for (int q = 0; q < 3; ++q) {
            nn[q] = mk<C>((T)nre[q * 75 + tid], (T)nim[q * 75 + tid]);
            uu[q] = ((const C*)a.U[q])[(size_t)rr * a.rstride + g];
            oo[q] = ((const C*)a.O[q])[(size_t)rr * a.rstride + g];
        }
        // the update without the forcing factor (ff = 1 here)
        double one[2] = {1.0, 1.0};
        update_mode<T>(kx, ky, kz, N, a.nek, 0, (T)a.dt, (T)a.rnu, one, nn, uu, oo, vv, nd);
        const double k2 = (double)(kx * kx + kyw * kyw + kzw * kzw);
        const int ik2 = (int)(sqrt(k2 == 0.0 ? 1.e-5 : k2) + 0.5);
        double e = 0.0;
        if (ik2 == 1 || ik2 == 2) {
            for (int q = 0; q < 3; ++q) e += (double)vv[q].x * (double)vv[q].x + (double)vv[q].y * (double)vv[q].y;
            if (kx == 0) e *= 0.5;
            e = (ik2 == 1) ? e : -e;      // sign tags the shell
        }
        emode[tid] = e;
    }
    __syncthreads();
    if (tid == 0) {
        double e1 = 0.0, e2 = 0.0;
        for (int i = 0; i < 75; ++i) {
            if (emode[i] > 0) e1 += emode[i];
            else e2 -= emode[i];
        }
        low[0] = sqrt((own ? low[LOW_PAR + 1] : a.force0) / e1);
        low[1] = sqrt((own ? low[LOW_PAR + 2] : a.force1) / e2);
        low[2] = e1;
        low[3] = e2;
    }
}

// ------------------------------------------------------------------ kx = 0 plane of u-hat
template <typename T, int N>
__global__ void k_sym(void* u0, void* u1, void* u2, size_t rstride, double* low)
{
    // the z stage before this kernel wrote every mode beyond the dealiasing sphere
    if (blockIdx.x == 0 && threadIdx.x == 0) low[(size_t)blockIdx.y * LOW_STRIDE + LOW_ZOUT] = 1.0;
    using C = cpx<T>;
    constexpr int M = N / 2;
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= N * N) return;
    const int ky = t / N, kz = t % N;
    const int mz = (N - kz) & (N - 1), my = (N - ky) & (N - 1);
    if (my * N + mz < t) return;           // the partner with the smaller index does the pair
    void* fs[3] = {u0, u1, u2};
#pragma unroll
    for (int q = 0; q < 3; ++q) {
        C* f = (C*)fs[q] + (size_t)blockIdx.y * rstride;     // realisation blockIdx.y
        const size_t gp = spec_index<T>(N, kz, ky, 0), gm = spec_index<T>(N, mz, my, 0);
        const C p = f[gp], m = f[gm];
        const C s = mk<C>((T)0.5 * (p.x + m.x), (T)0.5 * (p.y - m.y));
        f[gp] = s;
        f[gm] = cconj(s);
    }
}

// ------------------------------------------------------------------ initial field
// The random start of initial_flow (flowlib.f90:53-144) on the device.  The reference
// draws from Intel's IFPORT rand, which is not available; here every mode draws its own
// pair of uniforms from a counter-based generator, SplitMix64 (Steele, Lea and Flood,
// "Fast splittable pseudorandom number generators", OOPSLA 2014): output i of the
// stream with key s is the SplitMix64 finaliser of s + (i + 1) * 0x9E3779B97F4A7C15.
__device__ __forceinline__ double init_uniform(unsigned long long key, unsigned long long i)
{
    unsigned long long z = key + (i + 1ull) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    z ^= z >> 31;
    return (double)(z >> 11) * 0x1.0p-53;                      // [0, 1)
}

// Box-Muller pair of component c at mode (kz, ky, kx), as flowlib.f90:158-172 forms it
// from two uniforms (each held above 1e-10)
template <int N>
__device__ __forceinline__ double2 init_gauss(unsigned long long key, int c, int kz, int ky, int kx)
{
    const unsigned long long m = (((unsigned long long)c * N + kz) * N + ky) * (N / 2) + kx;
    double t1 = init_uniform(key, 2 * m), t2 = init_uniform(key, 2 * m + 1);
    if (t1 <= 1.e-10) t1 = 1.e-10;
    if (t2 <= 1.e-10) t2 = 1.e-10;
    const double a = sqrt(-2.0 * log(t1)), ph = 2.0 * 3.14159265358979323846 * t2;
    return make_double2(a * cos(ph), a * sin(ph));
}

// One thread per mode: the three Gaussian components, the Hermitian kx = 0 plane
// ((g(k) + conj g(-k)) / 2, computed from both draws so the two halves agree), the
// Nyquist planes and the mean set to zero, the projection onto k.u = 0 (flowlib.f90:
// 94-101); then twice the shell's mode count, 2 per mode with kx > 0 and 1 on the kx = 0
// plane (flowlib.f90:107-118).  The shell energies are summed afterwards by the E(k)
// reduction (kx = 0 modes at half weight), whose fixed order makes the field the same
// bits on every run.
template <typename T, int N>
__global__ void __launch_bounds__(256) k_init_modes(void* u0, void* u1, void* u2, unsigned long long key, int nek,
                                                    unsigned long long* cnt2)
{
    using C = cpx<T>;
    constexpr int M = N / 2;
    // the counts of a work-group's modes in LDS first: one global atomic per mode made this
    // kernel 6.5 ms at 256^3 and 131 ms at 1024^3
    __shared__ unsigned cnt[M];
    for (int i = threadIdx.x; i < M; i += 256) cnt[i] = 0;
    __syncthreads();
    for (size_t t = (size_t)blockIdx.x * 256 + threadIdx.x; t < (size_t)N * N * M; t += (size_t)gridDim.x * 256) {
        int kx, ky, kz;
        spec_mode<T>(N, t, kz, ky, kx);
        const int kyw = wave_index(ky, N), kzw = wave_index(kz, N);
        const bool zero = ky == N / 2 || kz == N / 2 || (kx == 0 && ky == 0 && kz == 0);
        double2 g[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            g[c] = init_gauss<N>(key, c, kz, ky, kx);
            if (kx == 0) {
                const double2 h = init_gauss<N>(key, c, (N - kz) & (N - 1), (N - ky) & (N - 1), 0);
                g[c] = make_double2(0.5 * (g[c].x + h.x), 0.5 * (g[c].y - h.y));
            }
            if (zero) g[c] = make_double2(0.0, 0.0);
        }
        const double k[3] = {(double)kx, (double)kyw, (double)kzw};
        double k2 = k[0] * k[0] + k[1] * k[1] + k[2] * k[2];
        if (kx == 0 && ky == 0 && kz == 0) k2 = 1.e-5;
        const double pr = (k[0] * g[0].x + k[1] * g[1].x + k[2] * g[2].x) / k2;
        const double pi = (k[0] * g[0].y + k[1] * g[1].y + k[2] * g[2].y) / k2;
        void* u[3] = {u0, u1, u2};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const double x = g[c].x - k[c] * pr, y = g[c].y - k[c] * pi;
            ((C*)u[c])[t] = mk<C>((T)x, (T)y);
        }
        const int ik2 = (int)(sqrt(k2) + 0.5);
        // twice the shell's mode count (kx = 0 modes count one half): integer sums, the same
        // in any order; the shell energies come from the fixed-tree E(k) reduction
        if (ik2 >= 1 && ik2 <= nek) atomicAdd(cnt + ik2 - 1, kx == 0 ? 1u : 2u);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < nek; i += 256)
        if (cnt[i]) atomicAdd(cnt2 + i, (unsigned long long)cnt[i]);
}

// the shell factors (flowlib.f90:119-137), and zero above nek (139-141)
template <typename T, int N>
__global__ void k_init_scale(void* u0, void* u1, void* u2, int nek, const double* fac)
{
    using C = cpx<T>;
    constexpr int M = N / 2;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)N * N * M) return;
    int kx, ky, kz;
    spec_mode<T>(N, t, kz, ky, kx);
    const int kyw = wave_index(ky, N), kzw = wave_index(kz, N);
    double k2 = (double)(kx * kx + kyw * kyw + kzw * kzw);
    if (k2 == 0.0) k2 = 1.e-5;
    const int ik2 = (int)(sqrt(k2) + 0.5);
    if (ik2 < 1) return;
    const double f = ik2 <= nek ? fac[ik2 - 1] : 0.0;
    void* u[3] = {u0, u1, u2};
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        C v = ((C*)u[c])[t];
        v = mk<C>((T)((double)v.x * f), (T)((double)v.y * f));
        ((C*)u[c])[t] = v;
    }
}

// ================================================================== host side
static size_t field_elems(int N) { return (size_t)N * N * (N / 2); }

int flow_alloc(FlowBuffers& fb, int N, int precision, int R)
{
    const size_t cs = (precision == DDNS_FP64) ? sizeof(double2) : sizeof(float2);
    const size_t rs = (precision == DDNS_FP64) ? sizeof(double) : sizeof(float);
    if (R < 1) R = 1;
    fb.R = R;
    fb.rstride = R > 1 ? field_elems(N) : 0;
    fb.pstride = R > 1 ? (size_t)N * N * N * 3 : 0;
    const size_t fe = field_elems(N) * R;
    for (int i = 0; i < 3; ++i) {
        DDNS_HIP(hipMalloc(&fb.U[i], fe * cs));
        DDNS_HIP(hipMalloc(&fb.O[i], fe * cs));
        DDNS_HIP(hipMalloc(&fb.B[i], fe * cs));
        DDNS_HIP(hipMemset(fb.U[i], 0, fe * cs));
        DDNS_HIP(hipMemset(fb.O[i], 0, fe * cs));
    }
    for (int i = 0; i < 6; ++i) DDNS_HIP(hipMalloc(&fb.A[i], fe * cs));
    DDNS_HIP(hipMalloc(&fb.uphys, (size_t)N * N * N * 3 * rs * R));
    DDNS_HIP(hipMemset(fb.uphys, 0, (size_t)N * N * N * 3 * rs * R));
    // twiddles exp(-2 pi i m / L), computed in double and rounded once
    for (int pass = 0; pass < 2; ++pass) {
        const int L = pass == 0 ? N : N / 2;
        std::vector<double> d(2 * (size_t)L);
        for (int m = 0; m < L; ++m) {
            const double ang = -2.0 * M_PI * (double)m / (double)L;
            d[2 * m] = std::cos(ang);
            d[2 * m + 1] = std::sin(ang);
        }
        void** dst = pass == 0 ? &fb.tw : &fb.twh;
        if (precision == DDNS_FP64) {
            DDNS_HIP(hipMalloc(dst, d.size() * sizeof(double)));
            DDNS_HIP(hipMemcpy(*dst, d.data(), d.size() * sizeof(double), hipMemcpyHostToDevice));
        } else {
            std::vector<float> f(d.begin(), d.end());
            DDNS_HIP(hipMalloc(dst, f.size() * sizeof(float)));
            DDNS_HIP(hipMemcpy(*dst, f.data(), f.size() * sizeof(float), hipMemcpyHostToDevice));
        }
    }
    DDNS_HIP(hipMalloc(&fb.low, (size_t)LOW_STRIDE * R * sizeof(double)));
    DDNS_HIP(hipMemset(fb.low, 0, (size_t)LOW_STRIDE * R * sizeof(double)));
    DDNS_HIP(hipMalloc(&fb.sth_state, (size_t)STH_STATE_STRIDE * R * sizeof(int)));
    DDNS_HIP(hipMemset(fb.sth_state, 0, (size_t)STH_STATE_STRIDE * R * sizeof(int)));
    DDNS_HIP(hipMalloc(&fb.sth_b, (size_t)STH_B_STRIDE * R * sizeof(double)));
    DDNS_HIP(hipMemset(fb.sth_b, 0, (size_t)STH_B_STRIDE * R * sizeof(double)));
    DDNS_HIP(hipMalloc(&fb.spec_part, ((size_t)SPEC_BLOCKS + 1) * SPEC_NEK_MAX * sizeof(double)));
    return 0;
}

FlowBuffers flow_view(const FlowBuffers& fb, int r, int precision)
{
    const size_t cs = (precision == DDNS_FP64) ? sizeof(double2) : sizeof(float2);
    const size_t rs = (precision == DDNS_FP64) ? sizeof(double) : sizeof(float);
    FlowBuffers v{};
    auto off = [&](void* p) { return p ? (void*)((char*)p + (size_t)r * fb.rstride * cs) : nullptr; };
    for (int i = 0; i < 3; ++i) { v.U[i] = off(fb.U[i]); v.O[i] = off(fb.O[i]); v.B[i] = off(fb.B[i]); }
    for (int i = 0; i < 6; ++i) v.A[i] = off(fb.A[i]);
    v.uphys = (char*)fb.uphys + (size_t)r * fb.pstride * rs;
    v.tw = fb.tw; v.twh = fb.twh;
    v.low = fb.low + (size_t)r * LOW_STRIDE;
    v.sth_state = fb.sth_state + (size_t)r * STH_STATE_STRIDE;
    v.sth_b = fb.sth_b + (size_t)r * STH_B_STRIDE;
    v.ky_tc = fb.ky_tc; v.kz_nt = fb.kz_nt;
    return v;
}

int flow_set_realisation(const FlowBuffers& fb, int r, int forcing, double force0, double force1, double ou_tf,
                         double ou_var)
{
    const double par[5] = {(double)forcing, force0, force1, ou_tf, ou_var};
    DDNS_HIP(hipMemcpy(fb.low + (size_t)r * LOW_STRIDE + LOW_PAR, par, sizeof(par), hipMemcpyHostToDevice));
    return 0;
}

void flow_free(FlowBuffers& fb)
{
    for (int i = 0; i < 3; ++i) { (void)hipFree(fb.U[i]); (void)hipFree(fb.O[i]); (void)hipFree(fb.B[i]); }
    for (int i = 0; i < 6; ++i) (void)hipFree(fb.A[i]);
    (void)hipFree(fb.uphys); (void)hipFree(fb.tw); (void)hipFree(fb.twh);
    (void)hipFree(fb.low); (void)hipFree(fb.sth_state); (void)hipFree(fb.sth_b);
    for (int q = 0; q < 8; ++q) if (fb.dg[q]) (void)hipFree(fb.dg[q]);
    if (fb.dg_part) (void)hipFree(fb.dg_part);
    if (fb.spec_part) (void)hipFree(fb.spec_part);
    if (fb.stage) (void)hipFree(fb.stage);
    if (fb.bounce.host) (void)hipHostFree(fb.bounce.host);
    fb = FlowBuffers{};
}

// the fused z stage (or, not FULL, the curl and inverse transforms) at tile width TC
template <typename T, int N, int TC, bool FULL>
static bool launch_z_tc(const KzArgs& a, int R, hipStream_t s)
{
    if constexpr (kz_fits<T, N, TC>()) {
        hipLaunchKernelGGL((k_z_full<T, N, TC, FULL>), dim3((unsigned)(N / 2 / TC * N * R)), dim3(kz_threads<T, N, TC>()), 0,
                           s, a);
        return true;
    } else {
        return false;
    }
}

template <typename T, int N>
static int launch_z(int mode, const FlowBuffers& fb, const FlowConst& fc, hipStream_t s,
                    const void* src = nullptr, void* dst = nullptr, double scale = 1.0)
{
    KzArgs a{};
    for (int i = 0; i < 3; ++i) { a.B[i] = fb.A[i]; a.U[i] = fb.U[i]; a.O[i] = fb.O[i]; }
    for (int i = 0; i < 6; ++i) a.A[i] = fb.A[i];
    a.tw = fb.tw; a.low = fb.low; a.dt = fc.dt; a.rnu = fc.rnu; a.nek = fc.nek; a.forcing = fc.forcing;
    a.scale = scale;
    a.rstride = fb.rstride;
    const int R = fb.R;
    if (mode == KZ_PLAIN_FWD || mode == KZ_PLAIN_INV) { a.B[0] = src; a.U[0] = dst; a.rstride = 0; }
    constexpr unsigned gp = (unsigned)(N / 2 / kz_tc_plain<T, N>() * N);
    constexpr unsigned np = kz_plain_threads<T, N>();
    if (mode == KZ_PLAIN_FWD || mode == KZ_PLAIN_INV) {
        if (mode == KZ_PLAIN_FWD) hipLaunchKernelGGL((k_z<T, N, false>), dim3(gp), dim3(np), 0, s, a);
        else hipLaunchKernelGGL((k_z<T, N, true>), dim3(gp), dim3(np), 0, s, a);
        DDNS_HIP(hipGetLastError());
        return 0;
    }
    static_assert(kz_fits<T, N, kz_tc<T, N>()>(), "the default z tile must fit");
    if (mode == KZ_FULL && fb.kz_nt == kz_threads<T, N, kz_cand<T, N>(1)>() && launch_z_tc<T, N, kz_cand<T, N>(1), true>(a, R, s))
        ;
    else if (mode == KZ_FULL) (void)launch_z_tc<T, N, kz_tc<T, N>(), true>(a, R, s);
    else (void)launch_z_tc<T, N, kz_tc<T, N>(), false>(a, R, s);
    DDNS_HIP(hipGetLastError());
    return 0;
}

template <typename T, int N, int TC>
static void launch_y_tc(bool inv, bool sym, const KyArgs& a, int nf, int planes, hipStream_t s)
{
    const dim3 grid(N / 2 / TC, planes, nf), nt(TC * (N / col_e<T, N>()));
    if (inv && sym) hipLaunchKernelGGL((k_y<T, N, true, true, TC>), grid, nt, 0, s, a);
    else if (inv) hipLaunchKernelGGL((k_y<T, N, true, false, TC>), grid, nt, 0, s, a);
    else hipLaunchKernelGGL((k_y<T, N, false, false, TC>), grid, nt, 0, s, a);
}

// candidate k of the y-stage tile widths (0 = half, 1 = default, 2 = twice the default)
template <typename T, int N, int K>
static bool launch_y_cand(bool inv, bool sym, const KyArgs& a, int nf, int planes, hipStream_t s)
{
    constexpr int TC = ky_cand<T, N>(K);
    if constexpr (ky_fits<T, N, TC>()) {
        launch_y_tc<T, N, TC>(inv, sym, a, nf, planes, s);
        return true;
    } else {
        return false;
    }
}

// the y stage of nf fields of planes planes at the tile width fb.ky_tc (0: the default); nek > 0:
// the stage of a step, which leaves out the rows beyond the dealiasing sphere
template <typename T, int N>
static int launch_y(bool inv, bool sym, void* const* f, const PlainRows& rows, int nf, const FlowBuffers& fb, int planes,
                    hipStream_t s, int nek = 0)
{
    KyArgs a{};
    for (int i = 0; i < nf; ++i) a.F[i] = f[i];
    a.L = rows;
    a.tw = fb.tw;
    a.scale = 1.0 / N;
    a.rstride = fb.rstride;
    a.low = nek > 0 ? fb.low : nullptr;
    a.nek = nek;
    static_assert(ky_fits<T, N, ky_tc<T, N>()>(), "the default y tile must fit");
    const int tc = fb.ky_tc;
    bool done = false;
    if (tc == ky_cand<T, N>(0)) done = launch_y_cand<T, N, 0>(inv, sym, a, nf, planes, s);
    else if (tc == ky_cand<T, N>(2)) done = launch_y_cand<T, N, 2>(inv, sym, a, nf, planes, s);
    if (!done) launch_y_tc<T, N, ky_tc<T, N>()>(inv, sym, a, nf, planes, s);
    DDNS_HIP(hipGetLastError());
    return 0;
}

// One field as plain rows.
template <int N> static PlainRows plain_field(void* p)
{
    PlainRows r{};
    r.p[0] = p;
    r.rs[0] = N / 2;
    return r;
}

// The step's fields between the y and x stages: u (and, after the x stage, u x w) in B, one
// after the other; w in the physical velocity's memory, the rows of its three components
// side by side, which are the line's three real components once the x stage has read them.
template <typename T, int N>
static PlainRows plain_rows(const FlowBuffers& fb)
{
    PlainRows r{};
    for (int i = 0; i < 3; ++i) {
        r.p[i] = fb.B[i];
        r.rs[i] = N / 2;
        r.p[3 + i] = (cpx<T>*)fb.uphys + i * (N / 2);
        r.rs[3 + i] = 3 * (N / 2);
    }
    return r;
}

template <typename T, int N>
static PreArgs pre_args(const FlowBuffers& fb, const FlowConst& fc)
{
    PreArgs a{};
    for (int i = 0; i < 3; ++i) { a.B[i] = fb.A[i]; a.U[i] = fb.U[i]; a.O[i] = fb.O[i]; }
    a.tw = fb.tw; a.low = fb.low; a.sth_state = fb.sth_state; a.sth_b = fb.sth_b;
    a.dt = fc.dt; a.rnu = fc.rnu; a.force0 = fc.force0; a.force1 = fc.force1;
    a.ou_tf = fc.ou_tf; a.ou_var = fc.ou_var; a.pi2 = fc.pi2; a.nek = fc.nek; a.forcing = fc.forcing;
    a.rstride = fb.rstride;
    return a;
}

// ou: the step's stochastic forcing as well, one more work-group for each realisation
template <typename T, int N>
static int launch_x(const FlowBuffers& fb, const FlowConst& fc, bool ou, hipStream_t s)
{
    KxArgs a{};
    for (int i = 0; i < 3; ++i) a.B[i] = fb.B[i];
    a.uphys = fb.uphys; a.tw = fb.tw; a.twh = fb.twh;
    const unsigned nb = (unsigned)((size_t)fb.R * N * N / kxf_lines<T, N>());
    const PreArgs p = pre_args<T, N>(fb, fc);
    if (ou) hipLaunchKernelGGL((k_x_fused<T, N, true>), dim3(nb + fb.R), dim3(NT), 0, s, a, p, fb.R);
    else hipLaunchKernelGGL((k_x_fused<T, N, false>), dim3(nb), dim3(NT), 0, s, a, p, 0);
    DDNS_HIP(hipGetLastError());
    return 0;
}

template <typename T, int N>
static int launch_pre(const FlowBuffers& fb, const FlowConst& fc, hipStream_t s)
{
    if (fc.forcing != 1 && fc.forcing != 2 && fc.forcing >= 0) return 0;
    const PreArgs a = pre_args<T, N>(fb, fc);
    if (fc.forcing == 1 || fc.forcing < 0) hipLaunchKernelGGL((k_pre_dft<T, N>), dim3(225, fb.R), dim3(NT), 0, s, a);
    hipLaunchKernelGGL((k_pre<T, N>), dim3(fb.R), dim3(NT), 0, s, a);
    DDNS_HIP(hipGetLastError());
    return 0;
}

template <typename T, int N>
static int launch_sym(const FlowBuffers& fb, hipStream_t s)
{
    const int tot = N * N;
    hipLaunchKernelGGL((k_sym<T, N>), dim3((tot + 255) / 256, fb.R), dim3(256), 0, s, fb.U[0], fb.U[1], fb.U[2],
                       fb.rstride, fb.low);
    DDNS_HIP(hipGetLastError());
    return 0;
}

template <typename T, int N>
static int step_impl(const FlowBuffers& fb, const FlowConst& fc, hipStream_t s, hipEvent_t* ev, int part,
                     unsigned evflags)
{
    // FLOW_INV: inverse y + fused x (produces the physical velocity);
    // FLOW_FWD: forward y + pre + z + sym (closes the step, opens the next), or its two
    // pieces FLOW_FWD_Y (forward y + pre) and FLOW_FWD_Z (z + sym).  Events: 0-2 around
    // the first half, 3 forward y, 4 pre, 5 end of pre, 8 start of z, 6 end of z, 7 end.
    // evflags = hipEventRecordExternal while the stream is being captured into a graph:
    // the timing events then become event-record nodes of the graph
    // FLOW_STEP: both halves; the stochastic forcing, which reads no field, then runs beside the x
    // stage.  (A first half alone may be queued for a step that does not follow: it leaves the
    // forcing's state alone.)
    const bool ou = part == FLOW_STEP && fc.forcing == 2;
    if (part == FLOW_INV || part == FLOW_STEP) {
        if (ev) DDNS_HIP(hipEventRecordWithFlags(ev[0], s, evflags));
        int st = launch_y<T, N>(true, true, fb.A, plain_rows<T, N>(fb), 6, fb, fb.R * N, s, fc.nek);
        if (st) return st;
        if (ev) DDNS_HIP(hipEventRecordWithFlags(ev[1], s, evflags));
        st = launch_x<T, N>(fb, fc, ou, s);
        if (st) return st;
        if (ev) DDNS_HIP(hipEventRecordWithFlags(ev[2], s, evflags));
        if (part == FLOW_INV) return 0;
    }
    int st = 0;
    if (part != FLOW_FWD_Z) {
        if (ev) DDNS_HIP(hipEventRecordWithFlags(ev[3], s, evflags));
        st = launch_y<T, N>(false, false, fb.A, plain_rows<T, N>(fb), 3, fb, fb.R * N, s, fc.nek);
        if (st) return st;
        if (ev) DDNS_HIP(hipEventRecordWithFlags(ev[4], s, evflags));
        if (!ou) st = launch_pre<T, N>(fb, fc, s);
        if (st) return st;
        if (ev) DDNS_HIP(hipEventRecordWithFlags(ev[5], s, evflags));
        if (part == FLOW_FWD_Y) return 0;
    }
    if (ev) DDNS_HIP(hipEventRecordWithFlags(ev[8], s, evflags));
    st = launch_z<T, N>(KZ_FULL, fb, fc, s);
    if (st) return st;
    if (ev) DDNS_HIP(hipEventRecordWithFlags(ev[6], s, evflags));
    st = launch_sym<T, N>(fb, s);
    if (st) return st;
    if (ev) DDNS_HIP(hipEventRecordWithFlags(ev[7], s, evflags));
    return 0;
}

#define DDNS_DISPATCH_N(N_, CALL)                         \
    switch (N_) {                                          \
    case 32: { constexpr int NN = 32; CALL; } break;       \
    case 64: { constexpr int NN = 64; CALL; } break;       \
    case 128: { constexpr int NN = 128; CALL; } break;     \
    case 256: { constexpr int NN = 256; CALL; } break;     \
    case 512: { constexpr int NN = 512; CALL; } break;     \
    case 1024: { constexpr int NN = 1024; CALL; } break;   \
    default: set_error("unsupported grid size"); return DDNS_ERR_ARG; \
    }

int flow_prologue(const FlowBuffers& fb, const FlowConst& fc, int precision, hipStream_t s)
{
    int st = 0;
    if (precision == DDNS_FP64) { DDNS_DISPATCH_N(fc.N, st = (launch_z<double, NN>(KZ_CURL_INV, fb, fc, s))) }
    else { DDNS_DISPATCH_N(fc.N, st = (launch_z<float, NN>(KZ_CURL_INV, fb, fc, s))) }
    return st;
}

int flow_step(const FlowBuffers& fb, const FlowConst& fc, int precision, int part, hipStream_t s, hipEvent_t* ev,
              bool capturing)
{
    const unsigned evflags = capturing ? hipEventRecordExternal : hipEventRecordDefault;
    int st = 0;
    if (precision == DDNS_FP64) { DDNS_DISPATCH_N(fc.N, st = (step_impl<double, NN>(fb, fc, s, ev, part, evflags))) }
    else { DDNS_DISPATCH_N(fc.N, st = (step_impl<float, NN>(fb, fc, s, ev, part, evflags))) }
    return st;
}

// ---------------------------------------------------------------- host conversion
// State transfers.  The reference's layouts are formed on the device, in a staging buffer of
// at most STAGE_BYTES (or one ky plane), and copied straight to or from the caller's arrays:
// converting in host loops, through arrays that were allocated and faulted in on each call,
// took 246 ms for the six fields of a 256^3 FP32 state against 45 ms for the copies.
constexpr size_t STAGE_BYTES = 128u << 20;

static int stage_buffer(FlowBuffers& fb, size_t bytes, double** out)
{
    if (fb.stage_bytes < bytes) {
        if (fb.stage) DDNS_HIP(hipFree(fb.stage));
        fb.stage = nullptr;
        fb.stage_bytes = 0;
        DDNS_HIP(hipMalloc(&fb.stage, bytes));
        fb.stage_bytes = bytes;
    }
    *out = (double*)fb.stage;
    return 0;
}

// Planes ky0 .. ky0 + gridDim.z of v(N+2, N+2, N) (kz fastest, then kx re/im, then ky) from
// a spectral field, with the padding rows zero (PACK), or the field from the planes.
// 32 x 32 tiles through LDS: kx is contiguous on one side, kz on the other.
template <typename T, bool PACK>
__global__ void __launch_bounds__(256) k_layout(cpx<T>* __restrict__ f, double* __restrict__ v, int N, int ky0)
{
    using C = cpx<T>;
    __shared__ C tile[32][33];
    const int L = N + 2, M = N / 2;
    const int kz0 = blockIdx.x * 32, kx0 = blockIdx.y * 32, ky = ky0 + blockIdx.z;
    const int a = threadIdx.x & 31, b = threadIdx.x >> 5;
    double* plane = v + (size_t)blockIdx.z * L * L;
    if constexpr (PACK) {
#pragma unroll
        for (int q = 0; q < 32; q += 8) {
            const int kz = kz0 + b + q, kx = kx0 + a;
            tile[b + q][a] = kz < N && kx < M ? f[spec_index<T>(N, kz, ky, kx)] : mk<C>((T)0, (T)0);
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 32; q += 8) {
            const int kz = kz0 + a, kx = kx0 + b + q;
            if (kz < L && kx <= M) {
                const C c = tile[a][b + q];
                plane[(size_t)(2 * kx) * L + kz] = (double)c.x;
                plane[(size_t)(2 * kx + 1) * L + kz] = (double)c.y;
            }
        }
    } else {
#pragma unroll
        for (int q = 0; q < 32; q += 8) {
            const int kz = kz0 + a, kx = kx0 + b + q;
            if (kz < N && kx < M)
                tile[a][b + q] = mk<C>((T)plane[(size_t)(2 * kx) * L + kz], (T)plane[(size_t)(2 * kx + 1) * L + kz]);
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 32; q += 8) {
            const int kz = kz0 + b + q, kx = kx0 + a;
            if (kz < N && kx < M) f[spec_index<T>(N, kz, ky, kx)] = tile[b + q][a];
        }
    }
}

// n planes of L x L doubles per chunk of the staging buffer
static int stage_planes(int N) { return (int)std::max<size_t>(1, std::min<size_t>(N, STAGE_BYTES / sizeof(double) / (N + 2) / (N + 2))); }

template <typename T>
static int upload_spectral(FlowBuffers& fb, void* dev, int N, const double* v, hipStream_t s)
{
    const size_t plane = (size_t)(N + 2) * (N + 2);
    const int np = stage_planes(N);
    double* st = nullptr;
    int rc = stage_buffer(fb, np * plane * sizeof(double), &st);
    if (rc) return rc;
    for (int ky = 0; ky < N; ky += np) {
        const int m = std::min(np, N - ky);
        DDNS_HIP(hipMemcpyAsync(st, v + (size_t)ky * plane, m * plane * sizeof(double), hipMemcpyHostToDevice, s));
        hipLaunchKernelGGL((k_layout<T, false>), dim3((N + 31) / 32, (N / 2 + 31) / 32, m), dim3(256), 0, s, (cpx<T>*)dev, st,
                           N, ky);
        DDNS_HIP(hipGetLastError());
    }
    DDNS_HIP(hipStreamSynchronize(s));
    return 0;
}

template <typename T>
static int download_spectral(FlowBuffers& fb, const void* dev, int N, double* v, hipStream_t s)
{
    const size_t plane = (size_t)(N + 2) * (N + 2);
    const int np = stage_planes(N);
    double* st = nullptr;
    int rc = stage_buffer(fb, np * plane * sizeof(double), &st);
    if (rc) return rc;
    for (int ky = 0; ky < N; ky += np) {
        const int m = std::min(np, N - ky);
        hipLaunchKernelGGL((k_layout<T, true>), dim3((N + 2 + 31) / 32, (N / 2 + 1 + 31) / 32, m), dim3(256), 0, s,
                           (cpx<T>*)dev, st, N, ky);
        DDNS_HIP(hipGetLastError());
        DDNS_HIP(hipMemcpyAsync(v + (size_t)ky * plane, st, m * plane * sizeof(double), hipMemcpyDeviceToHost, s));
    }
    DDNS_HIP(hipStreamSynchronize(s));
    return 0;
}

// the state's modes beyond the dealiasing sphere may be nonzero again (an upload, a new
// field): the next inverse y stage reads every column, the next z stage stores the zeros
static int mark_dense(const FlowBuffers& fb)
{
    static const double zero = 0.0;
    DDNS_HIP(hipMemcpy(fb.low + LOW_ZOUT, &zero, sizeof(double), hipMemcpyHostToDevice));
    return 0;
}

int flow_upload_state(FlowBuffers& fb, int N, int precision, const double* const src[6], hipStream_t s)
{
    DDNS_HIP(hipStreamSynchronize(s));
    const int sm = mark_dense(fb);
    if (sm) return sm;
    for (int f = 0; f < 6; ++f) {
        if (!src[f]) continue;
        void* dev = f < 3 ? fb.U[f] : fb.O[f - 3];
        const int st = precision == DDNS_FP64 ? upload_spectral<double>(fb, dev, N, src[f], s)
                                              : upload_spectral<float>(fb, dev, N, src[f], s);
        if (st) return st;
    }
    return 0;
}

int flow_download_state(FlowBuffers& fb, int N, int precision, double* const dst[6], hipStream_t s)
{
    const size_t each = (size_t)N * (N + 2) * (N + 2);
    size_t nf = 0;
    for (int f = 0; f < 6; ++f) nf += dst[f] != nullptr;
    if (nf > 0 && nf * each * sizeof(double) <= BOUNCE_FIELDS) {
        double* st = nullptr;
        int rc = bounce_room(fb.bounce, nf * each * sizeof(double));
        if (!rc) rc = stage_buffer(fb, nf * each * sizeof(double), &st);
        if (rc) return rc;
        size_t at = 0;
        for (int f = 0; f < 6; ++f) {
            if (!dst[f]) continue;
            void* dev = f < 3 ? fb.U[f] : fb.O[f - 3];
            const dim3 g((N + 2 + 31) / 32, (N / 2 + 1 + 31) / 32, N);
            if (precision == DDNS_FP64)
                hipLaunchKernelGGL((k_layout<double, true>), g, dim3(256), 0, s, (cpx<double>*)dev, st + at, N, 0);
            else
                hipLaunchKernelGGL((k_layout<float, true>), g, dim3(256), 0, s, (cpx<float>*)dev, st + at, N, 0);
            at += each;
        }
        DDNS_HIP(hipGetLastError());
        DDNS_HIP(hipMemcpyAsync(fb.bounce.host, st, at * sizeof(double), hipMemcpyDeviceToHost, s));
        DDNS_HIP(hipStreamSynchronize(s));
        at = 0;
        for (int f = 0; f < 6; ++f) {
            if (!dst[f]) continue;
            std::memcpy(dst[f], fb.bounce.host + at, each * sizeof(double));
            at += each;
        }
        return 0;
    }
    for (int f = 0; f < 6; ++f) {
        if (!dst[f]) continue;
        const void* dev = f < 3 ? fb.U[f] : fb.O[f - 3];
        const int st = precision == DDNS_FP64 ? download_spectral<double>(fb, dev, N, dst[f], s)
                                              : download_spectral<float>(fb, dev, N, dst[f], s);
        if (st) return st;
    }
    return 0;
}

// components c = 0, 1, 2 of nodes [i0, i0 + n) of the physical velocity, one after the other
template <typename T>
__global__ void __launch_bounds__(256) k_phys_planes(const T* __restrict__ u, double* __restrict__ out, size_t i0, size_t n)
{
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
#pragma unroll
    for (int c = 0; c < 3; ++c) out[c * n + i] = (double)u[3 * (i0 + i) + c];
}

template <typename T>
static int download_phys_t(FlowBuffers& fb, int N, double* ux, double* uy, double* uz, hipStream_t s)
{
    const size_t n3 = (size_t)N * N * N;
    const size_t chunk = std::min(n3, STAGE_BYTES / (3 * sizeof(double)) / 256 * 256);
    double* st = nullptr;
    const bool small = 3 * n3 * sizeof(double) <= BOUNCE_FIELDS;          // then one chunk
    int rc = stage_buffer(fb, 3 * chunk * sizeof(double), &st);
    if (!rc && small) rc = bounce_room(fb.bounce, 3 * n3 * sizeof(double));
    if (rc) return rc;
    double* d[3] = {ux, uy, uz};
    for (size_t i = 0; i < n3; i += chunk) {
        const size_t m = std::min(chunk, n3 - i);
        hipLaunchKernelGGL((k_phys_planes<T>), dim3((unsigned)((m + 255) / 256)), dim3(256), 0, s, (const T*)fb.uphys, st, i, m);
        DDNS_HIP(hipGetLastError());
        if (small) DDNS_HIP(hipMemcpyAsync(fb.bounce.host, st, 3 * m * sizeof(double), hipMemcpyDeviceToHost, s));
        for (int c = 0; c < 3; ++c)
            if (d[c] && !small) DDNS_HIP(hipMemcpyAsync(d[c] + i, st + c * m, m * sizeof(double), hipMemcpyDeviceToHost, s));
    }
    DDNS_HIP(hipStreamSynchronize(s));
    for (int c = 0; c < 3; ++c)
        if (d[c] && small) std::memcpy(d[c], fb.bounce.host + c * n3, n3 * sizeof(double));
    return 0;
}

int flow_download_phys(FlowBuffers& fb, int N, int precision, double* ux, double* uy, double* uz, hipStream_t s)
{
    return precision == DDNS_FP64 ? download_phys_t<double>(fb, N, ux, uy, uz, s)
                                  : download_phys_t<float>(fb, N, ux, uy, uz, s);
}

// ---------------------------------------------------------------- initial field
template <typename T, int N>
static int init_impl(FlowBuffers& fb, int nek, int kind, int seed, double k0, double urms, double force0,
                     hipStream_t s)
{
    const size_t tot = field_elems(N);
    const unsigned g = (unsigned)((tot + 255) / 256);
    double* d = nullptr;                       // twice the mode counts (integers), then the factors (2 nek)
    DDNS_HIP(hipMalloc(&d, 2 * (size_t)nek * sizeof(double)));
    DDNS_HIP(hipMemsetAsync(d, 0, (size_t)nek * sizeof(double), s));
    const unsigned long long key = (unsigned long long)(long long)seed;
    hipLaunchKernelGGL((k_init_modes<T, N>), dim3(std::min(g, 4096u)), dim3(256), 0, s, fb.U[0], fb.U[1], fb.U[2], key, nek,
                       (unsigned long long*)d);
    DDNS_HIP(hipGetLastError());
    std::vector<unsigned long long> c2(nek);
    std::vector<double> h(2 * (size_t)nek), fac(nek, 1.0);
    DDNS_HIP(hipMemcpyAsync(c2.data(), d, c2.size() * sizeof(unsigned long long), hipMemcpyDeviceToHost, s));
    // shell energies of the unscaled field (kx = 0 modes at half weight), by the same
    // fixed-order reduction as E(k): the same bits on every run
    int sst = flow_spectrum(fb, N, nek, sizeof(T) == 8 ? DDNS_FP64 : DDNS_FP32_MIXED, h.data(), s);
    if (sst) { (void)hipFree(d); return sst; }
    for (int i = 0; i < nek; ++i) h[nek + i] = 0.5 * (double)c2[i];
    const double* e_t = h.data();
    const double* enumv = h.data() + nek;
    const double pi = 4. * std::atan(1.);
    if (kind == DDNS_SPEC_K4_GAUSS) {
        // E(k) proportional to (k/k0)^4 exp(-2 (k/k0)^2), total 3/2 urms^2
        std::vector<double> target(nek);
        double sum = 0.0;
        for (int i = 1; i <= nek; ++i) {
            const double q = (double)i / k0;
            target[i - 1] = q * q * q * q * std::exp(-2.0 * q * q);
            sum += target[i - 1];
        }
        for (int i = 1; i <= nek; ++i) {
            const double tg = target[i - 1] * 1.5 * urms * urms / sum;
            fac[i - 1] = e_t[i - 1] > 0 ? std::sqrt(tg / e_t[i - 1]) : 0.0;
        }
    } else {
        // initial_flow's own scaling: shell 1 at force(1) per shell volume, k^(-5/3) above
        const double ccc = force0 * 4. / 3. * pi * (1.5 * 1.5 * 1.5 - 0.5 * 0.5 * 0.5) / enumv[0];
        for (int i = 1; i <= nek; ++i) {
            const double vol = 4. / 3. * pi * ((i + 0.5) * (i + 0.5) * (i + 0.5) - (i - 0.5) * (i - 0.5) * (i - 0.5));
            fac[i - 1] = e_t[i - 1] > 0 ? std::sqrt(ccc / e_t[i - 1] * enumv[i - 1] / vol) / std::pow((double)i, 0.833333)
                                        : 0.0;
        }
    }
    DDNS_HIP(hipMemcpyAsync(d + nek, fac.data(), nek * sizeof(double), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL((k_init_scale<T, N>), dim3(g), dim3(256), 0, s, fb.U[0], fb.U[1], fb.U[2], nek,
                       (const double*)(d + nek));
    DDNS_HIP(hipGetLastError());
    // the history starts equal to the velocity (turb.f90:452-454)
    for (int c = 0; c < 3; ++c)
        DDNS_HIP(hipMemcpyAsync(fb.O[c], fb.U[c], tot * sizeof(cpx<T>), hipMemcpyDeviceToDevice, s));
    DDNS_HIP(hipStreamSynchronize(s));
    DDNS_HIP(hipFree(d));
    return 0;
}

int flow_init(FlowBuffers& fb, int N, int nek, int precision, int kind, int seed, double k0, double urms, double force0,
              hipStream_t s)
{
    int st = 0;
    DDNS_HIP(hipStreamSynchronize(s));
    st = mark_dense(fb);
    if (st) return st;
    if (precision == DDNS_FP64) { DDNS_DISPATCH_N(N, st = (init_impl<double, NN>(fb, nek, kind, seed, k0, urms, force0, s))) }
    else { DDNS_DISPATCH_N(N, st = (init_impl<float, NN>(fb, nek, kind, seed, k0, urms, force0, s))) }
    return st;
}

// ---------------------------------------------------------------- stand-alone FFTs
// One field src (spectral) to real lines dst ([z][y][x]) through tmp (intermediate layout);
// dst may be src.
template <typename T, int N>
static int c2r_dev(const FlowBuffers& fb, const void* src, void* tmp, void* dst, hipStream_t s)
{
    FlowConst fc{};
    fc.N = N;
    int st = launch_z<T, N>(KZ_PLAIN_INV, fb, fc, s, src, tmp, 1.0);
    if (st) return st;
    st = launch_y<T, N>(true, false, &tmp, plain_field<N>(dst), 1, fb, N, s);
    if (st) return st;
    hipLaunchKernelGGL((k_x_plain<T, N, true>), dim3((unsigned)((size_t)N * N / kx_lines<N>())), dim3(NT), 0, s,
                       (const void*)dst, dst, fb.tw, fb.twh);
    DDNS_HIP(hipGetLastError());
    return 0;
}

// Real lines src to the spectral field dst through tmp (plain rows) and mid (intermediate
// layout); dst may be src or tmp.
template <typename T, int N>
static int r2c_dev(const FlowBuffers& fb, const void* src, void* tmp, void* mid, void* dst, hipStream_t s)
{
    hipLaunchKernelGGL((k_x_plain<T, N, false>), dim3((unsigned)((size_t)N * N / kx_lines<N>())), dim3(NT), 0, s, src, tmp,
                       fb.tw, fb.twh);
    DDNS_HIP(hipGetLastError());
    int st = launch_y<T, N>(false, false, &mid, plain_field<N>(tmp), 1, fb, N, s);
    if (st) return st;
    FlowConst fc{};
    fc.N = N;
    return launch_z<T, N>(KZ_PLAIN_FWD, fb, fc, s, mid, dst, 1.0 / N);
}

template <typename T, int N>
static int r2c_impl(FlowBuffers& fb, double* v, hipStream_t s)
{
    using C = cpx<T>;
    const int L = N + 2;
    const size_t n3 = (size_t)N * N * N;
    std::vector<T> h(n3);
    for (int z = 0; z < N; ++z)
        for (int y = 0; y < N; ++y)
            for (int x = 0; x < N; ++x)
                h[((size_t)z * N + y) * N + x] = (T)v[(size_t)x + (size_t)L * ((size_t)y + (size_t)L * z)];
    // A[0] holds the real input (same byte size as one complex field), A[2] the output
    DDNS_HIP(hipMemcpyAsync(fb.A[0], h.data(), n3 * sizeof(T), hipMemcpyHostToDevice, s));
    const int st = r2c_dev<T, N>(fb, fb.A[0], fb.B[0], fb.A[1], fb.A[2], s);
    if (st) return st;
    return download_spectral<T>(fb, fb.A[2], N, v, s);
}

template <typename T, int N>
static int c2r_impl(FlowBuffers& fb, double* v, hipStream_t s)
{
    const int L = N + 2;
    const size_t n3 = (size_t)N * N * N;
    int st = upload_spectral<T>(fb, fb.A[1], N, v, s);
    if (st) return st;
    st = c2r_dev<T, N>(fb, fb.A[1], fb.B[0], fb.A[0], s);
    if (st) return st;
    std::vector<T> h(n3);
    DDNS_HIP(hipMemcpyAsync(h.data(), fb.A[0], n3 * sizeof(T), hipMemcpyDeviceToHost, s));
    DDNS_HIP(hipStreamSynchronize(s));
    std::memset(v, 0, sizeof(double) * (size_t)L * L * N);
    for (int z = 0; z < N; ++z)
        for (int y = 0; y < N; ++y)
            for (int x = 0; x < N; ++x)
                v[(size_t)x + (size_t)L * ((size_t)y + (size_t)L * z)] = (double)h[((size_t)z * N + y) * N + x];
    return 0;
}

int fft_r2c_host(FlowBuffers& fb, int N, int precision, double* v, hipStream_t s)
{
    int st = 0;
    if (precision == DDNS_FP64) { DDNS_DISPATCH_N(N, st = (r2c_impl<double, NN>(fb, v, s))) }
    else { DDNS_DISPATCH_N(N, st = (r2c_impl<float, NN>(fb, v, s))) }
    return st;
}

int fft_c2r_host(FlowBuffers& fb, int N, int precision, double* v, hipStream_t s)
{
    int st = 0;
    if (precision == DDNS_FP64) { DDNS_DISPATCH_N(N, st = (c2r_impl<double, NN>(fb, v, s))) }
    else { DDNS_DISPATCH_N(N, st = (c2r_impl<float, NN>(fb, v, s))) }
    return st;
}

// ---------------------------------------------------------------- diagnostics
// POSTPROC (postprocessing.f90:76-272) and TRANSPOSTPROC (275-315) on the current
// u-hat.  Spectral fields are formed by the kernels below, taken to physical space by
// the plain z / y / x transforms into scratch fields, and reduced with fixed grids.

// dst = i k_c src (c = 0, 1, 2: x, y, z), the derivative of component src along c
// (postprocessing.f90:97-111)
template <typename T, int N>
__global__ void k_mul_ik(const void* src, void* dst, int c)
{
    using C = cpx<T>;
    constexpr int M = N / 2;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)N * N * M) return;
    int kx, ky, kz;
    spec_mode<T>(N, t, kz, ky, kx);
    const T k = (T)(c == 0 ? kx : (c == 1 ? wave_index(ky, N) : wave_index(kz, N)));
    const C v = ((const C*)src)[t];
    ((C*)dst)[t] = mk<C>(-(k * v.y), k * v.x);
}

// dst = i (k x u)_c for c < 3 (the vorticity, turb.f90:506-517), or i k . u for c = 3
// (the divergence, postprocessing.f90:219-223)
template <typename T, int N>
__global__ void k_curl_div(const void* u0, const void* u1, const void* u2, void* dst, int c)
{
    using C = cpx<T>;
    constexpr int M = N / 2;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)N * N * M) return;
    int kx, ky, kz;
    spec_mode<T>(N, t, kz, ky, kx);
    const T fx = (T)kx, fy = (T)wave_index(ky, N), fz = (T)wave_index(kz, N);
    const C a = ((const C*)u0)[t], b = ((const C*)u1)[t], d = ((const C*)u2)[t];
    C w;
    if (c == 0) w = csub(cscale(d, fy), cscale(b, fz));
    else if (c == 1) w = csub(cscale(a, fz), cscale(d, fx));
    else if (c == 2) w = csub(cscale(b, fx), cscale(a, fy));
    else w = cadd(cadd(cscale(a, fx), cscale(b, fy)), cscale(d, fz));
    ((C*)dst)[t] = mk<C>(-w.y, w.x);
}

// in place: (w0, w1, w2) <- u x w, the nonlinear term in physical space (turb.f90:634-637)
template <typename T>
__global__ void k_cross(const T* __restrict__ u0, const T* __restrict__ u1, const T* __restrict__ u2,
                        T* w0, T* w1, T* w2, size_t n)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const T ux = u0[i], uy = u1[i], uz = u2[i], wx = w0[i], wy = w1[i], wz = w2[i];
    w0[i] = uy * wz - uz * wy;
    w1[i] = uz * wx - ux * wz;
    w2[i] = ux * wy - uy * wx;
}

constexpr int DG_BLOCKS = 256;   // fixed grid of the diagnostic reductions: one work-group per CU, of
constexpr int DG_T = 1024;       // 16 wavefronts (with 4 the loads in flight held it to 1.7 TB/s at 256^3)

// per work-group sums over a real field: mode 0: f^2, f^3, f^4 of one field;
// mode 1: the max of |f0| + |f1| + |f2|; mode 2: sum |g|, |g|^2 and |g| f0 with
// |g| = sqrt(f1^2 + f2^2 + f3^2) (vorticity magnitude against the divergence f0);
// mode 3: f, f^2 of one field
template <typename T>
__global__ void __launch_bounds__(DG_T) k_dg_reduce(const T* f0, const T* f1, const T* f2, const T* f3, size_t n,
                                                  int mode, double* part)
{
    __shared__ double sh[3][DG_T];
    double a0 = 0.0, a1 = 0.0, a2 = 0.0;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
        if (mode == 0) {
            const double v = (double)f0[i], v2 = v * v;
            a0 += v2; a1 += v2 * v; a2 += v2 * v2;
        } else if (mode == 1) {
            const double v = fabs((double)f0[i]) + fabs((double)f1[i]) + fabs((double)f2[i]);
            a0 = fmax(a0, v);
        } else if (mode == 3) {
            const double v = (double)f0[i];
            a0 += v; a1 += v * v;
        } else {
            const double w1 = (double)f1[i], w2 = (double)f2[i], w3 = (double)f3[i];
            const double g = sqrt(w1 * w1 + w2 * w2 + w3 * w3);
            a0 += g; a1 += g * g; a2 += g * (double)f0[i];
        }
    }
    sh[0][threadIdx.x] = a0; sh[1][threadIdx.x] = a1; sh[2][threadIdx.x] = a2;
    __syncthreads();
    for (int o = DG_T / 2; o > 0; o >>= 1) {
        if (threadIdx.x < o) {
            if (mode == 1) sh[0][threadIdx.x] = fmax(sh[0][threadIdx.x], sh[0][threadIdx.x + o]);
            else {
                sh[0][threadIdx.x] += sh[0][threadIdx.x + o];
                sh[1][threadIdx.x] += sh[1][threadIdx.x + o];
                sh[2][threadIdx.x] += sh[2][threadIdx.x + o];
            }
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[blockIdx.x] = sh[0][0];
        part[gridDim.x + blockIdx.x] = sh[1][0];
        part[2 * gridDim.x + blockIdx.x] = sh[2][0];
    }
}

// partials of a k_dg_reduce launch summed (or maxed) on the host in block order
template <typename T>
static int dg_reduce(const T* f0, const T* f1, const T* f2, const T* f3, size_t n, int mode, double* part, double out[3],
                     hipStream_t s)
{
    hipLaunchKernelGGL((k_dg_reduce<T>), dim3(DG_BLOCKS), dim3(DG_T), 0, s, f0, f1, f2, f3, n, mode, part);
    DDNS_HIP(hipGetLastError());
    double h[3 * DG_BLOCKS];
    DDNS_HIP(hipMemcpyAsync(h, part, sizeof(h), hipMemcpyDeviceToHost, s));
    DDNS_HIP(hipStreamSynchronize(s));
    for (int q = 0; q < 3; ++q) {
        double a = 0.0;
        for (int b = 0; b < DG_BLOCKS; ++b) a = mode == 1 ? fmax(a, h[q * DG_BLOCKS + b]) : a + h[q * DG_BLOCKS + b];
        out[q] = a;
    }
    return 0;
}

template <typename T, int N>
static int diag_impl(FlowBuffers& fb, int nek, double rnu, int want, double* ek, double* dk, double* tk, double* mom,
                     hipStream_t s)
{
    const size_t n3 = (size_t)N * N * N, nc = field_elems(N);
    const size_t fbytes = n3 * sizeof(T);                    // one real field = one complex field
    if (!fb.dg[0]) {
        for (int q = 0; q < 8; ++q) DDNS_HIP(hipMalloc(&fb.dg[q], fbytes));
        // the 3 nek shell sums (nek < N / 2) and their partials, or the 3 DG_BLOCKS partials of
        // a reduction over a real field
        DDNS_HIP(hipMalloc(&fb.dg_part, 3 * (size_t)std::max(DG_BLOCKS, (SPEC_BLOCKS + 1) * (N / 2)) * sizeof(double)));
    }
    T* R[6];
    for (int q = 0; q < 6; ++q) R[q] = (T*)fb.dg[q];
    void* ctmp = fb.dg[6];
    void* cout = fb.dg[7];
    const unsigned gc = (unsigned)((nc + 255) / 256), gr = (unsigned)((n3 + 255) / 256);
    int st;
    // physical u and w
    for (int c = 0; c < 3; ++c) {
        st = c2r_dev<T, N>(fb, fb.U[c], ctmp, R[c], s);
        if (st) return st;
        hipLaunchKernelGGL((k_curl_div<T, N>), dim3(gc), dim3(256), 0, s, fb.U[0], fb.U[1], fb.U[2], cout, c);
        st = c2r_dev<T, N>(fb, cout, ctmp, R[3 + c], s);
        if (st) return st;
    }
    if (want & 1) {
        // max |u| + |v| + |w| (the CFL number, postprocessing.f90:204-207)
        double o[3];
        st = dg_reduce<T>(R[0], R[1], R[2], nullptr, n3, 1, fb.dg_part, o, s);
        if (st) return st;
        mom[0] = o[0];
        // longitudinal velocity derivatives: sums of d^2, d^3, d^4 over the three
        // components (postprocessing.f90:97-137), into the ctmp / cout scratch
        double s2 = 0.0, s3 = 0.0, s4 = 0.0;
        for (int c = 0; c < 3; ++c) {
            hipLaunchKernelGGL((k_mul_ik<T, N>), dim3(gc), dim3(256), 0, s, fb.U[c], cout, c);
            // the derivative field replaces nothing needed later: use the second half of R
            // only after the vorticity moments (below) have been taken
            st = c2r_dev<T, N>(fb, cout, ctmp, cout, s);
            if (st) return st;
            st = dg_reduce<T>((const T*)cout, nullptr, nullptr, nullptr, n3, 0, fb.dg_part, o, s);
            if (st) return st;
            s2 += o[0]; s3 += o[1]; s4 += o[2];
        }
        mom[1] = s2; mom[2] = s3; mom[3] = s4;
    }
    if (want & 2) {
        // divergence and vorticity statistics (postprocessing.f90:217-270)
        hipLaunchKernelGGL((k_curl_div<T, N>), dim3(gc), dim3(256), 0, s, fb.U[0], fb.U[1], fb.U[2], cout, 3);
        st = c2r_dev<T, N>(fb, cout, ctmp, cout, s);
        if (st) return st;
        double o[3], g[3];
        st = dg_reduce<T>((const T*)cout, nullptr, nullptr, nullptr, n3, 3, fb.dg_part, o, s);
        if (st) return st;
        st = dg_reduce<T>((const T*)cout, R[3], R[4], R[5], n3, 2, fb.dg_part, g, s);
        if (st) return st;
        mom[4] = o[0]; mom[5] = o[1];                  // sum div, sum div^2
        mom[6] = g[0]; mom[7] = g[1]; mom[8] = g[2];   // sum |w|, sum |w|^2, sum |w| div
    }
    // spectra; the transfer needs the nonlinear term F = FFT(u x w) (turb.f90:634-650)
    double* dd = fb.dg_part;           // 3 nek shell sums
    const void* F[3] = {nullptr, nullptr, nullptr};
    if (tk) {
        hipLaunchKernelGGL((k_cross<T>), dim3(gr), dim3(256), 0, s, R[0], R[1], R[2], R[3], R[4], R[5], n3);
        DDNS_HIP(hipGetLastError());
        for (int c = 0; c < 3; ++c) {
            st = r2c_dev<T, N>(fb, R[3 + c], ctmp, R[c], R[3 + c], s);     // through u_c, no longer needed
            if (st) return st;
            F[c] = R[3 + c];
        }
    }
    st = flow_shell_sums(fb, F, N, nek, rnu, sizeof(T) == 8 ? DDNS_FP64 : DDNS_FP32_MIXED, dd + 3 * (size_t)nek, dd, s);
    if (st) return st;
    std::vector<double> h(3 * (size_t)nek);
    DDNS_HIP(hipMemcpyAsync(h.data(), dd, h.size() * sizeof(double), hipMemcpyDeviceToHost, s));
    DDNS_HIP(hipStreamSynchronize(s));
    for (int i = 0; i < nek; ++i) {
        if (ek) ek[i] = h[i];
        if (dk) dk[i] = h[nek + i];
        if (tk) tk[i] = h[2 * nek + i];
    }
    return 0;
}

int flow_diagnostics(FlowBuffers& fb, int N, int nek, double rnu, int precision, int want, double* ek, double* dk,
                     double* tk, double* mom, hipStream_t s)
{
    if (nek > N / 2) { set_error("too many shells for the diagnostics"); return DDNS_ERR_ARG; }
    int st = 0;
    if (precision == DDNS_FP64) { DDNS_DISPATCH_N(N, st = (diag_impl<double, NN>(fb, nek, rnu, want, ek, dk, tk, mom, s))) }
    else { DDNS_DISPATCH_N(N, st = (diag_impl<float, NN>(fb, nek, rnu, want, ek, dk, tk, mom, s))) }
    return st;
}

// ---------------------------------------------------------------- per-kernel timing
template <typename T, int N>
static int profile_impl(const FlowBuffers& fb, const FlowConst& fc, int k, double* ms, int nk, hipStream_t s)
{
    hipEvent_t ev[FLOW_EVENTS];
    for (int i = 0; i < FLOW_EVENTS; ++i) DDNS_HIP(hipEventCreate(&ev[i]));
    double acc[7] = {0, 0, 0, 0, 0, 0, 0};
    for (int it = 0; it < k; ++it) {
        int st = step_impl<T, N>(fb, fc, s, ev, FLOW_INV, hipEventRecordDefault);
        if (st) return st;
        st = step_impl<T, N>(fb, fc, s, ev, FLOW_FWD, hipEventRecordDefault);
        if (st) return st;
        DDNS_HIP(hipEventSynchronize(ev[7]));
        float t;
        DDNS_HIP(hipEventElapsedTime(&t, ev[0], ev[1])); acc[0] += t;   // y inverse
        DDNS_HIP(hipEventElapsedTime(&t, ev[1], ev[2])); acc[1] += t;   // x fused
        DDNS_HIP(hipEventElapsedTime(&t, ev[3], ev[4])); acc[2] += t;   // y forward
        DDNS_HIP(hipEventElapsedTime(&t, ev[4], ev[5])); acc[3] += t;   // pre
        DDNS_HIP(hipEventElapsedTime(&t, ev[8], ev[6])); acc[4] += t;   // z stage
        DDNS_HIP(hipEventElapsedTime(&t, ev[6], ev[7])); acc[5] += t;   // sym
        DDNS_HIP(hipEventElapsedTime(&t, ev[0], ev[7])); acc[6] += t;   // whole
    }
    for (int i = 0; i < nk && i < 7; ++i) ms[i] = acc[i] / k;
    for (int i = 0; i < FLOW_EVENTS; ++i) (void)hipEventDestroy(ev[i]);
    return 0;
}

// plain streaming copy, 16 B per lane per iteration: the HBM reference kernel
__global__ void __launch_bounds__(256) k_copy_calibration(const float4* __restrict__ src, float4* __restrict__ dst, size_t n)
{
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) dst[i] = src[i];
}

int flow_profile_copy(const FlowBuffers& fb, int N, int precision, int reps, double* ms, double* bytes, hipStream_t s)
{
    const size_t cs = (precision == DDNS_FP64) ? sizeof(double2) : sizeof(float2);
    const size_t n4 = field_elems(N) * cs / sizeof(float4);
    hipEvent_t e0, e1;
    DDNS_HIP(hipEventCreate(&e0));
    DDNS_HIP(hipEventCreate(&e1));
    const unsigned grid = 256 * 32;
    hipLaunchKernelGGL(k_copy_calibration, dim3(grid), dim3(256), 0, s, (const float4*)fb.A[0], (float4*)fb.A[1], n4);
    DDNS_HIP(hipEventRecord(e0, s));
    for (int r = 0; r < reps; ++r)
        hipLaunchKernelGGL(k_copy_calibration, dim3(grid), dim3(256), 0, s, (const float4*)fb.A[0], (float4*)fb.A[1], n4);
    DDNS_HIP(hipGetLastError());
    DDNS_HIP(hipEventRecord(e1, s));
    DDNS_HIP(hipEventSynchronize(e1));
    float t = 0;
    DDNS_HIP(hipEventElapsedTime(&t, e0, e1));
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    *ms = (double)t / reps;
    *bytes = 2.0 * (double)n4 * sizeof(float4);
    return 0;
}

// ---------------------------------------------------------------- tile-shape tuner
// The role the FFTW_MEASURE plans play in the reference (mpifft.f90:36-56): at set-up,
// before any state is loaded, each candidate shape is timed on the handle's own buffers
// (cleared first), one untimed run and then the mean of three, and the fastest is kept:
//   - the y-stage tile width: the inverse stage over six fields and the forward stage
//     over three, as a step runs them;
//   - the z stage's tile width, by its work-group's threads.
// The choices are cached per grid and precision for the life of the process.
// DDNS_KY_TC / DDNS_KZ_NT in the environment force a shape (one that is not a candidate,
// or does not fit, means the default) and skip the timing; DDNS_TUNE=0 keeps the defaults.
// No choice changes the arithmetic of a column or of a mode, so every one gives the
// same bits.
template <typename T, int N>
static bool ky_cand_fits(int k)
{
    switch (k) {
    case 0: return ky_fits<T, N, ky_cand<T, N>(0)>();
    case 1: return ky_fits<T, N, ky_cand<T, N>(1)>();
    default: return ky_fits<T, N, ky_cand<T, N>(2)>();
    }
}

template <typename T, int N>
static bool kz_cand_fits(int k)
{
    return k == 0 || kz_fits<T, N, kz_cand<T, N>(1)>();
}
// threads of the fused z stage's work-group at candidate k (once or twice the default width)
template <typename T, int N> constexpr int kz_nt_cand(int k) { return kz_threads<T, N, kz_tc<T, N>()>() << k; }

struct TuneRecord {
    int ky_tc, kz_nt;
    float ky_ms[3], kz_ms[3];
};

// times `reps` runs of launch after one untimed run (ms per run), 0 on failure
template <typename F>
static float time_runs(F&& launch, int reps, hipStream_t s, hipEvent_t e0, hipEvent_t e1, int* st)
{
    for (int rep = 0; rep <= reps && !*st; ++rep) {
        if (rep == 1 && hipEventRecord(e0, s) != hipSuccess) *st = DDNS_ERR_HIP;
        if (!*st) *st = launch();
    }
    float ms = 0.f;
    if (!*st && (hipEventRecord(e1, s) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
                 hipEventElapsedTime(&ms, e0, e1) != hipSuccess))
        *st = DDNS_ERR_HIP;
    return *st ? 0.f : ms / (float)reps;
}

template <typename T, int N>
static int tune_impl(FlowBuffers& fb, const FlowConst& fc, hipStream_t s)
{
    static std::mutex mu;
    static std::map<int, TuneRecord> cache;          // key: N * 4096 + R, per precision (one map per T)
    fb.ky_tc = ky_tc<T, N>();
    fb.kz_nt = kz_nt_cand<T, N>(0);
    for (int k = 0; k < 3; ++k) fb.ky_ms[k] = fb.kz_ms[k] = 0.f;
    bool forced = false;
    if (const char* f = std::getenv("DDNS_KY_TC")) {
        const int want = std::atoi(f);
        for (int k = 0; k < 3; ++k)
            if (want == ky_cand<T, N>(k) && ky_cand_fits<T, N>(k)) fb.ky_tc = want;
        forced = true;
    }
    if (const char* f = std::getenv("DDNS_KZ_NT")) {
        const int want = std::atoi(f);
        for (int k = 0; k < 2; ++k)
            if (want == kz_nt_cand<T, N>(k) && kz_cand_fits<T, N>(k)) fb.kz_nt = want;
        forced = true;
    }
    if (forced) return 0;
    if (const char* t = std::getenv("DDNS_TUNE"))
        if (t[0] == '0') return 0;
    {
        std::lock_guard<std::mutex> lock(mu);
        auto it = cache.find(N * 4096 + fb.R);        // per grid and number of realisations
        if (it != cache.end()) {
            fb.ky_tc = it->second.ky_tc;
            fb.kz_nt = it->second.kz_nt;
            for (int k = 0; k < 3; ++k) {
                fb.ky_ms[k] = it->second.ky_ms[k];
                fb.kz_ms[k] = it->second.kz_ms[k];
            }
            return 0;
        }
    }
    const size_t bytes = field_elems(N) * sizeof(cpx<T>) * fb.R;
    for (int q = 0; q < 6; ++q) DDNS_HIP(hipMemsetAsync(fb.A[q], 0, bytes, s));
    for (int q = 0; q < 3; ++q) DDNS_HIP(hipMemsetAsync(fb.B[q], 0, bytes, s));
    hipEvent_t e0 = nullptr, e1 = nullptr;
    DDNS_HIP(hipEventCreate(&e0));
    DDNS_HIP(hipEventCreate(&e1));
    for (int q = 0; q < 3; ++q) {
        DDNS_HIP(hipMemsetAsync(fb.U[q], 0, bytes, s));
        DDNS_HIP(hipMemsetAsync(fb.O[q], 0, bytes, s));
    }
    // a step's stages skip what lies beyond the dealiasing sphere (LOW_ZOUT; every field is zero
    // here).  Timed as after an upload, the z stage stored twice as much of the state and the
    // inverse y stage read a quarter more: 0.303 ms for a z stage at 256^3 FP32, 0.261 now
    std::vector<double> low((size_t)LOW_STRIDE * fb.R, 0.0);
    for (int r = 0; r < fb.R; ++r) low[(size_t)r * LOW_STRIDE + LOW_ZOUT] = 1.0;
    DDNS_HIP(hipMemcpyAsync(fb.low, low.data(), low.size() * sizeof(double), hipMemcpyHostToDevice, s));
    DDNS_HIP(hipStreamSynchronize(s));
    float best = 0.f;
    int best_tc = ky_tc<T, N>(), best_nt = kz_nt_cand<T, N>(0);
    int st = 0;
    for (int k = 0; k < 3 && !st; ++k) {
        if (!ky_cand_fits<T, N>(k)) continue;
        fb.ky_tc = ky_cand<T, N>(k);
        fb.ky_ms[k] = time_runs([&]() {
            const PlainRows rows = plain_rows<T, N>(fb);
            const int r = launch_y<T, N>(true, true, fb.A, rows, 6, fb, fb.R * N, s, fc.nek);
            return r ? r : launch_y<T, N>(false, false, fb.A, rows, 3, fb, fb.R * N, s, fc.nek);
        }, 3, s, e0, e1, &st);
        if (!st && (best == 0.f || fb.ky_ms[k] < best)) {
            best = fb.ky_ms[k];
            best_tc = fb.ky_tc;
        }
    }
    {
        best = 0.f;
        for (int k = 0; k < 2 && !st; ++k) {
            if (!kz_cand_fits<T, N>(k)) continue;
            fb.kz_nt = kz_nt_cand<T, N>(k);
            fb.kz_ms[k] = time_runs([&]() { return launch_z<T, N>(KZ_FULL, fb, fc, s); }, 3, s, e0, e1, &st);
            if (!st && (best == 0.f || fb.kz_ms[k] < best)) {
                best = fb.kz_ms[k];
                best_nt = fb.kz_nt;
            }
        }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (st) {
        set_error("tile-width tuner: a HIP call failed");
        return st;
    }
    // the state the timing runs wrote is cleared again: a new handle starts at rest
    for (int q = 0; q < 3; ++q) {
        DDNS_HIP(hipMemsetAsync(fb.U[q], 0, bytes, s));
        DDNS_HIP(hipMemsetAsync(fb.O[q], 0, bytes, s));
    }
    DDNS_HIP(hipMemsetAsync(fb.low, 0, (size_t)LOW_STRIDE * fb.R * sizeof(double), s));
    DDNS_HIP(hipStreamSynchronize(s));
    fb.ky_tc = best_tc;
    fb.kz_nt = best_nt;
    std::lock_guard<std::mutex> lock(mu);
    TuneRecord r{};
    r.ky_tc = best_tc;
    r.kz_nt = best_nt;
    for (int k = 0; k < 3; ++k) {
        r.ky_ms[k] = fb.ky_ms[k];
        r.kz_ms[k] = fb.kz_ms[k];
    }
    cache[N * 4096 + fb.R] = r;
    return 0;
}

int flow_tune(FlowBuffers& fb, const FlowConst& fc, int precision, hipStream_t s)
{
    int st = 0;
    if (precision == DDNS_FP64) { DDNS_DISPATCH_N(fc.N, st = (tune_impl<double, NN>(fb, fc, s))) }
    else { DDNS_DISPATCH_N(fc.N, st = (tune_impl<float, NN>(fb, fc, s))) }
    return st;
}

int flow_default_kz_nt(int N, int precision)
{
    int nt = 0;
    if (precision == DDNS_FP64) { DDNS_DISPATCH_N(N, nt = (kz_nt_cand<double, NN>(0))) }
    else { DDNS_DISPATCH_N(N, nt = (kz_nt_cand<float, NN>(0))) }
    return nt;
}

int flow_default_ky_tc(int N, int precision)
{
    int tc = 0;
    if (precision == DDNS_FP64) { DDNS_DISPATCH_N(N, tc = (ky_tc<double, NN>())) }
    else { DDNS_DISPATCH_N(N, tc = (ky_tc<float, NN>())) }
    return tc;
}

int flow_profile(const FlowBuffers& fb, const FlowConst& fc, int precision, int k, double* ms, int nk, hipStream_t s)
{
    int st = 0;
    if (precision == DDNS_FP64) { DDNS_DISPATCH_N(fc.N, st = (profile_impl<double, NN>(fb, fc, k, ms, nk, s))) }
    else { DDNS_DISPATCH_N(fc.N, st = (profile_impl<float, NN>(fb, fc, k, ms, nk, s))) }
    return st;
}

}  // namespace ddns
