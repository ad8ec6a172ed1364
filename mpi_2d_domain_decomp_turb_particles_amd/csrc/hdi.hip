// hdi.hip -- hydrodynamic interactions between droplets.
//
// Reference: NEI_LIST_PRECOMP partlib.f90:3218-3371 (neighbours within HDI_trunc
// radii of the *source* droplet, Stokes-sphere coefficients M = gamma r r + beta I),
// AFUN_PRECOMP 3375-3510 (A x = x + M x and b = M (V - U)), HDI_GMRES 2795-3005
// (unrestarted GMRES: modified Gram-Schmidt Arnoldi, explicit Givens factor Qn,
// back substitution, tolerance relaxed at iteration maxiter/2 and from maxiter-2,
// warm start from the previous disturbance velocity) and EUC_NORM 2756-2791.
//
// The system is solved in cell-sorted droplet order: row t is the droplet at sorted
// position t, so the neighbours a row gathers sit in the few cells around it and
// their vector entries are close in memory.  The solution is scattered back to the
// reference's droplet order at the end.  Neighbour lists are ELL, slot-major: slot s
// of row t holds the neighbour's sorted position and the 6 distinct entries of its
// symmetric 3x3 block, at s * n + t, so a wavefront reads each slot as one run.  One
// pass over the coarse cells fills them; the slot width grows when a row needs more.
// Krylov vectors use the reference's blocked order x(1:n), x(n+1:2n), x(2n+1:3n).
// In FP32-mixed mode the matrix and the Krylov basis are float, every inner product
// and norm accumulates in double, and the small least-squares problem is double.
// Reductions use a fixed grid and a fixed summation tree, and the last work-group to
// finish does the final sum, so results do not depend on timing.
#include "ddns_internal.h"

#include <algorithm>
#include <cmath>
#include <cstring>

namespace ddns {

constexpr int HT = 256;
constexpr int RED_BLOCKS = 256;    // reduction grids: at most one work-group per CU
constexpr int ELL_STEP = 8;        // the ELL width grows in multiples of this


// deterministic wavefront sum: lane 0 holds the butterfly result
__device__ __forceinline__ double wave_sum(double x)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    return x;
}

// ------------------------------------------------------------------ neighbour lists
// Row t (sorted position): every droplet p != t in the 27 cells around t with
// |x_t - x_p| < trunc * r_p (partlib.f90:3280-3330).  The walk only
// decides, from the squared distance (the square root is taken where rounding could decide),
// and leaves the accepted candidates in the list; a second, short loop forms their blocks.  In
// the walk a wavefront of 64 rows met an accepted candidate on nearly every turn, and took the
// blocks' divisions and six scattered stores there for one or two lanes each time (1M droplets
// 274 us, now 202; 100 000: 42, now 27).  Four lanes share a row up to NEI_SHARED droplets, where
// the rows alone leave the SIMDs short of wavefronts and each row's walk is a serial chain: the
// 16 realisations of 9 000 to 60 000 droplets 105 -> 46 us a launch (two lanes: 64^3 with 60 000
// droplets 0.76 ms a solve, four 0.73, eight 0.73), at 100 000 no difference.
constexpr int NT_NEI = 128, NEI_SHARED = 131072;

template <typename T, int L>
__global__ void __launch_bounds__(NT_NEI) k_nei(const double4* __restrict__ pk, const int* __restrict__ cell_start,
                                                int n, int G, double hc, double pi2, double trunc, int width,
                                                int* __restrict__ cnt, int* __restrict__ idx, T* __restrict__ mm,
                                                int* flags)
{
    __shared__ RunList<NT_NEI> runs;
    const int t = (xcd_chunk(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x) / L;
    const int sub = threadIdx.x & (L - 1), first = threadIdx.x & 63 & ~(L - 1);    // among the row's lanes; its first lane
    int k = 0;
    if (t < n) {
        const double4 me = pk[t];
        const double xi = me.x, yi = me.y, zi = me.z, ri = me.w;
        int cc[3];
        const double xs[3] = {xi, yi, zi};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            int q = (int)(xs[c] / hc);
            cc[c] = q < 0 ? 0 : (q >= G ? G - 1 : q);
        }
        const size_t ld = (size_t)n;
        bool overlap = false;
        // sqrt(d2) < l, decided without the root where d2 is not within rounding of l^2
        auto closer = [](double d2, double l) {
            const double l2 = l * l;
            if (fabs(d2 - l2) > 1e-12 * l2) return d2 < l2;
            return sqrt(d2) < l;
        };
        for_each_candidate<L>(runs, cell_start, G, pi2, cc, pk, (const int*)nullptr,
                           [&](int p, int w, double sx, double sy, double sz, const double4& o, int) {
            const double d0 = xi - (o.x + sx), d1 = yi - (o.y + sy), d2 = zi - (o.z + sz);
            const double dd = d0 * d0 + d1 * d1 + d2 * d2;
            if (p != t && closer(dd, ri + o.w)) overlap = true;             // 3294-3299
            const bool hit = p != t && closer(dd, trunc * o.w);             // 3302-3305
            // the row's lanes append in the order of their candidates
            const unsigned m = L == 1 ? (unsigned)hit : (unsigned)(__ballot(hit) >> first) & ((1u << L) - 1);
            if (L > 1) k = __shfl(k, first, 64);     // the first lane has a candidate on every turn
            const int j = k + __popc(m & ((1u << sub) - 1));
            if (hit && j < width) idx[(size_t)j * ld + t] = (int)((unsigned)p | ((unsigned)w << 27));
            k += __popc(m);
        });
        if (L > 1) k = __shfl(k, first, 64);
        if (overlap) atomicOr(flags, 1);
        if (k > DDNS_MAXNEI) atomicOr(flags, 2);
        // a row with more neighbours than the lists hold keeps what fits: the products that
        // may run before the host has read the width flag stay inside the lists, and the
        // host fills them again, wider, before it uses any result
        const int kk = k < width ? k : width;
        if (sub == 0) cnt[t] = kk;
        if (L > 1) __threadfence_block();            // entries that other lanes of the row wrote
        for (int j = sub; j < kk; j += L) {
            const unsigned v = (unsigned)idx[(size_t)j * ld + t];
            const int p = (int)(v & ((1u << 27) - 1));
            int wx, wy, wz;
            shift_of((int)(v >> 27), &wx, &wy, &wz);
            const double4 o = pk[p];
            const double d0 = xi - (o.x + (double)wx * pi2);
            const double d1 = yi - (o.y + (double)wy * pi2);
            const double d2 = zi - (o.z + (double)wz * pi2);
            const double dnij = sqrt(d0 * d0 + d1 * d1 + d2 * d2);
            double fact1 = o.w / dnij;                                      // 3312-3324
            const double fact2 = fact1 * fact1 * fact1;
            fact1 = 0.75 * fact1;
            const double gamma = (fact1 - 0.75 * fact2) / (dnij * dnij);
            const double beta = fact1 + 0.25 * fact2;
            idx[(size_t)j * ld + t] = p;
            T* m = mm + (size_t)(6 * j) * ld + t;
            m[0] = (T)(gamma * (d0 * d0) + beta);
            m[ld] = (T)(gamma * d0 * d1);
            m[2 * ld] = (T)(gamma * d0 * d2);
            m[3 * ld] = (T)(gamma * (d1 * d1) + beta);
            m[4 * ld] = (T)(gamma * d1 * d2);
            m[5 * ld] = (T)(gamma * (d2 * d2) + beta);
        }
    }
    // the widest row of the wavefront, for the width check
    int km = k;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) km = max(km, __shfl_xor(km, o, 64));
    if ((threadIdx.x & 63) == 0 && km > width) atomicMax(flags + 4, km);
}

// y = x + M x (AFUN_PRECOMP).  MODE 0: x = x0 in double, y0d = A x0 and b = M w.
// MODE 1: x is a basis vector.  MODE 2: x = v / h for the previous work vector v; the
// row's own entries of x are also stored as the next basis vector (q = v / h,
// partlib.f90:2897).  In modes 1 and 2 the Arnoldi step runs on M, y = M x: A = I + M
// spans the same Krylov spaces and its Hessenberg matrix is M's plus the identity
// (added to H(it, it) with the first projection), so the projections no longer cancel
// the large identity part of A x against q_it.
template <typename T, int MODE>
__device__ __forceinline__ void k_spmv_body(const int* __restrict__ cnt, const int* __restrict__ idx,
                                             const T* __restrict__ mm, int n, const T* __restrict__ x,
                                             const double* __restrict__ hx, T* __restrict__ qout, T* __restrict__ y,
                                             const double* __restrict__ x0d, double* __restrict__ y0d,
                                             const double* __restrict__ w, double* __restrict__ b,
                                             const double* __restrict__ stop, int bx, int nbx)
{
    if (stop && *stop != 0.0) return;   // converged in an earlier iteration of this batch
    const int t = xcd_chunk(bx, nbx) * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const size_t N = (size_t)n;
    const double h = MODE == 2 ? *hx : 1.0;
    auto xv = [&](size_t q) -> double {
        if (MODE == 0) return x0d[q];
        if (MODE == 1) return (double)x[q];
        return (double)(T)((double)x[q] / h);
    };
    const int kk = cnt[t];
    double r0 = 0.0, r1 = 0.0, r2 = 0.0, b0 = 0.0, b1 = 0.0, b2 = 0.0;
    for (int s = 0; s < kk; ++s) {
        const size_t q = (size_t)s * N + t;
        const int j = idx[q];
        const T* m = mm + (size_t)(6 * s) * N + t;
        const double m0 = m[0], m1 = m[N], m2 = m[2 * N], m3 = m[3 * N], m4 = m[4 * N], m5 = m[5 * N];
        const double v0 = xv(j), v1 = xv(N + j), v2 = xv(2 * N + j);
        r0 = r0 + m0 * v0 + m1 * v1 + m2 * v2;
        r1 = r1 + m1 * v0 + m3 * v1 + m4 * v2;
        r2 = r2 + m2 * v0 + m4 * v1 + m5 * v2;
        if (MODE == 0) {
            const double q0 = w[j], q1 = w[N + j], q2 = w[2 * N + j];
            b0 = b0 + m0 * q0 + m1 * q1 + m2 * q2;
            b1 = b1 + m1 * q0 + m3 * q1 + m4 * q2;
            b2 = b2 + m2 * q0 + m4 * q1 + m5 * q2;
        }
    }
    const double s0 = xv(t), s1 = xv(N + t), s2 = xv(2 * N + t);
    if (MODE == 0) {
        y0d[t] = r0 + s0; y0d[N + t] = r1 + s1; y0d[2 * N + t] = r2 + s2;
        b[t] = b0; b[N + t] = b1; b[2 * N + t] = b2;
    } else {
        y[t] = (T)r0; y[N + t] = (T)r1; y[2 * N + t] = (T)r2;   // M x: the identity is added to H
        if (MODE == 2) { qout[t] = (T)s0; qout[N + t] = (T)s1; qout[2 * N + t] = (T)s2; }
    }
}
template <typename T, int MODE>
__global__ void __launch_bounds__(HT) k_spmv(const int* __restrict__ cnt, const int* __restrict__ idx,
                                             const T* __restrict__ mm, int n, const T* __restrict__ x,
                                             const double* __restrict__ hx, T* __restrict__ qout, T* __restrict__ y,
                                             const double* __restrict__ x0d, double* __restrict__ y0d,
                                             const double* __restrict__ w, double* __restrict__ b,
                                             const double* __restrict__ stop)
{
    k_spmv_body<T, MODE>(cnt, idx, mm, n, x, hx, qout, y, x0d, y0d, w, b, stop, blockIdx.x, gridDim.x);
}

// ------------------------------------------------------------------ vector kernels
// r0 = b - A x0 into the first Krylov column, with the work-group partial sums of b.b
// and r0.r0 (part[blk], part[RED_BLOCKS + blk]) on a fixed grid
template <typename T>
__global__ void __launch_bounds__(HT) k_residual0(const double* __restrict__ b, const double* __restrict__ ax0,
                                                  T* __restrict__ q, long long n, double* __restrict__ part)
{
    __shared__ double sb[HT], sq[HT];
    double ab = 0.0, aq = 0.0;
    for (long long i = (long long)blockIdx.x * HT + threadIdx.x; i < n; i += (long long)gridDim.x * HT) {
        const double bi = b[i];
        const T r = (T)(bi - ax0[i]);
        q[i] = r;
        ab += bi * bi;
        aq += (double)r * (double)r;
    }
    sb[threadIdx.x] = ab;
    sq[threadIdx.x] = aq;
    __syncthreads();
    for (int o = HT / 2; o > 0; o >>= 1) {
        if (threadIdx.x < o) {
            sb[threadIdx.x] += sb[threadIdx.x + o];
            sq[threadIdx.x] += sq[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        part[blockIdx.x] = sb[0];
        part[RED_BLOCKS + blockIdx.x] = sq[0];
    }
}

// The small problem cleared (ntot values), then norm_b = |b| and norm_rhs = |r0| from the
// np partials of k_residual0 (fixed order), the tolerance, and the stop flag when the
// initial residual is below 1e-5 (2866-2868); the head and the lists' flags to the host's copy
__global__ void __launch_bounds__(HT) k_gm_start(double* sm, int ntot, double tol, const double* __restrict__ part,
                                                 int np, const int* __restrict__ flags, double* host)
{
    __shared__ double sb[HT], sq[HT];
    for (int i = threadIdx.x; i < ntot; i += HT) sm[i] = 0.0;
    double ab = 0.0, aq = 0.0;
    for (int i = threadIdx.x; i < np; i += HT) {
        ab += part[i];
        aq += part[RED_BLOCKS + i];
    }
    sb[threadIdx.x] = ab;
    sq[threadIdx.x] = aq;
    __syncthreads();
    for (int o = HT / 2; o > 0; o >>= 1) {
        if (threadIdx.x < o) {
            sb[threadIdx.x] += sb[threadIdx.x + o];
            sq[threadIdx.x] += sq[threadIdx.x + o];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {                // after the barriers of the tree: the clearing is done
        const double head[6] = {sqrt(sb[0]), sqrt(sq[0]), 0.0, tol, sqrt(sq[0]) < 1e-5 ? -1.0 : 0.0, 0.0};
#pragma unroll
        for (int k = 0; k < 6; ++k) sm[k] = host[k] = head[k];
    }
    if (threadIdx.x < 8) ((int*)(host + 8))[threadIdx.x] = flags[threadIdx.x];
}

template <typename T>
__global__ void k_scale(T* q, const double* den, long long n)
{
    const long long i = (long long)blockIdx.x * HT + threadIdx.x;
    if (i < n) q[i] = (T)((double)q[i] / *den);
}

// ---- Arnoldi step: classical Gram-Schmidt applied twice, the second pass's update
// only where the first pass lost more than 1 - 1/sqrt(2) of the vector's norm (the
// DGKS criterion: otherwise its corrections are below rounding).  Each projection kernel
// runs on a fixed grid of P <= RED_BLOCKS work-groups and writes one partial sum per
// work-group and column (a fixed tree inside the work-group); the kernel that needs
// the sums adds the P partials itself, in a fixed order, at its start.  Every result
// is independent of scheduling.
constexpr int RT = 1024;          // threads per work-group of the projection kernels
constexpr int RW = RT / 64;       // wavefronts per work-group
constexpr int MD_J = 8;           // Krylov columns per pass of k_mdot

// Work-group sums of acc[0..J): red[jj] valid for all threads on return.
template <int J>
__device__ __forceinline__ void block_sums(double (&acc)[J], double (*sh)[J], double* red)
{
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
#pragma unroll
    for (int jj = 0; jj < J; ++jj) {
        const double v = wave_sum(acc[jj]);
        if (lane == 0) sh[wv][jj] = v;
    }
    __syncthreads();
    if (threadIdx.x < J) {
        double v = sh[0][threadIdx.x];
#pragma unroll
        for (int w = 1; w < RW; ++w) v += sh[w][threadIdx.x];
        red[threadIdx.x] = v;
    }
    __syncthreads();
}

// hs[j] = sum over b < P of part[j * P + b] for j < k (lane-strided in order, then a
// fixed wavefront tree), the same in every work-group.  Work-group 0 also sets
// (add = 0, with A's identity added to H(k, k)) or increments (add = 1) the Hessenberg
// column hcol.
__device__ void sum_partials(const double* __restrict__ part, int P, int k, double* hs, double* hcol, int add, int bx)
{
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int j = wv; j < k; j += RW) {
        double acc = 0.0;
        for (int b = lane; b < P; b += 64) acc += part[(size_t)j * P + b];
        acc = wave_sum(acc);
        if (lane == 0) {
            hs[j] = acc;
            if (bx == 0) hcol[j] = add ? hcol[j] + acc : acc + (j == k - 1 ? 1.0 : 0.0);
        }
    }
    __syncthreads();
}

// Krylov columns start every ld elements (ld a multiple of 64), so each lane moves
// 16 bytes per access: 4 floats or 2 doubles.  Element e of a vector sits at
// Q + j * ld + e for e < n3; the last, partial vector is done element by element.
template <typename T> struct kvec;
template <> struct kvec<float> { using V = float4; static constexpr int W = 4; };
template <> struct kvec<double> { using V = double2; static constexpr int W = 2; };

template <typename T>
__device__ __forceinline__ void vld(const T* p, T (&x)[kvec<T>::W])
{
    using V = typename kvec<T>::V;
    *(V*)x = *(const V*)p;
}
template <typename T>
__device__ __forceinline__ void vst(T* p, const T (&x)[kvec<T>::W])
{
    using V = typename kvec<T>::V;
    *(V*)p = *(const V*)x;
}

// partials of Q_j . v for j < k, and of v . v as column k
template <typename T>
__device__ __forceinline__ void k_mdot_body(const T* __restrict__ Q, const T* __restrict__ v, int k, long long n3,
                                             long long ld, double* __restrict__ part, const double* __restrict__ stop, int bx, int nbx)
{
    if (*stop != 0.0) return;
    constexpr int W = kvec<T>::W;
    __shared__ double sh[RW][MD_J + 1];
    __shared__ double red[MD_J + 1];
    const int tid = threadIdx.x;
    const long long nv = (n3 + W - 1) / W;
    for (int j0 = 0; j0 < k; j0 += MD_J) {
        double acc[MD_J + 1];
#pragma unroll
        for (int jj = 0; jj <= MD_J; ++jj) acc[jj] = 0.0;
        for (long long iv = (long long)bx * RT + tid; iv < nv; iv += (long long)nbx * RT) {
            const long long i = iv * W;
            if (i + W <= n3) {
                T x[W];
                vld(v + i, x);
                if (j0 == 0) {
#pragma unroll
                    for (int e = 0; e < W; ++e) acc[MD_J] += (double)x[e] * (double)x[e];
                }
#pragma unroll
                for (int jj = 0; jj < MD_J; ++jj)
                    if (j0 + jj < k) {
                        T q[W];
                        vld(Q + (size_t)(j0 + jj) * ld + i, q);
#pragma unroll
                        for (int e = 0; e < W; ++e) acc[jj] += (double)q[e] * (double)x[e];
                    }
            } else {
                for (long long e = i; e < n3; ++e) {
                    if (j0 == 0) acc[MD_J] += (double)v[e] * (double)v[e];
#pragma unroll
                    for (int jj = 0; jj < MD_J; ++jj)
                        if (j0 + jj < k) acc[jj] += (double)Q[(size_t)(j0 + jj) * ld + e] * (double)v[e];
                }
            }
        }
        block_sums<MD_J + 1>(acc, sh, red);
        if (tid < MD_J && j0 + tid < k) part[(size_t)(j0 + tid) * nbx + bx] = red[tid];
        if (j0 == 0 && tid == 0) part[(size_t)k * nbx + bx] = red[MD_J];
    }
}
template <typename T>
__global__ void __launch_bounds__(RT) k_mdot(const T* __restrict__ Q, const T* __restrict__ v, int k, long long n3,
                                             long long ld, double* __restrict__ part, const double* __restrict__ stop)
{
    k_mdot_body<T>(Q, v, k, n3, ld, part, stop, blockIdx.x, gridDim.x);
}

// First pass's update fused with the second pass's projections, for k <= KC columns:
// h = sum of the P_in part_in (first pass), v -= sum_j h_j Q_j, partials of Q_j . v into part_out
// and of v . v (the updated v) as its column k
template <typename T, int KC>
__device__ __forceinline__ void k_maxpy_mdot_body(T* __restrict__ v, const T* __restrict__ Q, int k, long long n3,
                                                   long long ld, const double* __restrict__ part_in, int P_in,
                                                   double* __restrict__ hcol, double* __restrict__ part_out,
                                                   const double* __restrict__ stop, int bx, int nbx)
{
    if (*stop != 0.0) return;
    constexpr int W = kvec<T>::W;
    __shared__ double hs[KC];
    __shared__ double sh[RW][KC + 1];
    __shared__ double red[KC + 1];
    const int tid = threadIdx.x;
    sum_partials(part_in, P_in, k, hs, hcol, 0, bx);
    double acc[KC + 1];
#pragma unroll
    for (int jj = 0; jj <= KC; ++jj) acc[jj] = 0.0;
    const long long nv = (n3 + W - 1) / W;
    for (long long iv = (long long)bx * RT + tid; iv < nv; iv += (long long)nbx * RT) {
        const long long i = iv * W;
        if (i + W <= n3) {
            T q[KC][W];
            T xv[W];
            vld(v + i, xv);
            double x[W];
#pragma unroll
            for (int e = 0; e < W; ++e) x[e] = (double)xv[e];
#pragma unroll
            for (int jj = 0; jj < KC; ++jj)
                if (jj < k) {
                    vld(Q + (size_t)jj * ld + i, q[jj]);
#pragma unroll
                    for (int e = 0; e < W; ++e) x[e] -= hs[jj] * (double)q[jj][e];
                }
#pragma unroll
            for (int e = 0; e < W; ++e) {
                xv[e] = (T)x[e];
                acc[KC] += (double)xv[e] * (double)xv[e];
            }
            vst(v + i, xv);
#pragma unroll
            for (int jj = 0; jj < KC; ++jj)
                if (jj < k) {
#pragma unroll
                    for (int e = 0; e < W; ++e) acc[jj] += (double)q[jj][e] * (double)xv[e];
                }
        } else {
            for (long long e = i; e < n3; ++e) {
                double x = (double)v[e];
                for (int jj = 0; jj < k; ++jj) x -= hs[jj] * (double)Q[(size_t)jj * ld + e];
                const T xt = (T)x;
                v[e] = xt;
                acc[KC] += (double)xt * (double)xt;
#pragma unroll
                for (int jj = 0; jj < KC; ++jj)
                    if (jj < k) acc[jj] += (double)Q[(size_t)jj * ld + e] * (double)xt;
            }
        }
    }
    block_sums<KC + 1>(acc, sh, red);
    if (tid < k) part_out[(size_t)tid * nbx + bx] = red[tid];
    if (tid == 0) part_out[(size_t)k * nbx + bx] = red[KC];
}
template <typename T, int KC>
__global__ void __launch_bounds__(RT) k_maxpy_mdot(T* __restrict__ v, const T* __restrict__ Q, int k, long long n3,
                                                   long long ld, const double* __restrict__ part_in, int P_in,
                                                   double* __restrict__ hcol, double* __restrict__ part_out,
                                                   const double* __restrict__ stop)
{
    k_maxpy_mdot_body<T, KC>(v, Q, k, n3, ld, part_in, P_in, hcol, part_out, stop, blockIdx.x, gridDim.x);
}

// sum over b < P of part[b] (lane-strided in order, then the wavefront tree), the same
// in every work-group; all threads get it
__device__ __forceinline__ double sum_one(const double* __restrict__ part, int P, double* sh1)
{
    if (threadIdx.x < 64) {
        double acc = 0.0;
        for (int b = threadIdx.x; b < P; b += 64) acc += part[b];
        acc = wave_sum(acc);
        if (threadIdx.x == 0) *sh1 = acc;
    }
    __syncthreads();
    return *sh1;
}

// The product of an Arnoldi step fused with the first pass's projections, for k <= KC
// columns: y = x + M x as k_spmv<T, MODE> (MODE 1: x = Q_0; MODE 2: x = v / h, stored as
// Q_(k-1)), and the partials of Q_j . y for j < k and of y . y (column k).  The grid is
// the projection kernels' (P <= RED_BLOCKS work-groups); work-group b takes a contiguous
// run of rows, the runs placed so that neighbouring ones share an XCD.
template <typename T, int MODE, int KC>
__device__ __forceinline__ void k_spmv_mdot_body(const int* __restrict__ cnt, const int* __restrict__ idx,
                                                  const T* __restrict__ mm, int n, const T* __restrict__ x,
                                                  const double* __restrict__ hx, T* __restrict__ qout,
                                                  T* __restrict__ y, const T* __restrict__ Q, long long ld, int k,
                                                  double* __restrict__ part, const double* __restrict__ stop, int bx, int nbx)
{
    if (*stop != 0.0) return;   // converged in an earlier iteration of this batch
    __shared__ double sh[RW][KC + 1];
    __shared__ double red[KC + 1];
    const size_t N = (size_t)n;
    const double h = MODE == 2 ? *hx : 1.0;
    auto xv = [&](size_t q) -> double {
        if (MODE == 1) return (double)x[q];
        return (double)(T)((double)x[q] / h);
    };
    double acc[KC + 1];
#pragma unroll
    for (int jj = 0; jj <= KC; ++jj) acc[jj] = 0.0;
    const int lb = xcd_chunk(bx, nbx);
    const int per = (n + (int)nbx - 1) / (int)nbx;
    const int t1 = min(n, (lb + 1) * per);
    for (int t = lb * per + threadIdx.x; t < t1; t += RT) {
        const int kk = cnt[t];
        double r0 = 0.0, r1 = 0.0, r2 = 0.0;
        for (int sl = 0; sl < kk; ++sl) {
            const size_t q = (size_t)sl * N + t;
            const int j = idx[q];
            const T* m = mm + (size_t)(6 * sl) * N + t;
            const double m0 = m[0], m1 = m[N], m2 = m[2 * N], m3 = m[3 * N], m4 = m[4 * N], m5 = m[5 * N];
            const double v0 = xv(j), v1 = xv(N + j), v2 = xv(2 * N + j);
            r0 = r0 + m0 * v0 + m1 * v1 + m2 * v2;
            r1 = r1 + m1 * v0 + m3 * v1 + m4 * v2;
            r2 = r2 + m2 * v0 + m4 * v1 + m5 * v2;
        }
        const double s0 = xv(t), s1 = xv(N + t), s2 = xv(2 * N + t);
        const T y0 = (T)r0, y1 = (T)r1, y2 = (T)r2;   // M x: the identity is added to H
        y[t] = y0; y[N + t] = y1; y[2 * N + t] = y2;
        if (MODE == 2) { qout[t] = (T)s0; qout[N + t] = (T)s1; qout[2 * N + t] = (T)s2; }
        const double d0 = (double)y0, d1 = (double)y1, d2 = (double)y2;
        acc[KC] += d0 * d0 + d1 * d1 + d2 * d2;
#pragma unroll
        for (int jj = 0; jj < KC; ++jj)
            if (jj < k) {
                double q0, q1, q2;
                if (jj == k - 1) {      // this row of x itself (Q_0 in MODE 1, the new column in MODE 2)
                    q0 = (double)(T)s0; q1 = (double)(T)s1; q2 = (double)(T)s2;
                } else {
                    const T* qc = Q + (size_t)jj * ld;
                    q0 = (double)qc[t]; q1 = (double)qc[N + t]; q2 = (double)qc[2 * N + t];
                }
                acc[jj] += q0 * d0 + q1 * d1 + q2 * d2;
            }
    }
    block_sums<KC + 1>(acc, sh, red);
    if ((int)threadIdx.x < k) part[(size_t)threadIdx.x * nbx + bx] = red[threadIdx.x];
    if (threadIdx.x == 0) part[(size_t)k * nbx + bx] = red[KC];
}
template <typename T, int MODE, int KC>
__global__ void __launch_bounds__(RT) k_spmv_mdot(const int* __restrict__ cnt, const int* __restrict__ idx,
                                                  const T* __restrict__ mm, int n, const T* __restrict__ x,
                                                  const double* __restrict__ hx, T* __restrict__ qout,
                                                  T* __restrict__ y, const T* __restrict__ Q, long long ld, int k,
                                                  double* __restrict__ part, const double* __restrict__ stop)
{
    k_spmv_mdot_body<T, MODE, KC>(cnt, idx, mm, n, x, hx, qout, y, Q, ld, k, part, stop, blockIdx.x, gridDim.x);
}

// Small least-squares update of HDI_GMRES (2904-2971), by one wavefront.
// sm layout: [0] norm_b [1] norm_rhs [2] res [3] maxerr [4] done [5] iter
//            H at 16 + (r-1) + M1*(c-1), Rn after it, Qn after it, then bn and y
struct GmSmall {
    int maxiter;
    __host__ __device__ int M1() const { return maxiter + 1; }
    __host__ __device__ size_t H0() const { return 16; }
    __host__ __device__ size_t R0() const { return H0() + (size_t)M1() * maxiter; }
    __host__ __device__ size_t Q0() const { return R0() + (size_t)M1() * M1(); }
    __host__ __device__ size_t B0() const { return Q0() + (size_t)M1() * M1(); }
    __host__ __device__ size_t Y0() const { return B0() + M1(); }
    __host__ __device__ size_t total() const { return Y0() + M1(); }
};

constexpr int LT = 64;           // one wavefront; maxiter + 1 <= LT
constexpr int LS_MAXITER = 50;   // the reference's value

// The part of the small problem that iteration iter reads, in LDS with columns of iter + 1
// entries: 16 head values, iter columns of H and of Rn, iter + 1 of Qn, and bn.
__host__ __device__ constexpr int ls_doubles(int iter)
{
    return 16 + 2 * iter * (iter + 1) + (iter + 1) * (iter + 1) + iter + 1;
}

// its copy by threads t of nt
__device__ __forceinline__ void ls_load(double* sm, const double* __restrict__ gsm, GmSmall L, int iter, int t, int nt)
{
    const int d = iter + 1, M1 = L.M1(), n1 = d * iter, n2 = 2 * n1, n3 = n2 + d * d, n4 = n3 + d;
    for (int j = t; j < 16 + n4; j += nt) {
        const int e = j - 16;
        size_t a;
        if (e < 0) a = j;
        else if (e < n1) a = L.H0() + e % d + (size_t)M1 * (e / d);
        else if (e < n2) a = L.R0() + (e - n1) % d + (size_t)M1 * ((e - n1) / d);
        else if (e < n3) a = L.Q0() + (e - n2) % d + (size_t)M1 * ((e - n2) / d);
        else a = L.B0() + (e - n3);
        sm[j] = gsm[a];
    }
}

// LDS accesses of one wavefront are served in order: only the compiler has to keep them so
__device__ __forceinline__ void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// x of lane l (the same l in every lane)
__device__ __forceinline__ double of_lane(double x, int l)
{
    const long long b = __double_as_longlong(x);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, l);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// One wavefront, sm as ls_load leaves it, hnext = H(iter + 1, iter).  Lane r owns row r + 1 of the
// triangular factor, of the solution and of the residual; what the iteration changes goes back
// to gsm, and the head to the host's copy as well (null: none).
__device__ void ls_solve(double* sm, double* __restrict__ gsm, GmSmall L, int iter, double hnext, double* host)
{
    const int lane = threadIdx.x & 63, d = iter + 1, M1 = L.M1();
    double* H = sm + 16;
    double* Rn = H + d * iter;
    double* Qn = Rn + d * iter;
    double* bn = Qn + d * d;
#define HH(r, c) H[((r) - 1) + d * ((c) - 1)]
#define RN(r, c) Rn[((r) - 1) + d * ((c) - 1)]
#define QN(r, c) Qn[((r) - 1) + d * ((c) - 1)]
    const double norm_rhs = sm[1];
    double* gH = gsm + L.H0() + (size_t)M1 * (iter - 1);
    double* gR = gsm + L.R0() + (size_t)M1 * (iter - 1);
    double* gQ = gsm + L.Q0();
    if (lane == 0) {
        HH(iter + 1, iter) = hnext;
        gH[iter] = hnext;
    }
    wave_sync();
    double b;                                   // bn(lane + 1)
    if (iter == 1) {
        const double nrm = sqrt(HH(1, 1) * HH(1, 1) + HH(2, 1) * HH(2, 1));
        const double q11 = HH(1, 1) / nrm, q21 = HH(2, 1) / nrm;
        b = q11 * norm_rhs;
        if (lane == 0) {
            gQ[0] = q11; gQ[1] = q21; gQ[M1] = q21; gQ[M1 + 1] = -q11;
            RN(1, 1) = gR[0] = nrm;
            gsm[L.B0()] = b;
        }
        wave_sync();
    } else {
        // new column of R: Qn(1:iter, 1:iter) H(1:iter, iter)
        double r = 0.0;
        if (lane < iter)
            for (int c = 1; c <= iter; ++c) r = r + QN(lane + 1, c) * HH(c, iter);
        const double aa = of_lane(r, iter - 1), bb = hnext;
        const double dd = sqrt(aa * aa + bb * bb);
        const double cc = aa / dd, ss = bb / dd;
        if (lane == iter - 1) r = dd;
        if (lane < iter) RN(lane + 1, iter) = gR[lane] = r;
        // rows iter and iter + 1 of Qn after the rotation
        const double qi = lane < iter ? QN(iter, lane + 1) : 0.0;
        const double qa = lane < iter ? cc * qi : ss, qb = lane < iter ? -ss * qi : cc;
        if (lane <= iter) {
            gQ[(iter - 1) + (size_t)M1 * lane] = qa;
            gQ[iter + (size_t)M1 * lane] = qb;
        }
        b = lane < iter ? bn[lane] : 0.0;
        if (lane == iter - 2) b = QN(iter - 1, 1) * norm_rhs;
        const double blast = of_lane(qa, 0) * norm_rhs;
        if (lane == iter - 1) b = blast;
        if (lane >= iter - 2 && lane < iter) gsm[L.B0() + lane] = b;
        wave_sync();
    }
    // back substitution by columns: lane r accumulates row r + 1
    double acc = 0.0, y = 0.0;
    const double diag = lane < iter ? RN(lane + 1, lane + 1) : 1.0;
    for (int c = iter; c >= 1; --c) {
        const double rc = lane < c - 1 ? RN(lane + 1, c) : 0.0;
        const double yc = of_lane((b - acc) / diag, c - 1);
        if (lane == c - 1) y = yc;
        if (lane < c - 1) acc = acc + yc * rc;
    }
    if (lane < iter) gsm[L.Y0() + lane] = y;
    // residual H y - |r0| e1 (2958-2966)
    double rv = 0.0;
    for (int c = 1; c <= iter; ++c) rv = rv + (lane <= iter ? HH(lane + 1, c) : 0.0) * of_lane(y, c - 1);
    if (lane == 0) rv = rv - norm_rhs;
    double x_c = 0.0;
    for (int r = 0; r <= iter; ++r) {
        const double v = of_lane(rv, r);
        x_c = x_c + v * v;
    }
    if (lane == 0) {
        const double res = sqrt(x_c) / sm[0];
        double maxerr = sm[3];
        int done = 0;
        if (res < maxerr) done = 1;
        else {
            if (iter == L.maxiter / 2) maxerr = maxerr * 10;
            if (iter >= L.maxiter - 2) maxerr = maxerr * 10;
        }
        gsm[2] = res; gsm[3] = maxerr; gsm[4] = done; gsm[5] = iter;
        if (host) { host[2] = res; host[3] = maxerr; host[4] = done; host[5] = iter; }
    }
#undef HH
#undef RN
#undef QN
}

// h = sum of the P_in part_in, v -= sum_j h[j] Q_j (hcol set or, with add, incremented); returns the
// work-group's partial of |v|^2 in every thread
template <typename T>
__device__ __forceinline__ double update_body(T* __restrict__ v, const T* __restrict__ Q, int k, long long n3,
                                               long long ld, const double* __restrict__ part_in, int P_in,
                                               double* hcol, int add, int bx, int nbx)
{
    constexpr int W = kvec<T>::W;
    __shared__ double hs[64];
    __shared__ double sh[RW][1];
    __shared__ double red[1];
    const int tid = threadIdx.x;
    sum_partials(part_in, P_in, k, hs, hcol, add, bx);
    double nacc[1] = {0.0};
    const long long nv = (n3 + W - 1) / W;
    for (long long iv = (long long)bx * RT + tid; iv < nv; iv += (long long)nbx * RT) {
        const long long i = iv * W;
        if (i + W <= n3) {
            T xv[W];
            vld(v + i, xv);
            double x[W];
#pragma unroll
            for (int e = 0; e < W; ++e) x[e] = (double)xv[e];
#pragma unroll 4
            for (int j = 0; j < k; ++j) {
                T q[W];
                vld(Q + (size_t)j * ld + i, q);
                const double hj = hs[j];
#pragma unroll
                for (int e = 0; e < W; ++e) x[e] -= hj * (double)q[e];
            }
#pragma unroll
            for (int e = 0; e < W; ++e) {
                xv[e] = (T)x[e];
                nacc[0] += (double)xv[e] * (double)xv[e];
            }
            vst(v + i, xv);
        } else {
            for (long long e = i; e < n3; ++e) {
                double x = (double)v[e];
                for (int j = 0; j < k; ++j) x -= hs[j] * (double)Q[(size_t)j * ld + e];
                const T xt = (T)x;
                v[e] = xt;
                nacc[0] += (double)xt * (double)xt;
            }
        }
    }
    block_sums<1>(nacc, sh, red);
    return red[0];
}

// The first pass's update where it has a kernel of its own (k > 12)
template <typename T>
__global__ void __launch_bounds__(RT) k_maxpy(T* __restrict__ v, const T* __restrict__ Q, int k, long long n3,
                                              long long ld, const double* __restrict__ part_in,
                                              double* __restrict__ hcol, const double* __restrict__ stop)
{
    if (*stop != 0.0) return;
    update_body<T>(v, Q, k, n3, ld, part_in, gridDim.x, hcol, 0, blockIdx.x, gridDim.x);
}

// The end of iteration k: the second pass's update, then the least-squares update with
// H(k + 1, k) = |v|.  gate_w and gate_v hold the P_w and nbx partials of |w|^2 before the first
// pass and of |v|^2 after it; when the first pass kept at least 1/sqrt(2) of the norm (|v|^2 >= |w|^2 / 2, the
// DGKS criterion) the second pass's corrections are below rounding, its update is skipped (v and
// hcol stay) and work-group 0 goes on by itself, its upper wavefronts having loaded the small
// problem while the lower ones summed the gate.  Otherwise the last work-group to arrive (arrive
// counts them and is left zero) sums the partials and goes on.  As two kernels the update and
// the single wavefront of the least squares took 5.2 + 7.8 us at 100 000 droplets.
// ls: ls_doubles(k) of LDS.
template <typename T>
__global__ void __launch_bounds__(RT) k_finish(T* __restrict__ v, const T* __restrict__ Q, int k, long long n3,
                                               long long ld, const double* __restrict__ part_in,
                                               double* hcol, double* normpart, const double* stop,
                                               const double* __restrict__ gate_w, int P_w,
                                               const double* __restrict__ gate_v, double* gsm, GmSmall L, int* arrive,
                                               double* host)
{
    extern __shared__ double ls[];
    __shared__ double g1[2];
    __shared__ int last;
    if (*stop != 0.0) return;
    const int tid = threadIdx.x, bx = blockIdx.x, nbx = gridDim.x;
    if (bx == 0 && tid >= RT / 2) ls_load(ls, gsm, L, k, tid - RT / 2, RT / 2);
    const double nw = sum_one(gate_w, P_w, &g1[0]);
    double nv2 = sum_one(gate_v, nbx, &g1[1]);
    if (nv2 >= 0.5 * nw) {
        if (bx != 0) return;
    } else {
        const double mine = update_body<T>(v, Q, k, n3, ld, part_in, nbx, hcol, 1, bx, nbx);
        if (tid == 0) {
            normpart[bx] = mine;
            __threadfence();                       // the partial and hcol, before the arrival
            last = atomicAdd(arrive, 1) == nbx - 1;
        }
        __syncthreads();
        if (!last) return;
        __threadfence();
        if (tid == 0) *arrive = 0;
        ls_load(ls, gsm, L, k, tid, RT);
        nv2 = sum_one(normpart, nbx, &g1[0]);
    }
    if (tid < LT) ls_solve(ls, gsm, L, k, sqrt(nv2), host);
}

// pertvel = x0 + Q y (2951-2956), scattered back to the reference's droplet order.  The
// number of Krylov columns is the small problem's count of the iterations that ran
// (*itp), read on the device, so the kernel can be queued before the host has seen it.
template <typename T>
__global__ void k_solution(const double* x0, const T* Q, long long ld, const double* y, const double* itp,
                           const int* sorted, double* pert, int n, int cap)
{
    // one droplet per thread: its three components go out as one 24-byte record
    const int t = blockIdx.x * HT + threadIdx.x;
    if (t >= n) return;
    const int iters = (int)*itp;
    double out[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const size_t i = (size_t)c * n + t;
        double acc = 0.0;
        for (int j = 0; j < iters; ++j) acc = acc + (double)Q[(size_t)j * ld + i] * y[j];
        out[c] = x0[i] + acc;
    }
    double* dst = pert + 3 * (size_t)sorted[t];
#pragma unroll
    for (int c = 0; c < 3; ++c) dst[c] = out[c];
}

// ------------------------------------------------------------------ driver
// NEI_LIST_PRECOMP (partlib.f90:3218-3371) queued without a host wait: the flags it
// raises are read with the solve's first convergence check (lists_outcome).
template <typename T>
static int queue_lists(PartBuffers& pb, const PartConst& pc, hipStream_t s)
{
    const int n = pc.n;
    if (!pb.nei_idx) {
        pb.ell_width = 2 * ELL_STEP;
        DDNS_HIP(hipMalloc(&pb.nei_idx, (size_t)pb.ell_width * pb.cap * sizeof(int)));
        DDNS_HIP(hipMalloc(&pb.nei_m, (size_t)6 * pb.ell_width * pb.cap * sizeof(T)));
    }
    // the flags are clear: from the step's start, or from lists_outcome when the lists are filled again
    auto launch = [&](auto kernel, int lanes) {
        hipLaunchKernelGGL(kernel, dim3((unsigned)(((long long)n * lanes + NT_NEI - 1) / NT_NEI)), dim3(NT_NEI), 0, s,
                           (const double4*)pb.pk, pb.cell_start, n, pb.G, pb.hc, pc.pi2, pc.hdi_trunc, pb.ell_width,
                           pb.nei_cnt, pb.nei_idx, (T*)pb.nei_m, pb.flags);
    };
    if (n <= NEI_SHARED) launch(k_nei<T, 4>, 4);
    else launch(k_nei<T, 1>, 1);
    DDNS_HIP(hipGetLastError());
    return 0;
}

// The flags of queue_lists, once read: an error (overlapping droplets, more than 100
// neighbours), 1 when some row had more neighbours than the lists hold (they have been
// widened; fill them again), else 0.
template <typename T>
static int lists_outcome(PartBuffers& pb, const int* f, hipStream_t s)
{
    if (f[0] & 1) { set_error("inside NEI_LIST_PRECOMP: overlapping is not allowed"); return DDNS_ERR_OVERLAP; }
    if (f[0] & 2) { set_error("more than 100 HI neighbours for a droplet"); return DDNS_ERR_NEIGHBOUR_OVERFLOW; }
    if (f[4] <= pb.ell_width) return 0;
    DDNS_HIP(hipMemsetAsync(pb.flags, 0, 8 * sizeof(int), s));     // what fills them again follows on s
    if (pb.nei_idx) { (void)hipFree(pb.nei_idx); (void)hipFree(pb.nei_m); pb.nei_idx = nullptr; pb.nei_m = nullptr; }
    pb.ell_width = std::min(DDNS_MAXNEI, (f[4] + ELL_STEP - 1) / ELL_STEP * ELL_STEP);
    DDNS_HIP(hipMalloc(&pb.nei_idx, (size_t)pb.ell_width * pb.cap * sizeof(int)));
    DDNS_HIP(hipMalloc(&pb.nei_m, (size_t)6 * pb.ell_width * pb.cap * sizeof(T)));
    return 1;
}

// The solve's start (2820-2868) queued on s without a host wait: the neighbour lists,
// b = M w and A x0, r0 = b - A x0 into the first Krylov column with the norms, the
// small problem cleared, the tolerance and the stop flag, and q_1 = r0 / |r0|.
template <typename T>
static int hdi_begin(PartBuffers& pb, const PartConst& pc, int maxiter, double tol, hipStream_t s)
{
    const int n = pc.n;
    const long long n3 = 3LL * n;
    static_assert(LS_MAXITER + 1 <= LT && ls_doubles(LS_MAXITER) * sizeof(double) <= 63 * 1024, "least squares in one wavefront, in LDS");
    if (maxiter > LS_MAXITER) { set_error("GMRES maxiter too large (at most 50)"); return DDNS_ERR_ARG; }
    GmSmall L{maxiter};
    if (!pb.gm_host) DDNS_HIP(hipHostMalloc((void**)&pb.gm_host, 16 * sizeof(double), hipHostMallocDefault));
    // Krylov storage
    if (!pb.gm_small) {
        DDNS_HIP(hipMalloc(&pb.gm_small, 16384 * sizeof(double)));
        DDNS_HIP(hipMalloc(&pb.gm_red, (size_t)(128 + 2) * RED_BLOCKS * sizeof(double)));
        DDNS_HIP(hipMalloc(&pb.gm_b, 3 * (size_t)pb.cap * sizeof(double)));
        DDNS_HIP(hipMalloc(&pb.gm_v, 3 * (size_t)pb.cap * sizeof(double)));
        DDNS_HIP(hipMalloc(&pb.gm_Q, (size_t)(maxiter + 2) * ((3LL * pb.cap + 63) / 64 * 64) * sizeof(T)));
    }
    double* sm = pb.gm_small;
    double* ax0 = (double*)pb.gm_v;
    T* Q = (T*)pb.gm_Q;
    const unsigned nb3 = (unsigned)((n3 + HT - 1) / HT);
    const unsigned nbr = (unsigned)((n + HT - 1) / HT);
    const int sq = queue_lists<T>(pb, pc, s);
    if (sq) return sq;
    // x0 (pertvel) and w = V - U in cell order were written by the interpolation
    hipLaunchKernelGGL((k_spmv<T, 0>), dim3(nbr), dim3(HT), 0, s, (const int*)pb.nei_cnt, (const int*)pb.nei_idx,
                       (const T*)pb.nei_m, n, (const T*)nullptr, (const double*)nullptr, (T*)nullptr, (T*)nullptr,
                       (const double*)pb.gm_x0, ax0, (const double*)pb.gm_w, pb.gm_b, (const double*)nullptr);
    const int nr0 = (int)std::min<long long>(RED_BLOCKS, (n3 + HT - 1) / HT);
    hipLaunchKernelGGL((k_residual0<T>), dim3(nr0), dim3(HT), 0, s, pb.gm_b, ax0, Q, n3, pb.gm_red);
    // the tolerance, and the stop flag when the initial residual is below 1e-5
    // (2866-2868): then no iteration runs and pertvel keeps its warm-start value
    hipLaunchKernelGGL(k_gm_start, dim3(1), dim3(HT), 0, s, sm, (int)L.total(), tol, (const double*)pb.gm_red, nr0,
                       (const int*)pb.flags, pb.gm_host);
    hipLaunchKernelGGL((k_scale<T>), dim3(nb3), dim3(HT), 0, s, Q, sm + 1, n3);
    DDNS_HIP(hipGetLastError());
    return 0;
}

// work-groups of the projection kernels of a system of n droplets: as many as have about 700
// rows each.  With twice the rows the 74 work-groups of 100 000 droplets left most CUs idle (a
// solve 0.37 against 0.33 ms at 78 000 droplets in FP64, 0.73 against 0.58 at 60 000); with half
// of them the merged launches of a batch grew from 4.6 to 5.2 ms a step.
static int hdi_nred(int n)
{
    return (int)std::min<long long>(RED_BLOCKS, (3LL * n + 2LL * RT - 1) / (2LL * RT));
}

// those of them that have a vector of 16 bytes for a thread: the work-groups of the kernels that
// go by vectors.  In single precision that is half of them; the others added nothing to any sum,
// but read all partials for it, in a batch of 48 systems 229 against 142 us a launch
template <typename T>
static int hdi_nvec(int n)
{
    constexpr long long per = (long long)kvec<T>::W * RT;
    return (int)std::min<long long>(hdi_nred(n), (3LL * n + per - 1) / per);
}

template <typename T>
static int hdi_impl(PartBuffers& pb, const PartConst& pc, int maxiter, double tol, int* iters_out, double* res_out,
                    hipStream_t s)
{
    const int n = pc.n;
    const long long n3 = 3LL * n;
    *iters_out = 0;
    *res_out = 0.0;
    if (n == 0) return 0;
    GmSmall L{maxiter};
    const long long ld = (n3 + 63) / 64 * 64;     // column stride of the Krylov vectors
    const unsigned nbr = (unsigned)((n + HT - 1) / HT);
    const unsigned nred = (unsigned)hdi_nred(n), nvec = (unsigned)hdi_nvec<T>(n);   // reduction grids
    // The neighbour lists are filled and the solve started without a host wait; the
    // first convergence check also reads the lists' flags, and when a row had more
    // neighbours than the lists hold they are widened and the solve starts over (its
    // inputs x0 and w are unchanged, and pertvel is written only at the end).
    int iter = 0;
    double st6[6] = {0, 0, 0, 0, 0, 0};
    double* sm = nullptr;
    T* Q = nullptr;
    for (int lists = 1; lists > 0;) {
        // the Krylov storage is allocated by the first hdi_begin of the handle: every
        // pointer into it is taken after the call
        const int sq = hdi_begin<T>(pb, pc, maxiter, tol, s);
        if (sq) return sq;
        lists = 0;
        sm = pb.gm_small;
        Q = (T*)pb.gm_Q;
        double* part1 = pb.gm_red;                          // first-pass projections
        double* part2 = part1 + (size_t)64 * RED_BLOCKS;    // second-pass projections
        double* normpart = part2 + (size_t)64 * RED_BLOCKS;
        T* work[2] = {Q + (size_t)maxiter * ld, Q + (size_t)(maxiter + 1) * ld};
        // Iterations are launched in batches; every kernel of an iteration returns at
        // once when the least-squares update of an earlier one has set the converged
        // flag sm[4], so the host checks it once per batch.  The first batch runs as many
        // iterations as the last solve needed (consecutive steps converge alike), the
        // later ones three at a time.
        constexpr int BATCH = 3;
        const double* stop = sm + 4;
        double* Hd = sm + L.H0();
        const int M1 = L.M1();
        iter = 0;
        for (double& v : st6) v = 0.0;
        bool first = true;
        while (iter < maxiter && st6[4] == 0.0) {
            const int last = std::min(maxiter, iter + (iter == 0 ? std::max(BATCH, pb.gm_last_iters) : BATCH));
            for (int it = iter + 1; it <= last; ++it) {
                T* v = work[it & 1];
                // v = A q_it, q_it = v_(it-1) / H(it, it-1) formed inside the product; up to
                // 12 columns the first pass's projections are summed in the same kernel
                const T* xin = it == 1 ? (const T*)Q : (const T*)work[(it - 1) & 1];
                const double* hx = it == 1 ? (const double*)nullptr : (const double*)(Hd + (size_t)M1 * (it - 2) + (it - 1));
                T* qo = it == 1 ? (T*)nullptr : Q + (size_t)(it - 1) * ld;
                const int* nc = (const int*)pb.nei_cnt;
                const int* ni = (const int*)pb.nei_idx;
                const T* nm = (const T*)pb.nei_m;
                if (it == 1)
                    hipLaunchKernelGGL((k_spmv_mdot<T, 1, 8>), dim3(nred), dim3(RT), 0, s, nc, ni, nm, n, xin, hx, qo, v,
                                       (const T*)Q, ld, it, part1, stop);
                else if (it <= 8)
                    hipLaunchKernelGGL((k_spmv_mdot<T, 2, 8>), dim3(nred), dim3(RT), 0, s, nc, ni, nm, n, xin, hx, qo, v,
                                       (const T*)Q, ld, it, part1, stop);
                else if (it <= 12)
                    hipLaunchKernelGGL((k_spmv_mdot<T, 2, 12>), dim3(nred), dim3(RT), 0, s, nc, ni, nm, n, xin, hx, qo,
                                       v, (const T*)Q, ld, it, part1, stop);
                else {
                    hipLaunchKernelGGL((k_spmv<T, 2>), dim3(nbr), dim3(HT), 0, s, nc, ni, nm, n, xin, hx, qo, v,
                                       (const double*)nullptr, (double*)nullptr, (const double*)nullptr, (double*)nullptr,
                                       stop);
                    hipLaunchKernelGGL((k_mdot<T>), dim3(nvec), dim3(RT), 0, s, (const T*)Q, (const T*)v, it, n3, ld, part1,
                                       stop);
                }
                // orthogonalise v against q_1..q_it: classical Gram-Schmidt, twice (the
                // reference's modified Gram-Schmidt, 2886-2894, in two block passes), the
                // second pass's update only where the DGKS criterion asks for it
                double* hcol = Hd + (size_t)M1 * (it - 1);
                if (it <= 8)
                    hipLaunchKernelGGL((k_maxpy_mdot<T, 8>), dim3(nvec), dim3(RT), 0, s, v, (const T*)Q, it, n3, ld,
                                       (const double*)part1, (int)nred, hcol, part2, stop);
                else if (it <= 12)
                    hipLaunchKernelGGL((k_maxpy_mdot<T, 12>), dim3(nvec), dim3(RT), 0, s, v, (const T*)Q, it, n3, ld,
                                       (const double*)part1, (int)nred, hcol, part2, stop);
                else {
                    hipLaunchKernelGGL((k_maxpy<T>), dim3(nvec), dim3(RT), 0, s, v, (const T*)Q, it, n3, ld,
                                       (const double*)part1, hcol, stop);
                    hipLaunchKernelGGL((k_mdot<T>), dim3(nvec), dim3(RT), 0, s, (const T*)Q, (const T*)v, it, n3, ld, part2,
                                       stop);
                }
                // the second pass's update, skipped where the first kept 1/sqrt(2) of |v|, and the
                // least squares
                const unsigned P1 = it <= 12 ? nred : nvec;        // partials of the first pass
                hipLaunchKernelGGL((k_finish<T>), dim3(nvec), dim3(RT), ls_doubles(it) * sizeof(double), s, v, (const T*)Q,
                                   it, n3, ld, (const double*)part2, hcol, normpart, stop,
                                   (const double*)(part1 + (size_t)it * P1), (int)P1,
                                   (const double*)(part2 + (size_t)it * nvec), sm, L, pb.flags + 56, pb.gm_host);
            }
            DDNS_HIP(hipGetLastError());
            iter = last;
            // the kernels leave the small problem's head, and the start the neighbour lists'
            // flags, in host memory (two copies took the stream 10 us)
            int f[8];
            const int* fh = (const int*)(pb.gm_host + 8);
            if (!pb.sync_ev) DDNS_HIP(hipEventCreateWithFlags(&pb.sync_ev, hipEventDisableTiming));
            DDNS_HIP(hipEventRecord(pb.sync_ev, s));
            // the solution as far as this batch got (pertvel = x0 where no iteration ran),
            // queued behind the event: when the batch converged, the usual case, it runs
            // while the host reads the check and queues what follows; a later batch is
            // followed by its own
            hipLaunchKernelGGL((k_solution<T>), dim3(nbr), dim3(HT), 0, s, pb.gm_x0, (const T*)Q, ld, sm + L.Y0(),
                               (const double*)(sm + 5), (const int*)pb.sorted, pb.pert, n, pb.cap);
            DDNS_HIP(spin_wait(pb.sync_ev));
            std::memcpy(st6, pb.gm_host, sizeof(st6));
            if (first) std::memcpy(f, fh, sizeof(f));
            if (first) {
                first = false;
                lists = lists_outcome<T>(pb, f, s);
                if (lists < 0) return lists;
                if (lists > 0) break;            // fill the widened lists and solve again
            }
        }
    }
    if (st6[4] < 0.0) return 0;     // initial residual below 1e-5: no iteration
    const bool done = st6[4] != 0.0;
    const int used = (int)st6[5];   // the last iteration that ran
    pb.gm_last_iters = used;
    DDNS_HIP(hipGetLastError());
    // the solution was queued behind the last check; the residual and its bound were
    // final then: the solution kernel reads the small problem but does not change it
    *iters_out = used;
    *res_out = st6[2];
    if (!done && st6[2] > st6[3]) return DDNS_WARN_GMRES;                   // 2980-2982
    return 0;
}

int part_hdi(PartBuffers& pb, const PartConst& pc, int maxiter, double tol, int* iters, double* res, hipStream_t s)
{
    if (pc.precision == DDNS_FP64) return hdi_impl<double>(pb, pc, maxiter, tol, iters, res, s);
    return hdi_impl<float>(pb, pc, maxiter, tol, iters, res, s);
}

int part_hdi_begin(PartBuffers& pb, const PartConst& pc, int maxiter, double tol, hipStream_t s)
{
    if (pc.n == 0) return 0;
    if (pc.precision == DDNS_FP64) return hdi_begin<double>(pb, pc, maxiter, tol, s);
    return hdi_begin<float>(pb, pc, maxiter, tol, s);
}

// ------------------------------------------------------------------ batched solve
// The GMRES iterations of several independent systems (one per realisation of a batch)
// run together: each kernel of an iteration is one launch whose work-group row y works
// on system y.  Every system keeps its own Krylov basis, small problem, stop flag and
// reduction partials, and its reductions run on the grid of nred work-groups its own
// solve would use, so each system gets the same bits as when solved alone; a converged
// system's work-groups return at once, as in a solve of its own.
template <typename T>
struct GmDesc {
    const int* cnt;
    const int* idx;
    const T* mm;
    const int* flags;          // the neighbour lists' flags (read at the first check)
    T* Q;                      // maxiter Krylov columns, then the two work vectors
    double* sm;                // the small problem (GmSmall layout)
    double* part1;             // first-pass projection partials
    double* part2;             // second-pass projection partials
    double* normpart;          // |v|^2 partials
    long long n3, ld;
    int n, nred, nvec, nbr;    // 0: the system takes no part (any more)
};

template <typename T>
struct GmIter {
    const T* xin;
    const double* hx;
    T* qo;
    T* v;
    double* hcol;
    const double* stop;
};

// the vectors and Hessenberg entries of iteration it, as hdi_impl forms them
template <typename T>
__device__ __forceinline__ GmIter<T> gm_iter(const GmDesc<T>& g, GmSmall L, int it)
{
    GmIter<T> r;
    T* w0 = g.Q + (size_t)L.maxiter * g.ld;
    T* w1 = w0 + g.ld;
    double* Hd = g.sm + L.H0();
    const size_t M1 = L.M1();
    r.v = (it & 1) ? w1 : w0;
    r.xin = it == 1 ? g.Q : (((it - 1) & 1) ? w1 : w0);
    r.hx = it == 1 ? nullptr : Hd + M1 * (it - 2) + (it - 1);
    r.qo = it == 1 ? nullptr : g.Q + (size_t)(it - 1) * g.ld;
    r.hcol = Hd + M1 * (it - 1);
    r.stop = g.sm + 4;
    return r;
}

template <typename T, int MODE, int KC>
__global__ void __launch_bounds__(RT) kb_spmv_mdot(const GmDesc<T>* __restrict__ d, GmSmall L, int it)
{
    const GmDesc<T>& g = d[blockIdx.y];
    if ((int)blockIdx.x >= g.nred) return;
    const GmIter<T> q = gm_iter(g, L, it);
    k_spmv_mdot_body<T, MODE, KC>(g.cnt, g.idx, g.mm, g.n, q.xin, q.hx, q.qo, q.v, g.Q, g.ld, it, g.part1, q.stop,
                                  blockIdx.x, g.nred);
}

template <typename T>
__global__ void __launch_bounds__(HT) kb_spmv2(const GmDesc<T>* __restrict__ d, GmSmall L, int it)
{
    const GmDesc<T>& g = d[blockIdx.y];
    if (g.nred == 0 || (int)blockIdx.x >= g.nbr) return;
    const GmIter<T> q = gm_iter(g, L, it);
    k_spmv_body<T, 2>(g.cnt, g.idx, g.mm, g.n, q.xin, q.hx, q.qo, q.v, nullptr, nullptr, nullptr, nullptr, q.stop,
                      blockIdx.x, g.nbr);
}

template <typename T>
__global__ void __launch_bounds__(RT) kb_mdot(const GmDesc<T>* __restrict__ d, GmSmall L, int it, int second)
{
    const GmDesc<T>& g = d[blockIdx.y];
    if ((int)blockIdx.x >= g.nvec) return;
    const GmIter<T> q = gm_iter(g, L, it);
    k_mdot_body<T>(g.Q, q.v, it, g.n3, g.ld, second ? g.part2 : g.part1, q.stop, blockIdx.x, g.nvec);
}

template <typename T, int KC>
__global__ void __launch_bounds__(RT) kb_maxpy_mdot(const GmDesc<T>* __restrict__ d, GmSmall L, int it)
{
    const GmDesc<T>& g = d[blockIdx.y];
    if ((int)blockIdx.x >= g.nvec) return;
    const GmIter<T> q = gm_iter(g, L, it);
    k_maxpy_mdot_body<T, KC>(q.v, g.Q, it, g.n3, g.ld, g.part1, g.nred, q.hcol, g.part2, q.stop, blockIdx.x, g.nvec);
}

template <typename T>
__global__ void __launch_bounds__(RT) kb_maxpy(const GmDesc<T>* __restrict__ d, GmSmall L, int it)
{
    const GmDesc<T>& g = d[blockIdx.y];
    if ((int)blockIdx.x >= g.nvec) return;
    const GmIter<T> q = gm_iter(g, L, it);
    if (*q.stop != 0.0) return;
    update_body<T>(q.v, g.Q, it, g.n3, g.ld, g.part1, g.nvec, q.hcol, 0, blockIdx.x, g.nvec);
}

// k_finish as two launches: the second pass's update, then the least squares of every system.  In
// one launch each of the systems' work-groups, 2000 to 12 000 in all, wrote back and invalidated
// its XCD's L2 for the arrival: 228 us a launch with 48 systems, 47 + 8 as two (a system alone has at most
// 256, and saves the second launch).
template <typename T>
__device__ __forceinline__ bool kb_gate(const GmDesc<T>& g, int it, double* g1, double* nv2)
{
    const int P1 = it <= 12 ? g.nred : g.nvec;
    const double nw = sum_one(g.part1 + (size_t)it * P1, P1, &g1[0]);
    *nv2 = sum_one(g.part2 + (size_t)it * g.nvec, g.nvec, &g1[1]);
    return *nv2 >= 0.5 * nw;                     // the first pass suffices
}

template <typename T>
__global__ void __launch_bounds__(RT) kb_second(const GmDesc<T>* __restrict__ d, GmSmall L, int it)
{
    __shared__ double g1[2];
    const GmDesc<T>& g = d[blockIdx.y];
    if ((int)blockIdx.x >= g.nvec) return;
    const GmIter<T> q = gm_iter(g, L, it);
    if (*q.stop != 0.0) return;
    double nv2;
    if (kb_gate(g, it, g1, &nv2)) return;
    const double mine = update_body<T>(q.v, g.Q, it, g.n3, g.ld, g.part2, g.nvec, q.hcol, 1, blockIdx.x, g.nvec);
    if (threadIdx.x == 0) g.normpart[blockIdx.x] = mine;
}

template <typename T>
__global__ void __launch_bounds__(HT) kb_ls(const GmDesc<T>* __restrict__ d, GmSmall L, int it)
{
    extern __shared__ double ls_lds[];
    __shared__ double g1[2], g2;
    const GmDesc<T>& g = d[blockIdx.x];
    if (g.nred == 0 || g.sm[4] != 0.0) return;
    ls_load(ls_lds, g.sm, L, it, threadIdx.x, HT);
    double nv2;
    if (!kb_gate(g, it, g1, &nv2)) nv2 = sum_one(g.normpart, g.nvec, &g2);
    if (threadIdx.x < LT) ls_solve(ls_lds, g.sm, L, it, sqrt(nv2), nullptr);
}

// each system's small-problem head sm[0..5] (and its lists' flags) into 16 doubles
template <typename T>
__global__ void kb_heads(const GmDesc<T>* __restrict__ d, double* out, int with_flags)
{
    const GmDesc<T>& g = d[blockIdx.x];
    double* o = out + 16 * (size_t)blockIdx.x;
    const int i = threadIdx.x;
    if (!g.sm) {                       // no droplets, no solve: reads as "no iteration"
        if (i < 6) o[i] = i == 4 ? -1.0 : 0.0;
        if (i < 8) ((int*)(o + 8))[i] = 0;
        return;
    }
    if (i < 6) o[i] = g.sm[i];
    if (with_flags && i < 8) ((int*)(o + 8))[i] = g.flags[i];
}

void part_hdi_batch_free(HdiBatch& hb)
{
    if (hb.table) (void)hipFree(hb.table);
    if (hb.heads) (void)hipFree(hb.heads);
    if (hb.table_host) (void)hipHostFree(hb.table_host);
    if (hb.heads_host) (void)hipHostFree(hb.heads_host);
    hb = HdiBatch{};
}

template <typename T>
static int hdi_batch_impl(HdiBatch& hb, PartBuffers* const* pbs, const PartConst* const* pcs, int R, int maxiter,
                          int* iters, double* res, int* status, int* redo, hipStream_t s)
{
    if (R <= 0) return 0;
    GmSmall L{maxiter};
    if (hb.cap < R) {
        part_hdi_batch_free(hb);
        DDNS_HIP(hipMalloc(&hb.table, (size_t)R * sizeof(GmDesc<T>)));
        DDNS_HIP(hipMalloc(&hb.heads, (size_t)R * 16 * sizeof(double)));
        DDNS_HIP(hipHostMalloc(&hb.table_host, (size_t)R * sizeof(GmDesc<double>), hipHostMallocDefault));
        DDNS_HIP(hipHostMalloc((void**)&hb.heads_host, (size_t)R * 16 * sizeof(double), hipHostMallocDefault));
        hb.cap = R;
    }
    GmDesc<T>* th = (GmDesc<T>*)hb.table_host;
    int nredmax = 0, nvecmax = 0, nbrmax = 0, first = 3;
    for (int r = 0; r < R; ++r) {
        PartBuffers& pb = *pbs[r];
        const int n = pcs[r]->n;
        iters[r] = 0; res[r] = 0.0; status[r] = 0; redo[r] = 0;
        GmDesc<T> g{};
        if (n == 0 || !pb.gm_small) {  // nothing to solve (part_hdi_begin queued nothing)
            th[r] = g;
            continue;
        }
        g.cnt = pb.nei_cnt; g.idx = pb.nei_idx; g.mm = (const T*)pb.nei_m; g.flags = pb.flags;
        g.Q = (T*)pb.gm_Q; g.sm = pb.gm_small;
        g.part1 = pb.gm_red; g.part2 = g.part1 + (size_t)64 * RED_BLOCKS; g.normpart = g.part2 + (size_t)64 * RED_BLOCKS;
        g.n3 = 3LL * n; g.ld = (g.n3 + 63) / 64 * 64; g.n = n;
        g.nred = hdi_nred(n); g.nvec = hdi_nvec<T>(n); g.nbr = (n + HT - 1) / HT;
        th[r] = g;
        nredmax = std::max(nredmax, g.nred);
        nvecmax = std::max(nvecmax, g.nvec);
        nbrmax = std::max(nbrmax, g.nbr);
        first = std::max(first, pb.gm_last_iters);
    }
    const GmDesc<T>* td = (const GmDesc<T>*)hb.table;
    DDNS_HIP(hipMemcpyAsync(hb.table, th, (size_t)R * sizeof(GmDesc<T>), hipMemcpyHostToDevice, s));
    constexpr int BATCH = 3;
    std::vector<double> st6((size_t)R * 6, 0.0);
    std::vector<char> done(R, 0);
    int iter = 0;
    bool firstcheck = true;
    while (iter < maxiter) {
        bool any = false;
        for (int r = 0; r < R; ++r) any = any || (!done[r] && !redo[r]);
        if (!any) break;
        const int last = std::min(maxiter, iter + (iter == 0 ? first : BATCH));
        const dim3 g(nredmax, R), gv(nvecmax, R);
        for (int it = iter + 1; it <= last; ++it) {
            if (it == 1) hipLaunchKernelGGL((kb_spmv_mdot<T, 1, 8>), g, dim3(RT), 0, s, td, L, it);
            else if (it <= 8) hipLaunchKernelGGL((kb_spmv_mdot<T, 2, 8>), g, dim3(RT), 0, s, td, L, it);
            else if (it <= 12) hipLaunchKernelGGL((kb_spmv_mdot<T, 2, 12>), g, dim3(RT), 0, s, td, L, it);
            else {
                hipLaunchKernelGGL((kb_spmv2<T>), dim3(nbrmax, R), dim3(HT), 0, s, td, L, it);
                hipLaunchKernelGGL((kb_mdot<T>), gv, dim3(RT), 0, s, td, L, it, 0);
            }
            if (it <= 8) hipLaunchKernelGGL((kb_maxpy_mdot<T, 8>), gv, dim3(RT), 0, s, td, L, it);
            else if (it <= 12) hipLaunchKernelGGL((kb_maxpy_mdot<T, 12>), gv, dim3(RT), 0, s, td, L, it);
            else {
                hipLaunchKernelGGL((kb_maxpy<T>), gv, dim3(RT), 0, s, td, L, it);
                hipLaunchKernelGGL((kb_mdot<T>), gv, dim3(RT), 0, s, td, L, it, 1);
            }
            hipLaunchKernelGGL((kb_second<T>), gv, dim3(RT), 0, s, td, L, it);
            hipLaunchKernelGGL((kb_ls<T>), dim3(R), dim3(HT), ls_doubles(it) * sizeof(double), s, td, L, it);
        }
        DDNS_HIP(hipGetLastError());
        iter = last;
        // one check for every system: the heads (and, the first time, the lists' flags)
        hipLaunchKernelGGL((kb_heads<T>), dim3(R), dim3(64), 0, s, td, hb.heads, firstcheck ? 1 : 0);
        DDNS_HIP(hipMemcpyAsync(hb.heads_host, hb.heads, (size_t)R * 16 * sizeof(double), hipMemcpyDeviceToHost, s));
        DDNS_HIP(hipStreamSynchronize(s));
        bool retable = false;
        for (int r = 0; r < R; ++r) {
            if (redo[r] || !th[r].sm) {
                done[r] = 1;
                st6[6 * (size_t)r + 4] = -1.0;
                continue;
            }
            const double* h = hb.heads_host + 16 * (size_t)r;
            for (int k = 0; k < 6; ++k) st6[6 * (size_t)r + k] = h[k];
            if (firstcheck) {
                int f[8];
                std::memcpy(f, h + 8, sizeof(f));
                // the system leaves the merged launches before its lists are reallocated
                if (f[0] & 3 || f[4] > pbs[r]->ell_width) {
                    th[r].nred = th[r].nvec = th[r].nbr = 0;
                    retable = true;
                }
                const int lo = lists_outcome<T>(*pbs[r], f, s);
                if (lo < 0) {
                    status[r] = lo;
                    DDNS_HIP(hipMemcpyAsync(hb.table, th, (size_t)R * sizeof(GmDesc<T>), hipMemcpyHostToDevice, s));
                    DDNS_HIP(hipStreamSynchronize(s));
                    return lo;
                }
                if (lo > 0) redo[r] = 1;        // widened: solved again on its own
            }
            done[r] = st6[6 * (size_t)r + 4] != 0.0;
        }
        if (retable) DDNS_HIP(hipMemcpyAsync(hb.table, th, (size_t)R * sizeof(GmDesc<T>), hipMemcpyHostToDevice, s));
        firstcheck = false;
    }
    for (int r = 0; r < R; ++r) {
        if (redo[r]) continue;
        PartBuffers& pb = *pbs[r];
        const double* h = &st6[6 * (size_t)r];
        if (h[4] < 0.0) continue;      // initial residual below 1e-5: no iteration
        const bool ok = h[4] != 0.0;
        const int used = (int)h[5];
        pb.gm_last_iters = used;
        const int n = pcs[r]->n;
        const long long ld = (3LL * n + 63) / 64 * 64;
        hipLaunchKernelGGL((k_solution<T>), dim3((n + HT - 1) / HT), dim3(HT), 0, s, pb.gm_x0, (const T*)pb.gm_Q, ld,
                           pb.gm_small + L.Y0(), (const double*)(pb.gm_small + 5), (const int*)pb.sorted, pb.pert, n,
                           pb.cap);
        iters[r] = used;
        res[r] = h[2];
        if (!ok && h[2] > h[3]) status[r] = DDNS_WARN_GMRES;                // 2980-2982
    }
    DDNS_HIP(hipGetLastError());
    return 0;
}

int part_hdi_batch(HdiBatch& hb, PartBuffers* const* pbs, const PartConst* const* pcs, int R, int maxiter,
                   int* iters, double* res, int* status, int* redo, hipStream_t s)
{
    if (R <= 0) return 0;
    if (pcs[0]->precision == DDNS_FP64) return hdi_batch_impl<double>(hb, pbs, pcs, R, maxiter, iters, res, status, redo, s);
    return hdi_batch_impl<float>(hb, pbs, pcs, R, maxiter, iters, res, status, redo, s);
}

}  // namespace ddns
