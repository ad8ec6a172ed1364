// particles.hip -- Lagrangian droplet step on one MI355X (everything but the pair
// searches, which live in collide.hip, and the HI solve in hdi.hip).
//
// Reference: PREPARE_INTERP / INTERPOLATE partlib.f90:305-520 (6-point Lagrange
// gather), PART_HISTORY_FVP/FDP 553-625, PART_ADVANCE 629-726, UPDATE_PART_POSITION
// 730-757, PERIODIC wrap 1142-1151, RELOCATE 1984-2012.  The reference's linked
// cell list (HEADLIST 2171-2444) is replaced by a counting sort of droplets into a
// coarse periodic grid; periodic images are formed on the fly by the pair kernels.
//
// Droplet state is structure-of-arrays in double, slot i = the reference's array
// index i+1, so every index-order rule of the reference (ih2 > ih1, the order of the
// removal list and of the relocation draws) is evaluated on slot numbers.
#include "ddns_internal.h"

#include <cstring>

#include <algorithm>
#include <cmath>

namespace ddns {

constexpr int PT = 256;
constexpr int CELL_GMAX = 256;   // finest pair-search grid per dimension

static inline unsigned nblk(long long n, int t = PT) { return (unsigned)((n + t - 1) / t); }

// ------------------------------------------------------------------ scans
// Exclusive scan of n ints in two launches: the totals of tiles of E * SCAN_T ints, then
// each tile scanned with the sum of the totals before it (every work-group adds those
// itself, at most a few thousand ints from L2).  No work-group waits for another.
// Work-groups are small (256 threads, no LDS tile): a scan runs beside the flow kernels,
// and a work-group of 1024 threads was seen to wait for a whole flow kernel to drain.
constexpr int SCAN_T = 256;
constexpr int SCAN_W = SCAN_T / 64;

// the work-group's sum of x, returned to every thread
__device__ __forceinline__ int block_sum_int(int x, int* sh)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    if (lane == 0) sh[wv] = x;
    __syncthreads();
    int t = 0;
#pragma unroll
    for (int w = 0; w < SCAN_W; ++w) t += sh[w];
    __syncthreads();
    return t;
}

// thread tid's E consecutive ints of the tile (zero past n)
template <int E>
__device__ __forceinline__ void scan_load(const int* in, long long i0, int n, int (&v)[E])
{
    if (i0 + E <= n) {
#pragma unroll
        for (int q = 0; q < E; q += 4) {
            const int4 x = *(const int4*)(in + i0 + q);
            v[q] = x.x; v[q + 1] = x.y; v[q + 2] = x.z; v[q + 3] = x.w;
        }
    } else {
#pragma unroll
        for (int q = 0; q < E; ++q) v[q] = i0 + q < n ? in[i0 + q] : 0;
    }
}

// One or two independent scans (grid y)
struct ScanArgs {
    const int* in[2];
    int* out[2];
    int* bsum[2];
    int* zin[2];
    int n[2];
};

template <int E>
__global__ void __launch_bounds__(SCAN_T) k_scan_tiles(ScanArgs a)
{
    __shared__ int sh[SCAN_W];
    const int k = blockIdx.y, n = a.n[k];
    if ((long long)blockIdx.x * SCAN_T * E >= n) return;
    int v[E];
    scan_load<E>(a.in[k], ((long long)blockIdx.x * SCAN_T + threadIdx.x) * E, n, v);
    int tot = 0;
#pragma unroll
    for (int q = 0; q < E; ++q) tot += v[q];
    tot = block_sum_int(tot, sh);
    if (threadIdx.x == 0) a.bsum[k][blockIdx.x] = tot;
}

// in may alias out: a thread reads its ints before it writes them.  zin (= in, not
// aliasing out, or null): the input is cleared as it is read.
template <int E>
__global__ void __launch_bounds__(SCAN_T) k_scan_apply(ScanArgs a)
{
    __shared__ int sh[SCAN_W];
    __shared__ int wsum[SCAN_W];
    const int k = blockIdx.y, n = a.n[k];
    if (blockIdx.x > 0 && (long long)blockIdx.x * SCAN_T * E >= n) return;
    const int* in = a.in[k];
    const int* bsum = a.bsum[k];
    int *out = a.out[k], *zin = a.zin[k];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    int pre = 0;
    for (int b = tid; b < (int)blockIdx.x; b += SCAN_T) pre += bsum[b];
    pre = block_sum_int(pre, sh);
    const long long i0 = ((long long)blockIdx.x * SCAN_T + tid) * E;
    int v[E];
    scan_load<E>(in, i0, n, v);
    if (zin) {
        if (i0 + E <= n) {
#pragma unroll
            for (int q = 0; q < E; q += 4) *(int4*)(zin + i0 + q) = make_int4(0, 0, 0, 0);
        } else {
            for (int q = 0; q < E; ++q)
                if (i0 + q < n) zin[i0 + q] = 0;
        }
    }
    int tot = 0;
#pragma unroll
    for (int q = 0; q < E; ++q) tot += v[q];
    int incl = tot;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const int y = __shfl_up(incl, o, 64);
        if (lane >= o) incl += y;
    }
    if (lane == 63) wsum[wv] = incl;
    __syncthreads();
    int run = pre + incl - tot;
#pragma unroll
    for (int w = 0; w < SCAN_W; ++w)
        if (w < wv) run += wsum[w];
    int r[E];
#pragma unroll
    for (int q = 0; q < E; ++q) {
        r[q] = run;
        run += v[q];
    }
    if (i0 + E <= n) {
#pragma unroll
        for (int q = 0; q < E; q += 4) *(int4*)(out + i0 + q) = make_int4(r[q], r[q + 1], r[q + 2], r[q + 3]);
    } else {
        for (int q = 0; q < E; ++q)
            if (i0 + q < n) out[i0 + q] = r[q];
    }
    // the last tile's last thread holds the total
    if (tid == SCAN_T - 1 && ((long long)blockIdx.x + 1) * SCAN_T * E >= n) out[n] = run;
}

// k scans (1 or 2) in two launches
static int scan_launch(const ScanArgs& a, int k, hipStream_t s)
{
    const long long n = std::max(a.n[0], k > 1 ? a.n[1] : 0);
    const int E = n <= 16LL * SCAN_T * 1024 ? 16 : 32;
    const unsigned nb = (unsigned)std::max<long long>(1, (n + (long long)E * SCAN_T - 1) / ((long long)E * SCAN_T));
    if (E == 16) {
        hipLaunchKernelGGL(k_scan_tiles<16>, dim3(nb, k), dim3(SCAN_T), 0, s, a);
        hipLaunchKernelGGL(k_scan_apply<16>, dim3(nb, k), dim3(SCAN_T), 0, s, a);
    } else {
        hipLaunchKernelGGL(k_scan_tiles<32>, dim3(nb, k), dim3(SCAN_T), 0, s, a);
        hipLaunchKernelGGL(k_scan_apply<32>, dim3(nb, k), dim3(SCAN_T), 0, s, a);
    }
    DDNS_HIP(hipGetLastError());
    return 0;
}

// out[0..n-1] = exclusive scan of in, out[n] = total (in may alias out); tmp holds
// scan_tmp_ints(n) ints; in and out 16-byte aligned.  clear_in (in not aliasing out):
// in[0..n-1] is left zero.
int exclusive_scan(const int* in, int* out, int n, int* tmp, hipStream_t s, bool clear_in)
{
    ScanArgs a{};
    a.in[0] = in;
    a.out[0] = out;
    a.bsum[0] = tmp;
    a.zin[0] = clear_in ? const_cast<int*>(in) : nullptr;
    a.n[0] = std::max(0, n);
    return scan_launch(a, 1, s);
}

// ints of scratch exclusive_scan needs for n elements
size_t scan_tmp_ints(long long n)
{
    size_t t = 0;
    long long m = n;
    do {
        m = (m + 1023) / 1024;
        t += (size_t)m + 1;
    } while (m > 1);
    return t + 16;
}

// ------------------------------------------------------------------ allocation
int part_alloc(PartBuffers& pb, int cap, int nset, int G)
{
    pb.cap = cap;
    const size_t c = (size_t)cap;
    DDNS_HIP(hipMalloc(&pb.pos, 3 * c * 8));
    DDNS_HIP(hipMalloc(&pb.vel, 3 * c * 8));
    DDNS_HIP(hipMalloc(&pb.rad, c * 8));
    DDNS_HIP(hipMalloc(&pb.gid, c * 8));
    DDNS_HIP(hipMalloc(&pb.fvp, 9 * c * 8));
    DDNS_HIP(hipMalloc(&pb.fdp, 12 * c * 8));
    DDNS_HIP(hipMalloc(&pb.dmove, 3 * c * 8));
    DDNS_HIP(hipMalloc(&pb.vp, 3 * c * 8));
    DDNS_HIP(hipMalloc(&pb.pert, 3 * c * 8));
    DDNS_HIP(hipMemset(pb.pert, 0, 3 * c * 8));
    DDNS_HIP(hipMemset(pb.dmove, 0, 3 * c * 8));
    DDNS_HIP(hipMemset(pb.vp, 0, 3 * c * 8));
    DDNS_HIP(hipMalloc(&pb.cell_of, c * sizeof(int)));
    DDNS_HIP(hipMalloc(&pb.cell_rank, c * sizeof(int)));
    DDNS_HIP(hipMalloc(&pb.rlist, c * sizeof(int)));
    DDNS_HIP(hipMalloc(&pb.sorted, c * sizeof(int)));
    DDNS_HIP(hipMalloc(&pb.pk, c * sizeof(double4)));
    DDNS_HIP(hipMalloc(&pb.mult, (c + 1) * sizeof(int)));
    DDNS_HIP(hipMalloc(&pb.draw_off, (c + 1) * sizeof(int)));
    DDNS_HIP(hipMalloc(&pb.nei_cnt, (c + 1) * sizeof(int)));
    DDNS_HIP(hipMalloc(&pb.flags, 64 * sizeof(int)));
    DDNS_HIP(hipMemset(pb.flags, 0, 64 * sizeof(int)));
    DDNS_HIP(hipMalloc(&pb.ext, 2 * EXT_WORDS * sizeof(unsigned long long)));
    DDNS_HIP(hipMemset(pb.ext, 0, 2 * EXT_WORDS * sizeof(unsigned long long)));
    DDNS_HIP(hipMalloc(&pb.tested, 4 * sizeof(long long)));
    const size_t nb = (size_t)nset * nset * DDNS_NBIN;
    DDNS_HIP(hipMalloc(&pb.nirbin, nb * sizeof(int)));
    DDNS_HIP(hipMalloc(&pb.bins, 7 * nb * sizeof(double)));
    DDNS_HIP(hipMalloc(&pb.counts, 512 * sizeof(int)));
    pb.pair_cap = 1 << 16;
    DDNS_HIP(hipMalloc(&pb.pairs, (size_t)pb.pair_cap * DDNS_PAIR_REC * sizeof(long long)));
    pb.draw_cap = 1 << 16;
    DDNS_HIP(hipMalloc(&pb.draws, (size_t)pb.draw_cap * sizeof(double)));
    DDNS_HIP(hipMalloc(&pb.rng_state, 64 * sizeof(int)));
    DDNS_HIP(hipMemset(pb.rng_state, 0, 64 * sizeof(int)));
    DDNS_HIP(hipMalloc(&pb.red, 8192 * sizeof(double)));
    pb.scan_tmp_bytes = scan_tmp_ints(std::max((long long)G * G * G + 1, (long long)c + 1)) * sizeof(int);
    DDNS_HIP(hipMalloc(&pb.scan_tmp, pb.scan_tmp_bytes));
    pb.G = 0;
    return 0;
}

void part_free(PartBuffers& pb)
{
    void* ps[] = {pb.pos, pb.vel, pb.rad, pb.gid, pb.fvp, pb.fdp, pb.dmove, pb.vp, pb.pert,
                  pb.cell_count, pb.cell_start, pb.cell_of, pb.cell_rank, pb.sorted, pb.pk, pb.scan_tmp,
                  pb.nei_cnt, pb.nei_idx, pb.nei_m, pb.gm_Q, pb.gm_v, pb.gm_x0, pb.gm_b, pb.gm_w,
                  pb.gm_red, pb.gm_small, pb.mult, pb.cand, pb.hit, pb.flags, pb.tested, pb.nirbin, pb.bins, pb.counts,
                  pb.pairs, pb.contact, pb.draws, pb.draw_off, pb.rng_state, pb.red, pb.stage, pb.cell_rank2,
                  pb.rlist, pb.ext};
    for (void* p : ps) if (p) (void)hipFree(p);
    void* sp[] = {pb.spare.cell_count, pb.spare.cell_start, pb.spare.cell_of, pb.spare.sorted, pb.spare.pk};
    for (void* p : sp) if (p) (void)hipFree(p);
    if (pb.sync_ev) (void)hipEventDestroy(pb.sync_ev);
    if (pb.gm_host) (void)hipHostFree(pb.gm_host);
    if (pb.found_host) (void)hipHostFree(pb.found_host);
    if (pb.bounce.host) (void)hipHostFree(pb.bounce.host);
    if (pb.counts_host) (void)hipHostFree(pb.counts_host);
    pb = PartBuffers{};
}

// ------------------------------------------------------------------ state transfers
// The reference's arrays hold one droplet's K values side by side, the device one value of
// all droplets (column c of slot i at col[c] + i).  The change of layout runs on the device, in
// a staging buffer that is copied straight to or from the caller's array: nine columns-to-host
// copies, nine host arrays allocated per call and a host loop took 97 ms for 1M droplets.
struct Columns {
    double* col[12];        // null: zeros
};

template <bool PACK>
__global__ void __launch_bounds__(PT) k_columns(Columns a, int K, double* __restrict__ rec, int n)
{
    const long long e = (long long)blockIdx.x * PT + threadIdx.x;
    if (e >= (long long)n * K) return;
    const int i = (int)(e / K), c = (int)(e - (long long)i * K);
    if (PACK) rec[e] = a.col[c][i];
    else a.col[c][i] = rec[e];
}

static int stage_rows(PartBuffers& pb)
{
    const size_t all = std::min(35 * (size_t)pb.cap * sizeof(double), BOUNCE_ROWS);   // yp, fvp, fdp, vp, dmove
    if (!pb.stage) DDNS_HIP(hipMalloc(&pb.stage, std::max(12 * (size_t)pb.cap * sizeof(double), all)));
    return 0;
}

// host(K, n) <- columns
static int columns_out(PartBuffers& pb, const Columns& a, int K, double* host, int n, hipStream_t s)
{
    if (!host || n <= 0) return 0;
    hipLaunchKernelGGL(k_columns<true>, dim3(nblk((long long)n * K)), dim3(PT), 0, s, a, K, pb.stage, n);
    DDNS_HIP(hipGetLastError());
    DDNS_HIP(hipMemcpyAsync(host, pb.stage, (size_t)n * K * sizeof(double), hipMemcpyDeviceToHost, s));
    return 0;
}

// columns <- host(K, n)
static int columns_in(PartBuffers& pb, const Columns& a, int K, const double* host, int n, hipStream_t s)
{
    if (!host || n <= 0) return 0;
    DDNS_HIP(hipMemcpyAsync(pb.stage, host, (size_t)n * K * sizeof(double), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(k_columns<false>, dim3(nblk((long long)n * K)), dim3(PT), 0, s, a, K, pb.stage, n);
    DDNS_HIP(hipGetLastError());
    return 0;
}

static Columns yp_columns(const PartBuffers& pb)
{
    Columns a{};
    for (int c = 0; c < 3; ++c) {
        a.col[c] = pb.pos + (size_t)c * pb.cap;
        a.col[3 + c] = pb.vel + (size_t)c * pb.cap;
    }
    a.col[6] = pb.rad;
    a.col[7] = pb.gid;
    return a;
}

static Columns vec_columns(double* v, int cap)
{
    Columns a{};
    for (int c = 0; c < 3; ++c) a.col[c] = v + (size_t)c * cap;
    return a;
}

int part_upload3(PartBuffers& pb, int n, double* dst, const double* host, hipStream_t s)
{
    const int st = stage_rows(pb);
    return st ? st : columns_in(pb, vec_columns(dst, pb.cap), 3, host, n, s);
}

int part_upload(PartBuffers& pb, int n, const double* yp, const double* fvp, const double* fdp, const double* pertvel,
                hipStream_t s)
{
    int st = stage_rows(pb);
    if (st) return st;
    const size_t c = (size_t)pb.cap;
    // slots without a droplet, and arrays that are not given, read as zeros
    double* const base[7] = {pb.pos, pb.vel, pb.rad, pb.gid, pb.fvp, pb.fdp, pb.pert};
    const size_t cols[7] = {3, 3, 1, 1, 9, 12, 3};
    const bool full = (size_t)n == c;
    const bool given[7] = {full, full, full, full, full && fvp, full && fdp, full && pertvel};
    for (int k = 0; k < 7; ++k)
        if (!given[k]) DDNS_HIP(hipMemsetAsync(base[k], 0, cols[k] * c * sizeof(double), s));
    st = columns_in(pb, yp_columns(pb), 8, yp, n, s);
    if (st) return st;
    pb.hv_v = pb.hv_d = 0;                          // the levels are written in order
    pb.v0_stale = pb.d0_stale = false;
    Columns a{}, b{};
    for (int q = 0; q < 9; ++q) a.col[q] = pb.fvp + q * c;
    for (int q = 0; q < 12; ++q) b.col[q] = pb.fdp + q * c;
    st = columns_in(pb, a, 9, fvp, n, s);
    if (st) return st;
    st = columns_in(pb, b, 12, fdp, n, s);
    if (st) return st;
    // pertvel is droplet-major on the device too
    if (pertvel && n > 0) DDNS_HIP(hipMemcpyAsync(pb.pert, pertvel, 3 * (size_t)n * sizeof(double), hipMemcpyHostToDevice, s));
    DDNS_HIP(hipStreamSynchronize(s));
    return 0;
}

int part_download(PartBuffers& pb, int n, double* yp, double* fvp, double* fdp, double* pertvel, double* vp, double* dmove,
                  hipStream_t s)
{
    int st = stage_rows(pb);
    if (st) return st;
    const size_t c = (size_t)pb.cap;
    // history level t in its ring column (level 0 reads as level 1 after a shift)
    Columns a{}, b{};
    for (int t = 0; t < 3; ++t)
        for (int q = 0; q < 3; ++q) a.col[3 * t + q] = pb.fvp + (size_t)(pb.vcol(t == 0 && pb.v0_stale ? 1 : t) + q) * c;
    for (int t = 0; t < 4; ++t)
        for (int q = 0; q < 3; ++q) b.col[3 * t + q] = pb.fdp + (size_t)(pb.dcol(t == 0 && pb.d0_stale ? 1 : t) + q) * c;
    const Columns cols[5] = {yp_columns(pb), a, b, vec_columns(pb.vp, pb.cap), vec_columns(pb.dmove, pb.cap)};
    const int K[5] = {8, 9, 12, 3, 3};
    double* const host[5] = {yp, fvp, fdp, vp, dmove};
    size_t per = 0;                                 // values of a droplet that go through the staging buffer
    for (int k = 0; k < 5; ++k) per += host[k] ? K[k] : 0;
    const size_t m = (size_t)std::max(0, n), pv = pertvel ? 3 * m : 0, bytes = (per * m + pv) * sizeof(double);
    if (bytes > 0 && bytes <= BOUNCE_ROWS) {
        st = bounce_room(pb.bounce, bytes);
        if (st) return st;
        double* at = pb.stage;
        for (int k = 0; k < 5; ++k) {
            if (!host[k]) continue;
            hipLaunchKernelGGL(k_columns<true>, dim3(nblk((long long)n * K[k])), dim3(PT), 0, s, cols[k], K[k], at, n);
            at += K[k] * m;
        }
        DDNS_HIP(hipGetLastError());
        if (per) DDNS_HIP(hipMemcpyAsync(pb.bounce.host, pb.stage, per * m * sizeof(double), hipMemcpyDeviceToHost, s));
        if (pv) DDNS_HIP(hipMemcpyAsync(pb.bounce.host + per * m, pb.pert, pv * sizeof(double), hipMemcpyDeviceToHost, s));
        DDNS_HIP(hipStreamSynchronize(s));
        const double* from = pb.bounce.host;
        for (int k = 0; k < 5; ++k) {
            if (!host[k]) continue;
            std::memcpy(host[k], from, K[k] * m * sizeof(double));
            from += K[k] * m;
        }
        if (pv) std::memcpy(pertvel, from, pv * sizeof(double));
        return 0;
    }
    for (int k = 0; k < 5 && !st; ++k) st = columns_out(pb, cols[k], K[k], host[k], n, s);
    if (st) return st;
    if (pertvel && n > 0) DDNS_HIP(hipMemcpyAsync(pertvel, pb.pert, 3 * (size_t)n * sizeof(double), hipMemcpyDeviceToHost, s));
    DDNS_HIP(hipStreamSynchronize(s));
    return 0;
}

// ------------------------------------------------------------------ interpolation
// Lagrange weights for nodes node-2 .. node+3 at fractional position z (partlib.f90:333-338)
__device__ __forceinline__ void lagrange6(double z, double* bg)
{
    const double z2 = z * z, z3 = z2 * z, z4 = z3 * z, z5 = z4 * z;
    bg[0] = (6.0 * z - 5.0 * z2 - 5.0 * z3 + 5.0 * z4 - z5) / 120.0;
    bg[1] = (-12.0 * z + 16.0 * z2 - z3 - 4.0 * z4 + z5) / 24.0;
    bg[2] = (12.0 - 4.0 * z - 15.0 * z2 + 5.0 * z3 + 3.0 * z4 - z5) / 12.0;
    bg[3] = (12.0 * z + 8.0 * z2 - 7.0 * z3 - 2.0 * z4 + z5) / 12.0;
    bg[4] = (-6.0 * z - z2 + 7.0 * z3 + z4 - z5) / 24.0;
    bg[5] = (4.0 * z - 5.0 * z3 + z5) / 120.0;
}

// The physical velocity is stored node-major, [z][y][x][3] (u, v, w), so one node is one
// 12-byte (float) or three 8-byte (double) loads, and the six nodes of a stencil row are
// one contiguous run of 72 (144) bytes.
__device__ __forceinline__ void load_node(const float* p, double& a, double& b, double& c)
{
    const float3 v = *(const float3*)p;
    a = v.x; b = v.y; c = v.z;
}
__device__ __forceinline__ void load_node(const double* p, double& a, double& b, double& c)
{
    a = p[0]; b = p[1]; c = p[2];
}

// Six lanes per droplet, one per x offset of the 6 x 6 x 6 stencil: for each of the
// 36 (y, z) stencil rows the six lanes read the row's six nodes as one contiguous run,
// so a wavefront load touches about 10 cache lines instead of one line per lane.  Ten
// droplets share a wavefront (lanes 60..63 idle), taken in cell order (sorted[]) so
// that they read overlapping rows.  Each lane sums its 36 nodes with the weights
// bg(x) bg(y) bg(z) of partlib.f90:509; the six partial sums are added in x order.
constexpr int IG = 6;              // lanes per droplet
constexpr int IPW = 64 / IG;       // droplets per wavefront

// In cell order (order != null) it writes the result in cell order, us[c * n + t], and
// k_interp_scatter takes it to the droplets: the gather then shares L2 with nothing but
// the field, instead of with three droplet arrays read and one written a line per
// droplet each (which halved its L2 hit rate).  Without a cell order it writes vp.
template <typename T>
__global__ void __launch_bounds__(PT) k_interp(const T* __restrict__ u, int N, double pi2,
                                               const double* __restrict__ pos, const int* __restrict__ order,
                                               const double4* __restrict__ pk, double* __restrict__ vp, int n, int cap,
                                               double* __restrict__ us)
{
    const int lane = threadIdx.x & 63;
    const int wave = (xcd_chunk(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x) >> 6;
    const int g = lane / IG, a = lane - g * IG;
    const int t = wave * IPW + g;
    const bool active = g < IPW && t < n;
    const int i = active ? (order ? order[t] : t) : 0;
    double acc0 = 0.0, acc1 = 0.0, acc2 = 0.0;
    if (active) {
        const double dx = pi2 / (double)N;
        double wx[6], wy[6], wz[6];
        double y0, y1, y2;
        if (pk) {                         // the packed record of the cell order holds the same values
            const double4 r = pk[t];
            y0 = r.x; y1 = r.y; y2 = r.z;
        } else {
            y0 = pos[i]; y1 = pos[(size_t)cap + i]; y2 = pos[2 * (size_t)cap + i];
        }
        const int nx = (int)floor(y0 / dx), ny = (int)floor(y1 / dx), nz = (int)floor(y2 / dx);
        lagrange6((y0 - (double)nx * dx) / dx, wx);
        lagrange6((y1 - (double)ny * dx) / dx, wy);
        lagrange6((y2 - (double)nz * dx) / dx, wz);
        double wxa = wx[0];
#pragma unroll
        for (int m = 1; m < 6; ++m) wxa = a == m ? wx[m] : wxa;
        const size_t ix = (size_t)(((nx - 2 + a) % N + N) % N) * 3;
        size_t rowy[6], rowz[6];
#pragma unroll
        for (int m = 0; m < 6; ++m) {
            rowy[m] = (size_t)(((ny - 2 + m) % N + N) % N) * N;
            rowz[m] = (size_t)(((nz - 2 + m) % N + N) % N) * N * N;
        }
#pragma unroll
        for (int d = 0; d < 6; ++d) {
#pragma unroll
            for (int b2 = 0; b2 < 6; ++b2) {
                double u0, u1, u2;
                load_node(u + (rowz[d] + rowy[b2]) * 3 + ix, u0, u1, u2);
                const double w = wxa * wy[b2] * wz[d];
                acc0 += u0 * w;
                acc1 += u1 * w;
                acc2 += u2 * w;
            }
        }
    }
    // lane a == 0 of each group adds the group's six partial sums in x order
    const int g0 = g * IG;
    double s0 = acc0, s1 = acc1, s2 = acc2;
#pragma unroll
    for (int m = 1; m < IG; ++m) {
        const int src = g0 + m < 64 ? g0 + m : lane;
        const double p0 = __shfl(acc0, src, 64), p1 = __shfl(acc1, src, 64), p2 = __shfl(acc2, src, 64);
        s0 += p0; s1 += p1; s2 += p2;
    }
    if (active && a == 0) {
        if (us) {
            const size_t M = (size_t)n;
            us[t] = s0;
            us[M + t] = s1;
            us[2 * M + t] = s2;
        } else {
            const size_t C = (size_t)cap;
            vp[i] = s0;
            vp[C + i] = s1;
            vp[2 * C + i] = s2;
        }
    }
}

// The gathered velocities, in cell order in us, to the droplets (vp in the reference's
// order).  With HI on it also writes, in cell order, the inputs of the HI solve: the
// warm start x0 = pertvel and the velocity difference w = V - U, so the solve reads
// them contiguously; w may be us itself (each element is read before it is written).
__global__ void __launch_bounds__(PT) k_interp_scatter(const int* __restrict__ order, const double* us, double* vp,
                                                       int n, int cap, const double* __restrict__ vel,
                                                       const double* __restrict__ pert, double* __restrict__ x0,
                                                       double* w)
{
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const int i = order[t];
    const size_t C = (size_t)cap, M = (size_t)n;
    double s3[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) s3[c] = us[c * M + t];
#pragma unroll
    for (int c = 0; c < 3; ++c) vp[c * C + i] = s3[c];
    if (x0) {
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            x0[c * M + t] = pert[3 * (size_t)i + c];
            w[c * M + t] = vel[c * C + i] - s3[c];
        }
    }
}

int part_interp(PartBuffers& pb, const PartConst& pc, const void* uphys, hipStream_t s)
{
    if (pc.n == 0) return 0;
    const int* order = pb.G > 0 ? pb.sorted : nullptr;
    const double4* pk = order ? pb.pk : nullptr;
    // the HI solve works in the cell order of this grid
    if (pc.hdi && !order) { set_error("HI needs the cell grid before the interpolation"); return DDNS_ERR_ARG; }
    if (order && !pb.gm_w) DDNS_HIP(hipMalloc(&pb.gm_w, 3 * (size_t)pb.cap * sizeof(double)));
    if (pc.hdi && !pb.gm_x0) DDNS_HIP(hipMalloc(&pb.gm_x0, 3 * (size_t)pb.cap * sizeof(double)));
    double* us = order ? pb.gm_w : nullptr;       // cell-order result, then w in place
    const unsigned nb = (unsigned)(((long long)pc.n + IPW * (PT / 64) - 1) / (IPW * (PT / 64)));
    if (pc.precision == DDNS_FP64)
        hipLaunchKernelGGL(k_interp<double>, dim3(nb), dim3(PT), 0, s, (const double*)uphys, pc.N, pc.pi2,
                           pb.pos, order, pk, pb.vp, pc.n, pb.cap, us);
    else
        hipLaunchKernelGGL(k_interp<float>, dim3(nb), dim3(PT), 0, s, (const float*)uphys, pc.N, pc.pi2,
                           pb.pos, order, pk, pb.vp, pc.n, pb.cap, us);
    if (order)
        hipLaunchKernelGGL(k_interp_scatter, dim3(nblk(pc.n)), dim3(PT), 0, s, order, (const double*)us, pb.vp, pc.n,
                           pb.cap, (const double*)pb.vel, (const double*)pb.pert, pc.hdi ? pb.gm_x0 : nullptr,
                           pc.hdi ? pb.gm_w : nullptr);
    DDNS_HIP(hipGetLastError());
    return 0;
}

// ------------------------------------------------------------------ histories
// PART_HISTORY_FVP, partlib.f90:562-592, and the clearing of what this step's searches write
// (a launch of its own and four fills before: a small run's step is bound by its launches)
__global__ void k_hist_fvp(double* vel, const double* rad, double* fvp, int n, int cap, int newp, double Sv, int v0,
                           int v1, int v2, ZeroSpans z)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    zero_spans(z, i, (size_t)gridDim.x * blockDim.x);
    if (i >= n) return;
    if (newp) {
        const double a = rad[i];
        vel[i] = Sv * (a * a);
        vel[(size_t)cap + i] = 0.0;
        vel[2 * (size_t)cap + i] = 0.0;
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const double v = vel[(size_t)c * cap + i];
        fvp[(size_t)(v0 + c) * cap + i] = v;
        if (newp) { fvp[(size_t)(v1 + c) * cap + i] = v; fvp[(size_t)(v2 + c) * cap + i] = v; }
    }
}

int part_history_fvp(PartBuffers& pb, const PartConst& pc, hipStream_t s)
{
    pb.step_cleared = false;
    if (pc.n == 0) return 0;
    ZeroSpans z{};
    const int st = part_step_spans(pb, pc, z);
    if (st) return st;
    hipLaunchKernelGGL(k_hist_fvp, dim3(std::max(64u, nblk(pc.n))), dim3(PT), 0, s, pb.vel, pb.rad, pb.fvp, pc.n, pb.cap,
                       pc.new_particle, pc.Sv_const, pb.vcol(0), pb.vcol(1), pb.vcol(2), z);
    DDNS_HIP(hipGetLastError());
    pb.step_cleared = true;
    pb.v0_stale = false;
    return 0;
}

// ------------------------------------------------------------------ advance
// PART_HISTORY_FDP (599-625) + PART_ADVANCE (629-726): implicit Adams-Moulton
// velocity with Adams-Bashforth fluid history, Stokes or Schiller-Naumann drag,
// gravity along +x, displacement dmove.  It also raises the step's largest displacement and
// droplet radius (ext, cleared at the step's start), the reach of the collision search, which a
// separate reduction over the displacements read again.
__global__ void __launch_bounds__(PT) k_advance(double* vel, const double* rad, double* fvp, double* fdp, const double* vp,
                          const double* pert, double* dmove, int n, int cap, int newp, int hdi,
                          int ndrag, double dt, double rnu, double Sv, double tau2, int4 vc, int4 dc,
                          unsigned long long* ext)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    double far = 0.0, big = 0.0;
    if (i < n) {
        const size_t C = (size_t)cap;
        double f0[3], d2[3];
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            f0[c] = hdi ? vp[c * C + i] + pert[3 * (size_t)i + c] : vp[c * C + i];
            fdp[(dc.x + c) * C + i] = f0[c];
            if (newp) { fdp[(dc.y + c) * C + i] = f0[c]; fdp[(dc.z + c) * C + i] = f0[c]; fdp[(dc.w + c) * C + i] = f0[c]; }
        }
        const double a = rad[i];
        double FSN = 1.;
        if (ndrag == 1) {
            double d[3];
#pragma unroll
            for (int c = 0; c < 3; ++c)
                d[c] = hdi ? vel[c * C + i] - vp[c * C + i] - pert[3 * (size_t)i + c] : vel[c * C + i] - vp[c * C + i];
            const double Vrel = sqrt(d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
            FSN = 1. + 0.15 * pow(Vrel * 2. * a / rnu, 0.687);
        }
        const double taup = tau2 * (a * a);
        const double dtau = dt / (24.0 * taup) * FSN;
        const double wp_vel = Sv * (a * a);
        const double dtc = dt / 24.0;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const double unitv = c == 0 ? 1.0 : 0.0;
            const double fv0 = fvp[(vc.x + c) * C + i], fv1 = fvp[(vc.y + c) * C + i], fv2 = fvp[(vc.z + c) * C + i];
            const double tempv = 19.0 * fv0 - 5.0 * fv1 + fv2;
            const double tempd = 55.0 * f0[c] - 59.0 * fdp[(dc.y + c) * C + i] + 37.0 * fdp[(dc.z + c) * C + i] -
                                 9.0 * fdp[(dc.w + c) * C + i];
            const double vnew = (vel[c * C + i] + dt * unitv * wp_vel / taup * FSN - dtau * tempv + dtau * tempd) / (1.0 + 9.0 * dtau);
            const double dm = dtc * (9.0 * vnew + 19.0 * fv0 - 5.0 * fv1 + fv2);
            vel[c * C + i] = vnew;
            dmove[c * C + i] = dm;
            d2[c] = dm * dm;
        }
        // rounded up: the bound may be a little larger than the displacement the search computes
        far = sqrt(d2[0] + d2[1] + d2[2]) * (1.0 + 1e-14);
        big = a;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        far = fmax(far, __shfl_xor(far, o, 64));
        big = fmax(big, __shfl_xor(big, o, 64));
    }
    __shared__ double wm[2][PT / 64];
    if ((threadIdx.x & 63) == 0) {
        wm[0][threadIdx.x >> 6] = far;
        wm[1][threadIdx.x >> 6] = big;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < PT / 64; ++w) {
            far = fmax(far, wm[0][w]);
            big = fmax(big, wm[1][w]);
        }
        raise_extents(ext, far, big);
    }
}

int part_advance(PartBuffers& pb, const PartConst& pc, hipStream_t s)
{
    if (pc.n == 0) return 0;
    const int4 vc = make_int4(pb.vcol(0), pb.vcol(1), pb.vcol(2), 0);
    const int4 dc = make_int4(pb.dcol(0), pb.dcol(1), pb.dcol(2), pb.dcol(3));
    hipLaunchKernelGGL(k_advance, dim3(nblk(pc.n)), dim3(PT), 0, s, pb.vel, pb.rad, pb.fvp, pb.fdp, pb.vp, pb.pert,
                       pb.dmove, pc.n, pb.cap, pc.new_particle, pc.hdi, pc.ndrag, pc.dt, pc.rnu, pc.Sv_const, pc.tau2,
                       vc, dc, pb.ext);
    DDNS_HIP(hipGetLastError());
    pb.d0_stale = false;
    return 0;
}

// ------------------------------------------------------------------ position update, relocation, wrap
// UPDATE_PART_POSITION (741-751)
// PERIODIC wrap (1142-1151) of one coordinate
__device__ __forceinline__ double wrap_periodic(double y, double pi2)
{
    if (y >= pi2) y = y - pi2;
    if (y < 0.0) y = y + pi2;
    return y;
}

// UPDATE_PART_POSITION (730-757): the position, with the PERIODIC wrap of 608 applied at
// once (the relocation between them wraps the positions it draws itself); the history
// shift turns the rings (part_update_and_wrap)
__global__ void k_update_pos(double* pos, const double* dmove, int n, int cap, double pi2)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const size_t C = (size_t)cap;
#pragma unroll
    for (int c = 0; c < 3; ++c) pos[c * C + i] = wrap_periodic(pos[c * C + i] + dmove[c * C + i], pi2);
}


// ranff2, accesories.f90:107-147, sequential on one lane: the relocation draws of
// RELOCATE / OVERLAP_DET come from one stream in the reference's order.
__device__ double dev_ranff2(int* idum, int* iv, int* iy, int* idum2)
{
    const int IM1 = 2147483563, IM2 = 2147483399, IMM1 = IM1 - 1;
    const int IA1 = 40014, IA2 = 40692, IQ1 = 53668, IQ2 = 52774, IR1 = 12211, IR2 = 3791;
    const int NDIV = 1 + IMM1 / 32;
    const double AM = 1.0 / IM1, EPS = 1.2e-7, RNMX = 1.0 - EPS;
    int j, k;
    if (*idum <= 0) {
        *idum = (-*idum > 1) ? -*idum : 1;
        *idum2 = *idum;
        // 8 warm-up draws, then iv[31] .. iv[0]: the loop j = 40..1 with a store at
        // j <= 32, split so that no store index is ever outside the table
        for (j = 0; j < 8; ++j) {
            k = *idum / IQ1;
            *idum = IA1 * (*idum - k * IQ1) - k * IR1;
            if (*idum < 0) *idum += IM1;
        }
        for (j = 31; j >= 0; --j) {
            k = *idum / IQ1;
            *idum = IA1 * (*idum - k * IQ1) - k * IR1;
            if (*idum < 0) *idum += IM1;
            iv[j] = *idum;
        }
        *iy = iv[0];
    }
    k = *idum / IQ1;
    *idum = IA1 * (*idum - k * IQ1) - k * IR1;
    if (*idum < 0) *idum += IM1;
    k = *idum2 / IQ2;
    *idum2 = IA2 * (*idum2 - k * IQ2) - k * IR2;
    if (*idum2 < 0) *idum2 += IM2;
    j = 1 + *iy / NDIV;
    *iy = iv[j - 1] - *idum2;
    iv[j - 1] = *idum;
    if (*iy < 1) *iy += IMM1;
    const double r = AM * (double)(*iy);
    return r < RNMX ? r : RNMX;
}

// state layout: [0] idum, [1] iy, [2] idum2, [3..34] iv
// At most cap draws are made: a removal list that needs more sets *err (the host then
// reports a capacity error) and is cut short.
__global__ void k_draws(int* st, double* draws, const int* total, int cap, int* err)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    int idum = st[0], iy = st[1], idum2 = st[2];
    // shuffle table in LDS, not in a private array that the compiler turns into
    // indexed register moves
    __shared__ int iv[32];
    for (int q = 0; q < 32; ++q) iv[q] = st[3 + q];
    int nd = 3 * (*total);
    if (nd > cap) {
        atomicOr(err, 1);
        nd = cap - cap % 3;
    }
    for (int q = 0; q < nd; ++q) draws[q] = dev_ranff2(&idum, iv, &iy, &idum2);
    st[0] = idum; st[1] = iy; st[2] = idum2;
    for (int q = 0; q < 32; ++q) st[3 + q] = iv[q];
}

// A droplet that appears m times in the sorted removal list consumes 3m draws at
// offset off; the last triple is the position it keeps (RELOCATE, 1994-2006).
__global__ void k_apply_reloc(double* pos, const int* mult, const int* off, const double* draws, int n, int cap, double pi2,
                              long long draw_cap)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int m = mult[i];
    if (m <= 0) return;
    if (3 * ((long long)off[i] + m) > draw_cap) return;      // cut short by k_draws (capacity error)
    const double* d = draws + 3 * (size_t)(off[i] + m - 1);
    const double y[3] = {d[0] * pi2, d[1] * pi2 + 0.0 * pi2, d[2] * pi2 + 0.0 * pi2};
    pos[i] = y[0];
    pos[(size_t)cap + i] = y[1];
    pos[2 * (size_t)cap + i] = y[2];
}

__global__ void k_set_rng(int* st, int seed)
{
    if (threadIdx.x != 0) return;
    st[0] = seed; st[1] = 0; st[2] = 0;
    for (int q = 0; q < 32; ++q) st[3 + q] = 0;
}

int part_set_rng(const PartBuffers& pb, int iseedr, hipStream_t s)
{
    hipLaunchKernelGGL(k_set_rng, dim3(1), dim3(1), 0, s, pb.rng_state, iseedr);
    DDNS_HIP(hipGetLastError());
    return 0;
}

// relocate every droplet with mult > 0; returns the number of draws triples via *total_host
int relocate_by_mult(PartBuffers& pb, const PartConst& pc, int* total_host, hipStream_t s)
{
    int st = exclusive_scan(pb.mult, pb.draw_off, pc.n, (int*)pb.scan_tmp, s);
    if (st) return st;
    int total = 0;
    DDNS_HIP(hipMemcpyAsync(&total, pb.draw_off + pc.n, sizeof(int), hipMemcpyDeviceToHost, s));
    DDNS_HIP(hipStreamSynchronize(s));
    *total_host = total;
    if (total == 0) return 0;
    invalidate_cells(pb);                 // relocated droplets move
    if (3 * total > pb.draw_cap) {
        DDNS_HIP(hipFree(pb.draws));
        pb.draw_cap = 3 * total + 1024;
        DDNS_HIP(hipMalloc(&pb.draws, (size_t)pb.draw_cap * sizeof(double)));
    }
    hipLaunchKernelGGL(k_draws, dim3(1), dim3(1), 0, s, pb.rng_state, pb.draws, pb.draw_off + pc.n, pb.draw_cap,
                       pb.flags + 48);
    hipLaunchKernelGGL(k_apply_reloc, dim3(nblk(pc.n)), dim3(PT), 0, s, pb.pos, pb.mult, pb.draw_off, pb.draws,
                       pc.n, pb.cap, pc.pi2, (long long)pb.draw_cap);
    DDNS_HIP(hipGetLastError());
    return 0;
}

// The relocation of a step (RELOCATE, partlib.f90:1984-2012) by one work-group and without a
// host round trip: the droplets that the search listed (in any order) are sorted by index,
// which is the order of the reference's removal list, each takes 3 mult draws of the stream
// and keeps the last three.  A step relocates a handful of droplets: a scan of all
// multiplicities, the draws and the update as four launches took 40 us at 1M droplets.  For a list
// longer than the sort's room the multiplicities of all droplets are scanned in index order
// instead, RL_E of a thread side by side, and the listed ones moved: a sweep that relocates 5000
// of 1M droplets takes 2.57 ms (2.41 with the scan over all work-groups, 3.80 with one
// multiplicity a thread and a walk over all droplets to move them), 20 000 of them 8.4 (8.0, 9.6),
// most of it the serial draws.  At most draw_cap draws are made: a list that needs more sets *err
// (a capacity error) and is cut short.
constexpr int RL_T = 1024, RL_MAX = 4096, RL_E = 16;

struct RelocArgs {
    double* pos;
    const int* mult;
    const int* list;
    const int* nlist;
    int* off;               // cap + 1: the long list's offsets, by droplet
    double* draws;
    int* rng;
    int* total;             // list entries with their multiplicity
    int* err;
    int n, cap, draw_cap, wrap;
    double pi2;
};

__device__ __forceinline__ void reloc_apply(const RelocArgs& a, int i, int off, int m)
{
    if (3 * ((long long)off + m) > a.draw_cap) return;
    const double* d = a.draws + 3 * (size_t)(off + m - 1);
    double y[3] = {d[0] * a.pi2, d[1] * a.pi2 + 0.0 * a.pi2, d[2] * a.pi2 + 0.0 * a.pi2};
    for (int c = 0; c < 3; ++c) a.pos[(size_t)c * a.cap + i] = a.wrap ? wrap_periodic(y[c], a.pi2) : y[c];
}

__device__ __forceinline__ void reloc_draws(const RelocArgs& a, int total, int* iv)
{
    if (threadIdx.x == 0) {
        int* st = a.rng;
        int idum = st[0], iy = st[1], idum2 = st[2];
        for (int q = 0; q < 32; ++q) iv[q] = st[3 + q];
        long long nd = 3LL * total;
        if (nd > a.draw_cap) {
            atomicOr(a.err, 1);
            nd = a.draw_cap - a.draw_cap % 3;
        }
        for (long long q = 0; q < nd; ++q) a.draws[q] = dev_ranff2(&idum, iv, &iy, &idum2);
        st[0] = idum; st[1] = iy; st[2] = idum2;
        for (int q = 0; q < 32; ++q) st[3 + q] = iv[q];
    }
    __syncthreads();
}

__global__ void __launch_bounds__(RL_T) k_relocate(RelocArgs a)
{
    __shared__ int key[RL_MAX], off[RL_MAX], iv[32], wsum[RL_T / 64], run;
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int m = *a.nlist;
    if (m == 0) {
        if (tid == 0) *a.total = 0;
        return;
    }
    // exclusive sums of x over the work-group's threads, run carried from call to call
    auto scan = [&](int x) {
        int incl = x;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
            const int y = __shfl_up(incl, o, 64);
            if (lane >= o) incl += y;
        }
        if (lane == 63) wsum[wv] = incl;
        __syncthreads();
        int before = run;
        for (int w = 0; w < wv; ++w) before += wsum[w];
        __syncthreads();
        if (tid == RL_T - 1) run = before + incl;
        __syncthreads();
        return before + incl - x;
    };
    if (tid == 0) run = 0;
    if (m <= RL_MAX) {
        int P = 1;
        while (P < m) P <<= 1;
        for (int i = tid; i < P; i += RL_T) key[i] = i < m ? a.list[i] : 0x7fffffff;
        __syncthreads();
        for (int k = 2; k <= P; k <<= 1)
            for (int j = k >> 1; j > 0; j >>= 1) {
                for (int i = tid; i < P; i += RL_T) {
                    const int l = i ^ j;
                    if (l > i) {
                        const int x = key[i], y = key[l];
                        if ((x > y) == ((i & k) == 0)) { key[i] = y; key[l] = x; }
                    }
                }
                __syncthreads();
            }
        for (int b = 0; b < m; b += RL_T) {
            const int e = scan(b + tid < m ? a.mult[key[b + tid]] : 0);
            if (b + tid < m) off[b + tid] = e;
        }
        const int total = run;
        reloc_draws(a, total, iv);
        for (int e = tid; e < m; e += RL_T) reloc_apply(a, key[e], off[e], a.mult[key[e]]);
        if (tid == 0) *a.total = total;
        return;
    }
    __syncthreads();
    for (int b = 0; b < a.n; b += RL_T * RL_E) {
        const int i0 = b + tid * RL_E;
        int v[RL_E], sum = 0;
        if (i0 <= a.n - RL_E) {
#pragma unroll
            for (int q = 0; q < RL_E; q += 4) *(int4*)(v + q) = *(const int4*)(a.mult + i0 + q);
        } else {
#pragma unroll
            for (int q = 0; q < RL_E; ++q) v[q] = i0 + q < a.n ? a.mult[i0 + q] : 0;
        }
#pragma unroll
        for (int q = 0; q < RL_E; ++q) sum += v[q];
        int e = scan(sum);
#pragma unroll
        for (int q = 0; q < RL_E; ++q) {
            if (v[q] > 0) a.off[i0 + q] = e;
            e += v[q];
        }
    }
    const int total = run;
    reloc_draws(a, total, iv);                // its barrier also makes the offsets visible
    for (int e = tid; e < m; e += RL_T) {
        const int i = a.list[e];
        reloc_apply(a, i, a.off[i], a.mult[i]);
    }
    if (tid == 0) *a.total = total;
}

int relocate_list(PartBuffers& pb, const PartConst& pc, int nlist, bool wrap, hipStream_t s)
{
    invalidate_cells(pb);                 // relocated droplets move
    const int need = 3 * std::max(pb.cap, 1 << 16);
    if (pb.draw_cap < need) {
        DDNS_HIP(hipFree(pb.draws));
        pb.draw_cap = need;
        DDNS_HIP(hipMalloc(&pb.draws, (size_t)pb.draw_cap * sizeof(double)));
    }
    RelocArgs a{};
    a.pos = pb.pos; a.mult = pb.mult; a.list = pb.rlist; a.nlist = pb.flags + nlist; a.off = pb.draw_off;
    a.draws = pb.draws; a.rng = pb.rng_state; a.total = pb.flags + 50; a.err = pb.flags + 48;
    a.n = pc.n; a.cap = pb.cap; a.draw_cap = pb.draw_cap; a.wrap = wrap ? 1 : 0; a.pi2 = pc.pi2;
    hipLaunchKernelGGL(k_relocate, dim3(1), dim3(RL_T), 0, s, a);
    DDNS_HIP(hipGetLastError());
    return 0;
}

int part_update_and_wrap(PartBuffers& pb, const PartConst& pc, bool relocate, hipStream_t s)
{
    if (pc.n == 0) return 0;
    hipLaunchKernelGGL(k_update_pos, dim3(nblk(pc.n)), dim3(PT), 0, s, pb.pos, pb.dmove, pc.n, pb.cap, pc.pi2);
    DDNS_HIP(hipGetLastError());
    // fvp(2) = fvp(1), fvp(1) = fvp(0); fdp(3..1) = fdp(2..0): level t+1 takes level t's columns
    pb.hv_v = (pb.hv_v + 2) % 3;
    pb.hv_d = (pb.hv_d + 3) % 4;
    pb.v0_stale = true;
    pb.d0_stale = true;
    if (relocate) {
        int st = relocate_list(pb, pc, 51, true, s);
        if (st) return st;
    }
    return 0;
}

// ------------------------------------------------------------------ coarse cell grid
// A periodic grid of G^3 cells of width hc = 2pi/G >= the largest pair distance the
// caller needs, so a 27-cell neighbourhood holds every candidate.  Counting sort by
// cell, then each cell's slice is ordered by slot number (deterministic).
// One or two grids over the same positions (grid y): every kernel of a build covers both.
struct GridArgs {
    int *cell_of[2], *rank[2], *cnt[2], *start[2], *sorted[2];
    double4* pk[2];
    int G[2], ncell[2];
    double hc[2];
};

// cell of droplet i and its place among the droplets of that cell (the order in which
// the atomics were served; k_cell_order makes the final order deterministic)
__global__ void k_cell_key(const double* pos, GridArgs a, int n, int cap)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y;
    if (i >= n) return;
    const int G = a.G[k];
    const double hc = a.hc[k];
    int c3[3];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        int q = (int)(pos[(size_t)c * cap + i] / hc);
        q = q < 0 ? 0 : (q >= G ? G - 1 : q);
        c3[c] = q;
    }
    const int cell = cell_code(c3[0], c3[1], c3[2], G);
    a.cell_of[k][i] = cell;
    a.rank[k][i] = atomicAdd(a.cnt[k] + cell, 1);
}

// Droplet i (read in slot order, so the reads coalesce) takes the next free place of
// its cell and writes its index and its packed (x, y, z, radius) record there: the
// pair searches then read each candidate cell as one contiguous run.
__global__ void k_cell_fill(GridArgs a, const double* __restrict__ pos, const double* __restrict__ rad, int n, int cap)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y;
    if (i >= n) return;
    const int p = a.start[k][a.cell_of[k][i]] + a.rank[k][i];
    a.sorted[k][p] = i;
    a.pk[k][p] = make_double4(pos[i], pos[(size_t)cap + i], pos[2 * (size_t)cap + i], rad[i]);
}

// the order inside a cell is by droplet index, so it does not depend on the order in
// which the fill's atomics were served; the packed records move with their indices
__global__ void k_cell_order(GridArgs a)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x, k = blockIdx.y;
    if (c >= a.ncell[k]) return;
    const int* start = a.start[k];
    int* sorted = a.sorted[k];
    double4* pk = a.pk[k];
    const int b = start[c], e = start[c + 1];
    for (int i = b + 1; i < e; ++i) {
        const int v = sorted[i];
        const double4 r = pk[i];
        int j = i - 1;
        while (j >= b && sorted[j] > v) { sorted[j + 1] = sorted[j]; pk[j + 1] = pk[j]; --j; }
        sorted[j + 1] = v;
        pk[j + 1] = r;
    }
}

void invalidate_cells(PartBuffers& pb)
{
    pb.cells_valid = false;
    pb.spare.valid = false;
}

static void swap_cells(PartBuffers& pb)
{
    PartBuffers::CellSet& o = pb.spare;
    std::swap(pb.G, o.G);
    std::swap(pb.hc, o.hc);
    std::swap(pb.cell_count, o.cell_count);
    std::swap(pb.cell_count_zero, o.count_zero);
    std::swap(pb.cell_start, o.cell_start);
    std::swap(pb.cell_of, o.cell_of);
    std::swap(pb.sorted, o.sorted);
    std::swap(pb.pk, o.pk);
    std::swap(pb.cells_valid, o.valid);
}

static int alloc_spare(PartBuffers& pb)
{
    PartBuffers::CellSet& o = pb.spare;
    if (o.cell_count) return 0;
    const long long nmax = (long long)CELL_GMAX * CELL_GMAX * CELL_GMAX + 1;
    const size_t c = (size_t)pb.cap;
    DDNS_HIP(hipMalloc(&o.cell_count, nmax * sizeof(int)));
    DDNS_HIP(hipMalloc(&o.cell_start, nmax * sizeof(int)));
    DDNS_HIP(hipMalloc(&o.cell_of, c * sizeof(int)));
    DDNS_HIP(hipMalloc(&o.sorted, c * sizeof(int)));
    DDNS_HIP(hipMalloc(&o.pk, c * sizeof(double4)));
    o.valid = false;
    return 0;
}

// cells per dimension of a grid of width hmin or more (0: too few)
static int grid_cells(const PartConst& pc, double hmin)
{
    const int G = std::min(CELL_GMAX, (int)floor(pc.pi2 / hmin));
    if (G < 3) set_error("domain too small for the pair search grid (need 3 cells of the interaction radius)");
    return G < 3 ? 0 : G;
}

static int alloc_cells(PartBuffers& pb)
{
    if (pb.cell_count) return 0;
    // sized once for the finest grid, so switching between the collision and the overlap
    // grids never reallocates; the scratch of two scans at once
    const long long nmax = (long long)CELL_GMAX * CELL_GMAX * CELL_GMAX + 1;
    DDNS_HIP(hipMalloc(&pb.cell_count, nmax * sizeof(int)));
    DDNS_HIP(hipMalloc(&pb.cell_start, nmax * sizeof(int)));
    const size_t need = 2 * scan_tmp_ints(std::max(nmax, (long long)pb.cap + 1)) * sizeof(int);
    if (need > pb.scan_tmp_bytes) {
        (void)hipFree(pb.scan_tmp);
        pb.scan_tmp = nullptr;
        DDNS_HIP(hipMalloc(&pb.scan_tmp, need));
        pb.scan_tmp_bytes = need;
    }
    return 0;
}

// The cell kernels over k grids: the current one, then the spare.
static int build_grids(PartBuffers& pb, const PartConst& pc, int k, hipStream_t s)
{
    GridArgs a{};
    ScanArgs sc{};
    long long zero[2] = {0, 0};
    int ncmax = 0;
    const size_t half = pb.scan_tmp_bytes / sizeof(int) / 2;
    for (int g = 0; g < k; ++g) {
        PartBuffers::CellSet& o = pb.spare;
        a.cell_of[g] = g ? o.cell_of : pb.cell_of;
        a.cnt[g] = g ? o.cell_count : pb.cell_count;
        a.start[g] = g ? o.cell_start : pb.cell_start;
        a.sorted[g] = g ? o.sorted : pb.sorted;
        a.pk[g] = g ? o.pk : pb.pk;
        a.rank[g] = g ? pb.cell_rank2 : pb.cell_rank;
        a.G[g] = g ? o.G : pb.G;
        a.hc[g] = g ? o.hc : pb.hc;
        a.ncell[g] = cell_numbers(a.G[g]);
        ncmax = std::max(ncmax, a.ncell[g]);
        // the counts are left zero by the scan of the last build into this buffer
        long long& z = g ? o.count_zero : pb.cell_count_zero;
        if (z < a.ncell[g] + 1) {
            DDNS_HIP(hipMemsetAsync(a.cnt[g], 0, ((size_t)a.ncell[g] + 1) * sizeof(int), s));
            z = a.ncell[g] + 1;
        }
        zero[g] = z;
        z = 0;
        sc.in[g] = a.cnt[g];
        sc.out[g] = a.start[g];
        sc.zin[g] = a.cnt[g];
        sc.bsum[g] = (int*)pb.scan_tmp + g * half;
        sc.n[g] = a.ncell[g];
    }
    if (pc.n > 0) hipLaunchKernelGGL(k_cell_key, dim3(nblk(pc.n), k), dim3(PT), 0, s, (const double*)pb.pos, a, pc.n, pb.cap);
    const int st = scan_launch(sc, k, s);
    if (st) return st;
    pb.cell_count_zero = zero[0];
    if (k > 1) pb.spare.count_zero = zero[1];
    if (pc.n > 0) {
        hipLaunchKernelGGL(k_cell_fill, dim3(nblk(pc.n), k), dim3(PT), 0, s, a, (const double*)pb.pos, (const double*)pb.rad,
                           pc.n, pb.cap);
        hipLaunchKernelGGL(k_cell_order, dim3(nblk(ncmax), k), dim3(PT), 0, s, a);
    }
    DDNS_HIP(hipGetLastError());
    pb.cells_valid = true;
    if (k > 1) pb.spare.valid = true;
    return 0;
}

int part_build_cells(PartBuffers& pb, const PartConst& pc, double hmin, hipStream_t s)
{
    const int G = grid_cells(pc, hmin);
    if (!G) return DDNS_ERR_DOMAIN;
    int st = alloc_cells(pb);
    if (st) return st;
    if (pb.cells_valid && pb.G == G) return 0;                     // already built on these positions
    if (pb.spare.valid && pb.spare.G == G) {                      // kept from an earlier build
        swap_cells(pb);
        return 0;
    }
    if (pb.cells_valid) {
        // keep the current grid (another width) for a later search: build into the spare
        st = alloc_spare(pb);
        if (st) return st;
        swap_cells(pb);
    }
    pb.cells_valid = false;
    pb.G = G;
    pb.hc = pc.pi2 / G;
    return build_grids(pb, pc, 1, s);
}

int part_build_two(PartBuffers& pb, const PartConst& pc, double hmin, double other, hipStream_t s)
{
    const int G = grid_cells(pc, hmin), H = grid_cells(pc, other);
    if (!G || !H) return DDNS_ERR_DOMAIN;
    if (G == H || pb.cells_valid || pb.spare.valid) {
        const int st = part_build_cells(pb, pc, other, s);
        return st ? st : part_build_cells(pb, pc, hmin, s);
    }
    int st = alloc_cells(pb);
    if (!st) st = alloc_spare(pb);
    if (st) return st;
    if (!pb.cell_rank2) DDNS_HIP(hipMalloc(&pb.cell_rank2, (size_t)pb.cap * sizeof(int)));
    pb.G = G;
    pb.hc = pc.pi2 / G;
    pb.spare.G = H;
    pb.spare.hc = pc.pi2 / H;
    return build_grids(pb, pc, 2, s);
}

}  // namespace ddns
