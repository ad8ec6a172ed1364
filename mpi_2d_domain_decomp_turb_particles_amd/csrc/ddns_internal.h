// ddns_internal.h -- internal declarations shared by the HIP translation units of
// libddns.so: precision traits, complex helpers, device buffers of a handle and the
// host-side launch wrappers of every kernel family.
#pragma once

#include <hip/hip_runtime.h>
#include <chrono>
#include <cstddef>
#include <cstdint>
#include <string>
#include <vector>

#include "../../include/ddns.h"

#define DDNS_HIP(call)                                                              \
    do {                                                                            \
        hipError_t e_ = (call);                                                     \
        if (e_ != hipSuccess) return ddns::hip_fail(e_, #call, __FILE__, __LINE__); \
    } while (0)

namespace ddns {

// One detected collision pair on the device, in 64-bit words:
//   [0] canonical key (min gid << 32 | max gid << 2 | type)   [1] ih1 slot   [2] ih2 slot
//   [3] packed cell offsets   [4] ih2 image direction (0: the droplet itself, 5..8:
//   HEADLIST halo directions)   [5] radius of ih1, [6] radius of ih2 (bit patterns)
//   [7] the reference's visiting order of the pair (ih1, cell loop, linked list)
constexpr int DDNS_PAIR_REC = 8;

// One pair in contact (rcolla < d <= rcollb), in doubles: [0] ih1 slot and [1] the
// cell-loop / linked-list order of ih2 (bit patterns of 64-bit integers), then the
// reference's buffer(1:12, ij): index1, index2, va(3), vb(3), unit offset (3), Wr
constexpr int DDNS_CONTACT_REC = 14;

// Coarse-cell number of cell (x, y, z) of a G^3 grid, G <= 256: the rows along x are whole, so the
// candidates of a row's neighbouring cells are one run of the sorted droplets, and the rows
// follow the Morton (Z-curve) interleave of y and z, so droplets close in the order are close in
// space and the lanes of a wavefront touch overlapping field stencils and cells.
__host__ __device__ __forceinline__ unsigned cell_spread(unsigned v)
{
    v &= 0xffu;
    v = (v | (v << 4)) & 0x0f0fu;
    v = (v | (v << 2)) & 0x3333u;
    v = (v | (v << 1)) & 0x5555u;
    return v;
}
__host__ __device__ __forceinline__ int cell_row(int y, int z)
{
    return (int)(cell_spread((unsigned)y) | (cell_spread((unsigned)z) << 1));
}
__host__ __device__ __forceinline__ int cell_code(int x, int y, int z, int G) { return cell_row(y, z) * G + x; }
// the numbers of a G^3 grid lie below this (at most 256^3)
inline int cell_numbers(int G)
{
    int b = 0;
    while ((1 << b) < G) ++b;
    return G << (2 * b);
}
// Work-group b of a launch runs on XCD b % 8, and each of the 8 XCDs has its own L2.
// This gives the work-groups of one XCD a contiguous range of the nb logical blocks,
// so droplets that are close in cell order, which read the same field nodes and
// neighbour cells, share an L2.  A bijection of [0, nb).
__device__ __forceinline__ int xcd_chunk(int b, int nb)
{
    const int x = b & 7, r = b >> 3, q = nb >> 3, m = nb & 7;
    return x * q + (x < m ? x : m) + r;
}

// Offsets (-1 or 0 up to 0 or +1) of the neighbour cells to visit along each axis.
struct CellSpan {
    int lo[3] = {-1, -1, -1};
    int hi[3] = {1, 1, 1};
};

// The neighbour cells that can hold a point within distance reach of x, which lies in
// cell cc of width hc: along each axis the lower (upper) neighbour is needed only when
// x is closer than reach to the lower (upper) face.  The margin of 1e-9 hc covers the
// rounding of the cell index; clamped and periodic cells stay covered because the
// test only ever adds cells.
__device__ __forceinline__ CellSpan reach_span(const double x[3], const int cc[3], double hc, double reach)
{
    const double m = reach + 1e-9 * hc;
    CellSpan s;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        s.lo[c] = (x[c] - (double)cc[c] * hc < m) ? -1 : 0;
        s.hi[c] = ((double)(cc[c] + 1) * hc - x[c] < m) ? 1 : 0;
    }
    return s;
}

// The periodic shift of a run of candidates along each axis, -1, 0 or +1, in 5 bits
__device__ __forceinline__ int shift_code(int wx, int wy, int wz) { return 9 * (wx + 1) + 3 * (wy + 1) + wz + 1; }
__device__ __forceinline__ void shift_of(int w, int* wx, int* wy, int* wz)
{
    *wx = w / 9 - 1;
    *wy = (w / 3) % 3 - 1;
    *wz = w % 3 - 1;
}

// The candidates of the 27 neighbour cells (or of the part of them that span selects): for each
// (y, z) offset the cells x-1, x, x+1 are one run (across the periodic face in x two, the second
// in a pass of its own that only wavefronts at the face make).  The runs' ends load together,
// the non-empty ones go to the lane's column of the LDS list, and one loop walks them, the next
// record loading while f works on the current one: a wavefront takes as many turns as its
// fullest lane has candidates, where a loop for each run took the sum of the runs' longest,
// waiting for each run's ends.  At 1M droplets with half a droplet per cell the collision
// search took 246 us that way and takes 222, the overlap search 65 and 53; at
// 100 000 droplets 37 and 29, 10.8 and 7.0.  f(p, w, sx, sy, sz, rec, ib) gets the sorted
// position, the shift code, the shift in lengths (h the box), the record pk[p] and, when sorted
// is given, the droplet index sorted[p].  With L > 1, consecutive lanes of a wavefront share a
// droplet, and lane j of them takes every L-th candidate from the j-th on.
template <int NT>
struct RunList {
    int2 run[9][NT];
};
template <int L, int NT, typename F>
__device__ __forceinline__ void for_each_candidate(RunList<NT>& list, const int* __restrict__ cell_start, int G, double h,
                                                   const int cc[3], const double4* __restrict__ pk,
                                                   const int* __restrict__ sorted, F&& f, const CellSpan& span = CellSpan())
{
    const int tid = threadIdx.x, sub = tid & (L - 1);
    const int xl = cc[0] + span.lo[0], xh = cc[0] + span.hi[0];
    const bool edge = xl < 0 || xh >= G;
    const int passes = __any(edge) ? 2 : 1;
#pragma unroll 1
    for (int pass = 0; pass < passes; ++pass) {
        if (pass && !edge) break;
        // the cells a..b of each row: those inside the box, then the one beyond its face (G >= 3)
        const int wx = pass ? (xl < 0 ? -1 : 1) : 0;
        const int a = pass ? (xl < 0 ? G - 1 : 0) : max(xl, 0), b = pass ? a : min(xh, G - 1);
        int s[9], e[9], w[9];
#pragma unroll
        for (int r = 0; r < 9; ++r) {
            const int dy = r / 3 - 1, dz = r % 3 - 1;
            s[r] = e[r] = w[r] = 0;
            if (dy < span.lo[1] || dy > span.hi[1] || dz < span.lo[2] || dz > span.hi[2]) continue;
            const int qy = cc[1] + dy, qz = cc[2] + dz;
            const int wy = qy < 0 ? -1 : (qy >= G ? 1 : 0), wz = qz < 0 ? -1 : (qz >= G ? 1 : 0);
            const int* row = cell_start + cell_row(qy - wy * G, qz - wz * G) * G;
            w[r] = shift_code(wx, wy, wz);
            s[r] = row[a];
            e[r] = row[b + 1];
        }
        int n = 0;
#pragma unroll
        for (int r = 0; r < 9; ++r)
            if (e[r] > s[r]) list.run[n++][tid] = make_int2(s[r], ((e[r] - s[r]) << 5) | w[r]);
        if (n == 0) continue;
        int i = 0, p, end, wc, vx, vy, vz;
        // the run i, entered at its candidate number skip; a shorter run passes the rest on
        auto take = [&](int skip) {
            while (true) {
                const int2 r = list.run[i][tid];
                p = r.x + skip;
                end = r.x + (r.y >> 5);
                wc = r.y & 31;
                if (L == 1 || p < end) return true;
                if (++i == n) return false;
                skip = p - end;
            }
        };
        if (!take(sub)) continue;
        double4 next = pk[p];
        int inext = sorted ? sorted[p] : 0;
#pragma unroll 1
        while (true) {
            const int pc = p, w0 = wc;
            const double4 rec = next;
            const int ib = inext;
            p += L;
            bool more = p < end;
            if (!more && ++i < n) more = take(p - end);
            if (more) {
                next = pk[p];
                if (sorted) inext = sorted[p];
            }
            shift_of(w0, &vx, &vy, &vz);
            f(pc, w0, (double)vx * h, (double)vy * h, (double)vz * h, rec, ib);
            if (!more) break;
        }
    }
}

// Whether the collision and overlap searches of n droplets use the cells of a G^3 grid that is
// built in any case (the HI lists') instead of a finer grid of their own: the finer one saves
// candidates, but costs a build, whose scattered reads and writes move whole cache lines.  A step
// with one grid against two, by droplets per cell of the shared grid: 0.5 (128^3, 100 000) 0.59
// against 0.60 ms, 1.4 (256^3, 1M) 2.62 against 2.73, 4.1 (128^3, 800 000) 3.14 against 3.29,
// but 6 (64^3, 60 000, where a droplet's walk is a serial chain) 1.10 against 1.07.
inline bool grid_serves(int n, int G) { return (double)n <= 4.0 * G * (double)G * G; }

int hip_fail(hipError_t e, const char* what, const char* file, int line);
struct PartBuffers;
// droplet positions or slots changed: neither cell grid describes them any more
void invalidate_cells(PartBuffers& pb);
void set_error(const std::string& msg);

// ---------------------------------------------------------------- complex helpers
template <typename T> struct cpx_t;
template <> struct cpx_t<float>  { using type = float2; };
template <> struct cpx_t<double> { using type = double2; };
template <typename T> using cpx = typename cpx_t<T>::type;

template <typename C> __host__ __device__ __forceinline__ C mk(decltype(C{}.x) a, decltype(C{}.x) b) { C r; r.x = a; r.y = b; return r; }
template <typename C> __host__ __device__ __forceinline__ C cadd(C a, C b) { return mk<C>(a.x + b.x, a.y + b.y); }
template <typename C> __host__ __device__ __forceinline__ C csub(C a, C b) { return mk<C>(a.x - b.x, a.y - b.y); }
template <typename C> __host__ __device__ __forceinline__ C cmul(C a, C b) { return mk<C>(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x); }
template <typename C> __host__ __device__ __forceinline__ C cconj(C a) { return mk<C>(a.x, -a.y); }
template <typename C> __host__ __device__ __forceinline__ C cscale(C a, decltype(C{}.x) s) { return mk<C>(a.x * s, a.y * s); }
// fused forms, one rounding per product: c + a b, c - a b, c + a s (s real)
__host__ __device__ __forceinline__ float ffma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__host__ __device__ __forceinline__ double ffma(double a, double b, double c) { return __builtin_fma(a, b, c); }
template <typename C> __host__ __device__ __forceinline__ C cmadd(C c, C a, C b) { return mk<C>(ffma(a.x, b.x, ffma(-a.y, b.y, c.x)), ffma(a.x, b.y, ffma(a.y, b.x, c.y))); }
template <typename C> __host__ __device__ __forceinline__ C cmsub(C c, C a, C b) { return mk<C>(ffma(-a.x, b.x, ffma(a.y, b.y, c.x)), ffma(-a.x, b.y, ffma(-a.y, b.x, c.y))); }
template <typename C> __host__ __device__ __forceinline__ C csmadd(C c, C a, decltype(C{}.x) s) { return mk<C>(ffma(a.x, s, c.x), ffma(a.y, s, c.y)); }
// multiply by -i (forward) or +i (inverse)
template <typename C, bool INV> __host__ __device__ __forceinline__ C cmul_mi(C a) { return INV ? mk<C>(-a.y, a.x) : mk<C>(a.y, -a.x); }

// ---------------------------------------------------------------- flow layout
// Every field holds N x N x (N/2) complex values (kx < N/2: the kx = N/2 plane is identically
// zero and not stored), in rows of LW adjacent kx, one 128-byte line each:
//   - spectral fields (u-hat, the history): [ky][kx / LW][kz][LW], so the z stage finds a
//     column tile in one contiguous run;
//   - the fields between the z and y stages: [z / 8][kx / LW][y][z % 8][LW], so the z stage
//     meets N / 8 runs of 1 KB per column tile instead of N rows a whole plane apart, and the y
//     stage walks rows 1 KB apart, whose other parts the work-groups of the next planes read;
//   - the fields between the y and x stages: plain rows [z][y][kx].
// With plain rows in all three the z stage's traffic alone took 29.4 ms at 1024^3 FP32, where
// each row of a column lies on a page of its own, against 16.6 ms (256^3: 277 and 241 us).
// Physical velocity for the droplets: real [z][y][x][3] interleaved.
constexpr int LZB = 8;                               // z planes per block of an intermediate field
template <typename T> __host__ __device__ constexpr int lay_w() { return 128 / (2 * (int)sizeof(T)); }
template <typename T> __host__ __device__ __forceinline__ size_t spec_index(int N, int kz, int ky, int kx)
{
    constexpr int W = lay_w<T>();
    return (((size_t)ky * (N / 2 / W) + kx / W) * N + kz) * W + kx % W;
}
template <typename T> __host__ __device__ __forceinline__ size_t pipe_index(int N, int z, int y, int kx)
{
    constexpr int W = lay_w<T>();
    return ((((size_t)(z / LZB) * (N / 2 / W) + kx / W) * N + y) * LZB + z % LZB) * W + kx % W;
}
// the mode stored at position t of a spectral field
template <typename T> __device__ __forceinline__ void spec_mode(int N, size_t t, int& kz, int& ky, int& kx)
{
    constexpr int W = lay_w<T>();
    const int nb = N / 2 / W;
    const size_t row = t / W;
    const int kb = (int)((row / N) % nb);
    kz = (int)(row % N);
    ky = (int)(row / ((size_t)N * nb));
    kx = kb * W + (int)(t % W);
}
// Small outputs are formed side by side on the device, copied to pinned memory at once and from
// there to the caller's arrays by the host.  A copy straight to pageable memory waits for its
// kernel and takes 20 to 65 us however small it is, and an output has three to six of them: 1000
// droplets 178 us, now 64, 5000 250 and 130, the velocity at 32^3 FP32 82 and 66, the state there
// 236 and 140 (through host loops 245, 222, 54 and 217).  The host's second pass over the values
// eats the gain up with size, and a handle's first small output allocates the memory (0.1 to
// 0.4 ms).  Droplets: up to 2 MB, where a copy per array becomes as fast as the host loops were
// (with 8 MB the first pass of a new batch of 16 is 70 -> 81 ms).  Fields: up to 8 MB, so that the
// velocity at 64^3 FP32 is among them (475 and 430 us; 16 MB: no faster).
constexpr size_t BOUNCE_ROWS = 2u << 20, BOUNCE_FIELDS = 8u << 20;
struct Bounce {
    double* host = nullptr;                     // pinned, grown to the largest such output
    size_t bytes = 0;
};
inline int bounce_room(Bounce& b, size_t bytes)
{
    if (b.bytes >= bytes) return 0;
    if (b.host) DDNS_HIP(hipHostFree(b.host));
    b = Bounce{};
    DDNS_HIP(hipHostMalloc((void**)&b.host, bytes, hipHostMallocDefault));
    b.bytes = bytes;
    return 0;
}
struct FlowBuffers {
    void* U[3] = {nullptr, nullptr, nullptr};  // state u-hat
    void* O[3] = {nullptr, nullptr, nullptr};  // AB2 history
    void* A[6] = {};                            // between the z and y stages: u(3), w(3); (u x w)(3) in A[0..2]
    void* B[3] = {};                            // between the y and x stages, plain [z][y][kx]: u(3), then (u x w)(3)
    void* uphys = nullptr;                      // [z][y][x][3]: u, v, w (w-hat between the y and x stages)
    void* tw = nullptr;                         // N twiddles exp(-2 pi i m / N)
    void* twh = nullptr;                        // N/2 twiddles for the half-length x FFT
    double* low = nullptr;                      // pre-kernel scratch (1024): ff[2], energies, forcing table, DFT sums
    int* sth_state = nullptr;                   // ranff state on the device: iseedf, iyf, ivf[32]
    double* sth_b = nullptr;                    // b1r..b3r (450)
    void* dg[8] = {};                           // diagnostics scratch, 8 fields, allocated on first use
    double* dg_part = nullptr;                  // diagnostics reduction partials
    double* spec_part = nullptr;                // E(k): SPEC_BLOCKS partial rows of SPEC_NEK_MAX shells, then the result
    void* stage = nullptr;                      // state transfers: a part of a field in the reference's layout
    size_t stage_bytes = 0;                     // (allocated on first use, kept with the handle)
    Bounce bounce;                              // small outputs on their way to the caller's arrays
    int ky_tc = 0;                              // y-stage tile width chosen by flow_tune (0: the default)
    float ky_ms[3] = {0, 0, 0};                 // the tuner's time per y stage pair of each candidate (0: not valid)
    int kz_nt = 0;                              // threads of the fused z stage chosen by flow_tune (0: the default)
    float kz_ms[3] = {0, 0, 0};                 // the tuner's time per fused z stage of each candidate (0: not valid)
    // Independent realisations held side by side (a batch): every field above holds R
    // realisations, realisation r at r * rstride complex values (uphys: r * pstride reals,
    // low: r * 1024 doubles, sth_state: r * 64 ints, sth_b: r * 512 doubles), and every
    // flow launch covers all of them.  R = 1, rstride = pstride = 0 for one realisation.
    int R = 1;
    size_t rstride = 0, pstride = 0;
};
// The buffers of realisation r of a batch as a one-realisation FlowBuffers (pointers
// into the batch's arrays; nothing owned), for the transfers and diagnostics.
FlowBuffers flow_view(const FlowBuffers& fb, int r, int precision);

// E(k) shell sums (spectrum.hip): work-groups of the partial-sum kernel and the most
// shells any grid has (nek = 510 at N = 1024)
constexpr int SPEC_BLOCKS = 256;
constexpr int SPEC_NEK_MAX = 512;

struct FlowConst {
    int N;
    int nek;
    int forcing;
    double dt, rnu;
    double force0, force1;
    double ou_tf, ou_var;
    double pi2;
};

// launch wrappers (flow.hip)
int flow_alloc(FlowBuffers& fb, int N, int precision, int R = 1);
// the forcing kind and amplitudes of realisation r into its low-mode table (batches run
// with FlowConst::forcing = -1 and read them there)
int flow_set_realisation(const FlowBuffers& fb, int r, int forcing, double force0, double force1, double ou_tf,
                         double ou_var);
void flow_free(FlowBuffers& fb);
int flow_prologue(const FlowBuffers& fb, const FlowConst& fc, int precision, hipStream_t s);
// Parts of the flow step: the inverse stages (first half), the whole forward half, or the
// forward half in two pieces (forward y + pre, then z + sym) so that a wait can sit
// between them.  capturing: the stream is being captured into a graph (the events
// become graph nodes).
enum FlowPart { FLOW_INV = 0, FLOW_FWD = 1, FLOW_FWD_Y = 2, FLOW_FWD_Z = 3, FLOW_STEP = 4 };
int flow_step(const FlowBuffers& fb, const FlowConst& fc, int precision, int part, hipStream_t s,
              hipEvent_t* ev /* FLOW_EVENTS events or nullptr */, bool capturing = false);
constexpr int FLOW_EVENTS = 9;
int flow_upload_state(FlowBuffers& fb, int N, int precision, const double* const src[6], hipStream_t s);
int flow_download_state(FlowBuffers& fb, int N, int precision, double* const dst[6], hipStream_t s);
int flow_download_phys(FlowBuffers& fb, int N, int precision, double* ux, double* uy, double* uz, hipStream_t s);
// POSTPROC / TRANSPOSTPROC sums of the current u-hat.  want: 1 = CFL maximum and the
// velocity-derivative moments, 2 = divergence / vorticity sums.  ek, dk, tk (nek each,
// any may be null): energy, dissipation and transfer spectra.  mom: [0] max |u|+|v|+|w|,
// [1..3] sums of d^2, d^3, d^4 over the three longitudinal derivatives, [4..5] sums of
// div, div^2, [6..8] sums of |w|, |w|^2, |w| div
int flow_init(FlowBuffers& fb, int N, int nek, int precision, int kind, int seed, double k0, double urms, double force0,
              hipStream_t s);
int flow_diagnostics(FlowBuffers& fb, int N, int nek, double rnu, int precision, int want, double* ek, double* dk,
                     double* tk, double* mom, hipStream_t s);
int flow_spectrum(const FlowBuffers& fb, int N, int nek, int precision, double* ek, hipStream_t s);
// E, D and (F given) T shell sums on the device: part 3 SPEC_BLOCKS nek, sums_dev 3 nek doubles
int flow_shell_sums(const FlowBuffers& fb, const void* const F[3], int N, int nek, double rnu, int precision, double* part,
                    double* sums_dev, hipStream_t s);
// allocation-free E(k) (spectrum.hip): the partial rows in a file-scope device array whose
// address is resolved once per device by spectrum_scratch_init
int spectrum_scratch_init();
int flow_spectrum_device(const FlowBuffers& fb, int N, int nek, int precision, int dev, double* ek_dev, hipStream_t s);
int fft_r2c_host(FlowBuffers& fb, int N, int precision, double* v, hipStream_t s);
int fft_c2r_host(FlowBuffers& fb, int N, int precision, double* v, hipStream_t s);
int flow_profile(const FlowBuffers& fb, const FlowConst& fc, int precision, int k, double* ms, int nk, hipStream_t s);
// times the candidate y-stage tile widths and fused z-stage work-group sizes on fb's
// buffers (before any state is loaded) and keeps the fastest in fb.ky_tc, fb.kz_nt
// (cached per grid and precision); the defaults of a grid
int flow_tune(FlowBuffers& fb, const FlowConst& fc, int precision, hipStream_t s);
int flow_default_ky_tc(int N, int precision);
int flow_default_kz_nt(int N, int precision);
int flow_profile_copy(const FlowBuffers& fb, int N, int precision, int reps, double* ms, double* bytes, hipStream_t s);

// ---------------------------------------------------------------- droplets
struct PartBuffers {
    int cap = 0;
    // state, SoA FP64, slot order = the reference's droplet index order
    double* pos = nullptr;      // 3*cap
    double* vel = nullptr;      // 3*cap   yp(4:6)
    double* rad = nullptr;      // cap     yp(7)
    double* gid = nullptr;      // cap     yp(8)
    double* fvp = nullptr;      // 9*cap   fvp(:,0:2) as [t][c][cap]
    double* fdp = nullptr;      // 12*cap  fdp(:,0:3) as [t][c][cap]
    double* dmove = nullptr;    // 3*cap
    double* vp = nullptr;       // 3*cap
    double* pert = nullptr;     // 3*cap   pertvel(3, n), droplet-major as the reference stores it, so one
                                //         droplet's three components share a cache line
    // cell grid
    int G = 0;                  // coarse cells per dimension
    double hc = 0;
    int* cell_count = nullptr;  // G^3 + 1
    int* cell_start = nullptr;  // G^3 + 1
    int* cell_of = nullptr;     // cap
    int* sorted = nullptr;      // cap
    double4* pk = nullptr;      // cap: (x, y, z, radius) of sorted[p], refreshed with the cells
    int* cell_rank = nullptr;   // cap: place of a droplet among those of its cell (build scratch)
    int* cell_rank2 = nullptr;  // cap: the same for a second grid built in the same launches
    bool cells_valid = false;   // the grid above was built on the current positions
    hipEvent_t sync_ev = nullptr;   // waits of the droplet block (wait_stream)
    double* gm_host = nullptr;      // pinned: GMRES's small-problem head [0..5] and the list flags [8..11]
    // History levels as rings: level t of fvp (3 levels) is column block (t + hv_v) % 3,
    // of fdp (4 levels) (t + hv_d) % 4, so the step's history shift (level t+1 = level t)
    // only turns the rings.  After a shift level 0 holds the oldest level until it is
    // written again (fvp by the history step, fdp by the advance); until then it reads as
    // level 1, which the shift copied it to (v0_stale, d0_stale).
    int hv_v = 0, hv_d = 0;
    bool v0_stale = false, d0_stale = false;
    int vcol(int t) const { return 3 * ((t + hv_v) % 3); }   // first column of fvp level t
    int dcol(int t) const { return 3 * ((t + hv_d) % 4); }   // first column of fdp level t
    long long cell_count_zero = 0;  // cell_count[0 .. this) is zero (the last build's scan clears it)
    // the step's first overlap sweep is queued and its count not yet read; the validity
    // of the grids before its relocation, restored when it relocated nothing
    bool overlap_queued = false;
    bool overlap_cells_kept = false, overlap_spare_kept = false;
    // a second grid, kept from the last build of another width while it stays valid:
    // a search at that width then swaps it in instead of rebuilding
    struct CellSet {
        int G = 0;
        double hc = 0;
        int *cell_count = nullptr, *cell_start = nullptr, *cell_of = nullptr, *sorted = nullptr;
        double4* pk = nullptr;
        bool valid = false;
        long long count_zero = 0;
    } spare;
    void* scan_tmp = nullptr;
    size_t scan_tmp_bytes = 0;
    // HI, in cell-sorted droplet order: ELL neighbour lists, slot-major
    int* nei_cnt = nullptr;     // cap + 1
    int* nei_idx = nullptr;     // ell_width * cap: sorted position of neighbour s of row t at s * n + t
    void* nei_m = nullptr;      // 6 * ell_width * cap (float or double): entry c at (6 s + c) * n + t
    int ell_width = 0;
    void* gm_Q = nullptr;       // (maxiter+2) * 3 cap: Krylov basis, then two work vectors
    void* gm_v = nullptr;       // 3 cap
    double* gm_x0 = nullptr;    // 3 cap
    double* gm_b = nullptr;     // 3 cap
    double* gm_w = nullptr;     // 3 cap
    double* gm_red = nullptr;   // reduction partials
    double* gm_small = nullptr; // Hessenberg etc
    int gm_last_iters = 0;      // GMRES iterations of the last solve: the size of the next first batch
    // collisions
    int* mult = nullptr;        // cap: removal-list multiplicity
    void* cand = nullptr;       // cand_cap int2: pairs handed from the collision search to the pair kernel
    int cand_cap = 0;
    int last_ncand = 0;         // the last search's count: the size of the next pair-kernel grid
    int* hit = nullptr;         // cap: droplet already counted as ih1 of a collision
    // device flags / counters (64 ints): [0..7] HI lists and coalescence, [40..42] the collision search, [48] relocation draws ran out, [50] droplets relocated by an overlap
    // sweep, [51], [52] length of rlist (collision step, overlap sweep)
    int* flags = nullptr;
    unsigned long long* ext = nullptr;   // Extents: the step's displacement and radius, then overlap_setup's radius
    int* rlist = nullptr;       // cap: the droplets of a removal list, in no order
    bool step_cleared = false;  // the step's statistics, counters and flags were cleared with its history step
    long long* tested = nullptr;
    int* nirbin = nullptr;
    double* bins = nullptr;     // 7 * nset*nset*NBIN
    int* counts = nullptr;      // icc[3], colltype[100], nir[100]
    long long* pairs = nullptr; // pair_cap * DDNS_PAIR_REC: one record per detected pair
    int pair_cap = 0;
    double* contact = nullptr;  // contact_cap * DDNS_CONTACT_REC: one record per pair in contact
    int contact_cap = 0;
    int* found_host = nullptr;  // pinned: candidate and contact counts of the last collision search
    int* counts_host = nullptr; // pinned: the step's counts (512 ints) and tested pairs (4 long long)
    double* draws = nullptr;    // relocation draws
    int draw_cap = 0;
    int* draw_off = nullptr;    // cap + 1
    int* rng_state = nullptr;   // ranff2 state: idum, iy, idum2, iv[32]
    double* red = nullptr;      // generic reduction scratch
    double* stage = nullptr;    // droplet arrays in the reference's layout, made on the first transfer: one
                                // array of 12*cap, or several of a small output (Bounce)
    Bounce bounce;
};

struct PartConst {
    int N;            // flow grid (reference cell grid: ncdx = N)
    int n;            // droplets
    int nset;
    double radius[DDNS_MAXSET];
    double radmax;
    double dt, rnu, st;
    double Sv_const, tau2;
    double pi2;
    double d_coll, d_hdi, hdi_trunc;
    int nx_coll, nx_max, imax_stat;
    int hdi, nonoverlap, ndrag;
    int new_particle;
    int precision;
};

int part_alloc(PartBuffers& pb, int cap, int nset, int G);
// Droplet state to and from the reference's arrays on the host (any pointer may be null; an
// upload clears what it has no array for).  s must be ordered after the droplet block.
int part_upload(PartBuffers& pb, int n, const double* yp, const double* fvp, const double* fdp, const double* pertvel,
                hipStream_t s);
int part_download(PartBuffers& pb, int n, double* yp, double* fvp, double* fdp, double* pertvel, double* vp, double* dmove,
                  hipStream_t s);
// one 3-vector per droplet (dst(3,n), component-major slots) from the host's a(3, n)
int part_upload3(PartBuffers& pb, int n, double* dst, const double* a, hipStream_t s);
// Waits for event e: by polling it for POLL_MS, then as the runtime waits.  After a blocking
// wait the host thread ran again tens of microseconds after the GPU had finished, and the stream
// waited that long for the launches that follow; past POLL_MS that is a few per cent of the
// wait, and a program that has asked HIP for blocking waits (hipDeviceScheduleBlockingSync) gets
// its core back: 64 flow steps at 256^3 take 45 ms and held it for all of them when this polled
// to the end.
constexpr double POLL_MS = 2.0;
inline hipError_t spin_wait(hipEvent_t e)
{
    const auto t0 = std::chrono::steady_clock::now();
    for (;;) {
        const hipError_t r = hipEventQuery(e);
        if (r != hipErrorNotReady) return r;
        if (std::chrono::steady_clock::now() - t0 > std::chrono::duration<double, std::milli>(POLL_MS)) return hipEventSynchronize(e);
    }
}
// all work queued on s so far, waited for by spin_wait (pb.sync_ev, made on first use)
inline hipError_t wait_stream(PartBuffers& pb, hipStream_t s)
{
    if (!pb.sync_ev) {
        const hipError_t r = hipEventCreateWithFlags(&pb.sync_ev, hipEventDisableTiming);
        if (r != hipSuccess) return r;
    }
    const hipError_t r = hipEventRecord(pb.sync_ev, s);
    return r != hipSuccess ? r : spin_wait(pb.sync_ev);
}
void part_free(PartBuffers& pb);
// with HI on, also writes the HI solve's x0 and w in cell order (after part_history_fvp)
int part_interp(PartBuffers& pb, const PartConst& pc, const void* uphys, hipStream_t s);
// the history step; also clears what the step's searches write (ZeroSpans)
int part_history_fvp(PartBuffers& pb, const PartConst& pc, hipStream_t s);
int part_build_cells(PartBuffers& pb, const PartConst& pc, double hmin, hipStream_t s);
// The grid of width hmin as the current one and that of width other as the spare, both built in
// the same launches when neither is valid (as two part_build_cells calls would leave them, in
// the order other, hmin).
int part_build_two(PartBuffers& pb, const PartConst& pc, double hmin, double other, hipStream_t s);
// Several device spans (4-byte multiples) cleared by one launch instead of one fill per span.
struct ZeroSpans {
    unsigned* p[10];
    size_t words[10];
    int n;
};
int part_step_spans(PartBuffers& pb, const PartConst& pc, ZeroSpans& z);
__device__ __forceinline__ void zero_spans(const ZeroSpans& z, size_t at, size_t stride)
{
    for (int k = 0; k < z.n; ++k)
        for (size_t i = at; i < z.words[k]; i += stride) z.p[k][i] = 0u;
}
// The largest displacement and droplet radius, as the bits of non-negative doubles (whose order
// is the numeric order), in EXT_SLOTS slots of two that work-group b raises at slot b mod
// EXT_SLOTS; a reader takes the largest of all slots.  A single address served a million
// droplets' work-groups in 70 us (each XCD's atomics go to memory one after the other).
constexpr int EXT_SLOTS = 32, EXT_STRIDE = 16, EXT_WORDS = EXT_SLOTS * EXT_STRIDE;   // a slot per 128 bytes

// by one lane of a work-group; most find the slot as large already
__device__ __forceinline__ void raise_extents(unsigned long long* ext, double far, double big)
{
    unsigned long long* e = ext + (blockIdx.x % EXT_SLOTS) * EXT_STRIDE;
    const unsigned long long f = (unsigned long long)__double_as_longlong(far), b = (unsigned long long)__double_as_longlong(big);
    if (far > 0.0 && f > *(volatile unsigned long long*)e) atomicMax(e, f);
    if (big > 0.0 && b > *(volatile unsigned long long*)(e + 1)) atomicMax(e + 1, b);
}
// by all lanes of a wavefront; which: 0 the displacement, 1 the radius
__device__ __forceinline__ double read_extent(const unsigned long long* ext, int which)
{
    double m = __longlong_as_double((long long)ext[(threadIdx.x % EXT_SLOTS) * EXT_STRIDE + which]);
#pragma unroll
    for (int o = EXT_SLOTS / 2; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    return m;
}
int part_hdi(PartBuffers& pb, const PartConst& pc, int maxiter, double tol, int* iters, double* res, hipStream_t s);
// The start of a solve (neighbour lists, right-hand side, first Krylov vector) queued on s.
int part_hdi_begin(PartBuffers& pb, const PartConst& pc, int maxiter, double tol, hipStream_t s);
// The iterations of R started solves at once on stream s (every kernel one launch over
// the R systems), then each solution scattered to its droplets.  iters, res, status (0,
// DDNS_WARN_GMRES, or an error of the neighbour lists) per system; redo[r] = 1 where the
// lists had to be widened: that system is to be solved again on its own.
struct HdiBatch {
    void* table = nullptr;          // device: one descriptor per system
    double* heads = nullptr;        // device: 16 doubles per system
    void* table_host = nullptr;     // pinned staging of the descriptors
    double* heads_host = nullptr;   // pinned copy of the heads
    int cap = 0;
};
int part_hdi_batch(HdiBatch& hb, PartBuffers* const* pbs, const PartConst* const* pcs, int R, int maxiter,
                   int* iters, double* res, int* status, int* redo, hipStream_t s);
void part_hdi_batch_free(HdiBatch& hb);
int part_advance(PartBuffers& pb, const PartConst& pc, hipStream_t s);
int part_collide(PartBuffers& pb, const PartConst& pc, hipStream_t s);
// the collision search queued without a host wait, and its completion (waits for the
// search's counts, then queues the pair kernel)
int part_collide_search(PartBuffers& pb, const PartConst& pc, hipStream_t s);
// part_collide_finish / part_collide: some droplet's reach (its statistics window or
// its collision window) exceeds the cell width, so the walk may have missed partners:
// the caller builds wider cells and searches again
constexpr int DDNS_COLL_REGRID = 2;
int part_collide_finish(PartBuffers& pb, const PartConst& pc, hipStream_t s);
// queue the step's counts into pinned memory; read them after the stream was waited for
int part_queue_counts(PartBuffers& pb, hipStream_t s);
// exclusive scan of n ints into out[0..n-1], the total into out[n] (particles.hip);
// clear_in leaves in[0..n-1] zero (in must not alias out then)
int exclusive_scan(const int* in, int* out, int n, int* tmp, hipStream_t s, bool clear_in = false);
int part_take_counts(const PartBuffers& pb, const PartConst& pc, ddns_collision_counts* cc);
int part_update_and_wrap(PartBuffers& pb, const PartConst& pc, bool relocate, hipStream_t s);
// The droplets of rlist (flags[nlist] of them) relocated by one launch, no host round trip.
// wrap: the drawn positions get the PERIODIC wrap (the step's wrap follows its relocation)
int relocate_list(PartBuffers& pb, const PartConst& pc, int nlist, bool wrap, hipStream_t s);
int part_overlap(PartBuffers& pb, const PartConst& pc, int* sweeps, int* relocated, hipStream_t s);
// the step's overlap sweep: the first sweep queued without a host wait; the rest, if it
// relocated droplets, after the caller has waited for the stream
// next_width: the next step's first grid, built too, on the positions the sweep saw, and kept
// if the sweep moves nothing
// grown: coalescence has changed radii since the advance
int part_overlap_queue(PartBuffers& pb, const PartConst& pc, hipStream_t s, double next_width, bool grown);
int part_overlap_finish(PartBuffers& pb, const PartConst& pc, int* sweeps, int* relocated, hipStream_t s);
int part_read_counts(const PartBuffers& pb, const PartConst& pc, ddns_collision_counts* cc, hipStream_t s);
int part_read_bins(const PartBuffers& pb, const PartConst& pc, int* nirbin, double* const bins[7], hipStream_t s);
int part_read_pairs(PartBuffers& pb, const PartConst& pc, int64_t* triples, int cap, int* npairs, hipStream_t s);
int part_read_contacts(const PartBuffers& pb, double* rec, int cap, int* n, hipStream_t s);
int part_coalesce(PartBuffers& pb, const PartConst& pc, int* removed, hipStream_t s);
int part_set_rng(const PartBuffers& pb, int iseedr, hipStream_t s);

}  // namespace ddns
