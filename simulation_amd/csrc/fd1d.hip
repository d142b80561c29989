// fd1d.hip -- 1-D Ex/Hy kernels for gfx950.
//
// Semantics: the serial order of fd1d/clang/fd1d_1_2.c:151-167 and
// fd1d/clang/fd1d_1_5.c:25-41 (E update, source, two-step boundary, H update),
// in the expression order of the PyCUDA kernels fd1d/pycuda/fd1d_1_5.py:49-67.
// Built with -ffp-contract=off: every multiply and add rounds separately.
#include "fdtd_internal.h"
#include "lanes.h"

namespace fdtd {
namespace {

// E update of one cell.  ca == NULL means ca = 1 and cb == NULL means cb = 0.5:
// ca*ex == ex exactly for ca = 1, so one body covers the += forms of
// fd1d/pycuda/fd1d_1_2.py:47 and fd1d/pycuda/fd1d_1_3.py:50.
template <typename T>
__device__ __forceinline__ T e_cell(T e, T hl, T hr, const T *ca, const T *cb, int i)
{
    T d = hl - hr;
    if (ca) return ca[i] * e + cb[i] * d;
    if (cb) return e + cb[i] * d;
    return e + T(0.5) * d;
}

template <typename T>
__global__ void fd1d_exfield_kernel(int nx, const T *__restrict__ ca, const T *__restrict__ cb,
                                    T *__restrict__ ex, const T *__restrict__ hy,
                                    int src_mode, int src_pos, T src_val)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nx; i += blockDim.x * gridDim.x) {
        T v = ex[i];
        bool changed = false;
        if (i >= 1) { v = e_cell(v, hy[i - 1], hy[i], ca, cb, i); changed = true; }
        // the owner of the source cell applies the source after its update
        if (i == src_pos && src_mode == FDTD_SRC_HARD) { v = src_val; changed = true; }
        else if (i == src_pos && src_mode == FDTD_SRC_ADD) { v = v + src_val; changed = true; }
        if (changed) ex[i] = v;
    }
}

// Boundary + H update.  Thread i = 0 owns the low-end boundary (reads bc[0],
// bc[1], ex[1]; writes ex[0], bc[0], bc[1]) and thread i = nx-2 the high end
// (reads bc[2], bc[3], ex[nx-2]; writes ex[nx-1], bc[2], bc[3]); no other
// thread touches those words, and the H update of those two threads uses the
// new boundary values, as the serial program does.
template <typename T>
__global__ void fd1d_hyfield_kernel(int nx, T *__restrict__ ex, T *__restrict__ hy,
                                    T *__restrict__ bc)
{
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nx - 1; i += blockDim.x * gridDim.x) {
        T e0 = ex[i], e1 = ex[i + 1];
        if (bc) {
            if (i == 0) {
                T b0 = bc[0], b1 = bc[1];
                ex[0] = b0; bc[0] = b1; bc[1] = e1;
                e0 = b0;
            }
            if (i == nx - 2) {
                T b3 = bc[3], b2 = bc[2];
                ex[nx - 1] = b3; bc[3] = b2; bc[2] = e0;
                e1 = b3;
            }
        }
        hy[i] = hy[i] + T(0.5) * (e0 - e1);
    }
}

// All steps in one workgroup: ex and hy live in LDS, three barriers a step.
struct ProbeK { int n; int k[FDTD_MAX_PROBES]; };

template <typename T>
__global__ void __launch_bounds__(1024)
fd1d_run_kernel(int nx, int nsteps, const T *__restrict__ ca, const T *__restrict__ cb,
                T *__restrict__ ex_g, T *__restrict__ hy_g, T *__restrict__ bc_g,
                int src_mode, int src_pos, const T *__restrict__ src_wave,
                ProbeK pk, T *__restrict__ probe_out)
{
    extern __shared__ __align__(16) unsigned char smem[];
    T *ex = reinterpret_cast<T *>(smem);
    T *hy = ex + nx;
    const int tid = threadIdx.x, nt = blockDim.x;
    for (int i = tid; i < nx; i += nt) { ex[i] = ex_g[i]; hy[i] = hy_g[i]; }
    T b0 = 0, b1 = 0, b2 = 0, b3 = 0;
    if (tid == 0 && bc_g) { b0 = bc_g[0]; b1 = bc_g[1]; b2 = bc_g[2]; b3 = bc_g[3]; }
    __syncthreads();
    for (int s = 0; s < nsteps; ++s) {
        const T sv = src_wave ? src_wave[s] : T(0);
        for (int i = tid; i < nx; i += nt) {
            T v = ex[i];
            if (i >= 1) v = e_cell(v, hy[i - 1], hy[i], ca, cb, i);
            if (i == src_pos && src_mode == FDTD_SRC_HARD) v = sv;
            else if (i == src_pos && src_mode == FDTD_SRC_ADD) v = v + sv;
            ex[i] = v;
        }
        __syncthreads();
        if (tid == 0) {
            if (bc_g) {
                ex[0] = b0; b0 = b1; b1 = ex[1];
                ex[nx - 1] = b3; b3 = b2; b2 = ex[nx - 2];
            }
            for (int p = 0; p < pk.n; ++p) probe_out[(size_t)p * nsteps + s] = ex[pk.k[p]];
        }
        __syncthreads();
        for (int i = tid; i < nx - 1; i += nt) hy[i] = hy[i] + T(0.5) * (ex[i] - ex[i + 1]);
        __syncthreads();
    }
    for (int i = tid; i < nx; i += nt) { ex_g[i] = ex[i]; hy_g[i] = hy[i]; }
    if (tid == 0 && bc_g) { bc_g[0] = b0; bc_g[1] = b1; bc_g[2] = b2; bc_g[3] = b3; }
}

// Blocked run.  A wavefront holds 64 contiguous cells in registers, one a
// lane, and advances them with no barrier and no LDS: the cells beside a
// lane's own come from its neighbours through DPP wave shifts.  One step moves
// information one cell each way, so `halo` steps leave all but the outer
// `halo` cells of a wave exact.  The waves of a workgroup overlap by twice
// that; every `halo` steps each publishes the cells it has exact in LDS and
// takes its outer cells from there (one barrier; two buffers alternate).  In
// the same way workgroups overlap by twice the steps of a launch, each reading
// one state set and writing the cells it owns of the other; a grid that one
// workgroup holds takes all its steps in one launch, in place.
//
// What bounds it: one step is a chain of two neighbour shifts and five
// dependent floating-point instructions (about 35 ns a step for a single wave
// with nothing else to do), then the exchanges and launches.  Hence one cell a
// lane (two or four measured 1.3 and 1.6 times as long), and a loop body of
// its own for each kind of wave (edge, source, probe): deciding inside the
// step doubled it.  200 cells, FP32, 500 steps: 243 us as one workgroup with
// the fields in LDS and three barriers a step, 27 us now; 3001 cells, FP64,
// 1000 steps, lossy: 1827 -> 113 us; 38000 cells, FP32, 500 steps: 7.9 ms as
// two launches a step, 39 us now.
constexpr int W1D_MAX = 16;        // waves of a workgroup

template <typename T>
struct Run1d {
    int nx, n;                     // n: steps of this launch
    int own, depth, region;        // cells a workgroup owns, its outer halo, its region
    int stride, halo;              // of the waves inside a region
    const T *ca, *cb;              // NULL: 1, 0.5
    const T *ex_i, *hy_i, *bc_i;   // bc NULL: no boundary
    T *ex_o, *hy_o, *bc_o;
    int src_mode, src_pos;
    const T *src_wave;             // value of the launch's first step first
    ProbeK pk;
    T *probe_out;                  // the launch's first column
    int probe_len;
};

template <typename T>
struct Seg1d {                     // a wave's state and places
    T e, h, a, b;                  // lane's cell
    T b0, b1, b2, b3;              // two-step boundary: lane 0's and lane rl's
    int lane, rl;                  // rl: the lane of cell nx-1
    int sl, pl;                    // lanes of the source and of the first probe
    bool hard, many, mine;         // several waves; the lane's cell is published
    int chunk, at, pf;             // steps between exchanges; place in LDS; first probe
    unsigned long long pm;         // probes of the wave
    int from;                      // of probe `lane`: 4 times the lane of its cell
    bool rec;                      // probe `lane` is the wave's
};

enum { EDGE_L = 1, EDGE_R = 2, EDGE_ABC = 4 };   // cell 0, cell nx-1, two-step boundary

// One step; s: step of the chunk.  SRC: the wave holds the source cell (sw:
// its value of step l in lane l); PRB: it records one probe (tr: its trace,
// step l in lane l), or (2) several (out: probe `lane`'s trace).
template <typename T, bool COEF, int EDGE, bool SRC, int PRB>
__device__ __forceinline__ void step1d(Seg1d<T> &g, int s, T sw, T &tr, T *out)
{
    constexpr bool L = EDGE & EDGE_L, R = EDGE & EDGE_R, ABC = EDGE & EDGE_ABC;
    const T d = lane_left(g.h) - g.h;
    T v = COEF ? g.a * g.e + g.b * d : g.e + T(0.5) * d;
    if (L && !ABC) v = g.lane == 0 ? g.e : v;                   // cell 0: no update
    if (SRC) {
        const T sv = lane_get(sw, s);
        const T u = g.hard ? sv : v + sv;
        v = g.lane == g.sl ? u : v;
    }
    T er = T(0);
    if (ABC) {
        const T e1 = L ? lane_right(v) : T(0), e2 = R ? lane_left(v) : T(0);
        if (L) {
            v = g.lane == 0 ? g.b0 : v;
            g.b0 = g.b1;
            g.b1 = e1;
        }
        if (R) {
            v = g.lane == g.rl ? g.b3 : v;
            g.b3 = g.b2;
            g.b2 = e2;
        }
    }
    g.e = v;
    if (PRB == 1) {
        const T x = lane_get(v, g.pl);
        tr = g.lane == s ? x : tr;
    }
    if (PRB == 2) {
        // one exchange and one store for all probes (64 cells, 16 probes,
        // 400 steps, FP32 / FP64: 494 / 544 us with a loop over them, 46 / 61)
        const T x = lane_pick(v, g.from);
        if (g.rec) out[s] = x;
    }
    er = lane_right(v);
    const T w = g.h + T(0.5) * (v - er);
    g.h = R && g.lane == g.rl ? g.h : w;                        // cell nx-1: no update
}

template <typename T, bool COEF, int EDGE, bool SRC, int PRB>
__device__ __forceinline__ void chunk1d(Seg1d<T> &g, int n, T sw, T &tr, T *out)
{
    // unrolled by hand: the compiler does not unroll loops with lane shifts
    int s = 0;
#pragma unroll 1
    for (; s + 8 <= n; s += 8) {
        step1d<T, COEF, EDGE, SRC, PRB>(g, s, sw, tr, out);
        step1d<T, COEF, EDGE, SRC, PRB>(g, s + 1, sw, tr, out);
        step1d<T, COEF, EDGE, SRC, PRB>(g, s + 2, sw, tr, out);
        step1d<T, COEF, EDGE, SRC, PRB>(g, s + 3, sw, tr, out);
        step1d<T, COEF, EDGE, SRC, PRB>(g, s + 4, sw, tr, out);
        step1d<T, COEF, EDGE, SRC, PRB>(g, s + 5, sw, tr, out);
        step1d<T, COEF, EDGE, SRC, PRB>(g, s + 6, sw, tr, out);
        step1d<T, COEF, EDGE, SRC, PRB>(g, s + 7, sw, tr, out);
    }
#pragma unroll 1
    for (; s < n; ++s) step1d<T, COEF, EDGE, SRC, PRB>(g, s, sw, tr, out);
}

// All steps of a launch, `chunk` at a time.  One copy per kind of wave, with
// the exchange inside: choosing the body again for every chunk cost as much
// as eight steps.
template <typename T, bool COEF, int EDGE, bool SRC, int PRB>
__device__ __forceinline__ void run1d(Seg1d<T> &g, const Run1d<T> &P)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = g.lane;
    T sw = 0, sn = 0;
    if (SRC) sn = lane < P.n ? P.src_wave[lane] : T(0);
    T *es = reinterpret_cast<T *>(smem) + g.at;
    int flip = 2 * P.region;
    for (int done = 0; done < P.n;) {
        const int n = min(g.chunk, P.n - done);
        T tr = 0;
        T *out = P.probe_out + done;
        if (PRB == 2) out += (size_t)lane * P.probe_len;
        if (SRC) {
            // the next chunk's values, in flight during this one
            const int k = done + n + lane;
            sw = sn;
            sn = k < P.n ? P.src_wave[k] : T(0);
        }
        chunk1d<T, COEF, EDGE, SRC, PRB>(g, n, sw, tr, out);
        if (PRB == 1 && lane < n) out[(size_t)g.pf * P.probe_len + lane] = tr;
        done += n;
        if (g.many && done < P.n) {
            if (g.mine) { es[0] = g.e; es[P.region] = g.h; }
            __syncthreads();
            if (!g.mine) { g.e = es[0]; g.h = es[P.region]; }
            es += flip;
            flip = -flip;
        }
    }
}

template <typename T, bool COEF, int EDGE>
__device__ __forceinline__ void run1d_sp(Seg1d<T> &g, const Run1d<T> &P, bool src)
{
    const int prb = g.pm == 0 ? 0 : (g.pm & (g.pm - 1)) == 0 ? 1 : 2;
    if (prb == 2) {
        if (src) run1d<T, COEF, EDGE, true, 2>(g, P);
        else run1d<T, COEF, EDGE, false, 2>(g, P);
    } else if (prb) {
        if (src) run1d<T, COEF, EDGE, true, 1>(g, P);
        else run1d<T, COEF, EDGE, false, 1>(g, P);
    } else {
        if (src) run1d<T, COEF, EDGE, true, 0>(g, P);
        else run1d<T, COEF, EDGE, false, 0>(g, P);
    }
}

// ca NULL runs as ca = 1 (1 * ex is ex).
template <typename T, bool COEF>
__global__ void __launch_bounds__(64 * W1D_MAX) fd1d_wave_kernel(const Run1d<T> P)
{
    const int nx = P.nx, lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), nw = blockDim.x >> 6;
    const int wg = blockIdx.x;
    const bool last = wg == (int)gridDim.x - 1;
    // region of the workgroup, its owned cells, this wave's cells
    const int o0 = wg * P.own, o1 = last ? nx : o0 + P.own;
    const int g0 = max(0, min(o0 - P.depth, nx - P.region));
    const int st = g0 + max(0, min(wv * P.stride, P.region - 64));
    const int st1 = g0 + max(0, min((wv + 1) * P.stride, P.region - 64));
    const int i = st + lane;
    // cells this wave publishes, and those of them it writes out
    const int p0 = wv ? st + P.halo : st, p1 = wv + 1 < nw ? st1 + P.halo : g0 + P.region;
    const int w0 = max(p0, o0), w1 = min(p1, o1);
    Seg1d<T> g;
    g.lane = lane;
    const bool in = i < nx;
    g.e = in ? P.ex_i[i] : T(0);
    g.h = in ? P.hy_i[i] : T(0);
    g.a = COEF && in && P.ca ? P.ca[i] : T(1);
    g.b = COEF && in ? P.cb[i] : T(0.5);
    const bool left = st == 0, right = st + 64 >= nx, abc = P.bc_i != nullptr;
    g.rl = nx - 1 - st;
    g.b0 = g.b1 = g.b2 = g.b3 = T(0);
    if (abc && left) { g.b0 = P.bc_i[0]; g.b1 = P.bc_i[1]; }
    if (abc && right) { g.b2 = P.bc_i[2]; g.b3 = P.bc_i[3]; }
    const int edge = (left ? EDGE_L : 0) | (right ? EDGE_R : 0) | (abc && (left || right) ? EDGE_ABC : 0);
    g.sl = P.src_pos - st;
    const bool src = P.src_mode != FDTD_SRC_NONE && g.sl >= 0 && g.sl < 64;
    g.hard = P.src_mode == FDTD_SRC_HARD;
    // lane p holds probe p's cell; the wave that writes the cell records it
    const int pk = lane < P.pk.n ? P.pk.k[lane] : -1;
    g.pm = __builtin_amdgcn_ballot_w64(pk >= w0 && pk < w1);
    g.pf = g.pm ? __builtin_ctzll(g.pm) : 0;
    g.pl = (__builtin_amdgcn_readlane(pk, g.pf) - st) & 63;
    g.from = ((pk - st) & 63) * 4;
    g.rec = g.pm >> lane & 1;
    g.many = nw > 1;
    g.mine = i >= p0 && i < p1;
    g.chunk = nw > 1 ? P.halo : 64;
    g.at = i - g0;
    // every wave passes the same number of barriers (P.n, P.halo decide)
    switch (edge) {
    case 0: run1d_sp<T, COEF, 0>(g, P, src); break;
    case 1: run1d_sp<T, COEF, 1>(g, P, src); break;
    case 2: run1d_sp<T, COEF, 2>(g, P, src); break;
    case 3: run1d_sp<T, COEF, 3>(g, P, src); break;
    case 5: run1d_sp<T, COEF, 5>(g, P, src); break;
    case 6: run1d_sp<T, COEF, 6>(g, P, src); break;
    default: run1d_sp<T, COEF, 7>(g, P, src); break;
    }
    // in place: every wave has read its cells before any are written
    if (nw > 1) __syncthreads();
    if (i >= w0 && i < w1) { P.ex_o[i] = g.e; P.hy_o[i] = g.h; }
    if (abc && wg == 0 && left && lane == 0) { P.bc_o[0] = g.b0; P.bc_o[1] = g.b1; }
    if (abc && last && right && lane == g.rl) { P.bc_o[2] = g.b2; P.bc_o[3] = g.b3; }
}

// ca, cb of fd1d/pycuda/fd1d_1_5.py:71-78, in FP64, stored as T.
template <typename T>
__global__ void fd1d_dielectric_kernel(int nx, double dt, double epsr, double sigma,
                                       T *__restrict__ ca, T *__restrict__ cb)
{
    const double eps0 = 8.854e-12;
    const double epsf = dt * sigma / (2 * eps0 * epsr);
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < nx; i += blockDim.x * gridDim.x) {
        double a = 1.0, b = 0.5;
        if (i >= nx / 2) { a = (1 - epsf) / (1 + epsf); b = 0.5 / (epsr * (1 + epsf)); }
        ca[i] = (T)a;
        cb[i] = (T)b;
    }
}

constexpr int kLdsLimit = 64 * 1024;

inline int grid1d(int n, int block) { int g = (n + block - 1) / block; return g < 1 ? 1 : (g > 65535 ? 65535 : g); }

template <typename T>
int launch_wave(const Run1d<T> &p, int groups, int waves, hipStream_t s)
{
    const size_t lds = waves > 1 ? 4 * sizeof(T) * (size_t)p.region : 0;
    if (p.cb)
        hipLaunchKernelGGL((fd1d_wave_kernel<T, true>), dim3(groups), dim3(64 * waves), lds, s, p);
    else
        hipLaunchKernelGGL((fd1d_wave_kernel<T, false>), dim3(groups), dim3(64 * waves), lds, s, p);
    return hip_check(hipGetLastError(), "fd1d_run launch");
}

// Waves of a workgroup and their halo.  MI355X, us (waves, halo):
//   FP32 200 cells, 500 steps: (12,16) 27, (12,8) 31; 500 cells: (12,8) 34,
//     (16,16) 38; 38000 cells: (12,16) 39, (8,8) 41, (12,8) 44, (16,16) 42
//   FP64 200 cells, 500 steps, lossy: (12,8) 43, (12,16) 48; 500 cells: (12,8)
//     61, (16,12) 68; 3001 cells, 1000 steps: (8,8) 113, (12,8) 128,
//     (16,16) 163
// An FP64 step issues twice the instructions, so fewer waves share a SIMD.
struct Shape1d {
    int waves, halo;
    constexpr int stride() const { return 64 - 2 * halo; }
    constexpr int cells() const { return (waves - 1) * stride() + 64; }
};
constexpr Shape1d kWide1d{12, 8}, kDeep1d{12, 16}, kFew1d{8, 8};

}  // namespace

int fd1d_run_lds_limit() { return kLdsLimit; }

int fd1d_group_max_nx() { return kWide1d.cells(); }

template <typename T>
int launch_fd1d_blocked(int nx, int nsteps, const T *ca, const T *cb, T *ex, T *hy, T *bc,
                        int src_mode, int src_pos, const T *src_wave, int nprobe,
                        const int *probe_k, T *probe_out, int probe_len, T *work, hipStream_t s)
{
    constexpr bool f32 = sizeof(T) == 4;
    Run1d<T> p{};
    p.nx = nx;
    p.ca = ca; p.cb = cb;
    p.src_mode = src_wave ? src_mode : FDTD_SRC_NONE; p.src_pos = src_pos;
    p.pk.n = nprobe;
    for (int q = 0; q < nprobe; ++q) p.pk.k[q] = probe_k[q];
    p.probe_len = probe_len;
    if (nx <= fd1d_group_max_nx()) {
        // one workgroup, one launch, in place
        const Shape1d f = f32 && nx <= kDeep1d.cells() ? kDeep1d : kWide1d;
        p.halo = f.halo; p.stride = f.stride();
        p.n = nsteps; p.own = nx; p.depth = 0;
        p.region = nx > 64 ? nx : 64;
        p.ex_i = ex; p.hy_i = hy; p.bc_i = bc;
        p.ex_o = ex; p.hy_o = hy; p.bc_o = bc;
        p.src_wave = src_wave; p.probe_out = probe_out;
        return launch_wave<T>(p, 1, (p.region - 64 + p.stride - 1) / p.stride + 1, s);
    }
    if (!work) return fail("fd1d_run: several segments and no work buffer");
    // Several workgroups: a launch costs about as much as 80 steps, so the
    // launches are as deep as the region allows with 64 cells owned; once
    // that is more workgroups than CUs (256) the owned share grows, to half
    // of the region.
    const Shape1d f = f32 ? kDeep1d : kFew1d;
    p.halo = f.halo; p.stride = f.stride(); p.region = f.cells();
    int own = (nx + 255) / 256;
    own = own < 64 ? 64 : (own > p.region / 2 ? p.region / 2 : own);
    const int kmax = (p.region - own) / 2;
    int L = (nsteps + kmax - 1) / kmax;
    L += L % 2;                      // the result ends in the caller's arrays
    p.depth = nsteps / L + (nsteps % L ? 1 : 0);
    p.own = p.region - 2 * p.depth;
    T *w[3] = {work, work + nx, work + 2 * (size_t)nx};
    int done = 0;
    for (int l = 0; l < L; ++l) {
        p.n = nsteps / L + (l < nsteps % L ? 1 : 0);
        const bool odd = l % 2;
        p.ex_i = odd ? w[0] : ex; p.hy_i = odd ? w[1] : hy; p.bc_i = !bc ? nullptr : odd ? w[2] : bc;
        p.ex_o = odd ? ex : w[0]; p.hy_o = odd ? hy : w[1]; p.bc_o = !bc ? nullptr : odd ? bc : w[2];
        p.src_wave = src_wave ? src_wave + done : nullptr;
        p.probe_out = probe_out ? probe_out + done : nullptr;
        const int rc = launch_wave<T>(p, (nx + p.own - 1) / p.own, f.waves, s);
        if (rc) return rc;
        done += p.n;
    }
    return 0;
}

int preload_fd1d() { return preload_kernel(reinterpret_cast<const void *>(&fd1d_dielectric_kernel<float>)); }

template <typename T>
int launch_fd1d_exfield(int nx, const T *ca, const T *cb, T *ex, const T *hy,
                        int src_mode, int src_pos, T src_val, hipStream_t s)
{
    hipLaunchKernelGGL(fd1d_exfield_kernel<T>, dim3(grid1d(nx, 256)), dim3(256), 0, s,
                       nx, ca, cb, ex, hy, src_mode, src_pos, src_val);
    return hip_check(hipGetLastError(), "fd1d_exfield launch");
}

template <typename T>
int launch_fd1d_hyfield(int nx, T *ex, T *hy, T *bc, hipStream_t s)
{
    hipLaunchKernelGGL(fd1d_hyfield_kernel<T>, dim3(grid1d(nx - 1, 256)), dim3(256), 0, s,
                       nx, ex, hy, bc);
    return hip_check(hipGetLastError(), "fd1d_hyfield launch");
}

template <typename T>
int launch_fd1d_run(int nx, int nsteps, const T *ca, const T *cb, T *ex, T *hy, T *bc,
                    int src_mode, int src_pos, const T *src_wave,
                    int nprobe, const int *probe_k, T *probe_out, hipStream_t s)
{
    ProbeK pk{};
    pk.n = nprobe;
    for (int p = 0; p < nprobe; ++p) pk.k[p] = probe_k[p];
    int nt = ((nx + 63) / 64) * 64;
    if (nt > 1024) nt = 1024;
    const size_t lds = 2 * sizeof(T) * (size_t)nx;
    hipLaunchKernelGGL(fd1d_run_kernel<T>, dim3(1), dim3(nt), lds, s,
                       nx, nsteps, ca, cb, ex, hy, bc, src_mode, src_pos, src_wave, pk, probe_out);
    return hip_check(hipGetLastError(), "fd1d_run launch");
}

template <typename T>
int launch_fd1d_dielectric(int nx, double dt, double epsr, double sigma, T *ca, T *cb,
                           hipStream_t s)
{
    hipLaunchKernelGGL(fd1d_dielectric_kernel<T>, dim3(grid1d(nx, 256)), dim3(256), 0, s,
                       nx, dt, epsr, sigma, ca, cb);
    return hip_check(hipGetLastError(), "fd1d_dielectric launch");
}

template int launch_fd1d_dielectric<float>(int, double, double, double, float *, float *, hipStream_t);
template int launch_fd1d_dielectric<double>(int, double, double, double, double *, double *, hipStream_t);

template int launch_fd1d_blocked<float>(int, int, const float *, const float *, float *, float *, float *, int, int, const float *, int, const int *, float *, int, float *, hipStream_t);
template int launch_fd1d_blocked<double>(int, int, const double *, const double *, double *, double *, double *, int, int, const double *, int, const int *, double *, int, double *, hipStream_t);
template int launch_fd1d_exfield<float>(int, const float *, const float *, float *, const float *, int, int, float, hipStream_t);
template int launch_fd1d_exfield<double>(int, const double *, const double *, double *, const double *, int, int, double, hipStream_t);
template int launch_fd1d_hyfield<float>(int, float *, float *, float *, hipStream_t);
template int launch_fd1d_hyfield<double>(int, double *, double *, double *, hipStream_t);
template int launch_fd1d_run<float>(int, int, const float *, const float *, float *, float *, float *, int, int, const float *, int, const int *, float *, hipStream_t);
template int launch_fd1d_run<double>(int, int, const double *, const double *, double *, double *, double *, int, int, const double *, int, const int *, double *, hipStream_t);

}  // namespace fdtd
