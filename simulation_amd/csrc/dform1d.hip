// 1-D D/E form with lossy and Debye media and the 1-D running DFT
// (fd1d/pycuda/fd1d_2_1.py, fd1d_2_2.py, fd1d_2_3.py:73-158; serial semantics
// of fd1d/clang/test_2_3.c:26-90).
//
// Per step: D update with an additive source at one cell, E from D through
// the medium (nax, nbx; with ncx, ndx the Debye relaxation sx), the running
// DFT of ex, then the two-step absorbing boundary and the H update (the
// existing fd1d_hyfield).  FP32 in the reference's operand order without
// contraction; the DFT twiddles are evaluated on the host.
#include <hip/hip_runtime.h>
#include <math.h>

#include "fdtd_internal.h"
#include "lanes.h"

namespace fdtd {
namespace {

// dx[i] += 0.5 (hy[i-1] - hy[i]) for i in [1, nx); the thread that owns
// src_pos then adds the source (after its own update, as the serial loop).
__global__ void __launch_bounds__(256) dxfield_kernel(int nx, float *dx, const float *hy,
                                                      int src_pos, float src_val, int src_on)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < 1 || i >= nx) return;
    float d = dx[i] + 0.5f * (hy[i - 1] - hy[i]);
    if (src_on && i == src_pos) d = d + src_val;
    dx[i] = d;
}

// ex = nax (dx - ix [- ncx sx]); ix += nbx ex; [sx = ncx sx + ndx ex]
template <bool DEBYE>
__global__ void __launch_bounds__(256) exfield_kernel(int nx, const float *nax, const float *nbx,
                                                      const float *ncx, const float *ndx,
                                                      const float *dx, float *ix, float *sx,
                                                      float *ex)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < 1 || i >= nx) return;
    float e;
    if (DEBYE) {
        const float s = sx[i];
        e = nax[i] * (dx[i] - ix[i] - ncx[i] * s);
        ix[i] = ix[i] + nbx[i] * e;
        sx[i] = ncx[i] * s + ndx[i] * e;
    } else {
        e = nax[i] * (dx[i] - ix[i]);
        ix[i] = ix[i] + nbx[i] * e;
    }
    ex[i] = e;
}

struct Twiddle1 {
    int nf;
    float c[FDTD_MAX_FREQ], s[FDTD_MAX_FREQ];
};

__global__ void __launch_bounds__(256) fourier1d_kernel(int nx, Twiddle1 tw, const float *ex,
                                                        int probe, float *r_pt, float *i_pt,
                                                        float *r_in, float *i_in)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i == 0 && r_in) {
        const float e = ex[probe];
        for (int f = 0; f < tw.nf; ++f) {
            r_in[f] = r_in[f] + tw.c[f] * e;
            i_in[f] = i_in[f] - tw.s[f] * e;
        }
    }
    if (i >= nx) return;
    const float e = ex[i];
    for (int f = 0; f < tw.nf; ++f) {
        r_pt[(long)f * nx + i] = r_pt[(long)f * nx + i] + tw.c[f] * e;
        i_pt[(long)f * nx + i] = i_pt[(long)f * nx + i] - tw.s[f] * e;
    }
}

// Coefficients of fd1d/clang/test_2_3.c:75-90 (FP32 arithmetic; ncx_val =
// exp(-dt/tau) in double on the host, narrowed): free space below nx/2, the
// medium from nx/2 on.
__global__ void __launch_bounds__(256) debye_kernel(int nx, float dt, float chi, float tau,
                                                    float epsr, float sigma, float ncx_val,
                                                    float *nax, float *nbx, float *ncx, float *ndx)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nx) return;
    const float eps0 = 8.854e-12f;
    if (i < nx / 2) {
        nax[i] = 1.0f;
        nbx[i] = 0.0f;
        if (ncx) { ncx[i] = 0.0f; ndx[i] = 0.0f; }
        return;
    }
    const bool debye = ncx != nullptr;
    const float den = debye ? epsr + sigma * dt / eps0 + chi * dt / tau : epsr + sigma * dt / eps0;
    nax[i] = 1 / den;
    nbx[i] = sigma * dt / eps0;
    if (debye) {
        ncx[i] = ncx_val;
        ndx[i] = chi * dt / tau;
    }
}

// Fused run, as the blocked run of fd1d.hip: a wavefront holds 64 cells, one a
// lane, with every field and coefficient in registers and its neighbours'
// ex, hy by DPP shifts; the waves of a workgroup overlap by twice DF_HALO
// cells and exchange them through LDS every DF_HALO steps; workgroups overlap
// by twice the launch's steps.  A launch reads one state set and writes the
// other (dx ix sx ex hy bc), or works in place when one workgroup holds the
// grid.  The DFT planes and the incident-probe DFT are updated in place by
// their single owner: only the waves that own cells carry them (NF > 0).
// The steps' twiddles and source values go to LDS once a launch.
// Operands as the per-step kernels above, so the bits are theirs.
//
// What bounds it: instruction issue (14 a cell and step, 26 with three
// frequencies, two waves a SIMD).  38000 cells, Debye, three frequencies, 1024
// steps: 1590 us as 32-step launches with the fields in LDS and two barriers a
// step, 202 us now (218 with each row read when it is used).
struct SegD {
    float dx, ix, sx, ex, hy, na, nb, nc, nd;
    float b0, b1, b2, b3;
    int lane, rl, sl, pl;
    unsigned long long pm;
};

// A step's twiddles and source value, read from LDS a step ahead.
struct StepRow { float4 a, b; };

__device__ __forceinline__ StepRow step_row(const float *tab, int s)
{
    const float4 *t = reinterpret_cast<const float4 *>(tab + 8 * s);
    return StepRow{t[0], t[1]};
}

template <bool DEBYE, bool L, bool R, bool SP, int NF>
__device__ __forceinline__ void dform_step(SegD &g, const DformTbParams &P, const StepRow &row, int s,
                                           int pk, int st, bool inc, float (&fr)[NF ? NF : 1],
                                           float (&fi)[NF ? NF : 1], float (&rin)[NF ? NF : 1],
                                           float (&iin)[NF ? NF : 1], float &tr, float *out)
{
    float d = g.dx + 0.5f * (lane_left(g.hy) - g.hy);
    const float c[3] = {row.a.x, row.a.z, row.b.x}, sn[3] = {row.a.y, row.a.w, row.b.y};
    if (SP) {
        const float u = d + row.b.z;
        d = g.lane == g.sl ? u : d;
    }
    float e, ix, sx = g.sx;
    if (DEBYE) {
        e = g.na * (d - g.ix - g.nc * g.sx);
        ix = g.ix + g.nb * e;
        sx = g.nc * g.sx + g.nd * e;
    } else {
        e = g.na * (d - g.ix);
        ix = g.ix + g.nb * e;
    }
    if (L) {                                       // cell 0: no update
        const bool z = g.lane == 0;
        d = z ? g.dx : d;
        ix = z ? g.ix : ix;
        sx = z ? g.sx : sx;
        e = z ? g.ex : e;
    }
    g.dx = d;
    g.ix = ix;
    g.sx = sx;
#pragma unroll
    for (int f = 0; f < NF; ++f) {
        fr[f] = fr[f] + c[f] * e;
        fi[f] = fi[f] - sn[f] * e;
    }
    if (SP && NF > 0 && inc) {
#pragma unroll
        for (int f = 0; f < NF; ++f) {
            rin[f] = rin[f] + c[f] * e;
            iin[f] = iin[f] - sn[f] * e;
        }
    }
    const float e1 = L ? lane_right(e) : 0.f, e2 = R ? lane_left(e) : 0.f;
    if (L) {
        e = g.lane == 0 ? g.b0 : e;
        g.b0 = g.b1;
        g.b1 = e1;
    }
    if (R) {
        e = g.lane == g.rl ? g.b3 : e;
        g.b3 = g.b2;
        g.b2 = e2;
    }
    g.ex = e;
    if (SP && g.pm) {
        const float x = lane_get(e, g.pl);
        tr = g.lane == s ? x : tr;
        for (unsigned long long m = g.pm & (g.pm - 1); m; m &= m - 1) {
            const int p = __builtin_ctzll(m);
            if (g.lane == __builtin_amdgcn_readlane(pk, p) - st) out[(long)p * P.probe_len + s] = e;
        }
    }
    const float w = g.hy + 0.5f * (e - lane_right(e));
    g.hy = R && g.lane == g.rl ? g.hy : w;         // cell nx-1: no update
}

template <bool DEBYE, bool L, bool R, bool SP, int NF>
__device__ __forceinline__ void dform_steps(SegD &g, const DformTbParams &P, const float *tab,
                                            float *xch, int pk, int st, int i, int w0, int w1,
                                            bool many, bool mine)
{
    float fr[NF ? NF : 1], fi[NF ? NF : 1], rin[NF ? NF : 1], iin[NF ? NF : 1];
    const bool own = i >= w0 && i < w1;
    const bool inc = SP && NF > 0 && P.r_in && DF_INC_PROBE >= w0 && DF_INC_PROBE < w1;
#pragma unroll
    for (int f = 0; f < NF; ++f) {
        fr[f] = own ? P.r_pt[(long)f * P.nx + i] : 0.f;
        fi[f] = own ? P.i_pt[(long)f * P.nx + i] : 0.f;
        rin[f] = inc ? P.r_in[f] : 0.f;
        iin[f] = inc ? P.i_in[f] : 0.f;
    }
    const int pf = g.pm ? __builtin_ctzll(g.pm) : 0;
    int flip = 5 * P.region;
    const int chunk = many ? DF_HALO : 64;
    for (int done = 0; done < P.K;) {
        const int n = min(chunk, P.K - done);
        float tr = 0.f;
        float *out = P.probe_out + (P.t_first - 1 + done);
        const float *row = tab + 8 * done;
        int s = 0;
        StepRow r0 = step_row(row, 0), r1;
        // unrolled by hand: the compiler does not unroll loops with lane shifts
#pragma unroll 1
        for (; s + 4 <= n; s += 4) {
            r1 = step_row(row, s + 1);
            dform_step<DEBYE, L, R, SP, NF>(g, P, r0, s, pk, st, inc, fr, fi, rin, iin, tr, out);
            r0 = step_row(row, s + 2);
            dform_step<DEBYE, L, R, SP, NF>(g, P, r1, s + 1, pk, st, inc, fr, fi, rin, iin, tr, out);
            r1 = step_row(row, s + 3);
            dform_step<DEBYE, L, R, SP, NF>(g, P, r0, s + 2, pk, st, inc, fr, fi, rin, iin, tr, out);
            r0 = step_row(row, s + 4);
            dform_step<DEBYE, L, R, SP, NF>(g, P, r1, s + 3, pk, st, inc, fr, fi, rin, iin, tr, out);
        }
#pragma unroll 1
        for (; s < n; ++s) {
            r1 = step_row(row, s + 1);
            dform_step<DEBYE, L, R, SP, NF>(g, P, r0, s, pk, st, inc, fr, fi, rin, iin, tr, out);
            r0 = r1;
        }
        if (SP && g.pm && g.lane < n) out[(long)pf * P.probe_len + g.lane] = tr;
        done += n;
        if (many && done < P.K) {
            if (mine) {
                xch[0] = g.dx;
                xch[P.region] = g.ix;
                if (DEBYE) xch[2 * P.region] = g.sx;
                xch[3 * P.region] = g.ex;
                xch[4 * P.region] = g.hy;
            }
            __syncthreads();
            if (!mine) {
                g.dx = xch[0];
                g.ix = xch[P.region];
                if (DEBYE) g.sx = xch[2 * P.region];
                g.ex = xch[3 * P.region];
                g.hy = xch[4 * P.region];
            }
            xch += flip;
            flip = -flip;
        }
    }
#pragma unroll
    for (int f = 0; f < NF; ++f) {
        if (own) {
            P.r_pt[(long)f * P.nx + i] = fr[f];
            P.i_pt[(long)f * P.nx + i] = fi[f];
        }
        if (inc && i == DF_INC_PROBE) {
            P.r_in[f] = rin[f];
            P.i_in[f] = iin[f];
        }
    }
}

template <bool DEBYE, int NF>
__global__ void __launch_bounds__(64 * DF_WAVES) dform_tb_kernel(const DformTbParams P)
{
    extern __shared__ __align__(16) float sm[];    // steps' table, then the exchange buffers
    const int nx = P.nx, lane = threadIdx.x & 63;
    const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), nw = blockDim.x >> 6;
    const int wg = blockIdx.x;
    const bool last = wg == (int)gridDim.x - 1;
    constexpr int stride = 64 - 2 * DF_HALO;
    const int o0 = wg * P.own, o1 = last ? nx : o0 + P.own;
    const int g0 = max(0, min(o0 - P.depth, nx - P.region));
    const int st = g0 + max(0, min(wv * stride, P.region - 64));
    const int st1 = g0 + max(0, min((wv + 1) * stride, P.region - 64));
    const int i = st + lane;
    const int p0 = wv ? st + DF_HALO : st, p1 = wv + 1 < nw ? st1 + DF_HALO : g0 + P.region;
    const int w0 = max(p0, o0), w1 = min(p1, o1);
    for (int k = threadIdx.x; k < 8 * P.K; k += blockDim.x) sm[k] = P.tab[k / 8][k % 8];
    SegD g;
    g.lane = lane;
    const bool in = i < nx;
    g.dx = in ? P.dx_i[i] : 0.f;
    g.ix = in ? P.ix_i[i] : 0.f;
    g.ex = in ? P.ex_i[i] : 0.f;
    g.hy = in ? P.hy_i[i] : 0.f;
    g.na = in ? P.nax[i] : 0.f;
    g.nb = in ? P.nbx[i] : 0.f;
    g.sx = DEBYE && in ? P.sx_i[i] : 0.f;
    g.nc = DEBYE && in ? P.ncx[i] : 0.f;
    g.nd = DEBYE && in ? P.ndx[i] : 0.f;
    const bool left = st == 0, right = st + 64 >= nx;
    g.rl = nx - 1 - st;
    g.b0 = g.b1 = g.b2 = g.b3 = 0.f;
    if (left) { g.b0 = P.bc_i[0]; g.b1 = P.bc_i[1]; }
    if (right) { g.b2 = P.bc_i[2]; g.b3 = P.bc_i[3]; }
    g.sl = P.src_pos - st;
    const bool src = P.src_pos >= 1 && g.sl >= 0 && g.sl < 64;
    if (!src) g.sl = -1;
    const int pk = lane < P.nprobe ? P.probe_k[lane] : -1;
    g.pm = __builtin_amdgcn_ballot_w64(pk >= w0 && pk < w1);
    g.pl = (__builtin_amdgcn_readlane(pk, g.pm ? __builtin_ctzll(g.pm) : 0) - st) & 63;
    const bool inc = NF > 0 && P.r_in && DF_INC_PROBE >= w0 && DF_INC_PROBE < w1;
    const bool sp = src || g.pm || inc;
    const bool own = w0 < w1;                      // the wave carries DFT planes
    const bool many = nw > 1, mine = i >= p0 && i < p1;
    float *xch = sm + 8 * (DF_MAXK + 1) + (i - g0);
    __syncthreads();
    // every wave passes the same number of barriers (P.K decides)
#define DFORM_RUN(l, r, x, nf) \
    dform_steps<DEBYE, l, r, x, nf>(g, P, sm, xch, pk, st, i, w0, w1, many, mine)
    if (left || right) {
        if (left && right) DFORM_RUN(true, true, true, NF);
        else if (left) DFORM_RUN(true, false, true, NF);
        else DFORM_RUN(false, true, true, NF);
    } else if (sp) {
        DFORM_RUN(false, false, true, NF);
    } else if (NF > 0 && own) {
        DFORM_RUN(false, false, false, NF);
    } else {
        DFORM_RUN(false, false, false, 0);
    }
#undef DFORM_RUN
    // in place: every wave has read its cells before any are written
    if (many) __syncthreads();
    if (i >= w0 && i < w1) {
        P.dx_o[i] = g.dx;
        P.ix_o[i] = g.ix;
        if (DEBYE) P.sx_o[i] = g.sx;
        P.ex_o[i] = g.ex;
        P.hy_o[i] = g.hy;
    }
    if (wg == 0 && left && lane == 0) { P.bc_o[0] = g.b0; P.bc_o[1] = g.b1; }
    if (last && right && lane == g.rl) { P.bc_o[2] = g.b2; P.bc_o[3] = g.b3; }
}

inline int nblk(long n) { return (int)((n + 255) / 256); }

}  // namespace

int preload_dform1d() { return preload_kernel(reinterpret_cast<const void *>(&dxfield_kernel)); }

int launch_dxfield(int nx, float *dx, const float *hy, int src_pos, float src_val, int src_on,
                   hipStream_t s)
{
    hipLaunchKernelGGL(dxfield_kernel, dim3(nblk(nx)), dim3(256), 0, s, nx, dx, hy, src_pos,
                       src_val, src_on);
    return hip_check(hipGetLastError(), "dxfield");
}

int launch_exfield_dform(int nx, const fdtd_medium1d &md, const float *dx, float *ix, float *sx,
                         float *ex, hipStream_t s)
{
    if (md.ncx)
        hipLaunchKernelGGL(exfield_kernel<true>, dim3(nblk(nx)), dim3(256), 0, s, nx, md.nax,
                           md.nbx, md.ncx, md.ndx, dx, ix, sx, ex);
    else
        hipLaunchKernelGGL(exfield_kernel<false>, dim3(nblk(nx)), dim3(256), 0, s, nx, md.nax,
                           md.nbx, md.ncx, md.ndx, dx, ix, sx, ex);
    return hip_check(hipGetLastError(), "exfield (D form)");
}

int launch_fourier1d(int t, int nf, int nx, float dt, const float *freq, const float *ex, int probe,
                     const fdtd_ftrans &ft, hipStream_t s)
{
    Twiddle1 tw{};
    tw.nf = nf;
    for (int f = 0; f < nf; ++f) dft_twiddle(t, freq[f], dt, &tw.c[f], &tw.s[f]);
    hipLaunchKernelGGL(fourier1d_kernel, dim3(nblk(nx)), dim3(256), 0, s, nx, tw, ex, probe,
                       ft.r_pt, ft.i_pt, ft.r_in, ft.i_in);
    return hip_check(hipGetLastError(), "fourier (1-D)");
}

int launch_debye(int nx, float dt, float chi, float tau, float epsr, float sigma,
                 const fdtd_medium1d &md, hipStream_t s)
{
    const float ncx_val = (float)exp((double)(-dt / tau));
    hipLaunchKernelGGL(debye_kernel, dim3(nblk(nx)), dim3(256), 0, s, nx, dt, chi, tau, epsr, sigma,
                       ncx_val, md.nax, md.nbx, md.ncx, md.ndx);
    return hip_check(hipGetLastError(), "dielectric (Debye)");
}

template <bool DEBYE>
static int launch_dform_nf(const DformTbParams &p, int groups, int waves, hipStream_t s)
{
    const size_t lds = sizeof(float) * (8 * (DF_MAXK + 1) + (waves > 1 ? 10 * (size_t)p.region : 0));
    const dim3 grid(groups), nt(64 * waves);
    switch (p.nf) {
    case 0: hipLaunchKernelGGL((dform_tb_kernel<DEBYE, 0>), grid, nt, lds, s, p); break;
    case 1: hipLaunchKernelGGL((dform_tb_kernel<DEBYE, 1>), grid, nt, lds, s, p); break;
    case 2: hipLaunchKernelGGL((dform_tb_kernel<DEBYE, 2>), grid, nt, lds, s, p); break;
    default: hipLaunchKernelGGL((dform_tb_kernel<DEBYE, 3>), grid, nt, lds, s, p); break;
    }
    return hip_check(hipGetLastError(), "fd1d_dform_run launch");
}

int launch_dform_tb(const DformTbParams &p, int groups, int waves, hipStream_t s)
{
    return p.ncx ? launch_dform_nf<true>(p, groups, waves, s) : launch_dform_nf<false>(p, groups, waves, s);
}

}  // namespace fdtd
