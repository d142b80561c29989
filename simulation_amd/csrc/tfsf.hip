// Plane-wave total-field/scattered-field (TF/SF) injection and the running
// DFT of the reference's 2-D TM programs with an incident plane wave
// (fd2d/pycuda/fd2d_3_3.py:80-169, fd2d/pycuda/fd2d_3_4.py:121-226; serial
// semantics as fd2d/clang/test_3_4.c:38-147).
//
// The incident wave is a 1-D grid along y (ezi, hxi, ny cells) with the
// two-step absorbing boundary at both ends; the TF/SF box is rows and
// columns npml-1 .. n-npml.  Per step the reference runs ezinct, dfield (which
// also sets the incident source ezi[3]), inctdz, efield, fourier, hxinct,
// hfield, incthx, incthy; the kernels below are those steps, FP32, in the
// reference's operand order without contraction (bit-exact with its C
// program).  The DFT's twiddles cos/sin(2 pi f dt t) are evaluated on the
// host with the host libm, as the C program evaluates them, and passed to
// the kernel by value.
#include <hip/hip_runtime.h>
#include <math.h>

#include "fdtd_internal.h"
#include "lanes.h"

namespace fdtd {
namespace {

// ezi[j] += 0.5 (hxi[j-1] - hxi[j]) for j in [1, ny), then the two-step
// boundary at both ends (after every update: one workgroup), then the
// incident source (set_inc).
__global__ void __launch_bounds__(1024) ezinct_kernel(int ny, float *ezi, const float *hxi,
                                                      float *bc, int set_inc, int inc_pos,
                                                      float inc_val)
{
    for (int j = threadIdx.x + 1; j < ny; j += blockDim.x) ezi[j] = ezi[j] + 0.5f * (hxi[j - 1] - hxi[j]);
    __syncthreads();
    if (threadIdx.x == 0) {
        ezi[0] = bc[0];
        bc[0] = bc[1];
        bc[1] = ezi[1];
        ezi[ny - 1] = bc[3];
        bc[3] = bc[2];
        bc[2] = ezi[ny - 2];
        if (set_inc) ezi[inc_pos] = inc_val;
    }
}

__global__ void set_kernel(float *p, int pos, float v) { p[pos] = v; }

// hxi[j] += 0.5 (ezi[j] - ezi[j+1]) for j in [0, ny-1)
__global__ void __launch_bounds__(256) hxinct_kernel(int ny, const float *ezi, float *hxi)
{
    const int j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j < ny - 1) hxi[j] = hxi[j] + 0.5f * (ezi[j] - ezi[j + 1]);
}

// dz at columns npml-1 and ny-npml of rows npml-1 .. nx-npml
__global__ void __launch_bounds__(256) inctdz_kernel(int nx, int ny, int npml, const float *hxi,
                                                     float *dz)
{
    const int i = npml - 1 + (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i > nx - npml) return;
    float *row = dz + (size_t)i * ny;
    row[npml - 1] = row[npml - 1] + 0.5f * hxi[npml - 2];
    row[ny - npml] = row[ny - npml] - 0.5f * hxi[ny - npml];
}

// hx at columns npml-2 and ny-npml of rows npml-1 .. nx-npml
__global__ void __launch_bounds__(256) incthx_kernel(int nx, int ny, int npml, const float *ezi,
                                                     float *hx)
{
    const int i = npml - 1 + (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (i > nx - npml) return;
    float *row = hx + (size_t)i * ny;
    row[npml - 2] = row[npml - 2] + 0.5f * ezi[npml - 1];
    row[ny - npml] = row[ny - npml] - 0.5f * ezi[ny - npml];
}

// hy at rows npml-2 and nx-npml of columns npml-1 .. ny-npml
__global__ void __launch_bounds__(256) incthy_kernel(int nx, int ny, int npml, const float *ezi,
                                                     float *hy)
{
    const int j = npml - 1 + (int)(blockIdx.x * blockDim.x + threadIdx.x);
    if (j > ny - npml) return;
    float *a = hy + (size_t)(npml - 2) * ny + j;
    float *b = hy + (size_t)(nx - npml) * ny + j;
    *a = *a - 0.5f * ezi[j];
    *b = *b + 0.5f * ezi[j];
}

struct Twiddle {
    int nf;
    float c[FDTD_MAX_FREQ], s[FDTD_MAX_FREQ];
};

// r_pt[f][m] += c_f ez[m], i_pt[f][m] -= s_f ez[m] (frequency-major planes
// of n cells); the first thread also transforms the incident probe
// ezi[probe] into r_in, i_in.
__global__ void __launch_bounds__(256) fourier_kernel(long n, Twiddle tw, const float *ez,
                                                      const float *ezi, int probe, float *r_pt,
                                                      float *i_pt, float *r_in, float *i_in)
{
    const long m = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (m == 0 && r_in) {
        const float e = ezi[probe];
        for (int f = 0; f < tw.nf; ++f) {
            r_in[f] = r_in[f] + tw.c[f] * e;
            i_in[f] = i_in[f] - tw.s[f] * e;
        }
    }
    if (m >= n) return;
    const float e = ez[m];
    for (int f = 0; f < tw.nf; ++f) {
        r_pt[f * n + m] = r_pt[f * n + m] + tw.c[f] * e;
        i_pt[f * n + m] = i_pt[f * n + m] - tw.s[f] * e;
    }
}

inline int blocks(long n, int b) { return (int)((n + b - 1) / b); }

// The incident grid for a chunk of steps (one workgroup: every phase waits
// for the previous), recording per step what the fused 2-D launches read:
// table[s] = {hxi[npml-2], hxi[ny-npml] (before this step's hxinct),
// ezi[npml-1 .. ny-npml] (after ezinct and the source)}; also the incident
// probe's DFT (r_in, i_in; the reference's fourier after efield).
__global__ void __launch_bounds__(1024) inc_chunk_kernel(int ny, float *ezi, float *hxi, float *bc,
                                                         float *r_in, float *i_in, float *table,
                                                         IncChunk a)
{
    const int tid = threadIdx.x, m = a.npml, nbox = ny - 2 * m + 2;
    for (int s = 0; s < a.n; ++s) {
        for (int j = tid + 1; j < ny; j += blockDim.x) ezi[j] = ezi[j] + 0.5f * (hxi[j - 1] - hxi[j]);
        __syncthreads();
        if (tid == 0) {
            ezi[0] = bc[0];
            bc[0] = bc[1];
            bc[1] = ezi[1];
            ezi[ny - 1] = bc[3];
            bc[3] = bc[2];
            bc[2] = ezi[ny - 2];
            ezi[a.inc_pos] = a.wave[s];
        }
        __syncthreads();
        float *row = table + (size_t)s * a.stride;
        if (tid == 0) {
            row[0] = hxi[m - 2];
            row[1] = hxi[ny - m];
            if (r_in) {
                const float e = ezi[a.probe];
                for (int f = 0; f < a.nf; ++f) {
                    r_in[f] = r_in[f] + a.c[s][f] * e;
                    i_in[f] = i_in[f] - a.s[s][f] * e;
                }
            }
        }
        for (int k = tid; k < nbox; k += blockDim.x) row[2 + k] = ezi[m - 1 + k];
        __syncthreads();
        for (int j = tid; j < ny - 1; j += blockDim.x) hxi[j] = hxi[j] + 0.5f * (ezi[j] - ezi[j + 1]);
        __syncthreads();
    }
}

// The same with the incident grid in registers: a wave holds 64 M cells, M a
// lane, and owns all but the outer INC_HALO on either side it shares with a
// neighbour.  A step then needs DPP shifts only; every INC_HALO steps the
// waves pass their owned edge cells through LDS.  The chunk's source values
// and twiddles sit one step a lane.  What bounds it is the chain of one step
// (some 25 dependent operations) and the two barriers every INC_HALO steps.
// MI355X, ny 1024, three frequencies, 64 steps: 72 us with the grid in LDS
// (four barriers a step, the probe's transforms through memory), 27 us with
// branches around the table's stores, 21 us.
constexpr int INC_HALO = 8;

// LDS traffic done, then the barrier: the table's stores stay in flight
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <int M>
__global__ void __launch_bounds__(1024) inc_chunk_reg_kernel(int ny, float *ezi, float *hxi,
                                                             float *bc, float *r_in, float *i_in,
                                                             float *table, IncChunk a)
{
    constexpr int H = INC_HALO, S = 64 * M;
    // owned edge cells: [wave][left, right][ezi, hxi][cell]
    __shared__ float xch[16][2][2][H];
    const int lane = (int)threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), W = (int)blockDim.x >> 6;
    const int base = w * (S - 2 * H), k0 = lane * M, j0 = base + k0;
    const int o0 = w ? base + H : 0, o1 = w == W - 1 ? ny : base + S - H;
    const int m = a.npml;
    float e[M], h[M];
#pragma unroll
    for (int c = 0; c < M; ++c) {
        const int j = min(j0 + c, ny - 1);
        e[c] = ezi[j];
        h[c] = hxi[j];
    }
    float b0 = bc[0], b1 = bc[1], b2 = bc[2], b3 = bc[3];
    float wv = 0.f, twc[TB_MAX_FREQ], tws[TB_MAX_FREQ], ri[TB_MAX_FREQ], ii[TB_MAX_FREQ];
    static_assert(INC_CHUNK <= 64, "one step a lane");
    if (lane < a.n) wv = a.wave[lane];
    const bool dft = r_in && a.probe >= o0 && a.probe < o1;      // the wave owns the probe
#pragma unroll
    for (int f = 0; f < TB_MAX_FREQ; ++f) {
        twc[f] = tws[f] = ri[f] = ii[f] = 0.f;
        if (dft && f < a.nf) {
            if (lane < a.n) { twc[f] = a.c[lane][f]; tws[f] = a.s[lane][f]; }
            ri[f] = r_in[f];
            ii[f] = i_in[f];
        }
    }
    const bool src = a.inc_pos >= base && a.inc_pos < base + S;
    const bool right = ny - 1 < base + S;                        // the window holds cell ny-1
    // a step's table row: byte offsets of the lane's cells in it, past its end
    // where a cell is not the wave's to store (the range check drops those:
    // no branches in a step)
    unsigned eoff[M], hoff[M];
#pragma unroll
    for (int c = 0; c < M; ++c) {
        const int j = j0 + c;
        const bool own = j >= o0 && j < o1;
        eoff[c] = own && j >= m - 1 && j <= ny - m ? (unsigned)(2 + j - (m - 1)) * 4u : 0xFFFFFFFCu;
        hoff[c] = own && j == m - 2 ? 0u : own && j == ny - m ? 4u : 0xFFFFFFFCu;
    }
    const bool side = (m - 2 >= o0 && m - 2 < o1) || (ny - m >= o0 && ny - m < o1);
    // cell j's value (in the window), in every lane
    auto cell = [&](const float (&v)[M], int j) __attribute__((always_inline)) {
        const int k = j - base;
        float x = v[0];
#pragma unroll
        for (int c = 1; c < M; ++c) x = k % M == c ? v[c] : x;
        return lane_get(x, k / M);
    };
#pragma unroll 1
    for (int s = 0; s < a.n; ++s) {
        const float hl = lane_left(h[M - 1]);
#pragma unroll
        for (int c = M - 1; c >= 0; --c) e[c] = e[c] + 0.5f * ((c ? h[c ? c - 1 : 0] : hl) - h[c]);
        // two-step boundary (it replaces cells 0 and ny-1), then the source
        if (w == 0) {
            e[0] = lane == 0 ? b0 : e[0];
            b0 = b1;
            b1 = cell(e, 1);
        }
        if (right) {
#pragma unroll
            for (int c = 0; c < M; ++c) e[c] = j0 + c == ny - 1 ? b3 : e[c];
            b3 = b2;
            b2 = cell(e, ny - 2);
        }
        if (src) {
            const float v = lane_get(wv, s);
#pragma unroll
            for (int c = 0; c < M; ++c) e[c] = j0 + c == a.inc_pos ? v : e[c];
        }
        const auto row = __builtin_amdgcn_make_buffer_rsrc(table + (size_t)s * a.stride, (short)0,
                                                           a.stride * 4, 0x00020000);
#pragma unroll
        for (int c = 0; c < M; ++c)
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, e[c]), row, eoff[c], 0, 0);
        if (side) {
#pragma unroll
            for (int c = 0; c < M; ++c)
                __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, h[c]), row, hoff[c], 0, 0);
        }
        if (dft) {
            const float v = cell(e, a.probe);
#pragma unroll
            for (int f = 0; f < TB_MAX_FREQ; ++f) {
                ri[f] = ri[f] + lane_get(twc[f], s) * v;
                ii[f] = ii[f] - lane_get(tws[f], s) * v;
            }
        }
        const float er = lane_right(e[0]);
#pragma unroll
        for (int c = 0; c < M; ++c) {
            const float v = h[c] + 0.5f * (e[c] - (c + 1 < M ? e[c + 1 < M ? c + 1 : 0] : er));
            h[c] = j0 + c == ny - 1 ? h[c] : v;
        }
        if (W > 1 && s % H == H - 1) {
#pragma unroll
            for (int c = 0; c < M; ++c) {
                const int k = k0 + c;
                if (k >= H && k < 2 * H) { xch[w][0][0][k - H] = e[c]; xch[w][0][1][k - H] = h[c]; }
                if (k >= S - 2 * H && k < S - H) {
                    xch[w][1][0][k - (S - 2 * H)] = e[c];
                    xch[w][1][1][k - (S - 2 * H)] = h[c];
                }
            }
            lds_barrier();
#pragma unroll
            for (int c = 0; c < M; ++c) {
                const int k = k0 + c;
                if (w > 0 && k < H) { e[c] = xch[w - 1][1][0][k]; h[c] = xch[w - 1][1][1][k]; }
                if (w < W - 1 && k >= S - H) {
                    e[c] = xch[w + 1][0][0][k - (S - H)];
                    h[c] = xch[w + 1][0][1][k - (S - H)];
                }
            }
            lds_barrier();
        }
    }
    // in place: every wave has read its cells (and bc) before any are written
    if (W > 1) __syncthreads();
#pragma unroll
    for (int c = 0; c < M; ++c) {
        const int j = j0 + c;
        if (j >= o0 && j < o1) { ezi[j] = e[c]; hxi[j] = h[c]; }
    }
    if (lane == 0) {
        if (w == 0) { bc[0] = b0; bc[1] = b1; }
        if (w == W - 1) { bc[2] = b2; bc[3] = b3; }
        if (dft) {
#pragma unroll
            for (int f = 0; f < TB_MAX_FREQ; ++f)
                if (f < a.nf) { r_in[f] = ri[f]; i_in[f] = ii[f]; }
        }
    }
}

// Launches the register form with M cells a lane if 16 waves hold ny cells.
template <int M>
bool inc_chunk_reg(int ny, float *ezi, float *hxi, float *bc, float *r_in, float *i_in,
                   float *table, const IncChunk &a, hipStream_t s)
{
    constexpr int S = 64 * M, O = S - 2 * INC_HALO;
    const int waves = ny <= S ? 1 : 1 + (ny - S + O - 1) / O;
    if (waves > 16) return false;
    hipLaunchKernelGGL((inc_chunk_reg_kernel<M>), dim3(1), dim3(64 * waves), 0, s, ny, ezi, hxi, bc,
                       r_in, i_in, table, a);
    return true;
}

}  // namespace

int preload_tfsf() { return preload_kernel(reinterpret_cast<const void *>(&set_kernel)); }

int launch_inc_chunk(int ny, float *ezi, float *hxi, float *bc, float *r_in, float *i_in,
                     float *table, const IncChunk &a, hipStream_t s)
{
    // the fewest cells a lane that 16 waves allow; past 16144 cells (and on
    // grids whose two ends share cells) the form in global memory
    if (ny < 4 || !(inc_chunk_reg<1>(ny, ezi, hxi, bc, r_in, i_in, table, a, s) ||
                    inc_chunk_reg<2>(ny, ezi, hxi, bc, r_in, i_in, table, a, s) ||
                    inc_chunk_reg<4>(ny, ezi, hxi, bc, r_in, i_in, table, a, s) ||
                    inc_chunk_reg<8>(ny, ezi, hxi, bc, r_in, i_in, table, a, s) ||
                    inc_chunk_reg<16>(ny, ezi, hxi, bc, r_in, i_in, table, a, s)))
        hipLaunchKernelGGL(inc_chunk_kernel, dim3(1), dim3(1024), 0, s, ny, ezi, hxi, bc, r_in, i_in,
                           table, a);
    return hip_check(hipGetLastError(), "incident chunk");
}

// The reference's twiddle: cosf/sinf of 2*M_PI*freq*dt*t evaluated in double
// and narrowed to float (fd2d/clang/test_3_4.c:42-43).
void dft_twiddle(int t, float freq, float dt, float *c, float *s)
{
    const float a = (float)(2 * M_PI * (double)freq * (double)dt * (double)t);
    *c = cosf(a);
    *s = sinf(a);
}

int launch_ezinct(int ny, float *ezi, const float *hxi, float *bc, int set_inc, int inc_pos,
                  float inc_val, hipStream_t s)
{
    hipLaunchKernelGGL(ezinct_kernel, dim3(1), dim3(1024), 0, s, ny, ezi, hxi, bc, set_inc, inc_pos,
                       inc_val);
    return hip_check(hipGetLastError(), "ezinct");
}

int launch_set(float *p, int pos, float v, hipStream_t s)
{
    hipLaunchKernelGGL(set_kernel, dim3(1), dim3(1), 0, s, p, pos, v);
    return hip_check(hipGetLastError(), "incident source");
}

int launch_hxinct(int ny, const float *ezi, float *hxi, hipStream_t s)
{
    hipLaunchKernelGGL(hxinct_kernel, dim3(blocks(ny, 256)), dim3(256), 0, s, ny, ezi, hxi);
    return hip_check(hipGetLastError(), "hxinct");
}

int launch_inctdz(int nx, int ny, int npml, const float *hxi, float *dz, hipStream_t s)
{
    hipLaunchKernelGGL(inctdz_kernel, dim3(blocks(nx - 2 * npml + 2, 256)), dim3(256), 0, s, nx, ny,
                       npml, hxi, dz);
    return hip_check(hipGetLastError(), "inctdz");
}

int launch_incthx(int nx, int ny, int npml, const float *ezi, float *hx, hipStream_t s)
{
    hipLaunchKernelGGL(incthx_kernel, dim3(blocks(nx - 2 * npml + 2, 256)), dim3(256), 0, s, nx, ny,
                       npml, ezi, hx);
    return hip_check(hipGetLastError(), "incthx");
}

int launch_incthy(int nx, int ny, int npml, const float *ezi, float *hy, hipStream_t s)
{
    hipLaunchKernelGGL(incthy_kernel, dim3(blocks(ny - 2 * npml + 2, 256)), dim3(256), 0, s, nx, ny,
                       npml, ezi, hy);
    return hip_check(hipGetLastError(), "incthy");
}

int launch_fourier(int t, int nf, int nx, int ny, float dt, const float *freq, const float *ezi,
                   int probe, const float *ez, const fdtd_ftrans &ft, hipStream_t s)
{
    Twiddle tw{};
    tw.nf = nf;
    for (int f = 0; f < nf; ++f) dft_twiddle(t, freq[f], dt, &tw.c[f], &tw.s[f]);
    const long n = (long)nx * ny;
    hipLaunchKernelGGL(fourier_kernel, dim3(blocks(n, 256)), dim3(256), 0, s, n, tw, ez, ezi, probe,
                       ft.r_pt, ft.i_pt, ft.r_in, ft.i_in);
    return hip_check(hipGetLastError(), "fourier");
}

}  // namespace fdtd
