// fd2d_rt.hip -- fused 2-D TM time stepping of small grids: register tiles
// (gfx950).
//
// One launch advances the grid by K leapfrog steps (K a run-time number).
// Semantics per step are those of the reference's per-step kernels dfield ->
// hard source -> efield -> hfield (fd2d/pycuda/fd2d_3_2.py:219-260,
// fd2d/pycuda/fd2d_3_4.py:175-226 with the plane wave and the running DFT),
// operand for operand: the bits of tm_tb_kernel (fd2d_tb_impl.h).
//
// Why another form.  tm_tb_kernel's wave sweeps a strip row by row through K
// levels: a launch lasts (rows + 2K) positions of K dependent levels however
// few tiles there are, and short row blocks recompute 2K warm-up rows each.
// That pays on grids that fill the chip with tall strips; on a grid of up to
// some 1600 cells a side it leaves most SIMDs idle or busy with warm-up rows.
//
// Here a workgroup of up to 16 waves holds a tile of 64 columns by waves * R
// rows in registers for the whole launch: a wave has R = 4 rows, one column a
// lane, every field and coefficient of its cells in VGPRs.  Columns beside a
// lane's come by DPP shifts, the rows above and below a wave's from LDS (one
// row of hy down, one row of ez up), so a step costs two barriers and no
// memory.  Tiles overlap by K cells on either side of the cut they share
// (recomputed, never written twice).  Waves whose rows have left the cone of
// the tile's own rows skip the rest of the launch's steps but their barriers.
// Two rows a wave, 16 waves (the same tile) measured within 6%; eight rows
// spill and lose on every grid.
//
// Two bodies a wave chooses from: rows and columns inside the band of default
// profile values (constants, no edge tests; the terms 0 * ihx and 0 * ihy
// left out as in tm_tb_kernel), or the general one.
//
// What bounds it: on small grids the step itself (about 0.7 us a step for a
// 32-row tile at two waves a SIMD: instruction issue, then the two barriers)
// and some 4 us a launch for the loads, stores and the gap; from 1000^2 on
// the overlap (a third to a half of the cells computed) and the tiles' loads.
// MI355X, strips before -> tiles, 192 steps, lossy, npml 8: 100^2 1055 -> 190
// us, 400^2 1070 -> 235, 700^2 1085 -> 308, 1024^2 1120 -> 563, 1600^2 1181
// -> 1050.
#include "fdtd_internal.h"
#include "lanes.h"

#include <climits>

namespace fdtd {
namespace {

using gfloat = const __attribute__((address_space(1))) float;
using cfloat = const __attribute__((address_space(4))) float;

__device__ __forceinline__ float ldg(const float *p, unsigned i) { return ((gfloat *)p)[i]; }
// a row's profile value: a scalar load (the same index in every lane)
__device__ __forceinline__ float ldu(const float *p, int i)
{
    return ((cfloat *)p)[__builtin_amdgcn_readfirstlane(i)];
}
// LDS traffic done, then the barrier (global loads and stores stay in flight)
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <int N> struct Int { static constexpr int v = N; };

constexpr int R = RT_ROWS;

struct RtSmem {
    float up[RT_WAVES + 1][64];   // up[w]: hy of the row above wave w's first
    float dn[RT_WAVES + 1][64];   // dn[w]: ez of wave w's first row
    float src[FDTD_MAX_SOURCES * RT_MAX_STEPS];
};

// Tiles along n cells: spans of `span` cells that share 2H with each neighbour.
__host__ __device__ inline int rt_along(int n, int span, int H)
{
    return n <= span ? 1 : 1 + (n - span + span - 2 * H - 1) / (span - 2 * H);
}

// Tile (by, bx) of nsy x nsx, P.K steps; H >= P.K: the overlap the tiles are
// cut with.  PR: RtParams or RtGrid.
// SPLIT: one copy of the step loop per body.  Choosing the body again in every
// phase took a seventh of a step (MI355X, 192 steps: 60^2 215 -> 185 us, 400^2
// 265 -> 231, 1024^2 617 -> 563; plane wave 1024^2, three frequencies, 256
// steps 1692 -> 1428), but the copies take 95 registers a lane instead of 78:
// a batch of many tiles, which lives by three 8-wave or two 12-wave tiles a
// CU, keeps the one loop (112 steps: 4.5 million cells 1563 us, 1870 split).
template <bool LOSSY, bool PML, bool TF, int NF, bool SPLIT, class PR>
__device__ __forceinline__ void rt_tile(PR &P, int H, int bx, int by, int nsx, int nsy,
                                        RtSmem &S)
{
    auto &up = S.up;
    auto &dn = S.dn;
    auto &srcv = S.src;
    const int nx = P.nx, ny = P.ny, K = P.K;
    const int W = (int)blockDim.x >> 6, T = W * R;
    const int lane = (int)threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    // the tile's window starts at (bi, bj) -- the last one of a row or column
    // ends with the grid -- and its own cells are rows [o0, o1), columns [c0, c1)
    const int bi = min(by * (T - 2 * H), max(nx - T, 0));
    const int bj = min(bx * (64 - 2 * H), max(ny - 64, 0));
    const int o0 = by ? by * (T - 2 * H) + H : 0, o1 = by == nsy - 1 ? nx : by * (T - 2 * H) + T - H;
    const int c0 = bx ? bx * (64 - 2 * H) + H : 0, c1 = bx == nsx - 1 ? ny : bx * (64 - 2 * H) + 64 - H;
    const int i0 = bi + w * R, j = bj + lane, jc = min(j, ny - 1);
    const bool own_col = j >= c0 && j < c1;

    float dz[R], iz[LOSSY ? R : 1], hx[R], hy[R], ax[PML ? R : 1], ay[PML ? R : 1];
    float na[R], nb[LOSSY ? R : 1], e[R];
    float fr[NF ? NF : 1][R], fi[NF ? NF : 1][R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const unsigned o = (unsigned)min(i0 + r, nx - 1) * (unsigned)ny + (unsigned)jc;
        dz[r] = ldg(P.dz_i, o);
        hx[r] = ldg(P.hx_i, o);
        hy[r] = ldg(P.hy_i, o);
        na[r] = ldg(P.naz, o);
        if constexpr (LOSSY) { iz[r] = ldg(P.iz_i, o); nb[r] = ldg(P.nbz, o); }
        if constexpr (PML) { ax[r] = ldg(P.ihx_i, o); ay[r] = ldg(P.ihy_i, o); }
        e[r] = 0.f;
        if constexpr (NF > 0) {
            // planes are read and written by the cell's owner alone
            const bool own = own_col && i0 + r >= o0 && i0 + r < o1;
            const size_t plane = (size_t)nx * (size_t)ny;
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                fr[f][r] = own ? ldg(P.ft_r + f * plane, o) : 0.f;
                fi[f][r] = own ? ldg(P.ft_i + f * plane, o) : 0.f;
            }
        }
    }
    // profile values: columns in lanes, rows in scalar registers
    float gy2 = 1.f, gy3 = 1.f, fy1 = 0.f, fy2 = 1.f, fy3 = 1.f;
    float gx2[R], gx3[R], fx1[R], fx2[R], fx3[R];
    if constexpr (PML) {
        gy2 = ldg(P.pml.gy2, jc); gy3 = ldg(P.pml.gy3, jc);
        fy1 = ldg(P.pml.fy1, jc); fy2 = ldg(P.pml.fy2, jc); fy3 = ldg(P.pml.fy3, jc);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int i = min(i0 + r, nx - 1);
            gx2[r] = ldu(P.pml.gx2, i); gx3[r] = ldu(P.pml.gx3, i);
            fx1[r] = ldu(P.pml.fx1, i); fx2[r] = ldu(P.pml.fx2, i); fx3[r] = ldu(P.pml.fx3, i);
        }
    }
    const bool plain = i0 >= P.rlo && i0 + R <= P.rhi && bj >= P.clo && bj + 64 <= P.chi;
    const bool rows_own = i0 < o1 && i0 + R > o0;

    // sources and probes of the wave's cells: one a lane (row, column), and
    // those the wave has as a mask
    int sp_row = INT_MIN, sp_col = INT_MIN;
    if (lane < P.nsrc) {
        sp_row = P.src_i[lane]; sp_col = P.src_j[lane];
    } else if (lane >= FDTD_MAX_SOURCES && lane < FDTD_MAX_SOURCES + P.nprobe) {
        sp_row = P.probe_i[lane - FDTD_MAX_SOURCES]; sp_col = P.probe_j[lane - FDTD_MAX_SOURCES];
    }
    unsigned long long spm;
    {
        const bool in = sp_row >= i0 && sp_row < i0 + R && sp_col >= bj && sp_col < bj + 64;
        const bool mine = sp_row >= o0 && sp_row < o1 && sp_col >= c0 && sp_col < c1;
        spm = __builtin_amdgcn_ballot_w64(in && (lane < FDTD_MAX_SOURCES || mine));
    }
    const unsigned smask = (unsigned)spm & ((1u << FDTD_MAX_SOURCES) - 1u);
    const unsigned pmask = (unsigned)(spm >> FDTD_MAX_SOURCES);
    for (int k = (int)threadIdx.x; k < P.nsrc * K; k += (int)blockDim.x)
        srcv[k] = P.src_wave[(size_t)(k / K) * P.wave_len + (P.t_first - 1 + k % K)];
    // plane wave: whether the wave holds cells the TF/SF box corrects; the
    // step's four column values sit in lanes 0 .. 3, the row values one a
    // lane, both loaded a step ahead
    const int m = TF ? P.tf_npml : 0;
    bool tfw = false;
    float tfv = 0.f, tfr = 0.f;
    if constexpr (TF) {
        auto col_in = [&](int c) { return c >= bj && c < bj + 64; };
        auto row_in = [&](int i) { return i >= i0 && i < i0 + R; };
        tfw = i0 + R > m - 2 && i0 <= nx - m &&
              (col_in(m - 2) || col_in(m - 1) || col_in(ny - m) || row_in(m - 2) || row_in(nx - m));
    }
    auto load_tf = [&](int s) __attribute__((always_inline)) {
        const float *iv = P.inc + (size_t)(P.t_first + s - P.inc_t0 - 1) * P.inc_stride;
        tfv = ldg(iv, lane < 3 ? lane : 3 + ny - 2 * m);
        tfr = ldg(iv, (unsigned)(2 + min(max(j, m - 1), ny - m) - (m - 1)));
    };
    if (TF && tfw) load_tf(0);

    up[w + 1][lane] = hy[R - 1];
    if (w == 0) {
        up[0][lane] = 0.f;
        dn[W][lane] = 0.f;
    }
    lds_barrier();

    const bool colD = j >= 1, colH = j <= ny - 2;
    // D, source, E of the wave's rows; hu: hy of the row above
    auto e_phase = [&](auto G, auto SP, int s, float hu) __attribute__((always_inline)) {
        auto d_row = [&](int r, float hl) __attribute__((always_inline)) {
            const float hp = r ? hy[r ? r - 1 : 0] : hu;
            const float curl = hy[r] - hp - hx[r] + hl;
            if (PML && G.v) dz[r] = gx3[r] * gy3 * dz[r] + gx2[r] * gy2 * 0.5f * curl;
            else dz[r] = dz[r] + 0.5f * curl;
        };
        if (G.v) {
            // row 0 and column 0 have no update: one region of masked lanes
            // for all rows (a select per value costs more, and the compiler
            // makes a branch per row of it); the shifts need every lane
            float hl[R];
#pragma unroll
            for (int r = 0; r < R; ++r) hl[r] = lane_left(hx[r]);
            if (colD) {
#pragma unroll
                for (int r = R - 1; r >= 1; --r) d_row(r, hl[r]);
                if (i0 >= 1) d_row(0, hl[0]);
            }
        } else {
#pragma unroll
            for (int r = R - 1; r >= 0; --r) d_row(r, lane_left(hx[r]));
        }
        if (SP.v) {
            for (unsigned mk = smask; mk; mk &= mk - 1u) {
                const int k = __builtin_ctz(mk);
                const int rk = __builtin_amdgcn_readlane(sp_row, k) - i0;
                const bool at = j == __builtin_amdgcn_readlane(sp_col, k);
                const float v = srcv[k * K + s];
#pragma unroll
                for (int r = 0; r < R; ++r) dz[r] = at && r == rk ? v : dz[r];
            }
            if (TF && tfw) {
                const float h0 = lane_get(tfv, 0), h1 = lane_get(tfv, 1);
#pragma unroll
                for (int r = 0; r < R; ++r)
                    if (i0 + r >= m - 1 && i0 + r <= nx - m) {
                        if (j == m - 1) dz[r] = dz[r] + 0.5f * h0;
                        if (j == ny - m) dz[r] = dz[r] - 0.5f * h1;
                    }
            }
        }
#pragma unroll
        for (int r = R - 1; r >= 0; --r) {
            if constexpr (LOSSY) {
                e[r] = na[r] * (dz[r] - iz[r]);
                iz[r] = iz[r] + nb[r] * e[r];
            } else {
                e[r] = na[r] * dz[r];
            }
        }
        dn[w][lane] = e[0];
        if constexpr (NF > 0) {
            if (rows_own) {
#pragma unroll
                for (int f = 0; f < NF; ++f) {
                    const float c = P.tw[s][f], sn = P.tw[s][TB_MAX_FREQ + f];
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        fr[f][r] = fr[f][r] + c * e[r];
                        fi[f][r] = fi[f][r] - sn * e[r];
                    }
                }
            }
        }
        for (unsigned mk = SP.v ? pmask : 0u; mk; mk &= mk - 1u) {
            const int k = __builtin_ctz(mk);
            const int rk = __builtin_amdgcn_readlane(sp_row, FDTD_MAX_SOURCES + k) - i0;
            float v = e[0];
#pragma unroll
            for (int r = 1; r < R; ++r) v = r == rk ? e[r] : v;
            if (j == __builtin_amdgcn_readlane(sp_col, FDTD_MAX_SOURCES + k))
                P.probe_out[(size_t)k * P.probe_len + (P.t_first + s - 1)] = v;
        }
    };
    // H of the wave's rows; ed: ez of the row below
    auto h_phase = [&](auto G, auto SP, int s, float ed) __attribute__((always_inline)) {
        auto h_row = [&](int r, float eR, float heR) __attribute__((always_inline)) {
            const float ez = e[r], eD = r + 1 < R ? e[r + 1 < R ? r + 1 : 0] : ed;
            const float he = 0.5f * ez;
            if (PML && !G.v) {
                // profile values at their defaults: 0 * ihx and 0 * ihy add
                // nothing (tm_tb_kernel has the argument)
                ax[r] = ax[r] + (ez - eR);
                ay[r] = ay[r] + (ez - eD);
                hx[r] = hx[r] + (he - heR);
                hy[r] = hy[r] - (he - 0.5f * eD);
            } else if constexpr (PML) {
                ax[r] = ax[r] + (ez - eR);
                ay[r] = ay[r] + (ez - eD);
                hx[r] = fy3 * hx[r] + fy2 * (he - 0.5f * eR + fx1[r] * ax[r]);
                hy[r] = fx3[r] * hy[r] - fx2[r] * (he - 0.5f * eD + fy1 * ay[r]);
            } else {
                hx[r] = hx[r] + 0.5f * (ez - eR);
                hy[r] = hy[r] - 0.5f * (ez - eD);
            }
        };
        if (G.v) {
            // row nx-1 and column ny-1 have no update
            float eR[R];
#pragma unroll
            for (int r = 0; r < R; ++r) eR[r] = lane_right(e[r]);
            if (colH) {
                if (i0 + R <= nx - 1) {
#pragma unroll
                    for (int r = 0; r < R; ++r) h_row(r, eR[r], 0.f);
                } else {
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        if (i0 + r <= nx - 2) h_row(r, eR[r], 0.f);
                }
            }
        } else {
            // 0.5 * (right ez) is the right lane's 0.5 * ez, shifted as it is
#pragma unroll
            for (int r = 0; r < R; ++r) h_row(r, lane_right(e[r]), PML ? lane_right(0.5f * e[r]) : 0.f);
        }
        if (SP.v && TF && tfw) {
            const float e0 = lane_get(tfv, 2), e1 = lane_get(tfv, 3);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int i = i0 + r;
                if (i >= m - 1 && i <= nx - m) {
                    if (j == m - 2) hx[r] = hx[r] + 0.5f * e0;
                    if (j == ny - m) hx[r] = hx[r] - 0.5f * e1;
                }
                if (i == m - 2 || i == nx - m) {
                    const float sgn = i == nx - m ? 0.5f : -0.5f;
                    if (j >= m - 1 && j <= ny - m) hy[r] = hy[r] + sgn * tfr;
                }
            }
            if (s + 1 < K) load_tf(s + 1);
        }
        up[w + 1][lane] = hy[R - 1];
    };
    // steps in which a later own cell depends on the wave's rows (those within
    // K-s of [o0, o1) at step s); in the others it only keeps the barriers
    const int nact = i0 >= nx ? 0 : max(0, min(K, K - max(o0 - i0 - R, i0 - o1)));
    auto steps = [&](auto G, auto SP) __attribute__((always_inline)) {
#pragma unroll 1
        for (int s = 0; s < nact; ++s) {
            e_phase(G, SP, s, up[w][lane]);
            lds_barrier();
            h_phase(G, SP, s, dn[w + 1][lane]);
            lds_barrier();
        }
    };
    const bool sp = smask || pmask || tfw;
    // every wave passes the same number of barriers (K decides)
    if constexpr (SPLIT) {
        if (sp) steps(Int<1>{}, Int<1>{});
        else if (plain) steps(Int<0>{}, Int<0>{});
        else steps(Int<1>{}, Int<0>{});
    } else {
#pragma unroll 1
        for (int s = 0; s < nact; ++s) {
            const float hu = up[w][lane];
            if (sp) e_phase(Int<1>{}, Int<1>{}, s, hu);
            else if (plain) e_phase(Int<0>{}, Int<0>{}, s, hu);
            else e_phase(Int<1>{}, Int<0>{}, s, hu);
            lds_barrier();
            const float ed = dn[w + 1][lane];
            if (sp) h_phase(Int<1>{}, Int<1>{}, s, ed);
            else if (plain) h_phase(Int<0>{}, Int<0>{}, s, ed);
            else h_phase(Int<1>{}, Int<0>{}, s, ed);
            lds_barrier();
        }
    }
#pragma unroll 1
    for (int s = nact; s < K; ++s) {
        lds_barrier();
        lds_barrier();
    }
    if (!rows_own || !own_col) return;
    P.outputs();
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int i = i0 + r;
        if (i < o0 || i >= o1) continue;
        const unsigned o = (unsigned)i * (unsigned)ny + (unsigned)j;
        P.dz_o[o] = dz[r];
        P.hx_o[o] = hx[r];
        P.hy_o[o] = hy[r];
        if constexpr (LOSSY) P.iz_o[o] = iz[r];
        if constexpr (PML) { P.ihx_o[o] = ax[r]; P.ihy_o[o] = ay[r]; }
        if (P.ez_o) P.ez_o[o] = e[r];
        if constexpr (NF > 0) {
            const size_t plane = (size_t)nx * (size_t)ny;
#pragma unroll
            for (int f = 0; f < NF; ++f) {
                P.ft_r[f * plane + o] = fr[f][r];
                P.ft_i[f * plane + o] = fi[f][r];
            }
        }
    }
}

// workgroup b of n runs on XCD b % 8: the workgroups of one XCD take a
// contiguous run of tiles, which share their halos in its L2
__device__ __forceinline__ unsigned rt_slot(unsigned b, unsigned n)
{
    const unsigned xcd = b % 8u;
    return xcd * (n / 8u) + min(xcd, n % 8u) + b / 8u;
}

template <bool LOSSY, bool PML, bool TF, int NF>
__global__ void __launch_bounds__(64 * RT_WAVES) tm_rt_kernel(const RtParams P)
{
    __shared__ RtSmem S;
    const unsigned tile = rt_slot(blockIdx.x, gridDim.x), nsx = (unsigned)P.nsx;
    rt_tile<LOSSY, PML, TF, NF, true>(P, P.K, (int)(tile % nsx), (int)(tile / nsx), P.nsx,
                                (int)(gridDim.x / nsx), S);
}

// One grid of a batch (fd2d_grid): at most one source and one probe.
struct RtGrid {
    const fd2d_grid *g;
    bool swap, write_ez;            // odd launches read the partner set
    int nx, ny, K;
    const float *dz_i, *iz_i, *hx_i, *hy_i, *ihx_i, *ihy_i;
    float *dz_o, *iz_o, *hx_o, *hy_o, *ihx_o, *ihy_o, *ez_o;
    const float *naz, *nbz;
    PmlPtrs pml;
    int rlo, rhi, clo, chi;
    int t_first;
    struct One {
        int v;
        __device__ int operator[](int) const { return v; }
    };
    int nsrc;
    One src_i, src_j;
    const float *src_wave;
    int wave_len;
    int nprobe;
    One probe_i, probe_j;
    float *probe_out;
    int probe_len;
    static constexpr int tf_npml = 0, inc_t0 = 0, inc_stride = 0;
    static constexpr const float *inc = nullptr;
    // read from the record when the steps are done: kept over them, the
    // pointers cost 26 scalar registers, which spill into vector ones (88 of
    // those a lane instead of 80: two tiles a CU instead of three)
    __device__ __forceinline__ void outputs()
    {
        asm volatile("" : "+s"(g));
        dz_o = swap ? g->dz : g->dz2;
        iz_o = swap ? g->iz : g->iz2;
        hx_o = swap ? g->hx : g->hx2;
        hy_o = swap ? g->hy : g->hy2;
        ihx_o = swap ? g->ihx : g->ihx2;
        ihy_o = swap ? g->ihy : g->ihy2;
        ez_o = write_ez ? g->ez : nullptr;
    }
};

// Many grids, one workgroup a tile or fewer that take several; units: grid,
// tile column, tile row of tiles cut for H steps.  CUT: a launch of fewer steps
// K cuts its own, as a single grid's does; the units left without a tile lie
// evenly among the others, for at the end of a grid's they would idle whole
// XCDs.  An instance of its own: the map spills scalars of the step loop.
// MI355X, two launches of one step, cut for 8 steps / for one: 200 grids of
// 150^2 179 / 160 us, 100 of 30x1000 100 / 78 (with 12 / 8 waves a tile).
// Lossy PML form.  Six waves a SIMD: two 12-wave tiles a CU.
template <bool CUT>
__global__ void __launch_bounds__(64 * RT_WAVES) __attribute__((amdgpu_waves_per_eu(6)))
tm_rt_batch_kernel(const fd2d_grid *__restrict__ grids, const int *__restrict__ units, int nunits,
                   int K, int H, int parity, int t_first, int write_ez)
{
    __shared__ RtSmem S;
    const int T = ((int)blockDim.x >> 6) * R;
    for (int u = (int)rt_slot(blockIdx.x, gridDim.x); u < nunits; u += (int)gridDim.x) {
        const fd2d_grid &G = grids[units[4 * u]];
        int bx = units[4 * u + 1], by = units[4 * u + 2];
        int nsx = rt_along(G.ny, 64, H), nsy = rt_along(G.nx, T, H);
        if constexpr (CUT) {
            const long long q = (long long)by * nsx + bx, listed = (long long)nsx * nsy;
            nsx = rt_along(G.ny, 64, K);
            nsy = rt_along(G.nx, T, K);
            const long long n = (long long)nsx * nsy;
            const int tile = (int)(q * n / listed);
            if (tile == (int)((q + 1) * n / listed)) continue;
            by = tile / nsx;
            bx = tile % nsx;
        }
        RtGrid P;
        P.g = &G;
        P.swap = parity != 0;
        P.write_ez = write_ez != 0;
        P.nx = G.nx; P.ny = G.ny; P.K = K;
        P.dz_i = P.swap ? G.dz2 : G.dz;
        P.iz_i = P.swap ? G.iz2 : G.iz;
        P.hx_i = P.swap ? G.hx2 : G.hx;
        P.hy_i = P.swap ? G.hy2 : G.hy;
        P.ihx_i = P.swap ? G.ihx2 : G.ihx;
        P.ihy_i = P.swap ? G.ihy2 : G.ihy;
        P.naz = G.md.naz; P.nbz = G.md.nbz;
        P.pml = PmlPtrs{G.pml.fx1, G.pml.fx2, G.pml.fx3, G.pml.fy1, G.pml.fy2, G.pml.fy3,
                        G.pml.gx2, G.pml.gx3, G.pml.gy2, G.pml.gy3};
        const int *br = G.band_rows, *bc = G.band_cols;
        P.rlo = br[1] > br[0] ? max(br[0], 1) : 0;
        P.rhi = br[1] > br[0] ? min(br[1], G.nx - 1) : 0;
        P.clo = bc[1] > bc[0] ? max(bc[0], 1) : 0;
        P.chi = bc[1] > bc[0] ? min(bc[1], G.ny - 1) : 0;
        P.t_first = t_first;
        P.nsrc = G.src_i >= 0 ? 1 : 0;
        P.src_i.v = G.src_i; P.src_j.v = G.src_j;
        P.src_wave = G.src_wave; P.wave_len = G.wave_len;
        P.nprobe = G.probe_i >= 0 ? 1 : 0;
        P.probe_i.v = G.probe_i; P.probe_j.v = G.probe_j;
        P.probe_out = G.probe_out; P.probe_len = G.probe_len;
        rt_tile<true, true, false, 0, false>(P, CUT ? K : H, bx, by, nsx, nsy, S);
        lds_barrier();                        // the next tile rewrites S
    }
}

template <bool TF, int NF>
void launch_form(const RtParams &p, int waves, int tiles, bool lossy, bool pml, hipStream_t s)
{
    const dim3 g(tiles), b(64 * waves);
    if (pml && lossy) hipLaunchKernelGGL((tm_rt_kernel<true, true, TF, NF>), g, b, 0, s, p);
    else if (pml) hipLaunchKernelGGL((tm_rt_kernel<false, true, TF, NF>), g, b, 0, s, p);
    else if constexpr (!TF) {
        if (lossy) hipLaunchKernelGGL((tm_rt_kernel<true, false, false, 0>), g, b, 0, s, p);
        else hipLaunchKernelGGL((tm_rt_kernel<false, false, false, 0>), g, b, 0, s, p);
    }
}

}  // namespace

int rt_tiles(int nx, int ny, int waves, int K)
{
    return rt_along(nx, waves * R, K) * rt_along(ny, 64, K);
}

int preload_rt()
{
    return preload_kernel(reinterpret_cast<const void *>(&tm_rt_kernel<true, true, false, 0>));
}

int launch_fd2d_rt(const RtParams &p, int waves, int nf, bool lossy, bool pml, hipStream_t s)
{
    if (waves < 1 || waves > RT_WAVES || p.K < 1 || p.K > RT_MAX_STEPS || 2 * p.K >= waves * R ||
        2 * p.K >= 64)
        return fail("register tiles: %d steps a launch in tiles of %dx64", p.K, waves * R);
    const bool tf = nf || p.tf_npml;
    if (tf && !pml) return fail("register tiles: plane wave and DFT take the PML form");
    RtParams q = p;
    q.nsx = rt_tiles(1, p.ny, waves, p.K);
    const int tiles = rt_tiles(p.nx, p.ny, waves, p.K);
    if (!tf) launch_form<false, 0>(q, waves, tiles, lossy, pml, s);
    else if (nf == 0) launch_form<true, 0>(q, waves, tiles, lossy, pml, s);
    else if (nf == 1) launch_form<true, 1>(q, waves, tiles, lossy, pml, s);
    else if (nf == 2) launch_form<true, 2>(q, waves, tiles, lossy, pml, s);
    else if (nf == 3) launch_form<true, 3>(q, waves, tiles, lossy, pml, s);
    else return fail("register tiles: %d frequencies", nf);
    return hip_check(hipGetLastError(), "register tiles launch");
}

int launch_fd2d_rt_batch(const fd2d_grid *grids, const int *units, int nunits, int groups, int waves,
                         int K, int H, int parity, int t_first, int write_ez, hipStream_t s)
{
    if (waves < 1 || waves > RT_WAVES || K < 1 || K > H || H > RT_MAX_STEPS || 2 * H >= waves * R)
        return fail("register tiles: %d of %d steps a launch in tiles of %dx64", K, H, waves * R);
    // up to two tiles a CU, more and smaller tiles are as well
    const auto kernel = K < H && nunits > 512 ? tm_rt_batch_kernel<true> : tm_rt_batch_kernel<false>;
    hipLaunchKernelGGL(kernel, dim3(groups), dim3(64 * waves), 0, s, grids, units, nunits, K, H, parity,
                       t_first, write_ez);
    return hip_check(hipGetLastError(), "fd2d_batch_run launch");
}

}  // namespace fdtd
