// prop2d.hip -- device-resident 2-D propagation handles: CPML (the fused step
// of cpml2d.hip; fwdTimeCpmlFor2dAw_mex.c / rvsTimeCpmlFor2dAw_mex.c) and the
// Cerjan sponge (src/fwdTimeSpongeFor2dAw.m:69-106, src/rvsTimeSpongeFor2dAw.m).
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <numeric>
#include <type_traits>

#include "cpml2d.h"
#include "devbuf.h"
#include "tune.h"

namespace sssi {

// Sponge step: p_new = b p - g p_old + ax (pR+pL) + az (pD+pU) - v^2dt^2 s with
// b = 2 - 2ax - 2az, then multiplied by g.  ax, az, v^2dt^2 are formed from
// vdt = v*dt in-kernel.
// The reference damps both time levels after the rotation
// (fwdTimeSpongeFor2dAw.m:83-92); the stored level carries one factor and the
// second is applied when it is read back as p_old.
struct Sponge2dArgs {
    const float *pcur, *pold;  // levels before the first step
    float *ocur, *oold;        // levels after the last one (other buffers)
    const float *vdt;
    const float *g;  // g[m], m < nB
    int nz, nx, pitch, rows, nB;
    float idx2, idz2;  // 1/dx^2, 1/dz^2
    // time index of the first step and its direction, number of steps (<= kSpK)
    int t0, reverse, nsteps;
    const int *src_cell;
    const float *src_amp;  // [t*nsrc + k], t < src_nt (forward)
    int nsrc, src_nt;
    const float *surf;  // [t*nx + j], t < surf_nt (reverse)
    int surf_nt;
    float *rec;   // [t*nx + j] or null
    float *snap;  // slices at t % snap_stride == 0, slot t/stride - slot0; or null
    int snap_stride;
    int64_t snap_slot0;
    int *health;  // non-finite watchdog word (top row), or null
    int step;     // launch step reported to it (of the first step)
};

// Steps per launch of the sponge kernel, and the rows of its tile (64 columns
// wide); the inner cells are what a tile writes.
constexpr int kSpK = 8, kSpZ = 32;
constexpr int kSpCX = kTX - 2 * kSpK, kSpCZ = kSpZ - 2 * kSpK;

// Value of the lane before / after (DPP wave_shr:1 / wave_shl:1), 0 at the
// wavefront's edge.
__device__ __forceinline__ float lane_left(float v) {
    return __int_as_float(
        __builtin_amdgcn_mov_dpp(__float_as_int(v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float lane_right(float v) {
    return __int_as_float(
        __builtin_amdgcn_mov_dpp(__float_as_int(v), 0x130, 0xf, 0xf, true));
}

// Up to kSpK steps on the tile (ty, tx): see sponge2d_steps.  INNER: the whole
// tile lies inside the model and off its top row, and no damping strip touches
// it (every factor 1).
template <int R, bool INNER, bool MANY>
__device__ __forceinline__ void sponge2d_tile(const Sponge2dArgs &a, int tx, int ty,
                                              float (&edge)[2][kSpZ / R + 2][2][64]) {
    constexpr int K = kSpK;
    const int lane = threadIdx.x & 63, w = wave_id();
    const int j = tx * kSpCX - K + lane;
    const int q0 = w * R;                   // the wave's first row in the tile
    const int i0 = ty * kSpCZ - K + q0;     // and in the model
    const bool jin = INNER || (j >= 0 && j < a.nx);
    const bool jmine = jin && lane >= K && lane < 64 - K;
    const uint32_t rowb = (uint32_t)a.pitch * 4u;
    const uint32_t nbytes = rowb * (uint32_t)a.rows;
    const uint32_t vcol = jin ? (uint32_t)(j + kHX) * 4u : kOOB;
    auto iin = [&](int r) { return INNER || (i0 + r >= 0 && i0 + r < a.nz); };
    auto mine = [&](int r) { return iin(r) && q0 + r >= K && q0 + r < kSpZ - K; };
    auto srow = [&](int r) { return (uint32_t)(i0 + r + kHZ) * rowb; };

    float pa[R], pb[R], ax[R], az[R], gf[R];  // p (even steps), p_old, factors
    {
        const __amdgpu_buffer_rsrc_t rP = buf_rsrc(a.pcur, nbytes);
        const __amdgpu_buffer_rsrc_t rO = buf_rsrc(a.pold, nbytes);
        const __amdgpu_buffer_rsrc_t rV = buf_rsrc(a.vdt, nbytes);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            // rows outside the model: every lane out of range, so 0
            const uint32_t v = iin(r) ? vcol : kOOB, so = iin(r) ? srow(r) : 0u;
            pa[r] = buf_ld(rP, v, so);
            pb[r] = buf_ld(rO, v, so);
            ax[r] = buf_ld(rV, v, so);
        }
    }
    // all ones in the lanes and rows inside the model: ANDed to the update, it
    // keeps the cells outside 0 without a branch
    int keep[R];
#pragma unroll
    for (int r = 0; r < R; ++r) keep[r] = jin && iin(r) ? -1 : 0;
    // damping factor: the bottom strip's by row, else the side strips' by column
    float gx = 1.f;
    if constexpr (!INNER) {
        if (jin && j < a.nB) gx = a.g[j];
        else if (jin && j >= a.nx - a.nB) gx = a.g[a.nx - 1 - j];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const float v2 = ax[r] * ax[r];
        ax[r] = v2 * a.idx2;
        az[r] = v2 * a.idz2;
        gf[r] = gx;
        if constexpr (!INNER)
            if (iin(r) && i0 + r >= a.nz - a.nB) gf[r] = ld_uniform(a.g + (a.nz - 1 - i0 - r));
    }
    // sources in this wave's rows and columns
    WaveSources<R, MANY> src{a.src_cell, a.src_amp, a.nsrc, a.src_nt, a.nx, i0, tx * kSpCX - K};
    const bool has_src = !a.reverse && src.find(a.t0);
    const bool top = !INNER && i0 <= 0 && i0 + R > 0;  // the wave holds row 0
    const bool surf_here = top && a.reverse && a.surf;

    // source terms of a step, summed per cell in source order, then surface injection
    auto sources = [&](int t, float (&sv)[R]) {
#pragma unroll
        for (int r = 0; r < R; ++r) sv[r] = 0.f;
        if (has_src) src.add(t, j, sv);
        if (surf_here && t < a.surf_nt) {
            const float x = jin ? a.surf[(size_t)t * a.nx + j] : 0.f;
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (i0 + r == 0) sv[r] += x;
        }
    };
    const bool driven = has_src || surf_here;  // wave-uniform
    auto update = [&](float (&p)[R], float (&q)[R], float up, float below, int t, auto drive) {
        float sv[R];
        if constexpr (drive) sources(t, sv);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const float pc = p[r], dn = r + 1 < R ? p[r + 1] : below;
            // b p - p_old + ax (pR+pL) + az (pD+pU) regrouped as
            // p + (p - p_old) + ax((pR-p)+(pL-p)) + az((pD-p)+(pU-p)): the FP32
            // rounding then scales with the increments instead of with 2p.
            float lap = fmaf(ax[r], (lane_right(pc) - pc) + (lane_left(pc) - pc),
                             az[r] * ((dn - pc) + (up - pc)));
            if constexpr (drive) {
                const float vd = iin(r) && jin ? a.vdt[(size_t)(i0 + r + kHZ) * a.pitch + j + kHX]
                                               : 0.f;
                lap = fmaf(-sv[r], vd * vd, lap);
            }
            float pn = pc + (lap + (INNER ? pc - q[r] : fmaf(-gf[r], q[r], pc)));
            if constexpr (!INNER) {
                pn *= gf[r];
                pn = __int_as_float(__float_as_int(pn) & keep[r]);
            }
            q[r] = pn;
            up = pc;
        }
    };
    auto step = [&](int s, float (&p)[R], float (&q)[R]) {
        const int t = a.reverse ? a.t0 - s : a.t0 + s;
        float (&E)[kSpZ / R + 2][2][64] = edge[s & 1];
        E[w + 1][0][lane] = p[0];
        E[w + 1][1][lane] = p[R - 1];
        __syncthreads();
        const float up = E[w][1][lane], below = E[w + 2][0][lane];
        if (driven) update(p, q, up, below, t, std::true_type{});
        else update(p, q, up, below, t, std::false_type{});
        if (top) {
#pragma unroll
            for (int r = 0; r < R; ++r)
                if (i0 + r == 0 && mine(r)) {
                    if (a.rec && jmine) a.rec[(size_t)t * a.nx + j] = q[r];
                    if (a.health) report_nonfinite(a.health, jmine && nonfinite(q[r]), a.step + s);
                }
        }
        if (a.snap && t % a.snap_stride == 0) {
            const __amdgpu_buffer_rsrc_t rS = buf_rsrc(
                a.snap + (size_t)(t / a.snap_stride - a.snap_slot0) * a.nz * a.nx,
                (uint32_t)a.nz * (uint32_t)a.nx * 4u);
            const uint32_t vs = jmine ? (uint32_t)j * 4u : kOOB;
#pragma unroll
            for (int r = 0; r < R; ++r)
                buf_st(q[r], rS, mine(r) ? vs : kOOB,
                       mine(r) ? (uint32_t)(i0 + r) * (uint32_t)a.nx * 4u : 0u);
        }
    };
#pragma unroll 1
    for (int s = 0; s + 1 < a.nsteps; s += 2) {
        step(s, pa, pb);
        step(s + 1, pb, pa);
    }
    const bool odd = a.nsteps & 1;
    if (odd) step(a.nsteps - 1, pa, pb);  // the newest level ends in pb
    const __amdgpu_buffer_rsrc_t wP = buf_rsrc(odd ? a.oold : a.ocur, nbytes);
    const __amdgpu_buffer_rsrc_t wO = buf_rsrc(odd ? a.ocur : a.oold, nbytes);
    const uint32_t vst = jmine ? vcol : kOOB;
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t v = mine(r) ? vst : kOOB, so = mine(r) ? srow(r) : 0u;
        buf_st(pa[r], wP, v, so);
        buf_st(pb[r], wO, v, so);
    }
}

// nsteps <= kSpK time steps per launch.  A workgroup holds a tile of kSpZ rows
// x 64 columns in registers (lane = column, R rows per wavefront) and steps it
// without going back to memory: x neighbours by DPP, z neighbours from the
// lane's own registers and, at a wavefront's first and last row, through LDS
// (double-buffered, one barrier per step).  Cells at the tile's edge miss a
// neighbour and go wrong, and each step moves that error one cell inwards, so
// the tile's inner kSpCZ x kSpCX cells are exact after nsteps <= kSpK steps
// and are what it writes: two levels into buffers other than those it reads,
// as its neighbours still read their halos there.  Cells outside the model
// stay 0, which is the boundary.
// One step per launch was bound by the launch on small grids and by streaming
// four arrays per step on large ones; here 8 steps share a launch and one
// trip, at 12 VALU instructions per cell and step and 2.7 times the cells.
// 800 steps, whole call, one step per launch / this kernel: 100 x 150 2.59 /
// 1.14 ms, 301 x 450 with 58 snapshots 3.8 / 2.8, 515 x 1203 5.0 / 2.85,
// 1040 x 3080 12.0 / 8.3 (4 of them the model's way to the device).
// R = 4 (8 waves) has the shorter step, R = 8 (4 waves) the better use of a
// full chip: 100 x 150 1.14 against 1.50 ms, 515 x 1203 3.43 against 2.85.
// Blocks are 1-D over the tiles, XCD-banded: block b runs on XCD b % 8 and
// takes the next tile of that XCD's contiguous band.
template <int R, bool MANY>
__global__ void __launch_bounds__(64 * kSpZ / R) sponge2d_steps(Sponge2dArgs a, int ntx) {
    __shared__ float edge[2][kSpZ / R + 2][2][64];
    const int nb = (int)gridDim.x, b = (int)blockIdx.x;
    const int q = nb / 8, rem = nb % 8, x = b % 8;
    const int t = x * q + min(x, rem) + b / 8;
    const int ty = t / ntx, tx = t - ty * ntx;
    const int z0 = ty * kSpCZ - kSpK, x0 = tx * kSpCX - kSpK;  // first row and column held
    if (z0 > 0 && z0 + kSpZ <= a.nz - a.nB && x0 >= a.nB && x0 + 64 <= a.nx - a.nB)
        sponge2d_tile<R, true, MANY>(a, tx, ty, edge);
    else
        sponge2d_tile<R, false, MANY>(a, tx, ty, edge);
}

// One time step: for runs cut into pieces of a step or two, where the tiles of
// sponge2d_steps would compute 2.7 cells for each one they write and share
// their trip to memory with nobody.  A wavefront owns 64 columns x RZ rows
// (lane = column); every load is a raw buffer load with the wave-uniform row
// offset in the scalar offset: the column window p(i0-1 .. i0+RZ) once, the x
// neighbours as loads shifted by one column, then p_old and v*dt.  The new
// level goes where p_old was (ocur: each cell's is read by its own lane alone),
// with the arithmetic of sponge2d_tile cell by cell.  Rows i0-1 .. i0+RZ and
// columns j-1 .. j+1 of every wavefront with a row inside the model lie in the
// padded array, whose padding stays zero: lanes outside store nothing.
// Bound by the launch on small grids, by four arrays' streams on large ones.
// A step in pieces of one, this kernel / sponge2d_steps, us: 100 x 150 3.6 /
// 3.9, 515 x 1203 3.7 / 6.0, 1040 x 3080 7.6 / 15.5; in pieces of two 3.2 / 2.5,
// 3.6 / 4.0, 7.6 / 9.9; of three 3.0 / 2.0, 3.7 / 3.0, 7.6 / 7.2.
// 1-D over ntx * ntz block tiles, XCD-banded as sponge2d_steps.
constexpr int kSpRZ = 4;
template <int RZ>
__global__ void __launch_bounds__(256) sponge2d_step(Sponge2dArgs a, int ntx) {
    const int lane = threadIdx.x & 63, w = wave_id();
    const int nb = (int)gridDim.x, b = (int)blockIdx.x;
    const int q = nb / 8, rem = nb % 8, x = b % 8;
    const int tile = x * q + min(x, rem) + b / 8;
    const int ty = tile / ntx, tx = tile - ty * ntx;
    const int j = tx * 64 + lane;
    const int i0 = (ty * 4 + w) * RZ;
    if (i0 >= a.nz) return;
    const bool jin = j < a.nx;
    const uint32_t rowb = (uint32_t)a.pitch * 4u;
    const uint32_t nbytes = rowb * (uint32_t)a.rows;
    const __amdgpu_buffer_rsrc_t rP = buf_rsrc(a.pcur, nbytes);
    const __amdgpu_buffer_rsrc_t rO = buf_rsrc(a.ocur, nbytes);
    const __amdgpu_buffer_rsrc_t rV = buf_rsrc(a.vdt, nbytes);
    const uint32_t vcol = (uint32_t)(j + kHX) * 4u;
    const uint32_t srow = (uint32_t)(i0 + kHZ) * rowb;

    float col[RZ + 2], cl[RZ], cr[RZ], po[RZ], vd[RZ];
#pragma unroll
    for (int r = 0; r < RZ + 2; ++r) col[r] = buf_ld(rP, vcol, srow + (r - 1) * rowb);
#pragma unroll
    for (int r = 0; r < RZ; ++r) {
        cl[r] = buf_ld(rP, vcol - 4u, srow + r * rowb);
        cr[r] = buf_ld(rP, vcol + 4u, srow + r * rowb);
        po[r] = buf_ld(rO, vcol, srow + r * rowb);
        vd[r] = buf_ld(rV, vcol, srow + r * rowb);
    }

    // damping factor: the bottom strip's by row, else the side strips' by column
    const int nB = a.nB;
    float gx = 1.f;
    if (jin && j < nB) gx = a.g[j];
    else if (jin && j >= a.nx - nB) gx = a.g[a.nx - 1 - j];
    // source terms, summed per cell in source order, then surface injection
    const int t = a.t0;
    float s[RZ];
#pragma unroll
    for (int r = 0; r < RZ; ++r) s[r] = 0.f;
    if (!a.reverse && a.nsrc > 0) {
        WaveSources<RZ, true> src{a.src_cell, a.src_amp, a.nsrc, a.src_nt, a.nx, i0, tx * 64};
        if (src.find(t)) src.add(t, j, s);
    }
    if (a.reverse && a.surf && t < a.surf_nt && i0 == 0 && jin) s[0] += a.surf[(size_t)t * a.nx + j];
    float *snap = a.snap && t % a.snap_stride == 0
                      ? a.snap + (size_t)(t / a.snap_stride - a.snap_slot0) * a.nz * a.nx
                      : nullptr;

    float pn0 = 0.f;
#pragma unroll
    for (int r = 0; r < RZ; ++r) {
        const int i = i0 + r;
        if (i >= a.nz) break;
        const float gf = i >= a.nz - nB ? ld_uniform(a.g + (a.nz - 1 - i)) : gx;
        const float v2 = vd[r] * vd[r];
        const float ax = v2 * a.idx2, az = v2 * a.idz2;
        const float pc = col[r + 1];
        float lap = fmaf(ax, (cr[r] - pc) + (cl[r] - pc), az * ((col[r + 2] - pc) + (col[r] - pc)));
        lap = fmaf(-s[r], v2, lap);
        float pn = pc + (lap + fmaf(-gf, po[r], pc));
        pn *= gf;
        buf_st(pn, rO, jin ? vcol : kOOB, srow + r * rowb);
        if (r == 0) pn0 = pn;
        if (jin) {
            if (a.rec && i == 0) a.rec[(size_t)t * a.nx + j] = pn;
            if (snap) snap[(size_t)i * a.nx + j] = pn;
        }
    }
    if (a.health && i0 == 0) report_nonfinite(a.health, jin && nonfinite(pn0), a.step);
}

// One (slice, y) plane's 64 x 64 tile through LDS: rows of x in, columns of z
// out, both coalesced; 65 floats per LDS row keep the banks apart.
__global__ void __launch_bounds__(256) z_fastest(const float *__restrict__ in,
                                                 float *__restrict__ out, int64_t nz, int64_t nx,
                                                 int64_t ny, int64_t ntx, int64_t ntz,
                                                 int64_t ntiles) {
    __shared__ float t[64][65];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int64_t b = blockIdx.x; b < ntiles; b += gridDim.x) {
        const int64_t x0 = b % ntx * 64, z0 = b / ntx % ntz * 64, sy = b / (ntx * ntz);
        const int64_t y = sy % ny, base = sy / ny * (nz * nx * ny);
#pragma unroll 4
        for (int r = w; r < 64; r += 4)
            if (z0 + r < nz && x0 + lane < nx)
                t[r][lane] = in[base + ((z0 + r) * ny + y) * nx + x0 + lane];
        __syncthreads();
#pragma unroll 4
        for (int r = w; r < 64; r += 4)
            if (x0 + r < nx && z0 + lane < nz)
                out[base + (y * nx + x0 + r) * nz + z0 + lane] = t[lane][r];
        __syncthreads();
    }
}

void launch_z_fastest(const float *in, float *out, int64_t nz, int64_t nx, int64_t ny, int64_t ns,
                      hipStream_t s) {
    const int64_t ntx = (nx + 63) / 64, ntz = (nz + 63) / 64, n = ntx * ntz * ny * ns;
    if (n == 0) return;
    hipLaunchKernelGGL(z_fastest, dim3((unsigned)std::min<int64_t>(n, 1 << 20)), dim3(256), 0, s,
                       in, out, nz, nx, ny, ntx, ntz, n);
    SSSI_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
class Prop2D final : public Prop {
   public:
    // CPML
    std::unique_ptr<Cpml2dGrid> g;
    DevSources srcs;
    DevBuf<int2> order;
    int nblk = 0;
    // second set of levels and memory variables (several steps per launch:
    // a launch reads one set and writes the other)
    DevBuf<float> ap[2], azpsi, axpsi;
    StepGraph graph;   // captured time loop (re-captured when the descriptor changes)
    int64_t done = 0;  // steps since reset (parity of the current level)
    // sponge
    int64_t pitch = 0, rows = 0;
    // levels in pairs (current, old): a launch reads one pair, writes the other
    DevBuf<float> sp[2][2], vdt, gtab;
    DevBuf<int> sp_health;
    int cur = 0;  // pair that holds the present levels

    Prop2D(const double *v, int64_t nz_, int64_t nx_, int abc_, int N_, int nB_, double dz_,
           double dx_, double dt_) {
        dim = 2;
        abc = abc_;
        nz = nz_; nx = nx_; ny = 1; N = N_; nB = nB_; dz = dz_; dx = dx_; dt = dt_;
        SSSI_HIP(hipGetDevice(&device));
        stream = stream_acquire();
        {
            const double vmax = max_velocity(v, nz * nx);
            courant = vmax * dt * std::sqrt(1.0 / (dz * dz) + 1.0 / (dx * dx));
        }
        if (abc == SSSI_ABC_CPML) {
            g.reset(new Cpml2dGrid(v, nz, nx, N, nB, dz, dx, dt));
            if (autotune_enabled()) tune_layout();
            build_order();
        } else {
            validate_sponge_grid(nz, nx);
            pitch = round_up(kHX + round_up(nx, kTX) + 32, 64);
            rows = kHZ + round_up(nz, kTZmax) + kHZbot;
            const size_t np = (size_t)pitch * rows;
            for (auto &pair : sp)
                for (auto &level : pair) level.alloc(np);
            vdt.alloc(np);
            upload_model(v, nz, nx, 1, dt, false, vdt.p, vdt.n, pitch, 0, kHZ, 0, kHX, stream);
            std::vector<float> gg(std::max(nB, 1), 1.f);
            const double alpha = 0.015;
            for (int m = 0; m < nB; ++m) {
                const double e = std::exp(-((alpha * (nB - m)) * (alpha * (nB - m))));
                gg[m] = (float)std::pow(e, 10);
            }
            gtab.alloc(gg.size());
            SSSI_HIP(hipMemcpy(gtab.p, gg.data(), gtab.bytes(), hipMemcpyHostToDevice));
            sp_health.alloc(1);
        }
        reset();
    }

    ~Prop2D() override {
        graph.clear();  // before ~Prop destroys the stream its replays ran on
    }

    void build_order() {
        std::vector<int2> ord;
        build_block_order({g.get()}, ord);
        nblk = (int)ord.size();
        order.alloc(ord.size());
        SSSI_HIP(hipMemcpy(order.p, ord.data(), order.bytes(), hipMemcpyHostToDevice));
    }

    // Autotuner of the step kernel (small grids run most of their steps several to
    // a launch, where only the stencil forms of its tile height are kept): time
    // every instantiated layout (tile height, march groups) on this grid -- kTuneSteps launches after a short warm-up, HIP events on the
    // handle's stream -- keep the fastest, and cache it for the shape.
    void tune_layout() {
        const TuneKey key{2, nz, nx, 1, N, nB};
        static const int cand[][2] = {{4, 0}, {4, 2}, {4, 3}, {4, 4}, {4, 8},
                                      {8, 0}, {8, 2}, {8, 4}};
        int a = 0, b = 0;
        if (tune_lookup(key, a, b)) {
            // a cache entry is used only if it names an instantiated layout
            for (const auto &c : cand)
                if (c[0] == a && c[1] == b) {
                    g->set_layout(a, b);
                    return;
                }
        }
        // Layouts within a few percent of each other: every candidate is timed
        // over kTuneSteps launches in each of two passes (best pass kept), after
        // a first warm-up long enough for the clocks to settle.
        constexpr int kWarm = 20, kFirstWarm = 400, kTuneSteps = 200, kPasses = 2;
        hipEvent_t e0, e1;
        SSSI_HIP(hipEventCreate(&e0));
        SSSI_HIP(hipEventCreate(&e1));
        float best_ms = 1e30f;
        int best_a = g->rz, best_b = g->ng;
        try {
            for (int pass = 0; pass < kPasses; ++pass)
                for (const auto &c : cand) {
                    g->set_layout(c[0], c[1]);
                    build_order();
                    const Job2D J = g->job();  // no sources, receivers or snapshots
                    const int warm = pass == 0 && &c == &cand[0] ? kFirstWarm : kWarm;
                    for (int q = 0; q < warm; ++q)
                        launch_cpml2d_single(*g, J, order.p, nblk, q, stream);
                    SSSI_HIP(hipEventRecord(e0, stream));
                    for (int q = 0; q < kTuneSteps; ++q)
                        launch_cpml2d_single(*g, J, order.p, nblk, warm + q, stream);
                    SSSI_HIP(hipEventRecord(e1, stream));
                    SSSI_HIP(hipEventSynchronize(e1));
                    float ms = 0.f;
                    SSSI_HIP(hipEventElapsedTime(&ms, e0, e1));
                    if (ms < best_ms) {
                        best_ms = ms;
                        best_a = c[0];
                        best_b = c[1];
                    }
                }
        } catch (...) {
            (void)hipEventDestroy(e0);
            (void)hipEventDestroy(e1);
            throw;
        }
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        g->set_layout(best_a, best_b);
        tune_store(key, best_a, best_b);
    }

    void layout(int *a, int *b) const override {
        *a = g ? g->rz : 0;
        *b = g ? g->ng : 0;
    }

    void use_stream(hipStream_t s) override {
        graph.clear();  // its replays ran on the stream being replaced
        Prop::use_stream(s);
    }

    int64_t cells() const override { return nz * nx; }

    void reset() override {
        if (g) {
            g->zero_state(stream);
        } else {
            for (auto &pair : sp)
                for (auto &level : pair)
                    SSSI_HIP(hipMemsetAsync(level.p, 0, level.bytes(), stream));
            arm_health(sp_health.p, stream);
        }
        done = 0;
        steps_done = 0;
        cur = 0;
        SSSI_HIP(hipStreamSynchronize(stream));
    }

    void set_points(int n, const int *iz, const int *ix, const int *, const double *wavelet,
                    int64_t nt) override {
        if (g) {
            srcs.set(*g, n, iz, ix, wavelet, nt);
            nsrc = srcs.n;
            src_nt = nt;
            return;
        }
        if (n < 0 || nt < 1 || (n > 0 && (!iz || !ix || !wavelet)))
            fail(SSSI_EINVAL, "set_points: bad arguments");
        for (int k = 0; k < n; ++k)
            if (iz[k] < 0 || iz[k] >= nz || ix[k] < 0 || ix[k] >= nx)
                fail(SSSI_EINVAL, "set_points: source %d at (%d,%d) outside the %lldx%lld grid",
                     k, iz[k], ix[k], (long long)nz, (long long)nx);
        nsrc = n;
        src_nt = nt;
        std::vector<int> cell(std::max(n, 1), 0);
        for (int k = 0; k < n; ++k) cell[k] = iz[k] * (int)nx + ix[k];
        std::vector<float> amp((size_t)nt * std::max(n, 1), 0.f);
        for (int64_t t = 0; t < nt; ++t)
            for (int k = 0; k < n; ++k) amp[(size_t)t * n + k] = (float)wavelet[t * n + k];
        src_cell.alloc(cell.size());
        src_amp.alloc(amp.size());
        SSSI_HIP(hipMemcpy(src_cell.p, cell.data(), src_cell.bytes(), hipMemcpyHostToDevice));
        SSSI_HIP(hipMemcpy(src_amp.p, amp.data(), src_amp.bytes(), hipMemcpyHostToDevice));
    }

    void set_surface(const double *data, int64_t nt) override {
        if (!data || nt < 1) fail(SSSI_EINVAL, "set_surface: bad arguments");
        std::vector<float> h((size_t)nt * nx);
        for (size_t q = 0; q < h.size(); ++q) h[q] = (float)data[q];
        surf.alloc(h.size());
        surf_nt = nt;
        SSSI_HIP(hipMemcpy(surf.p, h.data(), surf.bytes(), hipMemcpyHostToDevice));
    }


    // Descriptor for `count` steps from time index t_first (see the kernel's
    // t / parity mapping): the level current now sits at parity rel_0 & 1.
    Job2D make_job(int64_t t_first, bool reverse, bool record, const SnapSink *sink,
                   int *step0) {
        Job2D J = g->job();
        const int curlev = (int)(done & 1);
        int rel0;
        if (!reverse) {
            J.start_step = (int)(done - t_first);
            J.nt = (int)(t_first + 1);
            rel0 = (int)t_first;
        } else {
            J.start_step = (int)done;
            J.nt = (int)(t_first + 1);
            rel0 = 0;
        }
        J.reverse = reverse ? 1 : 0;
        const int pa = rel0 & 1;
        J.p[pa] = g->p[curlev].p;
        J.p[pa ^ 1] = g->p[curlev ^ 1].p;
        J.zphi[pa] = g->zphi[curlev].p;
        J.zphi[pa ^ 1] = g->zphi[curlev ^ 1].p;
        J.xphi[pa] = g->xphi[curlev].p;
        J.xphi[pa ^ 1] = g->xphi[curlev ^ 1].p;
        if (srcs.n > 0) {
            J.src_ptr = srcs.ptr.p;
            J.src_cell = srcs.cell.p;
            J.src_amp = srcs.amp.p;
            J.nsrc = srcs.n;
            J.src_nt = srcs.nt;
        }
        if (surf.p) {
            J.surf = surf.p;
            J.surf_nt = (int)surf_nt;
        }
        if (record) J.rec = rec.p;
        if (sink && sink->dev) {
            J.snap = sink->dev;
            J.snap_stride = (int)sink->stride;
            J.snap_slot0 = (int)sink->slot0;
        }
        *step0 = (int)done;
        return J;
    }

    int *health_word() const override { return g ? g->health.p : sp_health.p; }

    void scan_field() override {
        if (g) g->scan_nonfinite((int)(done & 1), (int)done, stream);
        else launch_nonfinite_scan(sp[cur][0].p, sp[cur][0].n, sp_health.p, (int)done, stream);
    }

    // n <= kSpK sponge steps from time index t; the launches it took
    int steps_sponge(int64_t t, int n, bool reverse, bool record, const SnapSink *sink,
                      int step) {
        Sponge2dArgs a{};
        a.health = sp_health.p;
        a.step = step;
        a.pcur = sp[cur][0].p;
        a.pold = sp[cur][1].p;
        a.ocur = sp[cur ^ 1][0].p;
        a.oold = sp[cur ^ 1][1].p;
        a.vdt = vdt.p;
        a.g = gtab.p;
        a.nz = (int)nz; a.nx = (int)nx; a.pitch = (int)pitch; a.rows = (int)rows; a.nB = nB;
        a.idx2 = (float)(1.0 / (dx * dx));
        a.idz2 = (float)(1.0 / (dz * dz));
        a.t0 = (int)t;
        a.reverse = reverse ? 1 : 0;
        a.nsteps = n;
        if (!reverse && nsrc > 0) {
            a.src_cell = src_cell.p;
            a.src_amp = src_amp.p;
            a.nsrc = nsrc;
            a.src_nt = (int)src_nt;
        }
        if (reverse && surf.p) {
            a.surf = surf.p;
            a.surf_nt = (int)surf_nt;
        }
        if (record) a.rec = rec.p;
        if (sink && sink->dev) {
            a.snap = sink->dev;
            a.snap_stride = (int)sink->stride;
            a.snap_slot0 = sink->slot0;
        }
        const int ntx = (int)((nx + kSpCX - 1) / kSpCX);
        const int64_t ntz = (nz + kSpCZ - 1) / kSpCZ;
        // single steps: one at a time, and two where the chip is full (the
        // figures at sponge2d_step)
        if (n == 1 || (n == 2 && ntx * ntz >= 512)) {
            const int ntx1 = (int)((nx + 63) / 64);
            const int64_t ntz1 = (nz + 4 * kSpRZ - 1) / (4 * kSpRZ);
            for (int q = 0; q < n; ++q) {
                a.t0 = (int)(reverse ? t - q : t + q);
                a.step = step + q;
                a.nsteps = 1;
                a.pcur = sp[cur][0].p;
                a.ocur = sp[cur][1].p;  // (in place of the old level)
                hipLaunchKernelGGL(sponge2d_step<kSpRZ>, dim3((unsigned)(ntx1 * ntz1)), dim3(256),
                                   0, stream, a, ntx1);
                SSSI_HIP(hipGetLastError());
                std::swap(sp[cur][0], sp[cur][1]);
            }
            return n;
        }
        // 4 rows per wave while the tiles (8 waves each) leave the chip's 1024
        // SIMDs idle or nearly so, 8 rows from two blocks per CU
        const dim3 grid((unsigned)(ntx * ntz));
        const dim3 block(64 * kSpZ / (ntx * ntz < 512 ? 4 : 8));
        auto kernel = a.nsrc > kFewSources
                          ? (ntx * ntz < 512 ? sponge2d_steps<4, true> : sponge2d_steps<8, true>)
                          : (ntx * ntz < 512 ? sponge2d_steps<4, false> : sponge2d_steps<8, false>);
        hipLaunchKernelGGL(kernel, grid, block, 0, stream, a, ntx);
        SSSI_HIP(hipGetLastError());
        cur ^= 1;
        return 1;
    }

    void run(int64_t t_first, int64_t count, bool reverse, bool record, const SnapSink *sink,
             LaunchStats *st) override {
        if (count < 0) fail(SSSI_EINVAL, "run: negative step count");
        if (count == 0) return;
        if (record) ensure_rec(reverse ? t_first + 1 : t_first + count, nx);
        const int K = g && count > 1 && !graphs_enabled() && srcs.n <= kStepsMaxSrc
                          ? cpml2d_steps_per_launch(*g) : 0;
        if (K > 0) {
            run_steps(t_first, count, reverse, record, sink, K, st);
            return;
        }
        if (g) {
            int step0;
            const Job2D J = make_job(t_first, reverse, record, sink, &step0);
            graph.run(&J, sizeof(J), step0, count, stream,
                      [&](int step, const int *base, hipStream_t s) {
                          launch_cpml2d_single(*g, J, order.p, nblk, step, s, base);
                      });
            if (st) st->launches += count;
            done += count;
            steps_done = done;
            return;
        }
        for (int64_t q = 0; q < count; q += kSpK) {
            const int n = (int)std::min<int64_t>(kSpK, count - q);
            const int nl = steps_sponge(reverse ? t_first - q : t_first + q, n, reverse, record,
                                        sink, (int)(done + q));
            if (st) st->launches += nl;
        }
        done += count;
        steps_done = done;
    }

    // Up to K steps per launch.  The grid's buffers are swapped with the second
    // set so that the present levels and memory variables stay where make_job,
    // get_field and get_model look for them (by the parity of `done`).
    void run_steps(int64_t t_first, int64_t count, bool reverse, bool record,
                   const SnapSink *sink, int K, LaunchStats *st) {
        if (!ap[0].p) {
            // held only once all of it is there: the call may fail and come again
            DevBuf<float> p0(g->p[0].n), p1(g->p[1].n), zpsi, xpsi;
            if (nB > 0) {
                zpsi.alloc(g->zpsi.n);
                xpsi.alloc(g->xpsi.n);
            }
            for (auto *b : {&p0, &p1})  // (their padding stays 0)
                SSSI_HIP(hipMemsetAsync(b->p, 0, b->bytes(), stream));
            azpsi = std::move(zpsi);
            axpsi = std::move(xpsi);
            ap[0] = std::move(p0);
            ap[1] = std::move(p1);
        }
        for (int64_t q = 0; q < count;) {
            const int n = (int)std::min<int64_t>(K, count - q);
            int step;
            const Job2D J = make_job(reverse ? t_first - q : t_first + q, reverse, record, sink, &step);
            const int lev = (int)(done & 1), to = (int)((done + n) & 1);
            const Steps2DOut out{ap[0].p, ap[1].p, g->zphi[lev ^ 1].p, azpsi.p, g->xphi[lev ^ 1].p,
                                 axpsi.p};
            launch_cpml2d_steps(*g, J, out, step, n, stream);
            if (st) st->launches++;
            std::swap(g->p[to], ap[0]);
            std::swap(g->p[to ^ 1], ap[1]);
            std::swap(g->zpsi, azpsi);
            std::swap(g->xpsi, axpsi);
            if (to == lev) {  // the new Phi lies where the other parity's belongs
                std::swap(g->zphi[0], g->zphi[1]);
                std::swap(g->xphi[0], g->xphi[1]);
            }
            done += n;
            q += n;
        }
        steps_done = done;
    }

    void get_data(double *data, int64_t nt) override {
        if (nt > rec_nt || !rec.p)
            fail(SSSI_ESTATE, "get_data: no recorded traces for %lld steps", (long long)nt);
        widen_to_host(data, rec.p, (size_t)nt * nx, stream);  // [t][j] == data(nx,nt)
    }

    // sponge levels: interior of the current (0) or old (1) level, optionally times the second damping factor
    void download_sponge(int which, double *out, bool padded_model) {
        std::vector<float> h((size_t)pitch * rows);
        SSSI_HIP(hipMemcpyAsync(h.data(), sp[cur][which].p, h.size() * sizeof(float),
                                hipMemcpyDeviceToHost, stream));
        SSSI_HIP(hipStreamSynchronize(stream));
        std::vector<float> gf(std::max(nB, 1));
        SSSI_HIP(hipMemcpy(gf.data(), gtab.p, gtab.bytes(), hipMemcpyDeviceToHost));
        auto gfac = [&](int64_t i, int64_t j) -> float {
            if (i >= nz - nB) return gf[nz - 1 - i];
            if (j < nB) return gf[j];
            if (j >= nx - nB) return gf[nx - 1 - j];
            return 1.f;
        };
        if (!padded_model) {
            for (int64_t j = 0; j < nx; ++j)
                for (int64_t i = 0; i < nz; ++i)
                    out[j * nz + i] = h[(size_t)(i + kHZ) * pitch + j + kHX];
            return;
        }
        const int64_t mz = nz + 2, mx = nx + 2;
        for (int64_t q = 0; q < mz * mx; ++q) out[q] = 0.0;
        for (int64_t j = 0; j < nx; ++j)
            for (int64_t i = 0; i < nz; ++i)
                out[(j + 1) * mz + i + 1] = gfac(i, j) * h[(size_t)(i + kHZ) * pitch + j + kHX];
    }

    void get_field(double *field) override {
        if (g) g->download((int)(done & 1), field, stream);
        else download_sponge(0, field, false);
    }

    void get_model(double *model) override {
        if (!g) {
            download_sponge(1, model, true);
            return;
        }
        // reference model layout: (nz+2l) x (nx+2l), l-wide zero halo
        const int64_t l = 2 * N - 1, mz = nz + 2 * l, mx = nx + 2 * l;
        std::vector<double> in((size_t)nz * nx);
        g->download((int)((done & 1) ^ 1), in.data(), stream);
        for (int64_t q = 0; q < mz * mx; ++q) model[q] = 0.0;
        for (int64_t j = 0; j < nx; ++j)
            for (int64_t i = 0; i < nz; ++i) model[(j + l) * mz + i + l] = in[j * nz + i];
    }

    void alg_bytes(double *bytes, double *ncells) override {
        *ncells = (double)nz * nx;
        *bytes = g ? g->alg_bytes_per_step() : 16.0 * (double)nz * nx + 4.0 * nx;
    }
};

void Prop::check_health() {
    const int h = read_health(health_word(), stream);
    if (h != kHealthy)
        fail(SSSI_EUNSTABLE,
             "non-finite wavefield (NaN/Inf) at step %d of %lld since the last reset: the time "
             "step is likely beyond the scheme's stability limit (v_max dt sqrt(sum 1/d^2) = %.3f)",
             h + 1, (long long)steps_done, courant);
}

Prop *make_prop2d(const double *v, int64_t nz, int64_t nx, int abc, int N, int nB, double dz,
                  double dx, double dt) {
    return new Prop2D(v, nz, nx, abc, N, nB, dz, dx, dt);
}

}  // namespace sssi
