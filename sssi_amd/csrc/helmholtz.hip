// helmholtz.hip -- frequency-domain acoustic CPML Helmholtz solve on gfx950:
// freqCpmlFor2dAw (src/freqCpmlFor2dAw.m:43-133), A U = -S with A the
// (4k+1)-point impedance matrix (k = 2N-1) of squared slowness m, angular
// frequency w, CPML damping on the side and bottom strips.
//
// Matrix.  One thread per row cell computes the row's two complex damping
// factors (1j w / (s (1j w + d)))^2 in FP64 and writes the row into the band
// store (and, on request, CSR), in the reference's entry order.  Arithmetic
// is FP64 with contraction off, each operation rounded as the oracle rounds it.
//
// Solve.  A is banded in MATLAB's column-major cell order, kl = ku = k nz.
// The factorisation is LU with partial pivoting in LAPACK's band layout
// (A(i, j) at ab[kl + ku + i - j + j ldab], ldab = 2 kl + ku + 1; the top kl
// rows hold the fill of U), as panels of kNB columns.  Pivot = first row of
// maximal |re| + |im| within kl below the diagonal, scaling by the reciprocal
// of the pivot.  Each element receives the same operations in the same order
// as in the unblocked algorithm, and the factors equal the oracle's bit for
// bit.  No step is bound by bandwidth or arithmetic but by the chain of n
// pivot steps and, per source, 2 n substitution steps; the kernels shorten
// what lies on those chains.  120 x 140, nDiffOrder 2, 100 sources (kl = 360,
// 1050 panels): factorisation 67.1 ms with the panel in LDS and its steps
// replayed on every later column in a second launch, 36.1 ms as below (34 us
// per panel: 7 to load and prepare it, 6 for the panel before, 21 for its 16
// pivot steps); substitution 24.1 ms one step at a time, 11.0 ms by panels.
//   freq_lu      one launch per panel: workgroup 0 brings the next panel up to
//                date with the present one and factors it, rows in registers,
//                while the other workgroups update the columns behind it;
//   freq_subst   one workgroup per right-hand side, a panel at a time: forward
//                sweep with the interchanges, column-oriented backward sweep,
//                the band window of the right-hand side in LDS.
// Bands too wide for rows in registers (kl > kMaxBand) take the column replay:
//   freq_panel   one workgroup factors the panel, in LDS where its rows fit;
//   freq_trail(_lds)  workgroups of one to four later columns within reach
//                replay the panel's interchanges and updates in pivot order;
//   freq_solve   one workgroup per right-hand side, one step at a time.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <type_traits>
#include <vector>

#include "common.h"

namespace sssi {

struct alignas(16) cx {  // (16-byte LDS and global accesses)
    double re, im;
};

__device__ __forceinline__ cx cmul(cx a, cx b) {
#pragma clang fp contract(off)
    return {a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
__device__ __forceinline__ cx csub_mul(cx a, cx l, cx u) {  // a - l u
#pragma clang fp contract(off)
    return {a.re - (l.re * u.re - l.im * u.im), a.im - (l.re * u.im + l.im * u.re)};
}
__device__ __forceinline__ cx cdiv(cx a, cx b) {
#pragma clang fp contract(off)
    const double den = b.re * b.re + b.im * b.im;
    return {(a.re * b.re + a.im * b.im) / den, (a.im * b.re - a.re * b.im) / den};
}
__device__ __forceinline__ cx crecip(cx b) {
#pragma clang fp contract(off)
    const double den = b.re * b.re + b.im * b.im;
    return {b.re / den, -b.im / den};
}

constexpr int kNB = 16;      // panel width (columns)
constexpr int kMaxOff = 31;  // 2k + 1 summed coefficients, k <= 15

struct BandDesc {
    cx *ab;
    int64_t n, kl, ku, ldab;
    __device__ __forceinline__ cx &at(int64_t i, int64_t j) const {
        return ab[(kl + ku + i - j) + j * ldab];
    }
};

// (1j w / (s (1j w + d)))^2: t = (s d, s w); q = (0, w) / t; q^2
__device__ __forceinline__ cx freq_factor(double w, double s, double d) {
#pragma clang fp contract(off)
    const double tr = s * d, ti = s * w;
    const double den = tr * tr + ti * ti;
    const double qr = w * ti / den, qi = w * tr / den;
    return {qr * qr - qi * qi, qr * qi + qi * qr};
}

struct FreqCoef {
    double c[kMaxOff];
};

// Row r = j nz + i of A: x neighbours left, z above, centre, z below, x right
// (ascending column order).  ab (band) and/or CSR (rowptr given) are written.
__global__ void __launch_bounds__(256) freq_assemble(const double *__restrict__ m,
                                                     const double *__restrict__ xd,
                                                     const double *__restrict__ zd, FreqCoef fc,
                                                     int nz, int nx, int k, double w, double dz,
                                                     double dx, BandDesc B,
                                                     const int64_t *__restrict__ rowptr,
                                                     int64_t *__restrict__ col,
                                                     cx *__restrict__ val) {
#pragma clang fp contract(off)
    const int64_t n = (int64_t)nz * nx;
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < n;
         r += (int64_t)gridDim.x * blockDim.x) {
        const int j = (int)(r / nz), i = (int)(r - (int64_t)j * nz);
        const cx fz = freq_factor(w, dz, zd[r]), fx = freq_factor(w, dx, xd[r]);
        int64_t e = rowptr ? rowptr[r] : 0;
        auto emit = [&](int64_t cidx, cx v) {
            if (B.ab) B.at(r, cidx) = v;
            if (rowptr) {
                col[e] = cidx;
                val[e] = v;
                ++e;
            }
        };
        for (int o = -k; o <= -1; ++o)
            if (j + o >= 0) emit(r + (int64_t)o * nz, cx{fc.c[o + k] * fx.re, fc.c[o + k] * fx.im});
        for (int o = -k; o <= -1; ++o)
            if (i + o >= 0) emit(r + o, cx{fc.c[o + k] * fz.re, fc.c[o + k] * fz.im});
        {
            const double mw = m[r] * (w * w);
            emit(r, cx{(mw + fc.c[k] * fz.re) + fc.c[k] * fx.re, fc.c[k] * fz.im + fc.c[k] * fx.im});
        }
        for (int o = 1; o <= k; ++o)
            if (i + o < nz) emit(r + o, cx{fc.c[o + k] * fz.re, fc.c[o + k] * fz.im});
        for (int o = 1; o <= k; ++o)
            if (j + o < nx) emit(r + (int64_t)o * nz, cx{fc.c[o + k] * fx.re, fc.c[o + k] * fx.im});
    }
}

// State of the factorisation carried between launches (device resident).
struct LuState {
    int64_t ju;        // running reach of U (last column touched)
    int singular;      // first zero pivot column + 1 (0: none)
};

// Column-replay form: factor panel columns j0 .. j0+kNB-1 (256 threads).  With LDS, the panel's
// rows j0 .. j0+kNB-1+kl (R of them) are staged in dynamic LDS, column-major,
// for the whole factorisation; entries outside the band are neither read nor
// written (none of the steps touches them).  Per column: pivot search (wave
// reductions), the decision by thread 0, the row swap, then each thread
// scales its rows of the column and applies them to the later columns (the
// multiplier stays in a register: one pass, no barrier between the two).
// Measured per panel of 16 columns at kl = 360: 62.7 us with 256 threads,
// 75.7 us with 1024 (rank-1 split over column groups), 75.1 us with the rows
// batched through registers.
template <bool LDS>
__global__ void __launch_bounds__(256) freq_panel(BandDesc B, int64_t j0, int64_t *__restrict__ piv,
                                                  int64_t *__restrict__ juv, LuState *st,
                                                  int64_t R) {
#pragma clang fp contract(off)
    extern __shared__ cx P[];
    __shared__ double s_best[4];
    __shared__ int s_arg[4];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int64_t n = B.n, kl = B.kl, ku = B.ku;
    const int64_t jend = min(j0 + kNB, n);
    const int Ri = (int)R;
    auto inband = [&](int64_t i, int64_t j) {
        return i < n && j < n && i - j <= kl && j - i <= kl + ku;
    };
    auto A = [&](int64_t i, int64_t j) -> cx & {
        if constexpr (LDS) return P[(int)(j - j0) * Ri + (int)(i - j0)];
        else return B.at(i, j);
    };
    if constexpr (LDS) {
        // a row's kNB entries are loaded together, then stored to LDS: one
        // memory latency per row instead of one per entry
        for (int r = tid; r < Ri; r += 256) {
            cx v[kNB];
#pragma unroll
            for (int c = 0; c < kNB; ++c) {
                const int64_t i = j0 + r, j = j0 + c;
                v[c] = inband(i, j) ? B.at(i, j) : cx{0.0, 0.0};
            }
#pragma unroll
            for (int c = 0; c < kNB; ++c) P[c * Ri + r] = v[c];
        }
    }
    // furthest column any step so far reaches (kept by every thread alike)
    int64_t ju = st->ju;
    __syncthreads();
    for (int64_t j = j0; j < jend; ++j) {
        const int km = (int)min(kl, n - 1 - j);
        // pivot: first maximum of |re| + |im| over rows j .. j+km
        double best = -1.0;
        int arg = 0;
        for (int t = tid; t <= km; t += 256) {
            const cx a = A(j + t, j);
            const double s = fabs(a.re) + fabs(a.im);
            if (s > best) { best = s; arg = t; }
        }
        for (int off = 32; off >= 1; off >>= 1) {
            const double ob = __shfl_xor(best, off);
            const int oa = __shfl_xor(arg, off);
            if (ob > best || (ob == best && oa < arg)) { best = ob; arg = oa; }
        }
        if (lane == 0) { s_best[wv] = best; s_arg[wv] = arg; }
        __syncthreads();
        // every thread combines the four waves' candidates (the same first
        // maximum), so no second barrier hands the pivot out
        double b = s_best[0];
        int a = s_arg[0];
        for (int q = 1; q < 4; ++q)
            if (s_best[q] > b || (s_best[q] == b && s_arg[q] < a)) { b = s_best[q]; a = s_arg[q]; }
        const int64_t reach = min(j + ku + a, n - 1);
        if (reach > ju) ju = reach;
        if (tid == 0) {
            if (b == 0.0 && st->singular == 0) st->singular = (int)min<int64_t>(j + 1, INT32_MAX);
            piv[j] = j + a;
            juv[j] = ju;
        }
        const int jp = a;
        const int64_t cend = min(jend - 1, ju);  // panel columns within reach
        if (jp != 0 && j + tid <= cend) {
            const int64_t c = j + tid;
            const cx t = A(j, c);
            A(j, c) = A(j + jp, c);
            A(j + jp, c) = t;
        }
        __syncthreads();
        if (km > 0) {
            const cx r = crecip(A(j, j));
            for (int t = 1 + tid; t <= km; t += 256) {
                const cx l = cmul(A(j + t, j), r);
                A(j + t, j) = l;
                // columns four at a time: their loads are independent and go
                // out together (each entry's update is the same operation)
                int64_t c = j + 1;
                for (; c + 3 <= cend; c += 4) {
                    cx a[4], u[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        a[q] = A(j + t, c + q);
                        u[q] = A(j, c + q);
                    }
#pragma unroll
                    for (int q = 0; q < 4; ++q) A(j + t, c + q) = csub_mul(a[q], l, u[q]);
                }
                for (; c <= cend; ++c) A(j + t, c) = csub_mul(A(j + t, c), l, A(j, c));
            }
        }
        __syncthreads();
    }
    if constexpr (LDS) {
        for (int r = tid; r < Ri; r += 256) {
            cx v[kNB];
#pragma unroll
            for (int c = 0; c < kNB; ++c) v[c] = P[c * Ri + r];
#pragma unroll
            for (int c = 0; c < kNB; ++c) {
                const int64_t i = j0 + r, j = j0 + c;
                if (inband(i, j)) B.at(i, j) = v[c];
            }
        }
    }
    if (tid == 0) st->ju = ju;
}

// Replay the panel's swaps and updates on column c = j0 + kNB + blockIdx.x,
// for the steps whose reach includes it (general form: global memory).
__global__ void __launch_bounds__(256) freq_trail(BandDesc B, int64_t j0,
                                                  const int64_t *__restrict__ piv,
                                                  const int64_t *__restrict__ juv) {
#pragma clang fp contract(off)
    const int64_t n = B.n, kl = B.kl;
    const int64_t c = j0 + kNB + blockIdx.x;
    const int64_t jend = min(j0 + kNB, n);
    if (c >= n || c > juv[jend - 1]) return;  // beyond every step's reach: untouched
    const int tid = threadIdx.x;
    for (int64_t p = j0; p < jend; ++p) {
        if (c > juv[p]) continue;  // block-uniform
        const int64_t jp = piv[p] - p;
        if (jp != 0 && tid == 0) {
            const cx t = B.at(p, c);
            B.at(p, c) = B.at(p + jp, c);
            B.at(p + jp, c) = t;
        }
        __syncthreads();
        const int64_t km = min(kl, n - 1 - p);
        const cx u = B.at(p, c);
        for (int64_t t = 1 + tid; t <= km; t += blockDim.x)
            B.at(p + t, c) = csub_mul(B.at(p + t, c), B.at(p + t, p), u);
        __syncthreads();
    }
}

// The same with the column's rows j0 .. j0+R-1 staged in LDS, and all of a
// thread's multipliers of the panel (rows tid + 256 q, q < RPT), the panel's
// pivots and reaches loaded up front, so the 16 steps touch only LDS and
// registers.
template <int RPT, int NC>
__global__ void __launch_bounds__(256) freq_trail_lds(BandDesc B, int64_t j0,
                                                      const int64_t *__restrict__ piv,
                                                      const int64_t *__restrict__ juv, int64_t R) {
#pragma clang fp contract(off)
    __shared__ cx Cl[NC][RPT * 256];
    __shared__ int64_t s_jv[kNB], s_pv[kNB];
    const int64_t n = B.n, kl = B.kl, ku = B.ku;
    const int64_t c0 = j0 + kNB + (int64_t)blockIdx.x * NC;  // columns c0 .. c0+NC-1
    const int64_t jend = min(j0 + kNB, n);
    const int tid = threadIdx.x;
    auto inband = [&](int64_t i, int64_t c) {
        return c < n && i < n && i - c <= kl && c - i <= kl + ku;
    };
    // The reaches, pivots and the columns' rows go out together; the panel's
    // multipliers are loaded one step ahead of their use (two register sets)
    // and serve all NC columns of the workgroup.
    const int64_t reach = juv[jend - 1];
    if (tid < kNB) {
        s_jv[tid] = j0 + tid < jend ? juv[j0 + tid] : -1;
        s_pv[tid] = j0 + tid < jend ? piv[j0 + tid] : j0 + tid;
    }
    cx col[NC][RPT];
#pragma unroll
    for (int k = 0; k < NC; ++k)
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
            const int64_t r = tid + 256 * q;
            col[k][q] = r < R && inband(j0 + r, c0 + k) ? B.at(j0 + r, c0 + k) : cx{0.0, 0.0};
        }
    // multiplier of local row r at step p: L(j0 + r, p) when p < j0 + r <= p + km(p)
    auto lmul = [&](int pp, cx (&L)[RPT]) {
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
            const int64_t p = j0 + pp, i = j0 + tid + 256 * q;
            L[q] = (pp < kNB && p < jend && i > p && i <= p + min(kl, n - 1 - p)) ? B.at(i, p)
                                                                                : cx{0.0, 0.0};
        }
    };
    cx La[RPT], Lb[RPT];
    lmul(0, La);
    if (c0 >= n || c0 > reach) return;  // every column beyond every step's reach: untouched
#pragma unroll
    for (int k = 0; k < NC; ++k)
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
            const int64_t r = tid + 256 * q;
            if (r < R) Cl[k][r] = col[k][q];
        }
    __syncthreads();
    auto step = [&](int pp, const cx (&L)[RPT], cx (&Ln)[RPT]) {
        lmul(pp + 1, Ln);
        const int64_t p = j0 + pp, jv = s_jv[pp];
        if (c0 > jv) return;  // block-uniform: no column of the block within reach
        const int64_t jp = s_pv[pp] - p;
        // column k within reach (block-uniform; the columns within reach are a prefix)
        if (jp != 0 && tid < NC && c0 + tid <= jv && c0 + tid < n) {
            cx *C = Cl[tid];
            const cx t = C[pp];
            C[pp] = C[pp + jp];
            C[pp + jp] = t;
        }
        __syncthreads();
        const int64_t km = min(kl, n - 1 - p);
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            if (c0 + k > jv) break;
            const cx u = Cl[k][pp];
#pragma unroll
            for (int q = 0; q < RPT; ++q) {
                const int64_t r = tid + 256 * q, i = j0 + r;
                if (i > p && i <= p + km) Cl[k][r] = csub_mul(Cl[k][r], L[q], u);
            }
        }
        __syncthreads();
    };
#pragma unroll 1
    for (int pp = 0; pp < kNB; pp += 2) {
        step(pp, La, Lb);
        step(pp + 1, Lb, La);
    }
#pragma unroll
    for (int k = 0; k < NC; ++k)
        for (int64_t r = tid; r < R; r += 256)
            if (inband(j0 + r, c0 + k)) B.at(j0 + r, c0 + k) = Cl[k][r];
}

// ---------------------------------------------------------------------------
// Blocked form, rows in registers.
//
// Panel q holds columns j = q kNB + c, c < kNB, and rows q kNB + r, r < R =
// kNB + kl.  Rows are not moved while a panel is factored: pos[q][r] is the
// row (relative to the panel's first) at which row r ends up, and its
// multipliers are kept with it, apart from the band, as L[q][c][r] (rows
// fastest; 0 outside the band and where the row had become a row of U).
// Applying a panel to a column is then: the rows with pos < kNB, put in that
// order, go through a kNB x kNB unit triangular solve, every other row
// through kNB independent updates, and each is stored at its pos -- the
// operations of the interleaved interchanges and updates, in the same order
// for each element, with no barrier between the steps.
constexpr int kMaxRows = 512;                 // rows of a panel and the one before it
constexpr int kMaxBand = kMaxRows - 2 * kNB;  // widest kl of the blocked form
constexpr int kTrailCols = 4;                // columns per workgroup behind the next panel

struct LuPanels {
    cx *L;
    int *pos;
    int64_t *reach;  // [q] last column any step up to panel q touches
    int R;
};

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// Value of lane P of the lane's row of 16 (DPP row_newbcast).
template <int P>
__device__ __forceinline__ double row_lane(double v) {
    const long long u = __builtin_bit_cast(long long, v);
    const int lo = __builtin_amdgcn_mov_dpp((int)u, 0x150 + P, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_mov_dpp((int)(u >> 32), 0x150 + P, 0xf, 0xf, true);
    return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}
template <int P>
__device__ __forceinline__ cx row_lane(cx v) {
    return {row_lane<P>(v.re), row_lane<P>(v.im)};
}

__device__ __forceinline__ double read_lane(double v, int l) {
    const long long u = __builtin_bit_cast(long long, v);
    const int lo = __builtin_amdgcn_readlane((int)u, l);
    const int hi = __builtin_amdgcn_readlane((int)(u >> 32), l);
    return __builtin_bit_cast(double, ((long long)hi << 32) | (unsigned)lo);
}

// Maximum over the wavefront, uniform: DPP row shifts and broadcasts, then
// lane 63's value.
template <int CTL, int ROWS>
__device__ __forceinline__ int max_step(int v) {
    return max(v, __builtin_amdgcn_update_dpp(v, v, CTL, ROWS, 0xf, false));
}
__device__ __forceinline__ int wave_max(int v) {
    v = max_step<0x111, 0xf>(v);  // row_shr:1, 2, 4, 8
    v = max_step<0x112, 0xf>(v);
    v = max_step<0x114, 0xf>(v);
    v = max_step<0x118, 0xf>(v);
    v = max_step<0x142, 0xa>(v);  // row_bcast:15, 31
    v = max_step<0x143, 0xc>(v);
    return __builtin_amdgcn_readlane(v, 63);
}

// Unit triangular solve of a column held by 16 lanes (lane r: row r), with
// l[p] the row's multipliers (0 from the diagonal on).
__device__ __forceinline__ cx tri_lower(cx x, const cx (&l)[kNB]) {
    static_for<0, kNB - 1>([&](auto P) { x = csub_mul(x, l[P], row_lane<P>(x)); });
    return x;
}

// Lane of the first maximum of non-negative values v over the wavefront: of
// the lanes with the largest v the one with the least ps (distinct).  key is
// v's upper half, or negative for a lane without one (-1: the largest key and
// the least ps; below: any lane, there is none to choose).
__device__ __forceinline__ int first_max(int key, double v, int ps) {
    const int best = wave_max(key);
    unsigned long long k = __ballot(key == best);
    if ((k & (k - 1)) && best > -2) {  // several lanes: by the lower halves, 31 bits and 1, then by ps
        const int lane = threadIdx.x & 63;
        const unsigned lo = best >= 0 ? (unsigned)__builtin_bit_cast(long long, v) : 0u;
        const unsigned top = (unsigned)wave_max(k >> lane & 1 ? (int)(lo >> 1) : -1);
        k &= __ballot(lo >> 1 == top);
        if (const unsigned long long odd = k & __ballot(lo & 1u)) k = odd;
        const int least = -wave_max(k >> lane & 1 ? -ps : -0x7fffffff);
        k &= __ballot(ps == least);
    }
    return __ffsll(k) - 1;
}

// LDS of the two parts of freq_lu (NW wavefronts).
template <int NW>
struct LuShared {
    cx X[kNB][kNB];   // top rows of the columns being updated
    cx Ls[kNB][kNB];  // their multipliers, [p][r]
    struct alignas(16) Cand {  // a wavefront's pivot candidate
        double val;            // |re| + |im|
        int key, pos;          // its key (first_max), the row's position
    } cand[2][NW];
    cx row[2][kNB];  // the pivot's row from the pivot on
    cx rcp[2];       // and its reciprocal
};

// Pivot steps kNB-C .. kNB-C+3 of panel q: a[c] is column kNB-C+c of the
// thread's row, c < C; each step moves the columns down by one as it updates
// them, so the loop body is the same for every step.  Each wavefront leaves
// its candidate's value and position in LDS; after a barrier every wavefront
// picks the winner, whose owner alone writes its row (LDS accesses cost their
// full width with one lane as with 64: eight candidates' rows took longer than
// the second barrier); after that barrier each wavefront reads the row once,
// one column per lane, and takes it from there by readlane.
template <int C, int NW>
__device__ __forceinline__ void pivot_steps(const BandDesc &B, cx *Lq, int R, int64_t j1, int ncol,
                                            int p0, int &ps, cx (&a)[kNB], int64_t &ju, int &sing,
                                            LuShared<NW> &S) {
#pragma clang fp contract(off)
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kl = (int)B.kl, ku = (int)B.ku;
#pragma unroll 1
    for (int i = 0; i < 4; ++i) {
        const int jj = kNB - C + i, buf = i & 1;
        const int64_t j = j1 + jj;
        const int km = (int)min<int64_t>(kl, B.n - 1 - j);  // < 0: no such column
        // pivot: first maximum of |re| + |im| over positions jj .. jj+km
        const double v = fabs(a[0].re) + fabs(a[0].im);
        int t = ps - jj;
        const int key = t >= 0 && t <= km
                            ? (v >= 0.0 ? (int)(__builtin_bit_cast(long long, v) >> 32) : -1)
                            : -2;  // (a NaN below every value)
        const int cl = first_max(key, v, ps);
        if (lane == cl) S.cand[buf][wv] = {v, key, ps};
        __syncthreads();
        const auto win = S.cand[buf][lane & (NW - 1)];
        const int pw = first_max(lane < NW ? win.key : -3, win.val, win.pos);
        const int pp = km < 0 ? jj : __builtin_amdgcn_readlane(win.pos, pw);
        if (wv == pw) {
            const cx rc = crecip(a[0]);
            if (lane == cl) {
#pragma unroll
                for (int c = 0; c < C; ++c) S.row[buf][c] = a[c];
                S.rcp[buf] = rc;
            }
        }
        __syncthreads();
        const cx rcp = S.rcp[buf], mine = S.row[buf][lane & (kNB - 1)];  // (lanes < C)
        if (tid < C && jj + tid < ncol && tid <= kl + ku)  // the row of U
            B.ab[(j + tid) * B.ldab + kl + ku - tid] = mine;
        const int64_t rr = min<int64_t>(j + ku + (pp - jj), B.n - 1);
        if (rr > ju) ju = rr;
        if (__builtin_amdgcn_readlane(win.key, pw) == 0 && sing == 0 && read_lane(win.val, pw) == 0.0)
            sing = (int)min<int64_t>(j + 1, INT32_MAX);
        ps = ps == jj ? pp : ps == pp ? jj : ps;
        t = ps - jj;
        const cx w = cmul(a[0], rcp);
        const bool on = t > 0 && t <= km;
        const cx f = {on ? w.re : 0.0, on ? w.im : 0.0};
        if (p0 >= 0 && p0 < R) Lq[(int64_t)jj * R + p0] = f;
#pragma unroll
        for (int c = 1; c < C; ++c)
            a[c - 1] = csub_mul(a[c], f, cx{read_lane(mine.re, c), read_lane(mine.im, c)});
        a[C - 1] = cx{0.0, 0.0};
    }
    if constexpr (C > 4)
        pivot_steps<C - 4, NW>(B, Lq, R, j1, ncol, p0, ps, a, ju, sing, S);
}

// Workgroup 0: panel q-1 applied to panel q's columns (q > 0), then panel q
// factored.  Thread tid holds row tid of the window that starts kNB above the
// panel, all kNB columns in registers.  The code is kept in loops: run once
// per launch, straight-line code for the 16 steps (70 KB) was bound by its own
// fetch, at about a byte per cycle.
template <int NW>
__device__ __forceinline__ void lu_chain(const BandDesc &B, const LuPanels &W, int64_t q,
                                         LuState *st, LuShared<NW> &S) {
#pragma clang fp contract(off)
    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t n = B.n, j1 = q * kNB;
    const int kl = (int)B.kl, ku = (int)B.ku, ldab = (int)B.ldab, R = W.R;
    const int ncol = (int)min<int64_t>(kNB, n - j1);  // columns of the panel
    // Window row r in column c is the band's element kl + ku + r - kNB - c of
    // that column; rows outside the band read 0 (kOut), as do those past n.
    constexpr uint32_t kOut = 0x80000000u;
    const uint32_t colb = (uint32_t)ldab * (uint32_t)sizeof(cx);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        (void *)(B.ab + j1 * ldab), (short)0, (int)(ncol * colb), 0x00020000);
    cx a[kNB];
    const bool row = tid < R + kNB, old = q > 0 && tid < R;  // old: a row of panel q-1
    // position in the panel before its factorisation (negative: above it)
    const int p0 = row ? (old ? W.pos[(q - 1) * R + tid] : tid) - kNB : kMaxRows;
#pragma unroll
    for (int c = 0; c < kNB; ++c) {
        const int e = kl + ku - kNB + tid - c;
        const bool in = row && (uint32_t)e < (uint32_t)ldab && c < ncol;
        a[c] = __builtin_bit_cast(cx, __builtin_amdgcn_raw_buffer_load_b128(
                                          rs, (int)(in ? (uint32_t)e * (uint32_t)sizeof(cx) : kOut),
                                          (int)(c * colb), 0));
    }
    if (q > 0) {
        const cx *L = W.L + (q - 1) * (int64_t)kNB * R;
        const int rl = min(tid, R - 1);
        cx l[4];  // multipliers on their way, four steps ahead
#pragma unroll
        for (int d = 0; d < 4; ++d) l[d] = L[(int64_t)d * R + rl];
        if (p0 < 0) {
#pragma unroll
            for (int c = 0; c < kNB; ++c) S.X[p0 + kNB][c] = a[c];
#pragma unroll 4
            for (int p = 0; p < kNB; ++p) S.Ls[p][p0 + kNB] = L[(int64_t)p * R + tid];
        }
        __syncthreads();
        if (wv < 4) {  // four columns per wavefront
            const int c = 4 * wv + (lane >> 4), r = lane & 15;
            cx t[kNB];
#pragma unroll
            for (int p = 0; p < kNB; ++p) t[p] = S.Ls[p][r];
            const cx x = tri_lower(S.X[r][c], t);
            S.X[r][c] = x;
            // row j1 - kNB + r of column j1 + c
            if (c < ncol && c + kNB - r <= kl + ku)
                B.ab[(j1 + c) * ldab + kl + ku - kNB + r - c] = x;
        }
        __syncthreads();
        // a step's row of U is read half a step ahead (the wavefront is alone
        // on its SIMD, or nearly: it waits out the LDS latency itself)
        constexpr int HB = kNB / 2;
        cx ua[HB], ub[HB];
#pragma unroll
        for (int c = 0; c < HB; ++c) ua[c] = S.X[0][c];
#pragma unroll 1
        for (int g = 0; g < kNB; g += 4)
#pragma unroll
            for (int d = 0; d < 4; ++d) {
                const cx f = {old ? l[d].re : 0.0, old ? l[d].im : 0.0};
                l[d] = L[(int64_t)min(g + d + 4, kNB - 1) * R + rl];
#pragma unroll
                for (int c = 0; c < HB; ++c) ub[c] = S.X[g + d][HB + c];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int c = 0; c < HB; ++c) a[c] = csub_mul(a[c], f, ua[c]);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int c = 0; c < HB; ++c) ua[c] = S.X[min(g + d + 1, kNB - 1)][c];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int c = 0; c < HB; ++c) a[HB + c] = csub_mul(a[HB + c], f, ub[c]);
                __builtin_amdgcn_sched_barrier(0);
            }
    }
    int64_t ju = st->ju;
    int sing = 0, ps = p0;
    pivot_steps<kNB, NW>(B, W.L + q * (int64_t)kNB * R, R, j1, ncol, p0, ps, a, ju, sing, S);
    if (p0 >= 0 && p0 < R) W.pos[q * R + p0] = ps;
    if (tid == 0) {
        st->ju = ju;
        if (sing && st->singular == 0) st->singular = sing;
        W.reach[q] = ju;
    }
}

// Panel q applied to columns c0 .. c0+kTrailCols-1 behind the next panel.
template <int NW>
__device__ __forceinline__ void lu_trail(const BandDesc &B, const LuPanels &W, int64_t q,
                                         int64_t c0, LuShared<NW> &S) {
#pragma clang fp contract(off)
    constexpr int NC = kTrailCols;
    const int64_t n = B.n, j0 = q * kNB;
    const int kl = (int)B.kl, ku = (int)B.ku, ldab = (int)B.ldab;
    if (c0 >= n || c0 > W.reach[q]) return;  // beyond every step's reach: untouched
    const int tid = threadIdx.x, R = W.R;
    const cx *L = W.L + q * (int64_t)kNB * R;
    const int d0 = (int)(c0 - j0), ncol = (int)min<int64_t>(NC, n - c0);
    cx *col = B.ab + c0 * ldab;
    // panel row r in column c0 + k is element kl + ku + r - d0 - k of that column
    auto elem = [&](int r, int k) { return kl + ku + r - d0 - k; };
    const bool row = tid < R;
    const int rl = min(tid, R - 1), ps = W.pos[q * R + rl];
    // (0 outside the band, as in lu_chain)
    constexpr uint32_t kOut = 0x80000000u;
    const uint32_t colb = (uint32_t)ldab * (uint32_t)sizeof(cx);
    const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
        (void *)col, (short)0, (int)(ncol * colb), 0x00020000);
    cx x[NC];
#pragma unroll
    for (int k = 0; k < NC; ++k) {
        const bool in = row && k < ncol && elem(tid, k) >= 0;
        x[k] = __builtin_bit_cast(cx, __builtin_amdgcn_raw_buffer_load_b128(
                   rs, (int)(in ? (uint32_t)elem(tid, k) * (uint32_t)sizeof(cx) : kOut),
                   (int)(k * colb), 0));
    }
    cx l[4];  // multipliers on their way, four steps ahead
#pragma unroll
    for (int d = 0; d < 4; ++d) l[d] = L[(int64_t)d * R + rl];
    if (row && ps < kNB) {
#pragma unroll
        for (int k = 0; k < NC; ++k) S.X[ps][k] = x[k];
#pragma unroll 4
        for (int p = 0; p < kNB; ++p) S.Ls[p][ps] = L[(int64_t)p * R + tid];
    }
    __syncthreads();  // (also: every row is read before any is written)
    if (tid < 64) {
        const int k = tid >> 4, r = tid & 15;
        cx t[kNB];
#pragma unroll
        for (int p = 0; p < kNB; ++p) t[p] = S.Ls[p][r];
        const cx y = tri_lower(S.X[r][k], t);
        S.X[r][k] = y;
        if (k < ncol && elem(r, k) >= 0) col[k * ldab + elem(r, k)] = y;
    }
    __syncthreads();
    if (!row || ps < kNB || j0 + ps >= n) return;  // (the top rows are written)
#pragma unroll 1
    for (int g = 0; g < kNB; g += 4)
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            const cx f = l[d];
            l[d] = L[(int64_t)min(g + d + 4, kNB - 1) * R + rl];
            __builtin_amdgcn_sched_barrier(0);  // (bounds the registers)
#pragma unroll
            for (int k = 0; k < NC; ++k) x[k] = csub_mul(x[k], f, S.X[g + d][k]);
        }
#pragma unroll
    for (int k = 0; k < NC; ++k)
        if (k < ncol && elem(ps, k) >= 0) col[k * ldab + elem(ps, k)] = x[k];
}

// Launch q: workgroup 0 makes panel q (from panel q-1), the others apply panel
// q-1 to the columns behind panel q.
template <int NW>
__global__ void __launch_bounds__(64 * NW) freq_lu(BandDesc B, LuPanels W, int64_t q, LuState *st) {
    __shared__ LuShared<NW> S;
    if (blockIdx.x == 0)
        lu_chain<NW>(B, W, q, st, S);
    else
        lu_trail<NW>(B, W, q - 1, (q + 1) * kNB + (int64_t)(blockIdx.x - 1) * kTrailCols, S);
}

// a / b for y = 1 / b rounded: Markstein's quotient (corrections by the
// exactly computed remainder) is the correctly rounded one while nothing
// leaves the range of normal numbers (quot_ok).
__device__ __forceinline__ double quot(double a, double b, double y) {
    double q = a * y;
    q = __builtin_fma(__builtin_fma(-b, q, a), y, q);
    return __builtin_fma(__builtin_fma(-b, q, a), y, q);
}
__device__ __forceinline__ bool quot_ok(double a, double b) {
    const double m = fabs(a);
    return m > 0x1p-400 && m < 0x1p400 && b > 0x1p-400 && b < 0x1p400;
}

// One right-hand side per workgroup: b = -s, forward sweep panel by panel
// (window rows j0 .. j0+R-1), backward sweep by blocks of kNB columns (window
// rows jb-kl-ku .. jb+kNB-1), the windows a power-of-two ring in LDS (slot of
// b[i] = i & mask).  Per panel the first wavefront runs the kNB dependent
// steps on kNB lanes (values passed by DPP), then every thread applies them to
// its rows (one and QB per thread); a panel's factors are loaded into registers
// while the dependent steps before them run.
template <int QB>
__global__ void __launch_bounds__(512) freq_subst(BandDesc B, LuPanels W, const cx *__restrict__ S,
                                                  cx *__restrict__ U, int64_t mask) {
#pragma clang fp contract(off)
    extern __shared__ cx ring[];
    __shared__ cx us[2][kNB], xt[kNB], tri[2][kNB][kNB];
    const int64_t n = B.n;
    const int tid = threadIdx.x, T = blockDim.x, R = W.R;
    const bool first = tid < 64;
    const cx *s = S + (int64_t)blockIdx.x * n;
    cx *u = U + (int64_t)blockIdx.x * n;
    const int64_t np = (n + kNB - 1) / kNB;
    // element e of a column whose address is uniform (32-bit lane offset)
    auto at = [](const cx *col, int e) {
        return *(const cx *)((const char *)col + (uint32_t)e * (uint32_t)sizeof(cx));
    };

    // ---- forward
    for (int64_t i = tid; i < min<int64_t>(R, n); i += T) ring[i & mask] = cx{-s[i].re, -s[i].im};
    cx l[kNB];
    int ps = 0;
    auto load_f = [&](int64_t q) {  // the row's multipliers and position
        if (q >= np) return;
        const int r = min(tid, R - 1);
        ps = W.pos[q * R + r];
#pragma unroll
        for (int p = 0; p < kNB; ++p) l[p] = at(W.L + (q * kNB + p) * R, r);
    };
    load_f(0);
    __syncthreads();
    for (int64_t q = 0; q < np; ++q) {
        const int64_t j0 = q * kNB;
        const int buf = (int)(q & 1);
        // the value entering the window for the next panel
        const int64_t e = j0 + R + tid;
        cx in{0.0, 0.0};
        if (tid < kNB && e < n) in = cx{-s[e].re, -s[e].im};
        // (rows past the last are 0: a 0 multiplier must not meet a NaN)
        cx x = tid < R && j0 + tid < n ? ring[(j0 + tid) & mask] : cx{0.0, 0.0};
        if (tid < R && ps < kNB) {  // the top rows, in their final order
            xt[ps] = x;
#pragma unroll
            for (int p = 0; p < kNB; ++p) tri[0][p][ps] = l[p];
        }
        __syncthreads();  // the ring has been read
        if (first) {
            cx t[kNB];
#pragma unroll
            for (int p = 0; p < kNB; ++p) t[p] = tri[0][p][tid & (kNB - 1)];
            const cx y = tri_lower(xt[tid & (kNB - 1)], t);
            if (tid < kNB) {
                us[buf][tid] = y;
                if (j0 + tid < n) u[j0 + tid] = y;
            }
        }
        __syncthreads();
#pragma unroll
        for (int p = 0; p < kNB; ++p) x = csub_mul(x, l[p], us[buf][p]);
        if (tid < R && ps >= kNB) ring[(j0 + ps) & mask] = x;
        if (tid < kNB && e < n) ring[e & mask] = in;
        __builtin_amdgcn_sched_barrier(0);  // the next panel's loads reuse l's registers
        load_f(q + 1);
        __syncthreads();
    }

    // ---- backward
    // Row e of block jb's window is jb - H + e (H = kl + ku, e < H the rows
    // above the block); its entry in column jb + p is the band's
    // ab[(jb + p) ldab + e - p], inside the band from e = p on.
    const int H = (int)(B.kl + B.ku);
    const int64_t jl = (np - 1) * kNB;
    for (int64_t i = max<int64_t>(0, jl - H) + tid; i < n; i += T) ring[i & mask] = u[i];
    // Buffer loads give 0 outside the band, the matrix and the window without
    // a branch (offset kOut is past the 16 columns the resource covers).
    constexpr uint32_t kOut = 0x80000000u;
    const uint32_t colb = (uint32_t)B.ldab * (uint32_t)sizeof(cx);
    auto band = [&](int64_t jb, uint32_t voff, int p) {
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            (void *)(B.ab + jb * B.ldab), (short)0, (int)(kNB * colb), 0x00020000);
        const auto v = __builtin_amdgcn_raw_buffer_load_b128(
            rs, (int)voff, (int)((uint32_t)p * (colb - (uint32_t)sizeof(cx))), 0);
        return __builtin_bit_cast(cx, v);
    };
    auto entry = [&](int64_t jb, int e, int p) {  // p uniform
        const int lo = (int)max<int64_t>(p, H - jb);
        return band(jb, e >= lo && e < H && jb + p < n ? (uint32_t)e * (uint32_t)sizeof(cx) : kOut, p);
    };
    // loaded one block ahead: the rows' entries of the block's columns, the
    // pivots (lane p: column p's)
    cx w[QB][kNB], piv{1.0, 0.0};
    auto load_b = [&](int64_t jb) {
        if (jb < 0) return;
#pragma unroll
        for (int m = 0; m < QB; ++m)
#pragma unroll
            for (int p = 0; p < kNB; ++p) w[m][p] = entry(jb, tid + T * m, p);
        if (tid < kNB) piv = jb + tid < n ? at(B.ab + (jb + tid) * B.ldab, H) : cx{1.0, 0.0};
    };
    // two blocks ahead, through LDS: the block's own upper triangle, [p][r]
    const int dp = tid / kNB, dr = tid % kNB;  // (tid < kNB kNB)
    auto load_d = [&](int64_t jb) {
        const bool ok = tid < kNB * kNB && dp > dr && dp - dr <= H && jb + dp < n;
        const uint32_t o = (uint32_t)dp * (colb - (uint32_t)sizeof(cx)) +
                           (uint32_t)(H + dr) * (uint32_t)sizeof(cx);
        return jb >= 0 ? band(jb, ok ? o : kOut, 0) : cx{0.0, 0.0};
    };
    cx dn = load_d(jl);
    if (tid < kNB * kNB) tri[(jl / kNB) & 1][dp][dr] = dn;
    dn = load_d(jl - kNB);
    load_b(jl);
    __syncthreads();
    for (int64_t jb = jl; jb >= 0; jb -= kNB) {
        const int buf = (int)(jb / kNB) & 1;
        // the value entering the window for the next block
        const int64_t e = jb - H - kNB + tid;
        cx in{0.0, 0.0};
        if (tid < kNB && e >= 0) in = u[e];
        if (first) {
            const int r = tid & (kNB - 1);
            cx t[kNB];
#pragma unroll
            for (int p = 0; p < kNB; ++p) t[p] = tri[buf][p][r];
            cx x = tid < kNB && jb + tid < n ? ring[(jb + tid) & mask] : cx{0.0, 0.0};
            const double den = piv.re * piv.re + piv.im * piv.im, rden = 1.0 / den;
            static_for<0, kNB>([&](auto I) {
                constexpr int p = kNB - 1 - decltype(I)::value;
                // x / piv in lane p (cdiv with the reciprocal at hand)
                const double a = x.re * piv.re + x.im * piv.im, b = x.im * piv.re - x.re * piv.im;
                cx y = {quot(a, den, rden), quot(b, den, rden)};
                if (__any(tid == p && !(quot_ok(a, den) && quot_ok(b, den)))) y = {a / den, b / den};
                x = {tid == p ? y.re : x.re, tid == p ? y.im : x.im};
                x = csub_mul(x, t[p], row_lane<p>(x));  // (t is 0 at rows from p on)
            });
            if (tid < kNB) {
                us[buf][tid] = x;
                if (jb + tid < n) u[jb + tid] = x;
            }
        }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < QB; ++m) {
            const int r = tid + T * m;
            const int64_t i = jb - H + r;
            const bool live = r < H && i >= 0;
            cx x = live ? ring[i & mask] : cx{0.0, 0.0};
#pragma unroll
            for (int p = kNB - 1; p >= 0; --p)
                x = csub_mul(x, w[m][p], us[buf][p]);
            if (live) ring[i & mask] = x;
            __builtin_amdgcn_sched_barrier(0);  // (the next block's loads reuse w's registers)
        }
        load_b(jb - kNB);
        if (tid < kNB * kNB) tri[buf ^ 1][dp][dr] = dn;
        dn = load_d(jb - 2 * kNB);
        if (tid < kNB && e >= 0) ring[e & mask] = in;
        __syncthreads();
    }
}

// Column-replay form: one right-hand side per workgroup of 1024: b = -s, forward sweep with
// interchanges (window b[j .. j+kl]), backward sweep (window b[j-kl-ku .. j]),
// the windows a power-of-two ring in LDS (slot of b[q] = q & mask).  The
// values entering the window come from global memory in chunks of 1024 per
// sweep into a double-buffered LDS stage, and each thread loads its
// multipliers of step j+1 while step j runs (two register sets, alternating).
constexpr int kStage = 1024;

template <int RPT>
__global__ void __launch_bounds__(1024) freq_solve(BandDesc B, const int64_t *__restrict__ piv,
                                                   const cx *__restrict__ S, cx *__restrict__ U,
                                                   int64_t mask) {
#pragma clang fp contract(off)
    extern __shared__ cx W[];
    cx *St = W + (mask + 1);  // 2 x kStage
    const int64_t n = B.n, kl = B.kl, ku = B.ku;
    const cx *s = S + (int64_t)blockIdx.x * n;
    cx *u = U + (int64_t)blockIdx.x * n;
    const int tid = threadIdx.x;
    cx la[RPT], lb[RPT];

    // ---- forward: step j's rows j+t, t = 1 + tid + 1024 q <= lm(j); entering b[j+kl+1]
    auto lf = [&](int64_t j, cx (&l)[RPT]) {
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
            const int64_t t = 1 + tid + 1024 * q;
            l[q] = (j < n && t <= min(kl, n - 1 - j)) ? B.at(j + t, j) : cx{0.0, 0.0};
        }
    };
    auto fwd = [&](int64_t j, const cx (&cur)[RPT], cx (&nxt)[RPT]) {
        if (j % kStage == 0) {  // stage b[j+kl+1 ..] of the next chunk
            const int64_t q = j + kl + 1 + tid;
            St[((j / kStage) & 1) * kStage + tid] = q < n ? cx{-s[q].re, -s[q].im} : cx{0.0, 0.0};
        }
        lf(j + 1, nxt);
        if (tid == 0) {
            const int64_t l = piv[j];
            if (l != j) {
                const cx t = W[l & mask];
                W[l & mask] = W[j & mask];
                W[j & mask] = t;
            }
        }
        __syncthreads();
        const cx bj = W[j & mask];
        const int64_t lm = min(kl, n - 1 - j);
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
            const int64_t t = 1 + tid + 1024 * q;
            if (t <= lm) W[(j + t) & mask] = csub_mul(W[(j + t) & mask], cur[q], bj);
        }
        __syncthreads();
        if (tid == 0) {
            u[j] = bj;
            const int64_t q = j + kl + 1;
            if (q < n) W[q & mask] = St[((j / kStage) & 1) * kStage + (j % kStage)];
        }
    };
    for (int64_t q = tid; q <= min(kl, n - 1); q += blockDim.x) W[q & mask] = cx{-s[q].re, -s[q].im};
    lf(0, la);
    __syncthreads();
    int64_t j = 0;
    for (; j + 1 < n; j += 2) {
        fwd(j, la, lb);
        fwd(j + 1, lb, la);
    }
    if (j < n) fwd(j, la, lb);
    __syncthreads();

    // ---- backward: step j's rows i = max(0, j-kl-ku) + tid + 1024 q < j; entering
    // b[j-kl-ku-1], staged in chunks counted from the top (k = n-1-j)
    auto ub = [&](int64_t jj, cx (&l)[RPT]) {
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
            const int64_t i = max<int64_t>(0, jj - kl - ku) + tid + 1024 * q;
            l[q] = (jj >= 0 && i < jj) ? B.at(i, jj) : cx{0.0, 0.0};
        }
    };
    auto bwd = [&](int64_t jj, const cx (&cur)[RPT], cx (&nxt)[RPT]) {
        const int64_t k = n - 1 - jj;
        if (k % kStage == 0) {
            const int64_t q = jj - kl - ku - 1 - tid;
            St[((k / kStage) & 1) * kStage + tid] = q >= 0 ? u[q] : cx{0.0, 0.0};
        }
        ub(jj - 1, nxt);
        if (tid == 0) W[jj & mask] = cdiv(W[jj & mask], B.at(jj, jj));
        __syncthreads();
        const cx bj = W[jj & mask];
        const int64_t i0 = max<int64_t>(0, jj - kl - ku);
#pragma unroll
        for (int q = 0; q < RPT; ++q) {
            const int64_t i = i0 + tid + 1024 * q;
            if (i < jj) W[i & mask] = csub_mul(W[i & mask], cur[q], bj);
        }
        __syncthreads();
        if (tid == 0) {
            u[jj] = bj;
            const int64_t q = jj - kl - ku - 1;
            if (q >= 0) W[q & mask] = St[((k / kStage) & 1) * kStage + (k % kStage)];
        }
    };
    const int64_t w0 = max<int64_t>(0, n - 1 - kl - ku);
    for (int64_t q = w0 + tid; q < n; q += blockDim.x) W[q & mask] = u[q];
    ub(n - 1, la);
    __syncthreads();
    int64_t jj = n - 1;
    for (; jj - 1 >= 0; jj -= 2) {
        bwd(jj, la, lb);
        bwd(jj - 1, lb, la);
    }
    if (jj >= 0) bwd(jj, la, lb);
}

// ---------------------------------------------------------------------------
// Host side: damping and summed coefficients exactly as the oracle computes
// them (src/freqCpmlFor2dAw.m:52-89 with src/dampPml.m:16-18).
static void freq_host_setup(const double *m, int64_t nz, int64_t nx, int N, int nB, double dz,
                            double dx, std::vector<double> &xd, std::vector<double> &zd,
                            FreqCoef &fc) {
    std::vector<double> coeff(N);
    staggered_coefficients(N, coeff.data());
    const int k = 2 * N - 1;
    for (int o = 0; o < kMaxOff; ++o) fc.c[o] = 0;
    for (int ii = 1; ii <= N; ++ii)
        for (int jj = 1; jj <= N; ++jj) {
            const int o1 = ii + jj - 1, o2 = ii - jj;
            const double p = coeff[ii - 1] * coeff[jj - 1];
            fc.c[o1 + k] = fc.c[o1 + k] + p;
            fc.c[o2 + k] = fc.c[o2 + k] - p;
            fc.c[-o1 + k] = fc.c[-o1 + k] + p;
            fc.c[-o2 + k] = fc.c[-o2 + k] - p;
        }
    xd.assign(nz * nx, 0.0);
    zd.assign(nz * nx, 0.0);
    if (nB == 0) return;
    const double logR = std::log(1e-6);
    const double Lx = nB * dx, Lz = nB * dz;
    for (int j = 0; j < nB; ++j)
        for (int64_t i = 0; i < nz; ++i) {
            const int64_t jl = j, jr = nx - nB + j;
            const double ul = (nB - j) * dx, ur = (j + 1) * dx;
            const double vl = std::sqrt(1. / m[jl * nz + i]), vr = std::sqrt(1. / m[jr * nz + i]);
            const double d0l = -(3 * vl) / (2 * Lx) * logR, d0r = -(3 * vr) / (2 * Lx) * logR;
            const double sl = (ul / Lx) * (ul / Lx), sr = (ur / Lx) * (ur / Lx);
            xd[jl * nz + i] = d0l * sl;
            xd[jr * nz + i] = d0r * sr;
        }
    for (int64_t j = 0; j < nx; ++j)
        for (int i = 0; i < nB; ++i) {
            const int64_t ii = nz - nB + i;
            const double u = (i + 1) * dz;
            const double v = std::sqrt(1. / m[j * nz + ii]);
            const double d0 = -(3 * v) / (2 * Lz) * logR;
            zd[j * nz + ii] = d0 * ((u / Lz) * (u / Lz));
        }
}

static int64_t freq_nnz(int64_t nz, int64_t nx, int k, std::vector<int64_t> *rowptr) {
    std::vector<int64_t> cz(nz), cxn(nx);
    for (int64_t i = 0; i < nz; ++i) {
        int64_t t = 0;
        for (int o = -k; o <= k; ++o) t += (o != 0 && i + o >= 0 && i + o < nz);
        cz[i] = t;
    }
    for (int64_t j = 0; j < nx; ++j) {
        int64_t t = 0;
        for (int o = -k; o <= k; ++o) t += (o != 0 && j + o >= 0 && j + o < nx);
        cxn[j] = t;
    }
    int64_t e = 0;
    if (rowptr) rowptr->resize(nz * nx + 1);
    for (int64_t j = 0; j < nx; ++j)
        for (int64_t i = 0; i < nz; ++i) {
            if (rowptr) (*rowptr)[j * nz + i] = e;
            e += cz[i] + cxn[j] + 1;
        }
    if (rowptr) (*rowptr)[nz * nx] = e;
    return e;
}

static void freq_validate(const double *m, int64_t nz, int64_t nx, double w, int N, int nB,
                          double dz, double dx) {
    if (!m) fail(SSSI_EINVAL, "model must not be NULL");
    if (nz < 1 || nx < 1 || nz > (1 << 24) || nx > (1 << 24) || nz * nx > ((int64_t)1 << 28))
        fail(SSSI_EINVAL, "model %lldx%lld out of range", (long long)nz, (long long)nx);
    if (N < 1 || N > 8) fail(SSSI_EINVAL, "nDiffOrder must be in 1..8");
    if (nB < 0 || nB > nz || 2 * (int64_t)nB > nx)
        fail(SSSI_EINVAL, "nBoundary must satisfy 0 <= nBoundary <= nz and 2 nBoundary <= nx");
    if (!std::isfinite(w) || !(dz > 0) || !(dx > 0) || !std::isfinite(dz) || !std::isfinite(dx))
        fail(SSSI_EINVAL, "w must be finite and dz, dx positive");
    for (int64_t q = 0; q < nz * nx; ++q)
        if (!std::isfinite(m[q]) || !(m[q] > 0))
            fail(SSSI_EINVAL, "model (squared slowness) must be finite and positive (element %lld)",
                 (long long)q);
}

// Device matrix in band form (and CSR on request).
struct FreqSystem {
    int64_t nz, nx, n, kl, ku, ldab;
    int k;
    bool form_blocked = false;  // (chosen by factor)
    OwnedStream s;  // before the buffers: destroyed after them
    DevBuf<cx> ab;
    DevBuf<int64_t> piv, juv;  // column-replay form: per column
    DevBuf<cx> lp;             // blocked form (LuPanels)
    DevBuf<int> pos;
    DevBuf<int64_t> reach;
    DevBuf<LuState> st;
    // Blocked form up to kMaxBand, where a panel's rows still fit 512 threads
    // with all 16 columns in registers; the column replay beyond (1024 threads
    // have half the registers each: 145 spilled in the pivot chain).  Whole call
    // with 20 sources, ms, blocked / replay: band 246 13.7 / 21.5, 360 20.8 /
    // 36.8, 480 30.4 / 50.3; with 1024 threads 483 86.6 / 50.8, 600 120 / 86, 771
    // 161 / 154, 900 191 / 187.
    // SSSI_FREQ_NC = 1, 2 or 4: the column replay at every band, with that many
    // columns per workgroup.
    static int replay_columns() {
        const char *e = std::getenv("SSSI_FREQ_NC");
        const int v = e ? std::atoi(e) : 0;
        return v == 1 || v == 2 || v == 4 ? v : 0;
    }
    bool blocked() const { return form_blocked; }
    // Whether the panels of the blocked form (a third of the band's bytes on wide
    // bands, more than its bytes on narrow ones) fit beside what the replay needs
    // too; looked up where they are large enough to matter.
    bool panels_fit(int nsrc) const {
        const int64_t np = (n + kNB - 1) / kNB;
        const double need = (double)np * (kNB + kl) * (kNB * sizeof(cx) + sizeof(int));
        if (need < 1e9) return true;
        size_t free_now = 0, total = 0;
        SSSI_HIP(hipMemGetInfo(&free_now, &total));
        return need + 2.0 * n * nsrc * sizeof(cx) + 256e6 <= (double)free_now;
    }
    LuPanels panels() const { return LuPanels{lp.p, pos.p, reach.p, (int)(kNB + kl)}; }

    FreqSystem(const double *m, int64_t nz_, int64_t nx_, double w, int N, int nB, double dz,
               double dx, bool band, int64_t *rowptr_out, int64_t *col_out, double *val_out)
        : nz(nz_), nx(nx_), n(nz_ * nx_), k(2 * N - 1) {
        kl = (int64_t)k * nz;
        ku = kl;
        ldab = 2 * kl + ku + 1;
        if (band && (double)ldab * n * sizeof(cx) > 200e9)
            fail(SSSI_ENOMEM, "band storage of %.1f GB exceeds the device budget",
                 (double)ldab * n * sizeof(cx) / 1e9);
        std::vector<double> xd, zd;
        FreqCoef fc;
        freq_host_setup(m, nz, nx, N, nB, dz, dx, xd, zd, fc);
        s.create();
        DevBuf<double> dm(n), dxd(n), dzd(n);
        SSSI_HIP(hipMemcpyAsync(dm.p, m, dm.bytes(), hipMemcpyHostToDevice, s));
        SSSI_HIP(hipMemcpyAsync(dxd.p, xd.data(), dxd.bytes(), hipMemcpyHostToDevice, s));
        SSSI_HIP(hipMemcpyAsync(dzd.p, zd.data(), dzd.bytes(), hipMemcpyHostToDevice, s));
        std::vector<int64_t> rp;
        DevBuf<int64_t> drp, dcol;
        DevBuf<cx> dval;
        if (rowptr_out) {
            const int64_t nnz = freq_nnz(nz, nx, k, &rp);
            drp.alloc(n + 1);
            dcol.alloc(nnz);
            dval.alloc(nnz);
            SSSI_HIP(hipMemcpyAsync(drp.p, rp.data(), drp.bytes(), hipMemcpyHostToDevice, s));
        }
        BandDesc B{nullptr, n, kl, ku, ldab};
        if (band) {
            ab.alloc((size_t)ldab * n);
            SSSI_HIP(hipMemsetAsync(ab.p, 0, ab.bytes(), s));
            B.ab = ab.p;
        }
        const unsigned nb = (unsigned)std::min<int64_t>(65535, (n + 255) / 256);
        hipLaunchKernelGGL(freq_assemble, dim3(nb), dim3(256), 0, s, dm.p, dxd.p, dzd.p, fc,
                           (int)nz, (int)nx, k, w, dz, dx, B, rowptr_out ? drp.p : nullptr,
                           dcol.p, dval.p);
        SSSI_HIP(hipGetLastError());
        if (rowptr_out) {
            std::memcpy(rowptr_out, rp.data(), rp.size() * sizeof(int64_t));
            SSSI_HIP(hipMemcpyAsync(col_out, dcol.p, dcol.bytes(), hipMemcpyDeviceToHost, s));
            SSSI_HIP(hipMemcpyAsync(val_out, dval.p, dval.bytes(), hipMemcpyDeviceToHost, s));
        }
        SSSI_HIP(hipStreamSynchronize(s));
    }

    // dynamic LDS a workgroup may use on the current device
    static size_t lds_limit() {
        int dev = 0;
        SSSI_HIP(hipGetDevice(&dev));
        hipDeviceProp_t prop;
        SSSI_HIP(hipGetDeviceProperties(&prop, dev));
        return prop.sharedMemPerBlock;
    }

    float factor(int nsrc) {
        const int64_t np = (n + kNB - 1) / kNB;
        form_blocked = kl <= kMaxBand && replay_columns() == 0 && panels_fit(nsrc);
        if (blocked()) {
            lp.alloc((size_t)(np * kNB * (kNB + kl)));
            pos.alloc((size_t)(np * (kNB + kl)));
            reach.alloc((size_t)np);
        } else {
            piv.alloc(n);
            juv.alloc(n);
        }
        st.alloc(1);
        SSSI_HIP(hipMemsetAsync(st.p, 0, sizeof(LuState), s));
        BandDesc B{ab.p, n, kl, ku, ldab};
        hipEvent_t e0, e1;
        SSSI_HIP(hipEventCreate(&e0));
        SSSI_HIP(hipEventCreate(&e1));
        SSSI_HIP(hipEventRecord(e0, s));
        for (int64_t q = 0; blocked() && q < np; ++q) {
            // columns behind panel q that panel q-1 reaches
            const int64_t c0 = (q + 1) * kNB, c1 = std::min(n - 1, q * kNB - 1 + kl + ku);
            const int64_t nt = q > 0 && c1 >= c0 ? (c1 - c0 + kTrailCols) / kTrailCols : 0;
            const dim3 g((unsigned)(1 + nt));
            if (kl + 2 * kNB <= 256)
                hipLaunchKernelGGL(freq_lu<4>, g, dim3(256), 0, s, B, panels(), q, st.p);
            else
                hipLaunchKernelGGL(freq_lu<8>, g, dim3(512), 0, s, B, panels(), q, st.p);
        }
        const int64_t R = std::min<int64_t>(n, kNB + kl);  // panel rows (and a column's)
        const size_t plds = (size_t)kNB * R * sizeof(cx);
        const bool panel_lds = plds + 1024 <= lds_limit();
        const int rpt = R <= 256 ? 1 : R <= 512 ? 2 : R <= 1024 ? 4 : 0;
        // columns per workgroup of the replay: two share one load of the
        // panel's multipliers (every workgroup reads the same panel, so fewer
        // workgroups contend less for its cache lines): 1050 replays at kl = 360
        // take 67.2 ms at 2 columns, 77.3 ms at 1 and 78.5 ms at 4.
        const int trail_nc = replay_columns() ? replay_columns() : 2;
        for (int64_t j0 = 0; !blocked() && j0 < n; j0 += kNB) {
            if (panel_lds)
                hipLaunchKernelGGL(freq_panel<true>, dim3(1), dim3(256), plds, s, B, j0, piv.p,
                                   juv.p, st.p, R);
            else
                hipLaunchKernelGGL(freq_panel<false>, dim3(1), dim3(256), 0, s, B, j0, piv.p,
                                   juv.p, st.p, R);
            const int64_t c0 = j0 + kNB, c1 = std::min(n - 1, j0 + kNB - 1 + kl + ku);
            if (c1 < c0) continue;
            const dim3 g((unsigned)(c1 - c0 + 1));
            const dim3 g2((unsigned)((c1 - c0 + 2) / 2)), g4((unsigned)((c1 - c0 + 4) / 4));
            switch (rpt * (trail_nc == 4 ? 100 : trail_nc == 2 ? 10 : 1)) {
                case 1: hipLaunchKernelGGL((freq_trail_lds<1, 1>), g, dim3(256), 0, s, B, j0, piv.p, juv.p, R); break;
                case 2: hipLaunchKernelGGL((freq_trail_lds<2, 1>), g, dim3(256), 0, s, B, j0, piv.p, juv.p, R); break;
                case 4: hipLaunchKernelGGL((freq_trail_lds<4, 1>), g, dim3(256), 0, s, B, j0, piv.p, juv.p, R); break;
                case 10: hipLaunchKernelGGL((freq_trail_lds<1, 2>), g2, dim3(256), 0, s, B, j0, piv.p, juv.p, R); break;
                case 20: hipLaunchKernelGGL((freq_trail_lds<2, 2>), g2, dim3(256), 0, s, B, j0, piv.p, juv.p, R); break;
                case 40: hipLaunchKernelGGL((freq_trail_lds<4, 2>), g2, dim3(256), 0, s, B, j0, piv.p, juv.p, R); break;
                case 100: hipLaunchKernelGGL((freq_trail_lds<1, 4>), g4, dim3(256), 0, s, B, j0, piv.p, juv.p, R); break;
                case 200: hipLaunchKernelGGL((freq_trail_lds<2, 4>), g4, dim3(256), 0, s, B, j0, piv.p, juv.p, R); break;
                case 400: hipLaunchKernelGGL((freq_trail_lds<4, 4>), g4, dim3(256), 0, s, B, j0, piv.p, juv.p, R); break;
                default: hipLaunchKernelGGL(freq_trail, g, dim3(256), 0, s, B, j0, piv.p, juv.p);
            }
        }
        SSSI_HIP(hipGetLastError());
        SSSI_HIP(hipEventRecord(e1, s));
        LuState h{};
        SSSI_HIP(hipMemcpyAsync(&h, st.p, sizeof(h), hipMemcpyDeviceToHost, s));
        SSSI_HIP(hipStreamSynchronize(s));
        float ms = 0;
        SSSI_HIP(hipEventElapsedTime(&ms, e0, e1));
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        if (h.singular)
            fail(SSSI_EINVAL, "the impedance matrix is singular (zero pivot in column %d)",
                 h.singular);
        return ms;
    }

    float solve(const double *S, int nsrc, double *U) {
        // window of the wider sweep, the backward one, and (blocked) a block
        int64_t ring = 1;
        while (ring < kl + ku + (blocked() ? 2 * kNB : 1)) ring <<= 1;
        const size_t sh = (ring + (blocked() ? 0 : 2 * kStage)) * sizeof(cx);
        if (sh > lds_limit())
            fail(SSSI_EINVAL, "band too wide for the solve's LDS window (kl = (2 nDiffOrder - 1) "
                 "nz = %lld; the window of 2 kl + 1 values, rounded up to a power of two, and "
                 "the staging must fit %zu bytes of LDS)", (long long)kl, lds_limit());
        const int64_t rows = kl + ku;  // per step, the backward sweep's is the wider
        const int rpt = rows <= 1024 ? 1 : rows <= 2048 ? 2 : rows <= 4096 ? 4 : 8;
        DevBuf<cx> dS((size_t)n * nsrc), dU((size_t)n * nsrc);
        SSSI_HIP(hipMemcpyAsync(dS.p, S, dS.bytes(), hipMemcpyHostToDevice, s));
        BandDesc B{ab.p, n, kl, ku, ldab};
        hipEvent_t e0, e1;
        SSSI_HIP(hipEventCreate(&e0));
        SSSI_HIP(hipEventCreate(&e1));
        SSSI_HIP(hipEventRecord(e0, s));
        const dim3 g((unsigned)nsrc), blk(1024);
        const int64_t mask = ring - 1;
        if (blocked()) {
            // a thread per row of the backward window up to 512 rows, two rows
            // per thread beyond (kl <= kMaxBand: at most 960 rows)
            const dim3 bl((unsigned)std::max<int64_t>(kNB * kNB,
                                                      std::min<int64_t>(512, round_up(rows, 64))));
            if (rows <= 512)
                hipLaunchKernelGGL(freq_subst<1>, g, bl, sh, s, B, panels(), dS.p, dU.p, mask);
            else
                hipLaunchKernelGGL(freq_subst<2>, g, bl, sh, s, B, panels(), dS.p, dU.p, mask);
        } else
            switch (rpt) {
                case 1: hipLaunchKernelGGL(freq_solve<1>, g, blk, sh, s, B, piv.p, dS.p, dU.p, mask); break;
                case 2: hipLaunchKernelGGL(freq_solve<2>, g, blk, sh, s, B, piv.p, dS.p, dU.p, mask); break;
                case 4: hipLaunchKernelGGL(freq_solve<4>, g, blk, sh, s, B, piv.p, dS.p, dU.p, mask); break;
                default: hipLaunchKernelGGL(freq_solve<8>, g, blk, sh, s, B, piv.p, dS.p, dU.p, mask);
            }
        SSSI_HIP(hipGetLastError());
        SSSI_HIP(hipEventRecord(e1, s));
        copy_to_host(U, dU.p, dU.bytes(), s);
        float ms = 0;
        SSSI_HIP(hipEventElapsedTime(&ms, e0, e1));
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        return ms;
    }
};

}  // namespace sssi

using namespace sssi;

namespace {
template <class F>
int fguard(F &&f) {
    try {
        f();
        set_last_error("");
        return SSSI_OK;
    } catch (const Error &e) {
        set_last_error(e.what());
        return e.code;
    } catch (const std::bad_alloc &) {
        set_last_error("host allocation failed");
        return SSSI_ENOMEM;
    } catch (const std::exception &e) {
        set_last_error(e.what());
        return SSSI_EDEVICE;
    }
}
thread_local double g_factor_ms = 0, g_solve_ms = 0;
}  // namespace

extern "C" {

int sssi_freq_cpml_2d_matrix(const double *model, int64_t nz, int64_t nx, double w,
                             int nDiffOrder, int nBoundary, double dz, double dx, int64_t *nnz,
                             int64_t *rowptr, int64_t *col, double *val) {
    return fguard([&] {
        freq_validate(model, nz, nx, w, nDiffOrder, nBoundary, dz, dx);
        if (!nnz) fail(SSSI_EINVAL, "nnz must not be NULL");
        *nnz = freq_nnz(nz, nx, 2 * nDiffOrder - 1, nullptr);
        if (!rowptr) return;
        if (!col || !val) fail(SSSI_EINVAL, "col and val must not be NULL with rowptr");
        FreqSystem fs(model, nz, nx, w, nDiffOrder, nBoundary, dz, dx, false, rowptr, col, val);
    });
}

int sssi_freqCpmlFor2dAw(const double *model, int64_t nz, int64_t nx, const double *source,
                         int nsrc, double w, int nDiffOrder, int nBoundary, double dz, double dx,
                         double *snapshot) {
    return fguard([&] {
        freq_validate(model, nz, nx, w, nDiffOrder, nBoundary, dz, dx);
        if (nsrc < 1 || !source || !snapshot)
            fail(SSSI_EINVAL, "source and snapshot must hold at least one column");
        FreqSystem fs(model, nz, nx, w, nDiffOrder, nBoundary, dz, dx, true, nullptr, nullptr,
                      nullptr);
        g_factor_ms = fs.factor(nsrc);
        g_solve_ms = fs.solve(source, nsrc, snapshot);
    });
}

int sssi_freq_last_timing(double *factor_ms, double *solve_ms) {
    if (factor_ms) *factor_ms = g_factor_ms;
    if (solve_ms) *solve_ms = g_solve_ms;
    return SSSI_OK;
}

}  // extern "C"
