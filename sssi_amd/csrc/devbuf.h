// Device-side helpers shared by the 2-D kernels: raw buffer access with a
// wave-uniform scalar offset, scalar loads of uniform tables, and the
// wave index as a scalar.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace sssi {

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), (short)0, (int)bytes,
                                             0x00020000);
}
__device__ __forceinline__ float buf_ld(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, (int)voff, (int)soff, 0));
}
__device__ __forceinline__ void buf_st(float v, __amdgpu_buffer_rsrc_t r, uint32_t voff,
                                       uint32_t soff) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, (int)voff, (int)soff, 0);
}
// Byte offset marking a lane with no value in a buffer of fewer than 2^31
// bytes: the range check covers the vector offset, so a load there returns 0
// and a store is dropped.  Offsets of the form kOOB + k (k < 2^31) stay out
// of range.
constexpr uint32_t kOOB = 0x80000000u;

// Load of wave-uniform data that no launch of this kernel writes (source
// tables, checkpoint scales of earlier steps): through the constant address
// space the compiler emits a scalar load, which is waited for with lgkmcnt and
// leaves the in-order vmcnt of the prefetched field loads untouched.
template <class T>
__device__ __forceinline__ T ld_uniform(const T *p) {
    return *(const __attribute__((address_space(4))) T *)p;
}

// Index of the wavefront in its block, as a wave-uniform (scalar) value: the
// compiler cannot prove threadIdx.x >> 6 uniform, and a row offset derived
// from it would turn every buffer load into a waterfall loop.
__device__ __forceinline__ int wave_id() {
    return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
}

// Point sources of a wavefront that holds R rows from i0 and 64 columns from j0
// (lane = column) over the steps of one launch.
// Few (MANY false): a loop over all of them with scalar loads, which costs the
// wavefront 0.1 to 0.2 us per source and step whether or not it holds them.
// MANY: lanes test 64 at a time, and the wavefront adds its own in the order of
// the list; the first 64 sources' places stay in a register, and their
// amplitudes are loaded a step ahead.  The registers cost where they take a
// wavefront's place on its SIMD, so the two are compiled apart, and a launch
// takes MANY from where it pays: kFewSources, for CPML of order 2 (held to 128
// registers) 8.  us per step at 1, 4, 8 and 64 sources all over the model, few
// and many: sponge 100 x 150 1.06 1.46 2.30 11.6 and 1.00 1.04 1.05 1.36, sponge
// 1040 x 3080 at one 3.80 and 3.96, CPML 120 x 240 N=2 2.73 3.29 3.79 14.1 and
// (at 8, 64) 3.40 3.68, N=4 5.28 5.82 6.44 18.1 and 5.41 5.57 5.56 5.70.
constexpr int kFewSources = 4;
template <int R, bool MANY>
struct WaveSources {
    const int *cell;   // [k] = row * nx + column, k < n
    const float *amp;  // [t * n + k], t < nt
    int n, nt, nx, i0, j0;
    int first = -1;    // MANY: lane's place among the first 64, row * 64 + column, or -1
    float next = 0.f;  // MANY: its amplitude of the next step

    __device__ __forceinline__ int place(int k) const {
        if (k >= n) return -1;
        const int c = cell[k], ci = c / nx, i = ci - i0, j = c - ci * nx - j0;
        return i >= 0 && i < R && j >= 0 && j < 64 ? i * 64 + j : -1;
    }
    __device__ __forceinline__ void fetch(int t) {
        next = first >= 0 && t < nt ? amp[(size_t)t * n + (threadIdx.x & 63)] : 0.f;
    }
    // whether any lies here (wave-uniform); steps t0, t0 + 1, ... follow
    __device__ __forceinline__ bool find(int t0) {
        bool any = false;
        if constexpr (MANY) {
            const int lane = (int)(threadIdx.x & 63);
            first = place(lane);
            any = __ballot(first >= 0) != 0;
            for (int k = 64; k < n; k += 64) any |= __ballot(place(k + lane) >= 0) != 0;
            if (any) fetch(t0);
        } else {
            for (int k = 0; k < n; ++k) {
                const int c = ld_uniform(cell + k), ci = c / nx, cj = c - ci * nx;
                any |= ci >= i0 && ci < i0 + R && cj >= j0 && cj < j0 + 64;
            }
        }
        return any;
    }
    // adds step t's terms to sv (rows of column j, the lane's)
    __device__ __forceinline__ void add(int t, int j, float (&sv)[R]) {
        if (t >= nt) return;
        if constexpr (MANY) {
            const int lane = (int)(threadIdx.x & 63);
            auto chunk = [&](int at, float a) {
                for (unsigned long long m = __ballot(at >= 0); m; m &= m - 1) {
                    const int l = __ffsll(m) - 1;
                    const int u = __builtin_amdgcn_readlane(at, l);
                    const float x = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(a), l));
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        if (u == r * 64 + lane) sv[r] += x;
                }
            };
            chunk(first, next);
            fetch(t + 1);
            for (int k = 64; k < n; k += 64) {
                const int at = place(k + lane);
                chunk(at, at >= 0 ? amp[(size_t)t * n + k + lane] : 0.f);
            }
        } else {
            for (int k = 0; k < n; ++k) {
                const int c = ld_uniform(cell + k), ci = c / nx, cj = c - ci * nx;
                const float a = ld_uniform(amp + (size_t)t * n + k);
                if (cj == j) {
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        if (ci == i0 + r) sv[r] += a;
                }
            }
        }
    }
};

}  // namespace sssi
