// abd_block.h — workgroup-level building blocks (wave64 ballots, fixed-order
// reductions and scans through LDS).  Every helper ends with a barrier so the
// LDS it used can be reused immediately by the caller.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace abd {

constexpr int kWave = 64;

__device__ __forceinline__ int lane_id() { return (int)(threadIdx.x & (kWave - 1)); }
__device__ __forceinline__ int wave_id() { return (int)(threadIdx.x / kWave); }
__device__ __forceinline__ int n_waves() { return (int)((blockDim.x + kWave - 1) / kWave); }

// Sum over the workgroup, fixed pairing (deterministic); result returned to every thread.
// sh must hold blockDim.x doubles.
__device__ __forceinline__ double block_sum(double v, double* sh) {
    const int t = threadIdx.x;
    sh[t] = v;
    __syncthreads();
    for (int s = (int)blockDim.x / 2; s > 0; s >>= 1) {
        if (t < s) sh[t] = sh[t] + sh[t + s];
        __syncthreads();
    }
    double r = sh[0];
    __syncthreads();
    return r;
}
// Minimum over the workgroup (blockDim.x a multiple of 64; sh: n_waves() entries): a
// shuffle tree inside each wave, then the waves' minima (two barriers).  NaN never wins a
// comparison, so a NaN is kept only where every other value is NaN.
__device__ __forceinline__ double block_min(double v, double* sh) {
    double r = v;
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1) {
        const double y = __shfl_xor(r, off, kWave);
        r = y < r ? y : r;
    }
    if (lane_id() == 0) sh[wave_id()] = r;
    __syncthreads();
    r = sh[0];
    for (int k = 1; k < n_waves(); ++k) r = sh[k] < r ? sh[k] : r;
    __syncthreads();
    return r;
}

// Sums across lanes by the vector unit's own lane moves (DPP, and the half and row swaps),
// about 25 cycles a level where a shuffle through the LDS unit takes over 100.  The pairing
// is that of a shfl_down tree (lanes 32 apart first), every lane ending with lane 0's value.
// All lanes must be active.
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppRor4 = 0x124, kDppRor8 = 0x128;
constexpr int kDppPair0 = 0xA0, kDppPair1 = 0xF5;  // lane k of a pair to both
constexpr int kDppRowBcast = 0x150;  // + i: lane i of each row of 16 lanes to all of it
// v summed over each row of 16 lanes (8 apart first; a rotation by 4 is lane ^ 4 once lanes
// 8 apart hold the same value)
__device__ __forceinline__ double row_sum(double v) {
    v += dpp_move<kDppRor8>(v);
    v += dpp_move<kDppRor4>(v);
    v += dpp_move<kDppXor2>(v);
    v += dpp_move<kDppXor1>(v);
    return v;
}
__device__ __forceinline__ double wave_sum(double v) {
    {
        const auto lo = __builtin_amdgcn_permlane32_swap(__double2loint(v), __double2loint(v), false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap(__double2hiint(v), __double2hiint(v), false, false);
        v = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);  // lane i and i ^ 32
    }
    {
        const auto lo = __builtin_amdgcn_permlane16_swap(__double2loint(v), __double2loint(v), false, false);
        const auto hi = __builtin_amdgcn_permlane16_swap(__double2hiint(v), __double2hiint(v), false, false);
        v = __hiloint2double(hi[0], lo[0]) + __hiloint2double(hi[1], lo[1]);  // i ^ 16
    }
    return row_sum(v);
}
// The waves' sums (sh: one per wave, at most 16, absent ones 0) in the pairing 8, 4, 2, 1
// apart, by every wave.
__device__ __forceinline__ double waves_sum(const double* sh, int nw) {
    const int i = lane_id() & 15;
    return row_sum(i < nw ? sh[i] : 0.0);
}

// Sum over the workgroup with two barriers: wave_sum inside each wave, the wave sums through
// LDS, reduced in the same fixed order by every wave (alike, so all waves branch alike on
// it).  blockDim.x must be a multiple of 64 and at most 1024; sh must hold 16 doubles.
__device__ __forceinline__ double block_sum_fast(double v, double* sh) {
    v = wave_sum(v);
    if (lane_id() == 0) sh[wave_id()] = v;
    __syncthreads();
    const double r = waves_sum(sh, n_waves());
    __syncthreads();
    return r;
}

// Two independent sums with the reduction pattern of block_sum_fast (each result
// bit-identical to a block_sum_fast of that value alone) and the same two
// barriers.  sh must hold 34 doubles.
__device__ __forceinline__ void block_sum2_fast(double& a, double& b, double* sh) {
    a = wave_sum(a);
    b = wave_sum(b);
    if (lane_id() == 0) {
        sh[wave_id()] = a;
        sh[17 + wave_id()] = b;
    }
    __syncthreads();
    a = waves_sum(sh, n_waves());
    b = waves_sum(sh + 17, n_waves());
    __syncthreads();
}

// The extrema of a body's vertices over the T threads of its workgroup, valid in thread 0.
template <int T>
__device__ __forceinline__ void body_extrema(double (&mn)[3], double (&mx)[3], double* sh) {
#pragma unroll
    for (int off = kWave / 2; off > 0; off >>= 1)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const double a = __shfl_xor(mn[k], off, kWave), b = __shfl_xor(mx[k], off, kWave);
            mn[k] = a < mn[k] ? a : mn[k];
            mx[k] = b > mx[k] ? b : mx[k];
        }
    if (T > kWave) {
        if (lane_id() == 0)
            for (int k = 0; k < 3; ++k) {
                sh[6 * wave_id() + k] = mn[k];
                sh[6 * wave_id() + 3 + k] = mx[k];
            }
        __syncthreads();
        if (threadIdx.x == 0)
            for (int w = 1; w < T / kWave; ++w)
                for (int k = 0; k < 3; ++k) {
                    const double a = sh[6 * w + k], b = sh[6 * w + 3 + k];
                    mn[k] = a < mn[k] ? a : mn[k];
                    mx[k] = b > mx[k] ? b : mx[k];
                }
    }
}

// Exclusive prefix sum of one int64 per thread (sh: at least n_waves() entries): a
// shuffle scan inside each wave, then the totals of the waves before it (two barriers).
__device__ __forceinline__ int64_t block_exclusive_scan_i64(int64_t v, int64_t* sh) {
    const int lane = lane_id(), w = wave_id();
    int64_t incl = v;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const int64_t y = __shfl_up(incl, off, kWave);
        if (lane >= off) incl += y;
    }
    if (lane == kWave - 1) sh[w] = incl;
    __syncthreads();
    int64_t before = 0;
    for (int k = 0; k < w; ++k) before += sh[k];
    __syncthreads();  // sh is free again for the caller
    return before + incl - v;
}

// Ordered compaction rank inside the workgroup: returns the number of threads
// with a lower thread index whose predicate holds; *total = count over the
// workgroup.  sh_waves: n_waves() ints.
__device__ __forceinline__ int block_rank(bool pred, int* sh_waves, int* total) {
    unsigned long long mask = __ballot(pred ? 1 : 0);
    const int lane = lane_id();
    const int w = wave_id();
    unsigned long long below = lane == 0 ? 0ull : (mask & ((~0ull) >> (kWave - lane)));
    int r = __popcll(below);
    if (lane == 0) sh_waves[w] = __popcll(mask);
    __syncthreads();
    int off = 0, tot = 0;
    const int nw = n_waves();
    for (int k = 0; k < nw; ++k) {
        int c = sh_waves[k];
        if (k < w) off += c;
        tot += c;
    }
    __syncthreads();
    *total = tot;
    return off + r;
}

// Single workgroup (kScanThreads threads) exclusive scan of load(0), ..., load(n - 1) into out;
// each pass covers 1024 threads x 8 items.  total / total2 (either may be null) receive the sum.
constexpr int kScanThreads = 1024;
constexpr int kScanItems = 8;

template <class Load>
__device__ __forceinline__ void scan_block_exclusive_by(Load load, int64_t* __restrict__ out, int64_t n,
                                                        int64_t* __restrict__ total, int64_t* __restrict__ total2) {
    __shared__ int64_t sh[kScanThreads];
    int64_t carry = 0;
    const int t = threadIdx.x;
    for (int64_t base = 0; base < n; base += (int64_t)kScanThreads * kScanItems) {
        int64_t v[kScanItems];
        int64_t s = 0;
        int64_t i0 = base + (int64_t)t * kScanItems;
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) {
            int64_t i = i0 + k;
            v[k] = i < n ? load(i) : 0;
            s += v[k];
        }
        int64_t excl = block_exclusive_scan_i64(s, sh);
        int64_t run = carry + excl;
#pragma unroll
        for (int k = 0; k < kScanItems; ++k) {
            int64_t i = i0 + k;
            if (i < n) out[i] = run;
            run += v[k];
        }
        // last thread holds the tile total
        if (t == kScanThreads - 1) sh[0] = excl + s;
        __syncthreads();
        carry += sh[0];
        __syncthreads();
    }
    if (t == 0 && total) *total = carry;
    if (t == 0 && total2) *total2 = carry;
}

}  // namespace abd
