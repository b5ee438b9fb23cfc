// BM3D kernels for CDNA4 (gfx950): block matching, group filter with
// weighted fixed-point aggregation, and finish.
//
// Main path (the shapes whose working sets fit the LDS budget):
//   match_run_kernel<B, SMALL> one workgroup per run of 8 references on one
//   match_run_mid_kernel<B>    grid row; the union of their search windows is
//                              staged in LDS once; each half-wave owns one
//                              reference and each lane 2 x 7 tiles of
//                              candidates (one tile: SMALL; up to three: mid,
//                              keys held in registers); then the G-1 smallest
//                              keys (dist, y, x) by a threshold and a rank
//                              count (rounds of a half-wave min as fallback).
//   filter_tile_kernel<B, W>   one workgroup per tile of references; each wave
//                              filters whole groups (2-D DCT, Haar along the
//                              group, hard threshold or Wiener, inverse) and
//                              adds them into the tile's int64 fixed-point
//                              numerator sums in LDS (ds_add_u64: exact and
//                              order-free); the tile writes those sums as its
//                              partials and one weight per group.
//   finish_tiles_kernel        per pixel, the numerator partials of the tiles
//                              covering it, summed exactly; the weights rebuilt
//                              from the match records; then num / den or the
//                              source.
// General path (any legal shape):
//   match_wave_kernel<B, S>    one wave per reference, window in LDS (or read
//                              from global when it does not fit).
//   filter_atomic_kernel<B, W> one wave per group, device-scope int64 atomics
//                              into frame-sized sums (den at the corner).
//   finish_corner_kernel<B>    box-sums the corner weights, divides.
// Workgroups are dealt round-robin over the 8 XCDs; every kernel remaps its
// block index so that each XCD works on a contiguous part of the frame (its
// L2 then holds the overlapping windows, patches and partial rows).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "bm3d_jobs.hpp"

namespace nsship {

// True when an armed test hook refuses this launch (device_mem.cpp); the
// launch wrappers then return hipErrorLaunchFailure without launching.
bool launch_fault();

// Orthonormal DCT-II matrices (row = frequency) for B in {2,4,8,12,16,32},
// concatenated; filled from the host (double cosines rounded to float, as
// src/cpu/bm/dct8.cpp:71-89 DctTable).
__constant__ float c_dct[4 + 16 + 64 + 144 + 256 + 1024];

template <int B>
__device__ constexpr int dct_offset() {
    return B == 2 ? 0 : B == 4 ? 4 : B == 8 ? 20 : B == 12 ? 84 : B == 16 ? 228 : 484;
}

inline constexpr uint32_t kTaken = 0xffffffffu;
inline constexpr uint32_t kNonFinite = 0x7f800000u;
inline constexpr int kXcds = 8;

// Calls f(integral_constant<0>) .. f(integral_constant<N - 1>).
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// Block index such that each XCD (blockIdx % 8 on dispatch) covers a
// contiguous range of logical blocks; a bijection on [0, gridDim.x).
__device__ inline int xcd_block() {
    const int nb = static_cast<int>(gridDim.x), b = static_cast<int>(blockIdx.x);
    const int q = nb / kXcds, rem = nb % kXcds;
    const int xcd = b % kXcds, slot = b / kXcds;
    return xcd < rem ? xcd * (q + 1) + slot : rem * (q + 1) + (xcd - rem) * q + slot;
}

// Orders the calling wave's LDS accesses (one wave's DS operations execute
// in issue order; this keeps the compiler from moving accesses across).
__device__ inline void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// min(v, v of the lane DPP control `ctrl` selects); lanes whose source is
// outside the row (or rows outside row_mask) keep v.
template <int CTRL, int ROW_MASK>
__device__ inline unsigned long long dpp_min_u64(unsigned long long v) {
    const int lo = static_cast<int>(static_cast<uint32_t>(v));
    const int hi = static_cast<int>(static_cast<uint32_t>(v >> 32));
    const int olo = __builtin_amdgcn_update_dpp(lo, lo, CTRL, ROW_MASK, 0xf, false);
    const int ohi = __builtin_amdgcn_update_dpp(hi, hi, CTRL, ROW_MASK, 0xf, false);
    const unsigned long long o = (static_cast<unsigned long long>(static_cast<uint32_t>(ohi)) << 32) |
                                 static_cast<uint32_t>(olo);
    return o < v ? o : v;
}

// Minimum over each half-wave (lanes 0-31 and 32-63), returned to every lane
// of that half. Must be reached by all 64 lanes. DPP row_shr 1, 2, 4, 8 leaves
// each 16-lane row's minimum in its last lane; row_bcast15 folds row 0 into
// row 1 and row 2 into row 3; lanes 31 and 63 then hold the two minima.
__device__ inline unsigned long long half_min_u64(unsigned long long v) {
    v = dpp_min_u64<0x111, 0xf>(v);
    v = dpp_min_u64<0x112, 0xf>(v);
    v = dpp_min_u64<0x114, 0xf>(v);
    v = dpp_min_u64<0x118, 0xf>(v);
    v = dpp_min_u64<0x142, 0xa>(v);
    const int lo = static_cast<int>(static_cast<uint32_t>(v));
    const int hi = static_cast<int>(static_cast<uint32_t>(v >> 32));
    const uint32_t lo0 = static_cast<uint32_t>(__builtin_amdgcn_readlane(lo, 31));
    const uint32_t hi0 = static_cast<uint32_t>(__builtin_amdgcn_readlane(hi, 31));
    const uint32_t lo1 = static_cast<uint32_t>(__builtin_amdgcn_readlane(lo, 63));
    const uint32_t hi1 = static_cast<uint32_t>(__builtin_amdgcn_readlane(hi, 63));
    const bool upper = threadIdx.x & 32;
    return (static_cast<unsigned long long>(upper ? hi1 : hi0) << 32) | (upper ? lo1 : lo0);
}

// min(v, v of the lane DPP control `ctrl` selects); lanes whose source is
// outside the row (or rows outside row_mask) see the identity ~0, so the
// move folds into the min as one DPP instruction.
template <int CTRL, int ROW_MASK>
__device__ inline uint32_t dpp_min_u32(uint32_t v) {
    const int o = __builtin_amdgcn_update_dpp(-1, static_cast<int>(v), CTRL, ROW_MASK, 0xf, false);
    return min(v, static_cast<uint32_t>(o));
}

// Half-wave minimum of 32-bit values (the DPP steps of half_min_u64).
__device__ inline uint32_t half_min_u32(uint32_t v) {
    v = dpp_min_u32<0x111, 0xf>(v);
    v = dpp_min_u32<0x112, 0xf>(v);
    v = dpp_min_u32<0x114, 0xf>(v);
    v = dpp_min_u32<0x118, 0xf>(v);
    v = dpp_min_u32<0x142, 0xa>(v);
    const uint32_t lo = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), 31));
    const uint32_t hi = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), 63));
    return (threadIdx.x & 32) ? hi : lo;
}

// Half-wave minimum of 64-bit keys (dist << 32 | index) in two 32-bit
// passes: the smallest dist, then the smallest index among the lanes holding
// it. Equal to half_min_u64's result; all 64 lanes must call.
__device__ inline unsigned long long half_min_key(unsigned long long v) {
    const uint32_t d = static_cast<uint32_t>(v >> 32);
    const uint32_t md = half_min_u32(d);
    const uint32_t mc = half_min_u32(d == md ? static_cast<uint32_t>(v) : 0xffffffffu);
    return (static_cast<unsigned long long>(md) << 32) | mc;
}

// Minimum over the whole wave, returned to every lane (same DPP steps as
// half_min_u64, then the smaller of lanes 31 and 63). All 64 lanes must call.
__device__ inline unsigned long long wave_min_u64(unsigned long long v) {
    v = dpp_min_u64<0x111, 0xf>(v);
    v = dpp_min_u64<0x112, 0xf>(v);
    v = dpp_min_u64<0x114, 0xf>(v);
    v = dpp_min_u64<0x118, 0xf>(v);
    v = dpp_min_u64<0x142, 0xa>(v);
    const int lo = static_cast<int>(static_cast<uint32_t>(v));
    const int hi = static_cast<int>(static_cast<uint32_t>(v >> 32));
    const unsigned long long a =
        (static_cast<unsigned long long>(static_cast<uint32_t>(__builtin_amdgcn_readlane(hi, 31))) << 32) |
        static_cast<uint32_t>(__builtin_amdgcn_readlane(lo, 31));
    const unsigned long long b =
        (static_cast<unsigned long long>(static_cast<uint32_t>(__builtin_amdgcn_readlane(hi, 63))) << 32) |
        static_cast<uint32_t>(__builtin_amdgcn_readlane(lo, 63));
    return a < b ? a : b;
}

__device__ inline int wave_sum_i32(int v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

__device__ inline float wave_sum_f32(float v) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
    return v;
}

template <typename Table>
__device__ inline int find_job(const Table& tab, int block) {
    int j = 0;
    while (j + 1 < tab.n && block >= tab.job[j + 1].wg_begin) ++j;
    return j;
}

__device__ inline uint32_t dist_key(float d) {
    const uint32_t k = __float_as_uint(d);
    return (k & kNonFinite) == kNonFinite ? kNonFinite : k;
}

// floor(c / d) for 0 <= c < 2^20 and 1 <= d <= 256, from inv = 1.f / d:
// (c + 1/2) / d lies at least 1/(2d) away from an integer, far more than the
// float rounding of the product.
__device__ inline int div_small(int c, float inv) {
    return static_cast<int>((static_cast<float>(c) + 0.5f) * inv);
}

__device__ inline int ref_x(const Grid& g, int i, int width, int block) { return min(i * g.step, width - block); }
__device__ inline int ref_y(const Grid& g, int j, int height, int block) {
    return min((j + g.row0) * g.step, height - block);
}

// ---------------------------------------------------------------------------
// Block matching (src/cpu/bm/matcher.hpp:247-283 collect_spatial_coords:
// window [c - r, c + r] clamped to the plane, raster scan, self excluded,
// reference first; order src/cpu/bm/matcher.hpp:27-57 match_less).
// ---------------------------------------------------------------------------

// The value of lane (lane ^ J) within each group of 32 lanes: DPP quad
// permutes for J = 1, 2, a bit-mode ds_swizzle for J = 4, 8, 16.
template <int J>
__device__ inline uint32_t xor_lane(uint32_t v) {
    if constexpr (J == 1) {
        return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0xb1, 0xf, 0xf, false));
    } else if constexpr (J == 2) {
        return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x4e, 0xf, 0xf, false));
    } else {
        return static_cast<uint32_t>(__builtin_amdgcn_ds_swizzle(static_cast<int>(v), 0x1f | (J << 10)));
    }
}

// One compare-exchange stage (block K, distance J) of a bitonic sort that
// orders each 32-lane half ascending: a lane keeps the smaller value where
// its J bit equals its K bit (K = 32: the whole half ascends).
// One compare-exchange stage (block K, distance J) of a bitonic sort that
// orders each 32-lane half ascending: a lane keeps the smaller value where
// its J bit equals its K bit (K = 32: the whole half ascends).
template <int K, int J>
__device__ inline unsigned long long bitonic_u64(unsigned long long v) {
    const int lane = threadIdx.x & 31;
    const uint32_t plo = xor_lane<J>(static_cast<uint32_t>(v));
    const uint32_t phi = xor_lane<J>(static_cast<uint32_t>(v >> 32));
    const unsigned long long p = (static_cast<unsigned long long>(phi) << 32) | plo;
    const bool keep_min = ((lane & J) == 0) == (K == 32 || (lane & K) == 0);
    return keep_min == (p < v) ? p : v;
}

// Ascending sort of the 32 keys of each half-wave (lane i of the half holds
// the i-th smallest). All 64 lanes must call.
__device__ inline unsigned long long sort32_u64(unsigned long long v) {
    v = bitonic_u64<2, 1>(v);
    v = bitonic_u64<4, 2>(v);
    v = bitonic_u64<4, 1>(v);
    v = bitonic_u64<8, 4>(v);
    v = bitonic_u64<8, 2>(v);
    v = bitonic_u64<8, 1>(v);
    v = bitonic_u64<16, 8>(v);
    v = bitonic_u64<16, 4>(v);
    v = bitonic_u64<16, 2>(v);
    v = bitonic_u64<16, 1>(v);
    v = bitonic_u64<32, 16>(v);
    v = bitonic_u64<32, 8>(v);
    v = bitonic_u64<32, 4>(v);
    v = bitonic_u64<32, 2>(v);
    return bitonic_u64<32, 1>(v);
}

// Lane tiles (2 x 7 candidates) a half-wave needs per lane for a whole
// window of the range.
__host__ __device__ constexpr int run_tiles_per_lane(int range) {
    return (((2 * range + 1 + 6) / 7) * ((2 * range + 1 + 1) / 2) + 31) / 32;
}

// Windows whose lane tiles fit one per lane of a half-wave (a side of up to
// 20: ranges up to 9) keep each lane's keys in registers through a workgroup
// barrier; the window keys and the gathered keys then overlay the staged
// region in LDS. Up to kRunMidTiles tiles per lane (ranges up to 16) do the
// same with the keys of every tile in registers and a smaller gather area
// (kRunMidGather keys per reference), so that a 33 x 33 window's workgroup
// fits four to a CU. Larger windows keep both areas.
__host__ __device__ constexpr bool run_keys_in_regs(int range) { return run_tiles_per_lane(range) <= 1; }
inline constexpr int kRunMidTiles = 3;
inline constexpr int kRunMidGather = 64;
__host__ __device__ constexpr bool run_keys_mid(int range) {
    return run_tiles_per_lane(range) > 1 && run_tiles_per_lane(range) <= kRunMidTiles;
}

// Floats of the staged region the run matcher's LDS layout reserves: the 8
// windows' span + 6 padding columns with the pitch rounded up to 2 mod 4, by
// the windows' height + 1 row (every workgroup's region fits).
__host__ __device__ constexpr int run_region_floats(int block, int step, int range) {
    return (((kRunRefs - 1) * step + 2 * range + block + 9) * (2 * range + block + 1) + 3) & ~3;
}

// SSD of the 2 x 7 candidates of lane tile (dy0, dx0) against the reference
// patch at rp, in block-row order (one fmaf per pixel, the order every
// matcher uses): region rows dy0 + py + i, columns dx0 .. dx0 + B + 5.
// REUSE (large windows, several tiles per lane): row dy0 + py + 1 serves
// block rows py and py + 1 and is read once, and the 14 differences of a
// reference pixel are formed before their products; it costs registers, so
// the small-window form (one tile per lane, 8 waves per SIMD) reads each
// row pair per block row instead.
template <int B, bool REUSE>
__device__ inline void run_tile_ssd(const float* rp, const float* base, int RW, float (&acc)[2][7]) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 7; ++j) acc[i][j] = 0.f;
    if constexpr (!REUSE) {
        for (int py = 0; py < B; ++py) {
            float rrow[B];
#pragma unroll
            for (int px = 0; px < B; ++px) rrow[px] = rp[py * RW + px];
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const float* rowp = base + (py + i) * RW;
                float v[B + 6];
#pragma unroll
                for (int c = 0; c < B + 6; ++c) v[c] = rowp[c];
#pragma unroll
                for (int j = 0; j < 7; ++j)
#pragma unroll
                    for (int px = 0; px < B; ++px) {
                        const float d = rrow[px] - v[j + px];
                        acc[i][j] = fmaf(d, d, acc[i][j]);
                    }
            }
        }
    } else {
        float cur[B + 6];
#pragma unroll
        for (int c = 0; c < B + 6; ++c) cur[c] = base[c];
#pragma unroll 2
        for (int py = 0; py < B; ++py) {
            float rrow[B], nxt[B + 6];
#pragma unroll
            for (int px = 0; px < B; ++px) rrow[px] = rp[py * RW + px];
#pragma unroll
            for (int c = 0; c < B + 6; ++c) nxt[c] = base[(py + 1) * RW + c];
#pragma unroll
            for (int px = 0; px < B; ++px) {
                float d0[7], d1[7];
#pragma unroll
                for (int j = 0; j < 7; ++j) {
                    d0[j] = rrow[px] - cur[j + px];
                    d1[j] = rrow[px] - nxt[j + px];
                }
#pragma unroll
                for (int j = 0; j < 7; ++j) {
                    acc[0][j] = fmaf(d0[j], d0[j], acc[0][j]);
                    acc[1][j] = fmaf(d1[j], d1[j], acc[1][j]);
                }
            }
#pragma unroll
            for (int c = 0; c < B + 6; ++c) cur[c] = nxt[c];
        }
    }
}

// Run matcher: references i0 .. i0+7 of grid row j share one LDS region.
// NT = 1: every job's window takes one lane tile per lane
// (run_keys_in_regs); NT = kRunMidTiles: up to that many (run_keys_mid),
// keys in registers; NT = 0: keys in LDS as they are scored.
template <int B, int NT>
__device__ __forceinline__ void match_run_body(const MatchTable& tab) {
    constexpr bool SMALL = NT == 1;
    constexpr int NG = NT == kRunMidTiles ? kRunMidGather : kRunGather;  // gathered keys per reference
    extern __shared__ __align__(16) float lds[];
    const int lb = xcd_block();
    const MatchJob& jb = tab.job[find_job(tab, lb)];
    const int run = lb - jb.wg_begin;
    const int rpr = (jb.grid.nx + kRunRefs - 1) / kRunRefs;
    const int row = run / rpr, i0 = (run - row * rpr) * kRunRefs;
    const int nrun = min(kRunRefs, jb.grid.nx - i0);
    const int r = jb.range;
    const int cy = ref_y(jb.grid, row, jb.height, B);
    const int top = max(cy - r, 0), bottom = min(cy + r, jb.height - B);
    const int rx0 = max(ref_x(jb.grid, i0, jb.width, B) - r, 0);
    const int rx1 = min(ref_x(jb.grid, i0 + nrun - 1, jb.width, B) + r, jb.width - B) + B - 1;
    // Lane tiles of 2 x 7 candidates (2 rows, 7 columns): a 19 x 19 window
    // is 10 x 3 tiles, 448 lane slots for 361 candidates. Tile columns 7 tx
    // spread the lanes over the banks; the region keeps 6 columns after the
    // windows and 1 row below (candidates of an overhanging tile are
    // discarded), with a row pitch = 2 mod 4.
    const int need = rx1 - rx0 + 1 + 6;
    const int RW = need + (6 - need % 4) % 4;
    const int RH = bottom - top + B + 1;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    // Rows wave, wave + 4, ... by 64-column strips: the row address is
    // wave-uniform and each lane's column is clamped once per strip; cells
    // outside the plane repeat its edge (only discarded candidates of
    // overhanging tiles read them).
    // Each load goes straight to LDS (global_load_lds: lane l's word lands
    // at the wave-uniform row address + 4 l), so the staging holds no
    // registers and issues no LDS stores; the barrier below waits for them.
    // The row (and so its address) is wave-uniform: scalar arithmetic, the
    // lane's clamped column the only per-lane offset.
    const int wv = __builtin_amdgcn_readfirstlane(wave);
    for (int c0 = 0; c0 < RW; c0 += 64) {
        const int xx = c0 + lane;
        if (xx < RW) {
            const int gx = min(rx0 + xx, jb.width - 1);
            for (int yy = wv; yy < RH; yy += 4) {
                const float* row = jb.plane + static_cast<size_t>(min(top + yy, jb.height - 1)) * jb.stride;
                __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(row + gx),
                                                 (__attribute__((address_space(3))) void*)(lds + yy * RW + c0), 4, 0,
                                                 0);
            }
        }
    }
    const int wmax = 2 * r + 1;
    constexpr bool regs = NT > 0;
    // Window keys (wmax^2 per reference) and up to NG gathered keys
    // per reference. Keys waiting in registers: both over the region. Else
    // the window keys after the region and the gathered keys over it (or
    // after the window keys when the region is smaller).
    // (The offsets follow the reserved region size, the same in every
    // workgroup of the launch.)
    const int region = run_region_floats(B, jb.grid.step, r);
    uint32_t* dist = reinterpret_cast<uint32_t*>(lds + (regs ? 0 : region));
    unsigned long long* surv =
        regs || region * 4 < kRunRefs * NG * 8
            ? reinterpret_cast<unsigned long long*>(dist + kRunRefs * wmax * wmax)
            : reinterpret_cast<unsigned long long*>(lds);
    __syncthreads();

    const int half = threadIdx.x >> 5, hl = threadIdx.x & 31;
    const int cx = ref_x(jb.grid, i0 + half, jb.width, B);
    const int left = max(cx - r, 0), right = min(cx + r, jb.width - B);
    const int ww = right - left + 1, wh = bottom - top + 1;
    const int ncand = ww * wh;
    uint32_t* dk = dist + half * wmax * wmax;
    const int tw = (ww + 6) / 7, th = (wh + 1) >> 1;
    const int self = (cy - top) * ww + (cx - left);
    const float* rp = lds + (cy - top) * RW + (cx - rx0);
    const float* wbase = lds + (left - rx0);
    if (NT > 1) {
        // up to NT tiles per lane (t = hl, hl + 32, ...): their keys wait in
        // registers for the barrier, then go to the key area over the region
        uint32_t kr[NT > 1 ? NT : 1][2][7];
        const int nt = half < nrun ? tw * th : 0;
#pragma unroll
        for (int q = 0; q < NT; ++q) {
            const int t = hl + 32 * q;
            if (t < nt) {
                const int ty = t / tw, tx = t - ty * tw;
                float acc[2][7];
                run_tile_ssd<B, true>(rp, wbase + ty * 2 * RW + tx * 7, RW, acc);
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 7; ++j) kr[q][i][j] = dist_key(acc[i][j]);
            }
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < NT; ++q) {
            const int t = hl + 32 * q;
            if (t < nt) {
                const int ty = t / tw, tx = t - ty * tw;
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 7; ++j) {
                        const int dy = ty * 2 + i, dx = tx * 7 + j, c = dy * ww + dx;
                        if (dy < wh && dx < ww) dk[c] = c == self ? kTaken : kr[q][i][j];
                    }
            }
        }
    } else if (regs) {
        // one tile per lane: its keys wait in registers for the barrier,
        // then go to the key area over the region
        const int ty = hl / tw, tx = hl - ty * tw;
        const int dy0 = ty * 2, dx0 = tx * 7;
        const bool mine = half < nrun && hl < tw * th;
        float acc[2][7];
        if (mine) run_tile_ssd<B, !SMALL>(rp, wbase + dy0 * RW + dx0, RW, acc);
        __syncthreads();
        if (mine) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < 7; ++j) {
                    const int dy = dy0 + i, dx = dx0 + j, c = dy * ww + dx;
                    if (dy < wh && dx < ww) dk[c] = c == self ? kTaken : dist_key(acc[i][j]);
                }
        }
    } else {
        if (half < nrun) {
            for (int t = hl; t < tw * th; t += 32) {
                const int ty = t / tw, tx = t - ty * tw;
                const int dy0 = ty * 2, dx0 = tx * 7;
                float acc[2][7];
                run_tile_ssd<B, !SMALL>(rp, wbase + dy0 * RW + dx0, RW, acc);
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 7; ++j) {
                        const int dy = dy0 + i, dx = dx0 + j, c = dy * ww + dx;
                        if (dy < wh && dx < ww) dk[c] = c == self ? kTaken : dist_key(acc[i][j]);
                    }
            }
        }
        __syncthreads();  // the region is read; gathered keys may overlay it
    }
    wave_sync();
    // Selection, wave-uniform: both half-waves take part (a half with fewer
    // candidates, or no reference, idles) so that cross-lane steps see all
    // 64 lanes. Keys order as (dist, window index); lane hl owns the keys
    // c = hl mod 32.
    const int K = half < nrun ? min(jb.group - 1, ncand - 1) : 0;
    const int kmax = max(__builtin_amdgcn_readlane(K, 0), __builtin_amdgcn_readlane(K, 32));
    const float inv_ww = 1.f / static_cast<float>(ww);
    const int ref_id = row * jb.grid.nx + i0 + half;
    MatchRec* out = jb.out + static_cast<size_t>(ref_id) * jb.group;
    if (half < nrun && hl == 0) {
        out[0] = MatchRec{cx, cy, jb.t0, 0u};
        jb.counts[ref_id] = 1 + K;
    }
    // Threshold selection (K <= 31). T = the K-th smallest of the half's 32
    // lane minima: distinct candidates, so at least K keys are <= T and the
    // K winners all are. The keys <= T (self excluded) are gathered in LDS
    // and each is ranked against the others; rank k is record 1 + k. When
    // more than NG keys are <= T in either half the wave takes the
    // rounds below instead.
    if (kmax <= 31) {
        const int nc = K > 0 ? ncand : 0;
        const int nc_max = max(__builtin_amdgcn_readlane(nc, 0), __builtin_amdgcn_readlane(nc, 32));
        auto key_at = [&](int c) -> unsigned long long {
            const uint32_t d = c < nc ? dk[c] : kTaken;
            return d == kTaken ? ~0ull : (static_cast<unsigned long long>(d) << 32) | static_cast<uint32_t>(c);
        };
        unsigned long long lmin = ~0ull;
        for (int c0 = 0; c0 < nc_max; c0 += 128) {
            unsigned long long k[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) k[u] = key_at(c0 + 32 * u + hl);
#pragma unroll
            for (int u = 0; u < 4; ++u) lmin = k[u] < lmin ? k[u] : lmin;
        }
        const unsigned long long sorted = sort32_u64(lmin);
        const int k0 = __builtin_amdgcn_readlane(K, 0), k1 = __builtin_amdgcn_readlane(K, 32);
        const int s0 = max(k0 - 1, 0), s1 = 32 + max(k1 - 1, 0);
        const unsigned long long t0 =
            (static_cast<unsigned long long>(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(sorted >> 32), s0))) << 32) |
            static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(sorted), s0));
        const unsigned long long t1 =
            (static_cast<unsigned long long>(static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(sorted >> 32), s1))) << 32) |
            static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(sorted), s1));
        // ~0 (self, no candidate) is the largest key: clamping T below it
        // leaves it out of the gather
        const unsigned long long T = min((threadIdx.x & 32) ? t1 : t0, ~0ull - 1);
        const uint32_t below = (1u << hl) - 1u;  // lanes of this half below this one
        unsigned long long* sv = surv + half * NG;
        int n = 0;  // keys gathered so far by this half
        for (int c0 = 0; c0 < nc_max; c0 += 128) {
            unsigned long long k[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) k[u] = key_at(c0 + 32 * u + hl);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const bool take = k[u] <= T;
                const unsigned long long m = __ballot(take);
                if (m) {
                    const uint32_t mh = (threadIdx.x & 32) ? static_cast<uint32_t>(m >> 32) : static_cast<uint32_t>(m);
                    const int slot = n + __popc(mh & below);
                    if (take && slot < NG) sv[slot] = k[u];
                    n += __popc(mh);
                }
            }
        }
        const int n0 = __builtin_amdgcn_readlane(n, 0), n1 = __builtin_amdgcn_readlane(n, 32);
        if (n0 <= NG && n1 <= NG) {
            wave_sync();
            // lane hl ranks the gathered keys hl, hl + 32, ... of its half
            const int nmax = max(n0, n1), qn = (nmax + 31) >> 5;
            unsigned long long own[NG / 32];
            int rank[NG / 32];
#pragma unroll
            for (int q = 0; q < NG / 32; ++q) {
                own[q] = q < qn && hl + 32 * q < n ? sv[hl + 32 * q] : ~0ull;
                rank[q] = 0;
            }
            for (int j0 = 0; j0 < nmax; j0 += 8) {
                unsigned long long o[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) o[u] = j0 + u < n ? sv[j0 + u] : ~0ull;
#pragma unroll
                for (int q = 0; q < NG / 32; ++q)
                    if (q < qn) {
#pragma unroll
                        for (int u = 0; u < 8; ++u) rank[q] += o[u] < own[q] ? 1 : 0;
                    }
            }
#pragma unroll
            for (int q = 0; q < NG / 32; ++q)
                if (hl + 32 * q < n && rank[q] < K) {
                    const int c = static_cast<int>(static_cast<uint32_t>(own[q]));
                    const int dy = div_small(c, inv_ww), dx = c - dy * ww;
                    out[1 + rank[q]] = MatchRec{left + dx, top + dy, jb.t0, static_cast<uint32_t>(own[q] >> 32)};
                }
            return;
        }
    }
    // Each lane keeps the four smallest of its keys (window indices c = hl
    // mod 32) sorted in registers; a round's winner is the half-wave minimum
    // of the lanes' heads, and only the winning lane advances (rebuilding its
    // four from LDS, where given-away keys are marked taken, after its fourth).
    unsigned long long best4[4];
    auto insert = [&](uint32_t d, int c) {
        const unsigned long long x = (static_cast<unsigned long long>(d) << 32) | static_cast<uint32_t>(c);
        if (d != kTaken && x < best4[3]) {
            best4[3] = x;
            if (best4[3] < best4[2]) { const unsigned long long t = best4[2]; best4[2] = best4[3]; best4[3] = t; }
            if (best4[2] < best4[1]) { const unsigned long long t = best4[1]; best4[1] = best4[2]; best4[2] = t; }
            if (best4[1] < best4[0]) { const unsigned long long t = best4[0]; best4[0] = best4[1]; best4[1] = t; }
        }
    };
    auto rebuild = [&]() {
        best4[0] = best4[1] = best4[2] = best4[3] = ~0ull;
        // four keys read before any is inserted (their LDS loads overlap)
        for (int c0 = hl; c0 < ncand; c0 += 128) {
            uint32_t d[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) d[u] = c0 + 32 * u < ncand ? dk[c0 + 32 * u] : kTaken;
#pragma unroll
            for (int u = 0; u < 4; ++u) insert(d[u], c0 + 32 * u);
        }
    };
    if (K > 0) {
        rebuild();
    } else {
        best4[0] = best4[1] = best4[2] = best4[3] = ~0ull;
    }
    // Round k's winner is kept by lane k of the half (k < 32) and the
    // records are written together after the rounds.
    int given = 0;
    unsigned long long won = ~0ull;
    for (int k = 0; k < kmax; ++k) {
        const bool live = k < K;
        const unsigned long long head = live ? best4[0] : ~0ull;
        const uint32_t hd = static_cast<uint32_t>(head >> 32);
        const uint32_t md = half_min_u32(hd);
        // The lanes holding the smallest distance: one per half (the usual
        // case) gives the winner directly; a tie between lanes is broken by
        // the smallest window index, as match_tie_less does.
        const unsigned long long at_min = __ballot(live && hd == md);
        const uint32_t lo_mask = static_cast<uint32_t>(at_min), hi_mask = static_cast<uint32_t>(at_min >> 32);
        uint32_t mc;
        if (__popc(lo_mask) <= 1 && __popc(hi_mask) <= 1) {
            const int hc = static_cast<int>(static_cast<uint32_t>(head));
            const uint32_t c0 = static_cast<uint32_t>(__builtin_amdgcn_readlane(hc, lo_mask ? __builtin_ctz(lo_mask) : 0));
            const uint32_t c1 =
                static_cast<uint32_t>(__builtin_amdgcn_readlane(hc, hi_mask ? 32 + __builtin_ctz(hi_mask) : 32));
            mc = (threadIdx.x & 32) ? c1 : c0;
        } else {
            mc = half_min_u32(hd == md ? static_cast<uint32_t>(head) : 0xffffffffu);
        }
        const unsigned long long best = (static_cast<unsigned long long>(md) << 32) | mc;
        const int c = static_cast<int>(mc);
        if (hl == k) won = best;
        if (live && k >= 32 && hl == 0) {
            const int dy = div_small(c, inv_ww), dx = c - dy * ww;
            out[1 + k] = MatchRec{left + dx, top + dy, jb.t0, md};
        }
        if (live && hl == (c & 31)) {
            dk[c] = kTaken;
            best4[0] = best4[1];
            best4[1] = best4[2];
            best4[2] = best4[3];
            best4[3] = ~0ull;
            if (++given == 4) {
                given = 0;
                rebuild();
            }
        }
    }
    if (hl < K && hl < 32) {
        const int c = static_cast<int>(static_cast<uint32_t>(won));
        const int dy = div_small(c, inv_ww), dx = c - dy * ww;
        out[1 + hl] = MatchRec{left + dx, top + dy, jb.t0, static_cast<uint32_t>(won >> 32)};
    }
}

// SMALL: the one-tile-per-lane layout; else keys in LDS as they are scored.
template <int B, bool SMALL>
__global__ __launch_bounds__(256) void match_run_kernel(MatchTable tab) {
    match_run_body<B, SMALL ? 1 : 0>(tab);
}

// Up to kRunMidTiles lane tiles per lane, their keys in registers.
template <int B>
__global__ __launch_bounds__(256) void match_run_mid_kernel(MatchTable tab) {
    match_run_body<B, kRunMidTiles>(tab);
}

// General matcher: one wave per reference.
template <int B, bool STAGE>
__global__ __launch_bounds__(64) void match_wave_kernel(MatchTable tab) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x;
    const int lb = xcd_block();
    const MatchJob& jb = tab.job[find_job(tab, lb)];
    const int ref = lb - jb.wg_begin;
    if (ref >= jb.grid.nx * jb.grid.ny) return;
    const int cx = ref_x(jb.grid, ref % jb.grid.nx, jb.width, B);
    const int cy = ref_y(jb.grid, ref / jb.grid.nx, jb.height, B);
    const int r = jb.range;
    const int top = max(cy - r, 0), bottom = min(cy + r, jb.height - B);
    const int left = max(cx - r, 0), right = min(cx + r, jb.width - B);
    const int ww = right - left + 1, wh = bottom - top + 1;
    const int ncand = ww * wh;
    const int rw = ww + B - 1, rh = wh + B - 1;

    const float* reg;
    int rs;
    uint32_t* dk;
    if constexpr (STAGE) {
        // straight to LDS (global_load_lds: lane l's word at the uniform
        // address lreg + yy rw + x0 + 4 l), every row's loads in flight
        // together; the barrier below waits for them
        float* lreg = reinterpret_cast<float*>(smem);
        for (int yy = 0; yy < rh; ++yy) {
            const float* row = jb.plane + static_cast<size_t>(top + yy) * jb.stride + left;
            for (int x0 = 0; x0 < rw; x0 += 64)
                if (x0 + lane < rw)
                    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(row + x0 + lane),
                                                     (__attribute__((address_space(3))) void*)(lreg + yy * rw + x0), 4,
                                                     0, 0);
        }
        reg = lreg;
        rs = rw;
        dk = reinterpret_cast<uint32_t*>(smem) + ((rw * rh + 3) & ~3);
    } else {
        reg = jb.plane + static_cast<size_t>(top) * jb.stride + left;
        rs = jb.stride;
        dk = reinterpret_cast<uint32_t*>(smem);
    }
    __syncthreads();

    const float* refp = reg + (cy - top) * rs + (cx - left);
    const int self = (cy - top) * ww + (cx - left);
    for (int c = lane; c < ncand; c += 64) {
        const int dy = c / ww, dx = c - dy * ww;
        const float* cp = reg + dy * rs + dx;
        float acc = 0.f;
        for (int py = 0; py < B; ++py) {
#pragma unroll
            for (int px = 0; px < B; ++px) {
                const float d = refp[py * rs + px] - cp[py * rs + px];
                acc = fmaf(d, d, acc);
            }
        }
        dk[c] = c == self ? kTaken : dist_key(acc);
    }
    __syncthreads();

    const int K = min(jb.group - 1, ncand - 1);
    MatchRec* out = jb.out + static_cast<size_t>(ref) * jb.group;
    if (lane == 0) out[0] = MatchRec{cx, cy, jb.t0, 0u};
    for (int i = 0; i < K; ++i) {
        unsigned long long best = ~0ull;
        for (int c = lane; c < ncand; c += 64) {
            const uint32_t d = dk[c];
            const unsigned long long key = (static_cast<unsigned long long>(d) << 32) | static_cast<uint32_t>(c);
            best = (d != kTaken && key < best) ? key : best;
        }
        best = wave_min_u64(best);
        const int c = static_cast<int>(static_cast<uint32_t>(best));
        if (lane == (c & 63)) {
            dk[c] = kTaken;
            const int dy = c / ww, dx = c - dy * ww;
            out[1 + i] = MatchRec{left + dx, top + dy, jb.t0, static_cast<uint32_t>(best >> 32)};
        }
        __syncthreads();
    }
    if (lane == 0) jb.counts[ref] = 1 + K;
}

// ---------------------------------------------------------------------------
// MFMA matcher (B = 8, G <= 32): the role of the reference's tensor-core
// matcher (src/cuda/common/match.cu:1165-1620, spatial_match_tensor), built
// for CDNA4. A workgroup of four waves takes a block of 4 x 4 references.
// The union of their windows is staged in LDS in FP32 (when that leaves four
// workgroups per CU) and as fp16 values h = fp16((v - mu) 2^S), S a scale of
// the block that keeps them below 2^13. Dot products of reference and
// candidate patches run on v_mfma_f32_16x16x32_f16 (16 references x 16
// candidates of one row per tile), giving d' = |h_r|^2 + |h_c|^2 - 2 h_r.h_c
// for every pair; wave w takes the candidate rows w mod 4. A third MFMA adds
// the candidates' norms with the bound's slope, and the accumulators start at
// the reference's constant, +inf outside its window: the VALU sees finished
// bounds, one operation per pair and pass. Two passes over the tiles:
//   A. per reference, the smallest upper bound U of each of 64 classes of
//      candidates (a lane's column residue, a wave's rows): the (K + 1)-th
//      smallest of those (the reference itself is among them) bounds the K-th
//      exact key from above;
//   B. every candidate whose lower bound L does not exceed it is listed (at
//      most 128 per reference for G <= 16, 192 for G <= 32), from the sign bits
//      of L minus the bound.
// The listed candidates are then scored in the FP32 order of the other
// matchers (rows, then columns, one fmaf per pixel) and taken in order of
// (dist, y, x): the records are those of match_run_kernel bit for bit. A
// reference whose list overflows, or a block holding a value fp16 cannot
// carry (non-finite, or |v - mu| >= 8192 so that S would be negative), scores
// its whole window exactly. A region of one value needs no scores at all.
//
// What bounds it: VALU issue and the matrix unit together. Per wave of the 1080p
// YUV420, step-3, range-19, group-16 launch 3.25 k VALU instructions, 211 MFMAs
// among them (with the norms, masks and rank sums on the VALU 6.0 k at range 16
// already): 0.8 of the two a CU can issue per cycle, the matrix units busy 27 %
// of the time, 28 % of the wave cycles waiting. At range 30 (7.2 k, 737) 0.6,
// 34 % and 30 %: 56 KB of LDS leave two workgroups per CU. The bound of five
// workgroups per CU spills four registers (20 bytes of scratch per lane).
// Per 1080p YUV420 frame at step 3, range 16: group 16 on the noisy planes 627
// us (1115 before the norms and masks went into the MFMAs, the sums of ranks into
// row minima and the reference's patch into registers); gray 1080p, step 8, range
// 30, group 16: 244 us (468). Group 32 on denoised planes took 1060 us (1758);
// lists of 160 cost 1340 there (overflows), of 256 1126 (LDS: four workgroups per
// CU instead of five). A constant 1080p plane at step 3, range 16: 59 us (the run
// matcher 828).
//
// Error bound, in the scaled units (every distance times 2^2S; u = 2^-24):
//   per element, |(v - mu) 2^S - h| <= 2^-11 |h| (1 + 2^-11) for a normal h,
//     and < 2^-14 where h was flushed to 0 (below fp16's smallest normal);
//     over a patch, E_c^2 <= kappa (|h_c|^2 + 1), kappa = 1.002 2^-22;
//   |d' - d''| <= C1 (|h_r|^2 + |h_c|^2), d'' the exact SSD of the fp16
//     patches (squares exact, 64-term FP32 sums and the MFMA's FP32
//     accumulation, about 200 u), C1 = 512 u;
//   by the triangle inequality sqrt(d*) lies within E_r + E_c of
//     sqrt(d''), d* the real SSD; with (a + b)^2 <= (1 + t) a^2 +
//     (1 + 1/t) b^2, (a - b)^2 >= (1 - t) a^2 - (1/t - 1) b^2 (t = 2^-6)
//     and E^2 <= 2 E_r^2 + 2 E_c^2 both bounds are linear in (c, |h_c|^2),
//     c = |h_r|^2 - 2 h_r.h_c the fp16 products' sum;
//   the FP32 key differs from d* by at most 66 u d* (taken as 1e-4).
// ---------------------------------------------------------------------------

typedef _Float16 mm_h16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 mm_h16x2 __attribute__((ext_vector_type(2)));
typedef float mm_f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t mm_u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t mm_u32x2 __attribute__((ext_vector_type(2)));
typedef float mm_f32x2 __attribute__((ext_vector_type(2)));

inline constexpr float kMmC1 = 3.0517578125e-05f;    // 512 * 2^-24
inline constexpr float kMmInf = __builtin_inff();
inline constexpr float kMmT = 0.015625f;              // t = 2^-6
inline constexpr float kMmKappa = 2.3889e-07f;        // 1.002 * 2^-22, rounded up
inline constexpr float kMmGammaU = 2.f * kMmKappa * (1.f + 1.f / kMmT);  // E^2 weight, upper bound
inline constexpr float kMmGammaL = 2.f * kMmKappa / kMmT;                // E^2 weight, lower bound
// Per-pair slopes in |h_c|^2 of the bounds U / (1 + t) and L / (1 - t) (c has
// slope 1): (1 + C1) + gamma_U / (1 + t) and (1 - C1) - gamma_L / (1 - t).
inline constexpr float kMmSlopeU = 1.f + kMmC1 + kMmGammaU / (1.f + kMmT) + 1e-6f;
inline constexpr float kMmSlopeL = 1.f - kMmC1 - kMmGammaL / (1.f - kMmT) - 1e-6f;

// Two fp16 values of one region word (rounded to nearest even).
__device__ inline uint32_t mm_pack(float a, float b) {
    return __builtin_bit_cast(uint32_t, mm_h16x2{static_cast<_Float16>(a), static_cast<_Float16>(b)});
}

// Eight fp16 values at region row `row`, columns col .. col + 7 (two per
// word; odd columns realigned with a funnel shift).
__device__ inline mm_h16x8 mm_frag(const uint32_t* reg, int pitch, int row, int col) {
    const uint32_t* p = reg + row * pitch + (col >> 1);
    const uint32_t w0 = p[0], w1 = p[1], w2 = p[2], w3 = p[3], w4 = p[4];
    const uint32_t sh = static_cast<uint32_t>(col & 1) * 16u;
    const mm_u32x4 o = {__builtin_amdgcn_alignbit(w1, w0, sh), __builtin_amdgcn_alignbit(w2, w1, sh),
                        __builtin_amdgcn_alignbit(w3, w2, sh), __builtin_amdgcn_alignbit(w4, w3, sh)};
    return __builtin_bit_cast(mm_h16x8, o);
}

__device__ inline float mm_sq(mm_h16x8 f) {
    float s = __builtin_amdgcn_fdot2(mm_h16x2{f[0], f[1]}, mm_h16x2{f[0], f[1]}, 0.f, false);
    s = __builtin_amdgcn_fdot2(mm_h16x2{f[2], f[3]}, mm_h16x2{f[2], f[3]}, s, false);
    s = __builtin_amdgcn_fdot2(mm_h16x2{f[4], f[5]}, mm_h16x2{f[4], f[5]}, s, false);
    return __builtin_amdgcn_fdot2(mm_h16x2{f[6], f[7]}, mm_h16x2{f[6], f[7]}, s, false);
}

// Sum over lanes n, n + 16, n + 32, n + 48 (the four 16-lane rows), equal in
// all four: rows swapped pairwise, then halves (additions commute).
__device__ inline float mm_rows_sum(float v) {
    const uint32_t b = __float_as_uint(v);
    const auto p = __builtin_amdgcn_permlane16_swap(b, b, false, false);
    const float s = __uint_as_float(p[0]) + __uint_as_float(p[1]);
    const uint32_t c = __float_as_uint(s);
    const auto q = __builtin_amdgcn_permlane32_swap(c, c, false, false);
    return __uint_as_float(q[0]) + __uint_as_float(q[1]);
}

// v of the lane DPP control CTRL selects (controls that stay inside a row).
template <int CTRL>
__device__ inline float dpp_f32(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, false));
}

template <int CTRL>
__device__ inline uint32_t dpp_row_u32(uint32_t v) {
    return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), CTRL, 0xf, 0xf, true));
}

// The value of lane l (uniform).
__device__ inline float lane_f32(float v, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// Sum and maximum over the wave in a fixed order, the result in every lane:
// each 16-lane row by DPP (quad_perm [1,0,3,2] and [2,3,0,1], row_half_mirror,
// row_mirror), then the four rows' results. All 64 lanes must call.
__device__ inline float wave_sum_dpp(float v) {
    v += dpp_f32<0xb1>(v);
    v += dpp_f32<0x4e>(v);
    v += dpp_f32<0x141>(v);
    v += dpp_f32<0x140>(v);
    return (lane_f32(v, 0) + lane_f32(v, 16)) + (lane_f32(v, 32) + lane_f32(v, 48));
}

__device__ inline float wave_max_dpp(float v) {
    v = fmaxf(v, dpp_f32<0xb1>(v));
    v = fmaxf(v, dpp_f32<0x4e>(v));
    v = fmaxf(v, dpp_f32<0x141>(v));
    v = fmaxf(v, dpp_f32<0x140>(v));
    return fmaxf(fmaxf(lane_f32(v, 0), lane_f32(v, 16)), fmaxf(lane_f32(v, 32), lane_f32(v, 48)));
}

// Lane N's value of each 16-lane row, in all its lanes (row_newbcast).
template <int N>
__device__ __forceinline__ float row_bcast_f32(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + N, 0xf, 0xf, false));
}

// The FP32 key of the other matchers for B = 8 (rows, then columns, one fmaf
// per pixel) with the reference's patch held by the 16-lane row (pixel 4 n + i
// in lane n's patch[i]); b the candidate's first pixel, rows p apart. All 64
// lanes must call. The broadcasts are operands of the subtractions, and only
// the candidate is read: half the LDS words of reading both, which bound it.
template <class Pitch>
__device__ __forceinline__ uint32_t mm_exact_row(const float (&patch)[4], const float* b, Pitch p) {
    float acc = 0.f;
    static_for<8>([&](auto yc) {
        constexpr int py = decltype(yc)::value;
        float v[8];
#pragma unroll
        for (int px = 0; px < 8; ++px) v[px] = b[py * p + px];
        static_for<8>([&](auto xc) {
            constexpr int px = decltype(xc)::value;
            const float d = row_bcast_f32<2 * py + (px >> 2)>(patch[px & 3]) - v[px];
            acc = fmaf(d, d, acc);
        });
    });
    return dist_key(acc);
}

// Largest of the four 16-lane rows' values (each row's lanes hold the same).
__device__ inline int wave_rows_max(int v) {
    return max(max(__builtin_amdgcn_readlane(v, 0), __builtin_amdgcn_readlane(v, 16)),
               max(__builtin_amdgcn_readlane(v, 32), __builtin_amdgcn_readlane(v, 48)));
}

// Minimum over the 16 lanes of each DPP row, returned to every lane of the
// row (quad_perm, row_half_mirror, row_mirror: folded into the minima).
__device__ inline uint32_t row_min_u32(uint32_t v) {
    v = min(v, dpp_row_u32<0xb1>(v));
    v = min(v, dpp_row_u32<0x4e>(v));
    v = min(v, dpp_row_u32<0x141>(v));
    return min(v, dpp_row_u32<0x140>(v));
}

// Minimum over the wave, uniform. All 64 lanes must call.
__device__ inline uint32_t wave_min_u32_dpp(uint32_t v) {
    v = row_min_u32(v);
    const auto of = [&](int l) { return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), l)); };
    return min(min(of(0), of(16)), min(of(32), of(48)));
}

// Whether a 16-bit field of m has two bits set or more.
__device__ inline bool rows_with_two(unsigned long long m) {
    bool two = false;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const uint32_t f = static_cast<uint32_t>(m >> (16 * r)) & 0xffffu;
        two = two || (f & (f - 1u)) != 0u;
    }
    return two;
}

// Region row pitch in words: the smallest p >= 8 nt + 5 (16 nt + 8 halves
// and the fifth word of an odd-column read) at which the four 16-lane rows
// of a fragment read (each within 9 consecutive words, rows p apart) fall on
// disjoint banks, for 32 banks (two rows per half-wave) and for 64.
constexpr int mm_pitch_of(int nt) {
    for (int p = 8 * nt + 5;; ++p) {
        const int a = p % 32;
        if (a < 9 || a > 23) continue;
        const int o[4] = {0, p % 64, (2 * p) % 64, (3 * p) % 64};
        bool ok = true;
        for (int i = 0; i < 4; ++i)
            for (int j = i + 1; j < 4; ++j) {
                const int d = ((o[i] - o[j]) % 64 + 64) % 64;
                ok = ok && d >= 9 && d <= 55;
            }
        if (ok) return p;  // p = 16 mod 64 always qualifies
    }
}
inline constexpr int kMmTiles = 10;  // tile columns of the largest union (step 8, range 64)
struct MmPitches {
    int of[kMmTiles + 1];
};
constexpr MmPitches mm_pitches() {
    MmPitches t{};
    for (int i = 1; i <= kMmTiles; ++i) t.of[i] = mm_pitch_of(i);
    return t;
}
__device__ constexpr MmPitches d_mm_pitch = mm_pitches();
inline constexpr MmPitches h_mm_pitch = mm_pitches();

struct MmWin {
    int cx, cy, left, right, top, bottom;
};

__device__ inline MmWin mm_win(const MatchJob& jb, int i, int j) {
    MmWin w;
    w.cx = ref_x(jb.grid, i, jb.width, 8);
    w.cy = ref_y(jb.grid, j, jb.height, 8);
    w.left = max(w.cx - jb.range, 0);
    w.right = min(w.cx + jb.range, jb.width - 8);
    w.top = max(w.cy - jb.range, 0);
    w.bottom = min(w.cy + jb.range, jb.height - 8);
    return w;
}

__device__ inline uint32_t row_max_u32(uint32_t v) {
    v = max(v, dpp_row_u32<0xb1>(v));
    v = max(v, dpp_row_u32<0x4e>(v));
    v = max(v, dpp_row_u32<0x141>(v));
    return max(v, dpp_row_u32<0x140>(v));
}

// Pitch of the staged FP32 region for nt tile columns: its 16 nt + 8 columns,
// and rows that start on different banks.
__host__ __device__ constexpr int mm_pitch32(int nt) { return 16 * nt + 10; }

inline constexpr int kMmCounters = 48;  // words of the counters, K values and bounds

// LIST: listed candidates per reference (128 for G <= 16, 192 for G <= 32).
// STAGED: the FP32 region is held in LDS too, read from memory once (straight
// to LDS); the scaling pass, the fp16 values and the exact keys come from it.
// Without it (regions too large) those read the plane.
template <int LIST, bool STAGED>
__global__ __launch_bounds__(256, 5) void match_mfma_kernel(MatchTable tab) {
    extern __shared__ __align__(16) uint32_t mm_lds[];
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, n = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: row loops branch on scalars
    // Dispatch order, XCDs in turn: blocks cost what their content makes them
    // list, and an XCD's own band of the frame would leave the others waiting
    // (a band per XCD: 698 against 665 us on 1080p YUV420 at step 3, range 16,
    // group 16); the regions' overlap is read from the last-level cache.
    const int lb = static_cast<int>(blockIdx.x);
    const MatchJob& jb = tab.job[find_job(tab, lb)];
    const int blk = lb - jb.wg_begin;
    const int nbx = (jb.grid.nx + 3) >> 2;
    const int by = blk / nbx, bx = blk - by * nbx;
    const int i0 = 4 * bx, j0 = 4 * by;
    const int ncol = min(4, jb.grid.nx - i0), nrow = min(4, jb.grid.ny - j0);
    const float* plane = jb.plane;
    const size_t stride = static_cast<size_t>(jb.stride);
    const int G = jb.group;

    const MmWin w00 = mm_win(jb, i0, j0), wlast = mm_win(jb, i0 + ncol - 1, j0 + nrow - 1);
    const int ux0 = w00.left, ux1 = wlast.right, uy0 = w00.top, uy1 = wlast.bottom;
    const int nt = (ux1 - ux0 + 16) >> 4;
    const int UW = 16 * nt;
    const int RH = uy1 - uy0 + 8;
    const int pitch = d_mm_pitch.of[nt];
    const int reg_words = (max(RH * pitch, 16 * LIST) + 3) & ~3;
    uint32_t* reg = mm_lds;
    // One area serves, in turn, the staging reductions and the pass-A
    // exchange (xw), the candidate lists (pass B, ranking), and the
    // fallback's keys.
    constexpr int kUnion = 8 * LIST;                                    // words (at least the exchange's 1024)
    uint32_t* xw = mm_lds + reg_words;
    const int P32 = mm_pitch32(nt);
    float* f32 = reinterpret_cast<float*>(mm_lds + reg_words + kUnion + kMmCounters);  // STAGED: rows of P32 floats
    uint16_t* list = reinterpret_cast<uint16_t*>(xw);                   // [16][LIST]
    int* cnt = reinterpret_cast<int*>(mm_lds + reg_words + kUnion);     // 16
    int* kmv = cnt + 16;                                                // 16
    float* wl = reinterpret_cast<float*>(kmv + 16);                     // 16 (kMmCounters words in all)

    // Per-reference counts K = min(G - 1, window - 1); counters cleared.
    if (tid < 16) {
        const int c = tid >> 2, j = tid & 3;
        int k = 0;
        if (c < ncol && j < nrow) {
            const MmWin w = mm_win(jb, i0 + c, j0 + j);
            k = min(G - 1, (w.right - w.left + 1) * (w.bottom - w.top + 1) - 1);
        }
        kmv[tid] = k;
        cnt[tid] = 0;
    }

    // mu: the mean of the first reference's patch (every wave alike). Two
    // passes over the region: the largest |v - mu| as bits (a non-finite
    // value's are the largest), then the scaled fp16 values. A wave's lanes
    // take words_per consecutive words of rows_per rows (a whole row per
    // step when a row has more than 64).
    float mu;
    const int wpr = 8 * nt + 4;  // words of a row that the fragments read
    const int rows_per = wpr <= 64 ? 64 / wpr : 1;
    const int lr = wpr <= 64 ? div_small(lane, 1.f / static_cast<float>(wpr)) : 0;
    const int lw = wpr <= 64 ? lane - lr * wpr : lane;
    // f(row, word, pixel, next pixel) of the region's words, four rows' loads
    // in flight
    auto each_word = [&](auto f) {
        if (lr >= rows_per) return;
        for (int w0 = lw; w0 < wpr; w0 += 64)
            for (int y0 = wave * rows_per + lr; y0 < RH; y0 += 16 * rows_per) {
                mm_f32x2 v[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const int yy = min(y0 + 4 * i * rows_per, RH - 1);
                    if constexpr (STAGED) {
                        v[i] = *reinterpret_cast<const mm_f32x2*>(f32 + yy * P32 + 2 * w0);
                    } else {
                        const float* row = plane + static_cast<size_t>(uy0 + yy) * stride;
                        v[i][0] = row[min(ux0 + 2 * w0, jb.width - 1)];
                        v[i][1] = row[min(ux0 + 2 * w0 + 1, jb.width - 1)];
                    }
                }
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    if (y0 + 4 * i * rows_per < RH) f(y0 + 4 * i * rows_per, w0, v[i][0], v[i][1]);
            }
    };
    if constexpr (STAGED) {
        // Rows wave, wave + 4, ... by 64-column strips, each load straight to
        // LDS (lane l's word lands at the wave-uniform address + 4 l); columns
        // past the plane repeat its last (only masked candidates read them).
        for (int c0 = 0; c0 < 16 * nt + 8; c0 += 64) {
            const int xx = c0 + lane;
            if (xx < 16 * nt + 8) {
                const int gx = min(ux0 + xx, jb.width - 1);
                for (int yy = wave; yy < RH; yy += 4)
                    __builtin_amdgcn_global_load_lds(
                        (const __attribute__((address_space(1))) void*)(plane + static_cast<size_t>(uy0 + yy) * stride + gx),
                        (__attribute__((address_space(3))) void*)(f32 + yy * P32 + c0), 4, 0, 0);
            }
        }
        __syncthreads();
        mu = wave_sum_dpp(f32[(w00.cy - uy0 + (lane >> 3)) * P32 + w00.cx - ux0 + (lane & 7)]) * (1.f / 64.f);
    } else {
        mu = wave_sum_dpp(plane[static_cast<size_t>(w00.cy + (lane >> 3)) * stride + w00.cx + (lane & 7)]) * (1.f / 64.f);
    }
    // S = 12 serves a largest |v - mu| in [2^-6, 2) (planes in [0, 1] with
    // any structure): the first pass converts with it and finds the largest.
    // Others convert again with their own S = 13 - e, bmax < 2^e: below 2^13
    // either way (|-2 h| < 2^15 fits fp16).
    // (v - mu) 2^S in one rounding: mu 2^S is exact. A value below fp16's
    // smallest normal keeps an error below 2^-14 whether the products take it
    // as a denormal or as 0.
    uint32_t amax = __float_as_uint(mu) & 0x7fffffffu;
    amax = amax >= kNonFinite ? amax : 0u;
    each_word([&](int yy, int w, float v0, float v1) {
        const float a0 = fmaf(v0, 4096.f, -mu * 4096.f), a1 = fmaf(v1, 4096.f, -mu * 4096.f);
        amax = max(amax, __float_as_uint(a0) & 0x7fffffffu);
        amax = max(amax, __float_as_uint(a1) & 0x7fffffffu);
        reg[yy * pitch + w] = mm_pack(a0, a1);
    });
    amax = row_max_u32(amax);
    if (n == 0) xw[wave * 4 + g] = amax;
    __syncthreads();
    const uint32_t bmax_bits = __builtin_amdgcn_readfirstlane(row_max_u32(xw[n]));
    const float bmax = __uint_as_float(bmax_bits) * (1.f / 4096.f);
    // One value everywhere (mu is then exactly it, and no difference vanishes
    // in the scaling): every distance is 0, so the records are the first places
    // of the window, the reference's own left out. Lane n of row g of wave w
    // takes the records n + 1, n + 17 of reference 4 w + g. Scoring the windows
    // of such regions exactly cost more than the run matcher does: 1080p, group
    // 16, half the frame constant: step 3, range 9 452 us (run matcher 341), now
    // 236; step 4, range 9 252 (196), now 127.
    const bool flat_region = bmax_bits == 0u;
    if (flat_region) {
        const int m = 4 * wave + g, K = kmv[m];
        const int ri = i0 + min(m >> 2, ncol - 1), rj = j0 + min(m & 3, nrow - 1);
        const MmWin w = mm_win(jb, ri, rj);
        const int ww = w.right - w.left + 1, self = (w.cy - w.top) * ww + (w.cx - w.left);
        const float inv_ww = 1.f / static_cast<float>(ww);
        MatchRec* out = jb.out + (static_cast<size_t>(rj) * jb.grid.nx + ri) * G + 1;
        for (int k = n; k < K; k += 16) {
            const int c = k + (k >= self ? 1 : 0);
            const int dy = div_small(c, inv_ww), dx = c - dy * ww;
            out[k] = MatchRec{w.left + dx, w.top + dy, jb.t0, 0u};
        }
    }
    bool anybad = bmax_bits >= kNonFinite || !(bmax < 8192.f) || flat_region;
    if (!anybad && !(bmax >= 0.015625f && bmax < 2.f)) {
        int ex = 0;
        (void)frexpf(bmax, &ex);
        const int S = min(13 - ex, 40);
        anybad = S < 0;
        if (!anybad) {
            const float sc = ldexpf(1.f, S), msc = -mu * sc;
            each_word([&](int yy, int w, float v0, float v1) {
                reg[yy * pitch + w] = mm_pack(fmaf(v0, sc, msc), fmaf(v1, sc, msc));
            });
        }
    }
    __syncthreads();

    if (!anybad) {
        // A operand: reference n (column n >> 2, row n & 3), patch rows g
        // and g + 4.
        const int acol = n >> 2, arow = n & 3;
        mm_h16x8 A0 = {}, A1 = {};
        if (acol < ncol && arow < nrow) {
            const MmWin w = mm_win(jb, i0 + acol, j0 + arow);
            A0 = mm_frag(reg, pitch, w.cy - uy0 + g, w.cx - ux0);
            A1 = mm_frag(reg, pitch, w.cy - uy0 + 4 + g, w.cx - ux0);
        }
        const float nrA = mm_rows_sum(mm_sq(A0) + mm_sq(A1));  // |h_r|^2 of reference n
        // The reference operand enters as -2 h_r (exact in fp16) and the
        // accumulator starts at |h_r|^2: a tile then holds |h_r|^2 - 2 h_r.h_c.
        A0 *= static_cast<_Float16>(-2.f);
        A1 *= static_cast<_Float16>(-2.f);
        // C layout: lane (g, n) holds references 4 g + j (column g, row j)
        // against candidate n of the tile.
        float nr[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) nr[j] = __shfl(nrA, 4 * g + j, 64);
        const bool cval = g < ncol;
        const MmWin cw = mm_win(jb, i0 + min(g, ncol - 1), j0);
        const int cleft = cval ? cw.left - ux0 : (1 << 30), cright = cval ? cw.right - ux0 : -1;
        // Each wave takes the candidate rows uy0 + wave + 4 i, i < steps; row
        // j's windows hold the steps i with i - first[j] <= count[j] (unsigned;
        // uniform, so the tests below are scalar).
        const int steps = (uy1 - uy0 - wave + 4) >> 2;
        int first[4];
        uint32_t count[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const MmWin w = mm_win(jb, i0, j0 + min(j, nrow - 1));
            const int a = (max(w.top - uy0 - wave, 0) + 3) >> 2, b = (w.bottom - uy0 - wave) >> 2;
            const bool any = j < nrow && w.bottom - uy0 - wave >= 0 && b >= a;
            first[j] = __builtin_amdgcn_readfirstlane(any ? a : 1 << 30);
            count[j] = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(any ? b - a : 0));
        }
        auto holds = [&](int i, int j) { return static_cast<uint32_t>(i - first[j]) <= count[j]; };

        // The tiles of NC tile columns from t0 on, row step by row step. A
        // tile is three MFMAs on c0: slope |h_c|^2 (lane (g, n)'s rows g and
        // g + 4 squared, summed over g by a row of slopes), then the two halves
        // of -2 h_r.h_c. c0 is each reference's start value, +inf where the
        // candidate column lies outside its window: no masks, norms or scaling
        // are left for the VALU. use(i, c) sees step i's tiles.
        auto pass_cols = [&](auto nc_tag, int t0, float slope, const float (&start)[4], auto use) {
            constexpr int NC = decltype(nc_tag)::value;
            mm_f32x4 c0[NC];
            mm_h16x8 F[2][NC];
            float sq[2][NC];
#pragma unroll
            for (int q = 0; q < NC; ++q) {
                const int col = 16 * (t0 + q) + n;
                const bool in = col >= cleft && col <= cright;
#pragma unroll
                for (int j = 0; j < 4; ++j) c0[q][j] = in ? start[j] : kMmInf;
                F[0][q] = mm_frag(reg, pitch, wave + g, col);
                sq[0][q] = mm_sq(F[0][q]);
            }
            auto step = [&](int i, const mm_h16x8 (&fa)[NC], const float (&sa)[NC], mm_h16x8 (&fb)[NC],
                            float (&sb)[NC]) {
                mm_f32x4 c[NC];
#pragma unroll
                for (int q = 0; q < NC; ++q) {
                    fb[q] = mm_frag(reg, pitch, wave + 4 * i + 4 + g, 16 * (t0 + q) + n);
                    sb[q] = mm_sq(fb[q]);
                    c[q] = __builtin_amdgcn_mfma_f32_16x16x4f32(slope, sa[q] + sb[q], c0[q], 0, 0, 0);
                    c[q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A0, fa[q], c[q], 0, 0, 0);
                    c[q] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A1, fb[q], c[q], 0, 0, 0);
                }
                use(i, c);
            };
            for (int i = 0; i < steps; i += 2) {
                step(i, F[0], sq[0], F[1], sq[1]);
                if (i + 1 < steps) step(i + 1, F[1], sq[1], F[0], sq[0]);
            }
        };
        auto pass = [&](float slope, const float (&start)[4], auto use) {
            for (int t = 0; t < nt;) {
                const int left = nt - t;
                if (left == 3 || left > 4) {
                    pass_cols(std::integral_constant<int, 3>{}, t, slope, start,
                              [&](int i, const mm_f32x4 (&c)[3]) { use(std::integral_constant<int, 3>{}, t, i, c); });
                    t += 3;
                } else if (left >= 2) {
                    pass_cols(std::integral_constant<int, 2>{}, t, slope, start,
                              [&](int i, const mm_f32x4 (&c)[2]) { use(std::integral_constant<int, 2>{}, t, i, c); });
                    t += 2;
                } else {
                    pass_cols(std::integral_constant<int, 1>{}, t, slope, start,
                              [&](int i, const mm_f32x4 (&c)[1]) { use(std::integral_constant<int, 1>{}, t, i, c); });
                    t += 1;
                }
            }
        };

        // Pass A: U / (1 + t) up to a per-reference constant; each lane keeps
        // the smallest of its candidates per reference (the positions of one
        // residue mod 16 columns and 4 rows: 64 disjoint classes). The start
        // is raised by the bound's own C1 |h_r|^2, and 2^-4: d' + C1 (|h_r|^2 +
        // |h_c|^2) stays above the sums' rounding, so the sums are positive,
        // order as their bits do, and the minimum is an integer one.
        float raised[4];
        uint32_t s[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            raised[j] = fmaf(nr[j], 1.f + kMmC1, 0.0625f);
            s[j] = kNonFinite;
        }
        pass(kMmSlopeU, raised, [&](auto nc_tag, int, int i, const auto& c) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (holds(i, j))
#pragma unroll
                    for (int q = 0; q < decltype(nc_tag)::value; ++q) s[j] = min(s[j], __float_as_uint(c[q][j]));
        });
        uint32_t* xch = xw;  // [wave][j][lane]
#pragma unroll
        for (int j = 0; j < 4; ++j) xch[(wave * 4 + j) * 64 + lane] = s[j];
        __syncthreads();
        // Wave w: references of row j = w. The (K + 1)-th smallest of the 64
        // classes' minima (the reference itself is one of the candidates) by
        // rounds of a row minimum over each lane's sorted four.
        {
            uint32_t m4[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) m4[v] = xch[(v * 4 + wave) * 64 + lane];
            auto order = [&](int a, int b) {
                const uint32_t lo = min(m4[a], m4[b]), hi = max(m4[a], m4[b]);
                m4[a] = lo;
                m4[b] = hi;
            };
            order(0, 1), order(2, 3), order(0, 2), order(1, 3), order(1, 2);
            const int K = kmv[4 * g + wave];
            int taken = 0;
            uint32_t tdb = kNonFinite;
            bool open = K > 0;
            while (__builtin_amdgcn_ballot_w64(open) != 0) {  // at most 64 / 16 + K rounds: each takes a class
                const uint32_t mn = row_min_u32(m4[0]);
                const bool eq = m4[0] == mn;
                const unsigned long long bal = __builtin_amdgcn_ballot_w64(eq);
                taken += __popc(static_cast<uint32_t>(bal >> (16 * g)) & 0xffffu);
                m4[0] = eq ? m4[1] : m4[0];
                m4[1] = eq ? m4[2] : m4[1];
                m4[2] = eq ? m4[3] : m4[2];
                m4[3] = eq ? kNonFinite : m4[3];
                if (open && taken > K) {
                    open = false;
                    tdb = mn;
                }
            }
            const float td = __uint_as_float(tdb);
            if (n == 0) {
                const float nrm = wave == 0 ? nr[0] : wave == 1 ? nr[1] : wave == 2 ? nr[2] : nr[3];
                float wt = -kMmInf;
                if (K > 0) {
                    if (!(td < kMmInf)) {
                        wt = 3.402823466e38f;  // every finite d' (masked pairs are +inf)
                    } else {
                        // U = (1 + t) td + beta_U bounds the K-th key;
                        // a candidate survives while its L = (1 - t) v -
                        // beta_L does not exceed U.
                        // (td holds C1 nrm already)
                        const float betaU = kMmGammaU * (nrm + 2.f);
                        const float betaL = (1.f - kMmT) * kMmC1 * nrm + kMmGammaL * (nrm + 2.f);
                        const float U = ((1.f + kMmT) * td + betaU) * 1.0001f;
                        wt = (U * 1.0001f + betaL) / (1.f - kMmT) * 1.00001f;
                    }
                }
                wl[4 * g + wave] = wt;
            }
        }
        __syncthreads();
        // Pass B: L / (1 - t) likewise, started at minus the bound: a negative
        // sum survives (equality too: the bound's own margins are far above a
        // rounding). Its sign goes into the lane's word of the tile column,
        // newest lowest; every eight steps, and at the end, the words' bits are
        // listed.
        float below[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) below[j] = nr[j] - wl[4 * g + j];
        uint32_t word[3] = {0u, 0u, 0u}, valid = 0u;
        pass(kMmSlopeL, below, [&](auto nc_tag, int t, int i, const auto& c) {
            constexpr int NC = decltype(nc_tag)::value;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                valid = (valid << 1) | (holds(i, j) ? 1u : 0u);
#pragma unroll
                for (int q = 0; q < NC; ++q) word[q] = __builtin_amdgcn_alignbit(word[q], __float_as_uint(c[q][j]), 31);
            }
            if ((i & 7) != 7 && i + 1 != steps) return;
#pragma unroll
            for (int q = 0; q < NC; ++q) {
                uint32_t bits = word[q] & valid;
                while (bits) {
                    const int at = __builtin_ctz(bits);  // step i - at / 4, row j = 3 - at % 4
                    bits &= bits - 1u;
                    const int m = 4 * g + 3 - (at & 3);
                    const int u = (wave + 4 * (i - (at >> 2))) * UW + 16 * (t + q) + n;
                    const int k = atomicAdd(&cnt[m], 1);
                    if (k < LIST) list[m * LIST + k] = static_cast<uint16_t>(u);
                }
            }
            valid = 0u;
        });
    }
    __syncthreads();

    // The patch at (x, y) over the lanes of a 16-lane row, and the exact key of
    // such a patch against the one at region column ux, row uy.
    auto row_patch = [&](int x, int y, float (&patch)[4]) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int py = y + (n >> 1), px = x + 4 * (n & 1) + i;
            patch[i] = STAGED ? f32[(py - uy0) * P32 + px - ux0] : plane[static_cast<size_t>(py) * stride + px];
        }
    };
    auto exact = [&](const float (&patch)[4], int ux, int uy) {
        if constexpr (STAGED)
            return mm_exact_row(patch, f32 + uy * P32 + ux, P32);
        else
            return mm_exact_row(patch, plane + static_cast<size_t>(uy0 + uy) * stride + ux0 + ux, stride);
    };

    // Listed candidates: lane n of row g of wave w scores the entries n,
    // n + 16, ... of reference m = 4 w + g exactly, its patch spread over the
    // row's lanes (four pixels each, broadcast by DPP), and keeps its four
    // smallest by (distance, place). The records then come in order by rounds
    // of a row minimum; all of it inside the wave, every lane active.
    {
        const int m = 4 * wave + g;
        const int c0 = cnt[m];
        const int c = (!anybad && kmv[m] > 0 && c0 <= LIST) ? c0 : 0, K = c > 0 ? kmv[m] : 0;
        const int cmax = wave_rows_max(c), kmax = wave_rows_max(K);
        const float inv_uw = 1.f / static_cast<float>(UW);
        uint32_t* dk = reg + m * LIST;
        const uint16_t* lm = list + m * LIST;
        const int cx = ref_x(jb.grid, min(i0 + (m >> 2), jb.grid.nx - 1), jb.width, 8);
        const int cy = ref_y(jb.grid, min(j0 + (m & 3), jb.grid.ny - 1), jb.height, 8);
        const uint32_t self = (static_cast<uint32_t>(cy - uy0) << 16) | static_cast<uint32_t>(cx - ux0);
        float patch[4];
        row_patch(cx, cy, patch);
        unsigned long long best[4] = {~0ull, ~0ull, ~0ull, ~0ull};
        auto place = [&](int q) {  // region row and column of entry q, as one ordered word
            const int u = lm[q];
            const int uy = div_small(u, inv_uw);
            return (static_cast<uint32_t>(uy) << 16) | static_cast<uint32_t>(u - uy * UW);
        };
        auto insert = [&](uint32_t d, uint32_t at) {
            const unsigned long long x = (static_cast<unsigned long long>(d) << 32) | at;
            best[3] = min(best[3], x);
#pragma unroll
            for (int k = 3; k > 0; --k) {
                const unsigned long long lo = min(best[k], best[k - 1]), hi = max(best[k], best[k - 1]);
                best[k - 1] = lo;
                best[k] = hi;
            }
        };
        for (int q0 = 0; q0 < cmax; q0 += 16) {
            const int q = q0 + n;
            const uint32_t at = q < c ? place(q) : self;
            const int uy = static_cast<int>(at >> 16), ux = static_cast<int>(at & 0xffffu);
            uint32_t d = exact(patch, ux, uy);
            if (at == self) d = kTaken;  // listed with the rest, never taken
            if (q < c) dk[q] = d;
            insert(d, at);
        }
        MatchRec* out = jb.out + (static_cast<size_t>(j0 + (m & 3)) * jb.grid.nx + i0 + (m >> 2)) * G + 1;
        int given = 0;
        for (int k = 0; k < kmax; ++k) {
            const uint32_t d = static_cast<uint32_t>(best[0] >> 32), at = static_cast<uint32_t>(best[0]);
            const uint32_t mn = row_min_u32(d);
            bool mine = d == mn && k < K;
            const unsigned long long who = __builtin_amdgcn_ballot_w64(mine);
            if (rows_with_two(who)) {  // equal distances: the first place
                const uint32_t first = row_min_u32(mine ? at : ~0u);
                mine = mine && at == first;
            }
            if (mine) {
                out[k] = MatchRec{ux0 + static_cast<int>(at & 0xffffu), uy0 + static_cast<int>(at >> 16), jb.t0, d};
                best[0] = best[1], best[1] = best[2], best[2] = best[3], best[3] = ~0ull;
                if (++given == 4) {  // the lane's next four
                    given = 0;
                    const unsigned long long won = (static_cast<unsigned long long>(d) << 32) | at;
                    for (int q = n; q < c; q += 16) {
                        const unsigned long long x = (static_cast<unsigned long long>(dk[q]) << 32) | place(q);
                        if (x > won && x < best[3]) insert(dk[q], static_cast<uint32_t>(x));
                    }
                }
            }
        }
    }
    if (tid < 16 && (tid >> 2) < ncol && (tid & 3) < nrow) {
        const MmWin w = mm_win(jb, i0 + (tid >> 2), j0 + (tid & 3));
        const int ref_id = (j0 + (tid & 3)) * jb.grid.nx + i0 + (tid >> 2);
        jb.out[static_cast<size_t>(ref_id) * G] = MatchRec{w.cx, w.cy, jb.t0, 0u};
        jb.counts[ref_id] = 1 + kmv[tid];
    }

    if (flat_region) return;
    // (no reference of the block needs the rest: the usual case)
    if (__builtin_amdgcn_ballot_w64(kmv[n] > 0 && (anybad || cnt[n] > LIST)) == 0) return;
    __syncthreads();  // the regions and lists become the fallback's keys
    // Whole windows, exactly, for the references the bound could not serve:
    // up to four at a time, the workgroup scores each window's candidates (one
    // per thread) into LDS, then a wave per reference takes the G - 1 smallest
    // by rounds of a wave minimum over each lane's four best. Windows that do
    // not fit come in pieces; the lanes carry the best so far. A window whose
    // first places hold G - 1 copies of the patch (distance 0) is done with
    // those: no later place can displace one (flat areas). Windows of up to 400
    // places (range 9): a wave looks through the first 64 of its own reference's,
    // then all four through each other reference's next 256; against 256 by all
    // at once, 1080p at step 3, range 7, group 8: half the frame constant 239 ->
    // 181 us, squares of 100 pixels 450 -> 310. Wider ones go to the 256 at
    // once: theirs are mostly denoised planes, whose lists overflow without
    // copies, and the first look cost them 2 % (step 8, range 19, group 32:
    // 376 -> 386 us of both stages' matching).
    const int space = reg_words + kUnion;
    const int wcap = min((2 * jb.range + 1) * (2 * jb.range + 1), (ux1 - ux0 + 1) * (uy1 - uy0 + 1));
    const int at_once = max(1, min(4, space / wcap));
    const int piece = min(wcap, space);
    int* copies = reinterpret_cast<int*>(wl);  // per reference at work
    uint32_t todo = static_cast<uint32_t>(
        __builtin_amdgcn_ballot_w64(kmv[n] > 0 && (anybad || cnt[n] > LIST)) & 0xffffull);
    while (todo) {
        uint32_t refs = 0u;  // a reference per nibble
        int nref = 0;
        for (; nref < at_once && todo; ++nref, todo &= todo - 1u)
            refs |= static_cast<uint32_t>(__builtin_ctz(todo)) << (4 * nref);
        if (tid < 4) copies[tid] = 0;
        __syncthreads();
        unsigned long long kept = ~0ull;  // lane k: the k-th best of the pieces so far
        uint32_t flat = 0u;               // the references done after their first places, a bit each
        // keys of places from .. to - 1 (p0 the piece's first) of the r-th
        // reference, by one wave or by all four; returns the copies found
        auto score = [&](int r, int p0, int from, int to, bool alone) {
            const int m = (refs >> (4 * r)) & 15;
            const MmWin w = mm_win(jb, i0 + (m >> 2), j0 + (m & 3));
            const int ww = w.right - w.left + 1, end = min(ww * (w.bottom - w.top + 1), to);
            const int self = (w.cy - w.top) * ww + (w.cx - w.left);
            const float inv_ww = 1.f / static_cast<float>(ww);
            float patch[4];
            row_patch(w.cx, w.cy, patch);
            int zeros = 0;
            const int by = alone ? 64 : 256;
            for (int q0 = from + (alone ? 0 : 64 * wave); q0 < end; q0 += by) {
                const int c = min(q0 + lane, end - 1);
                const int dy = div_small(c, inv_ww), dx = c - dy * ww;
                const uint32_t d = exact(patch, w.left - ux0 + dx, w.top - uy0 + dy);
                mm_lds[r * piece + c - p0] = c == self ? kTaken : d;
                zeros += __popcll(__builtin_amdgcn_ballot_w64(d == 0u && c != self && q0 + lane < end));
            }
            return zeros;
        };
        // record k of reference m: a key (distance, place in the window)
        auto store = [&](int m, int k, unsigned long long key) {
            const MmWin w = mm_win(jb, i0 + (m >> 2), j0 + (m & 3));
            const int ww = w.right - w.left + 1, c = static_cast<int>(static_cast<uint32_t>(key));
            const int dy = div_small(c, 1.f / static_cast<float>(ww)), dx = c - dy * ww;
            jb.out[(static_cast<size_t>(j0 + (m & 3)) * jb.grid.nx + i0 + (m >> 2)) * G + 1 + k] =
                MatchRec{w.left + dx, w.top + dy, jb.t0, static_cast<uint32_t>(key >> 32)};
        };
        for (int p0 = 0; p0 < wcap && flat != (1u << nref) - 1u; p0 += piece) {
            int from = p0;
            if (p0 == 0) {
                // (a reference done after 64 places has its copies among them:
                // its keys from there to `from` are not written and not read)
                for (int pass = wcap <= 400 ? 0 : 1; pass < 2 && flat != (1u << nref) - 1u; ++pass) {
                    const int next = min(piece, pass == 0 ? 64 : from + 256);
                    for (int r = 0; r < nref; ++r)
                        if (pass == 0 ? r == wave : !((flat >> r) & 1u)) {
                            const int zeros = score(r, 0, from, next, pass == 0);
                            if (lane == 0) atomicAdd(&copies[r], zeros);
                        }
                    from = next;
                    __syncthreads();
                    for (int r = 0; r < nref; ++r)
                        flat |= copies[r] >= kmv[(refs >> (4 * r)) & 15] ? 1u << r : 0u;
                    flat = __builtin_amdgcn_readfirstlane(flat);
                    __syncthreads();
                }
            }
            const uint32_t skip = __builtin_amdgcn_readfirstlane(flat);
            for (int r = 0; r < nref; ++r)
                if (!((skip >> r) & 1u)) score(r, p0, from, p0 + piece, false);
            __syncthreads();
            const bool copied = (skip >> wave) & 1u;
            const int m = wave < nref ? (refs >> (4 * wave)) & 15 : 0;
            const MmWin w = mm_win(jb, i0 + (m >> 2), j0 + (m & 3));
            const int last = min((w.right - w.left + 1) * (w.bottom - w.top + 1), copied ? from : p0 + piece) - p0;
            const uint32_t* keys = mm_lds + wave * piece;
            const int K = wave < nref ? kmv[m] : 0;
            if (copied) {  // the first K copies, in order
                int rank = 0;
                for (int c0 = 0; p0 == 0 && c0 < last && rank < K; c0 += 64) {
                    const bool zero = c0 + lane < last && keys[min(c0 + lane, last - 1)] == 0u;
                    const unsigned long long z = __builtin_amdgcn_ballot_w64(zero);
                    const int k = rank + __builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(z >> 32),
                                                                   __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(z), 0u));
                    if (zero && k < K) store(m, k, static_cast<unsigned long long>(c0 + lane));
                    rank += __popcll(z);
                }
            } else if (wave < nref) {
                const unsigned long long carried = lane < K ? kept : ~0ull;
                unsigned long long best[4];
                auto insert = [&](unsigned long long x) {
                    best[3] = x;
#pragma unroll
                    for (int k = 3; k > 0; --k)
                        if (best[k] < best[k - 1]) {
                            const unsigned long long t = best[k];
                            best[k] = best[k - 1];
                            best[k - 1] = t;
                        }
                };
                // the lane's four smallest keys from `from` on
                auto collect = [&](unsigned long long from) {
                    best[0] = best[1] = best[2] = best[3] = ~0ull;
                    if (carried >= from) insert(carried);
                    for (int c = lane; c < last; c += 64) {
                        const uint32_t d = keys[c];
                        const unsigned long long x = (static_cast<unsigned long long>(d) << 32) | static_cast<uint32_t>(p0 + c);
                        if (d != kTaken && x >= from && x < best[3]) insert(x);
                    }
                };
                collect(0ull);
                int given = 0;
                for (int k = 0; k < K; ++k) {
                    const uint32_t d = static_cast<uint32_t>(best[0] >> 32), at = static_cast<uint32_t>(best[0]);
                    const uint32_t mn = wave_min_u32_dpp(d);
                    bool mine = d == mn;
                    const unsigned long long who = __builtin_amdgcn_ballot_w64(mine);
                    uint32_t first = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(at), __builtin_ctzll(who)));
                    if ((who & (who - 1u)) != 0) {  // equal distances: the first place
                        first = wave_min_u32_dpp(mine ? at : ~0u);
                        mine = mine && at == first;
                    }
                    const unsigned long long win = (static_cast<unsigned long long>(mn) << 32) | first;
                    if (lane == k) kept = win;
                    if (mine && win != ~0ull) {
                        best[0] = best[1], best[1] = best[2], best[2] = best[3], best[3] = ~0ull;
                        if (++given == 4) {
                            given = 0;
                            collect(win + 1u);
                        }
                    }
                }
            }
            __syncthreads();
        }
        if (wave < nref && !((flat >> wave) & 1u)) {
            const int m = (refs >> (4 * wave)) & 15;
            if (lane < kmv[m]) store(m, lane, kept);
        }
    }
}

// ---------------------------------------------------------------------------
// Group filter (src/cpu/bm/dct8.cpp:926-1133 Bm3dFilterGroup).
// ---------------------------------------------------------------------------

// Factor of position j of the in-place orthonormal Haar of n samples
// (src/cpu/bm/dct8.cpp:580-591 HaarScale).
__device__ inline float haar_scale(int n, int j) {
    int e;
    if (j == 0) {
        e = 31 - __builtin_clz(static_cast<unsigned>(n));
    } else {
        e = __builtin_ctz(static_cast<unsigned>(j)) + 1;
    }
    float f = 1.f;
    for (int i = 0; i < e / 2; ++i) f *= 0.5f;
    return (e & 1) ? f * 0.70710678118654752f : f;
}

// In-place orthonormal Haar along one line at base[i * stride], i < n
// (src/cpu/bm/dct8.cpp:600-625 HaarLines).
__device__ inline void haar_forward(float* base, int n, int stride) {
    for (int h = 1; h < n; h <<= 1)
        for (int i = 0; i < n; i += 2 * h) {
            const float a = base[i * stride], b = base[(i + h) * stride];
            base[i * stride] = a + b;
            base[(i + h) * stride] = a - b;
        }
    for (int j = 0; j < n; ++j) base[j * stride] *= haar_scale(n, j);
}

__device__ inline void haar_inverse(float* base, int n, int stride) {
    for (int j = 0; j < n; ++j) base[j * stride] *= haar_scale(n, j);
    for (int h = n >> 1; h >= 1; h >>= 1)
        for (int i = 0; i < n; i += 2 * h) {
            const float a = base[i * stride], b = base[(i + h) * stride];
            base[i * stride] = a + b;
            base[(i + h) * stride] = a - b;
        }
}

// DCT of the lines of every patch of a cube (patch stride ps floats), by the
// 64 lanes of one wave. ROWS: lines along x (sample stride 1); else along y.
template <int B, bool ROWS>
__device__ inline void dct_lines(float* cube, int group, int ps, bool inverse, int lane) {
    if constexpr (B > 1) {
        const float* m = c_dct + dct_offset<B>();
        const int lines = group * B;
        for (int L = lane; L < lines; L += 64) {
            const int p = L / B, q = L - p * B;
            float* base = cube + p * ps + (ROWS ? q * B : q);
            constexpr int ss = ROWS ? 1 : B;
            float v[B], o[B];
#pragma unroll
            for (int i = 0; i < B; ++i) v[i] = base[i * ss];
            if (inverse) {
#pragma unroll
                for (int k = 0; k < B; ++k) {
                    float acc = 0.f;
#pragma unroll
                    for (int i = 0; i < B; ++i) acc = fmaf(m[i * B + k], v[i], acc);
                    o[k] = acc;
                }
            } else {
#pragma unroll
                for (int k = 0; k < B; ++k) {
                    float acc = 0.f;
#pragma unroll
                    for (int i = 0; i < B; ++i) acc = fmaf(m[k * B + i], v[i], acc);
                    o[k] = acc;
                }
            }
#pragma unroll
            for (int i = 0; i < B; ++i) base[i * ss] = o[i];
        }
    }
}

// Gathers the k matched patches of a group into an LDS cube (patch stride
// B*B + 1), zero beyond k up to the configured group size G. src_of(t) and
// wref_of(t) give the plane of temporal slot t (the record's t).
template <int B, bool WIENER, typename SrcOf, typename WrefOf>
__device__ inline void gather_group_wave(const MatchRec* rec, int k, int G, int stride, int wref_stride, SrcOf src_of,
                                         WrefOf wref_of, float* cube, float* rc, int lane) {
    constexpr int A = B * B;
    constexpr int PS = A + 1;
    for (int j = 0; j < G; ++j) {
        int mx = 0, my = 0, mt = 0;
        if (j < k) {
            mx = rec[j].x;
            my = rec[j].y;
            mt = rec[j].t;
        }
        const float* sp = j < k ? src_of(mt) : nullptr;
        const float* wp = (WIENER && j < k) ? wref_of(mt) : nullptr;
        for (int e = lane; e < A; e += 64) {
            const int py = e / B, px = e - (e / B) * B;
            float v = 0.f, w = 0.f;
            if (j < k) {
                v = sp[static_cast<size_t>(my + py) * stride + mx + px];
                if constexpr (WIENER) w = wp[static_cast<size_t>(my + py) * wref_stride + mx + px];
            }
            cube[j * PS + e] = v;
            if constexpr (WIENER) rc[j * PS + e] = w;
        }
    }
    wave_sync();
}

// One group by one wave: gather (spatial: every patch from the job's own
// planes), then the transform. Returns the aggregation weight.
template <int B, bool WIENER>
__device__ inline float transform_group_wave(int G, float sigma, float* cube, float* rc, int lane);

template <int B, bool WIENER>
__device__ inline float filter_group_wave(const FilterJob& jb, const MatchRec* rec, int k, float* cube, float* rc,
                                          int lane) {
    gather_group_wave<B, WIENER>(
        rec, k, jb.group, jb.stride, jb.wref_stride, [&](int) { return jb.src; }, [&](int) { return jb.wref; }, cube,
        rc, lane);
    return transform_group_wave<B, WIENER>(jb.group, jb.sigma, cube, rc, lane);
}

// Forward 3-D transform of the cube (and of the Wiener reference cube),
// shrink, inverse; the filtered patches stay in `cube`. Returns the
// aggregation weight, the same in every lane.
template <int B, bool WIENER>
__device__ inline float transform_group_wave(int G, float sigma, float* cube, float* rc, int lane) {
    constexpr int A = B * B;
    constexpr int PS = A + 1;
    dct_lines<B, true>(cube, G, PS, false, lane);
    if constexpr (WIENER) dct_lines<B, true>(rc, G, PS, false, lane);
    wave_sync();
    dct_lines<B, false>(cube, G, PS, false, lane);
    if constexpr (WIENER) dct_lines<B, false>(rc, G, PS, false, lane);
    wave_sync();

    int kept = 0;
    float w2 = 0.f;
    const float thr = 2.7f * sigma;  // include/nss/params.hpp:46 kBmHardLambda
    const float sig2 = sigma * sigma;
    for (int f = lane; f < A; f += 64) {
        haar_forward(cube + f, G, PS);
        if constexpr (WIENER) haar_forward(rc + f, G, PS);
        for (int j = 0; j < G; ++j) {
            float& c = cube[j * PS + f];
            const bool dc = (j == 0 && f == 0);
            if constexpr (WIENER) {
                float w = 1.f;
                if (!dc) {
                    const float rr = rc[j * PS + f];
                    const float r2 = rr * rr;
                    const float den = r2 + sig2;
                    w = den > 0.f ? r2 / den : 0.f;
                }
                c *= w;
                w2 = fmaf(w, w, w2);
            } else {
                if (!dc && fabsf(c) < thr)
                    c = 0.f;
                else
                    ++kept;
            }
        }
        haar_inverse(cube + f, G, PS);
    }
    wave_sync();
    dct_lines<B, false>(cube, G, PS, true, lane);
    wave_sync();
    dct_lines<B, true>(cube, G, PS, true, lane);
    wave_sync();
    if constexpr (WIENER) {
        return 1.f / fmaxf(wave_sum_f32(w2), 1e-12f);
    } else {
        return 1.f / static_cast<float>(max(wave_sum_i32(kept), 1));
    }
}

__device__ inline unsigned long long to_fixed(float v) {
    return static_cast<unsigned long long>(__float2ll_rn(v * 4294967296.0f));
}

// to_fixed of N values. Below 2^19 the conversion is one double addition: at
// 1.5 * 2^20 a double's unit is 2^-32, so the sum rounds to nearest even there
// as __float2ll_rn does, and the words less the constant's are the integer.
// Three operations instead of twelve (the cast's high and low words), which
// were a sixth of the group filters' VALU time: 1080p YUV420 at group 8 hard
// 45.3 -> 42.6 us, Wiener (with quotient()) 63.0 -> 57.3 us; group 32 Wiener
// at step 3 1609 -> 1489 us. Larger or non-finite
// values (one test of the magnitudes' sum) take the cast.
template <int N>
__device__ __forceinline__ void to_fixed_n(const float (&v)[N], unsigned long long (&o)[N]) {
    float mag = 0.f;
#pragma unroll
    for (int i = 0; i < N; ++i) mag += fabsf(v[i]);
    if (mag < 524288.f) {
#pragma unroll
        for (int i = 0; i < N; ++i)
            o[i] = static_cast<unsigned long long>(__double_as_longlong(static_cast<double>(v[i]) + 1572864.0)) -
                   0x4138000000000000ull;
    } else {
#pragma unroll
        for (int i = 0; i < N; ++i) o[i] = to_fixed(v[i]);
    }
}

// n / d for d in [2^-60, 2^62] and 0 <= n <= d: Newton's step on the reciprocal
// and two residual corrections (the operations of the full division without
// its scaling and special cases). Correctly rounded for n = 0 and n >= 2^-101;
// below that (quotients below 2^-41) the residuals underflow and the last
// place may be off.
__device__ __forceinline__ float quotient(float n, float d) {
    float y = __builtin_amdgcn_rcpf(d);
    y = fmaf(fmaf(-d, y, 1.f), y, y);
    float q = n * y;
    q = fmaf(fmaf(-d, q, n), y, q);
    return fmaf(fmaf(-d, q, n), y, q);
}

// Wiener gains r^2 / (r^2 + sig2) applied to a lane's G coefficients (lane 0's
// first, the group's mean, keeps 1); the sum of their squares is returned.
// quotient() serves coefficients below 2^30 and sig2 in (2^-60, 2^61), so that
// the denominators stay in its range; any finite sigma is accepted, and its
// square may be infinite (gain 0).
template <int G>
__device__ __forceinline__ float wiener_shrink(float (&c)[G], const float (&r)[G], float sig2, int lane) {
    float mag = 0.f, w2 = 0.f;
#pragma unroll
    for (int j = 0; j < G; ++j) mag += fabsf(r[j]);
    auto shrink = [&](auto gain) {
#pragma unroll
        for (int j = 0; j < G; ++j) {
            float w = 1.f;
            if (!(lane == 0 && j == 0)) {
                const float r2 = r[j] * r[j];
                w = gain(r2, r2 + sig2);
            }
            c[j] *= w;
            w2 = fmaf(w, w, w2);
        }
    };
    if (mag < 1073741824.f && sig2 > 0x1p-60f && sig2 < 0x1p61f)
        shrink([](float n, float d) { return quotient(n, d); });
    else
        shrink([](float n, float d) { return d > 0.f ? n / d : 0.f; });
    return w2;
}

__device__ inline void lds_add(unsigned long long* p, unsigned long long v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Tile epilogue: the tile's exact int64 numerator sums as its partials (2^32
// units), so that the finish adds every pixel's sums exactly and the output
// does not depend on how the grid was cut into tiles. The weights are not
// written per pixel: each group's weight goes out once (FilterJob::gweight)
// and the finish box-sums them from the records. pn points at column ax0 & 3
// of the tile's first row (rows of `pitch` entries). Called by every thread
// of the block after the accumulation's barrier.
__device__ inline void partials_out(int aw, int ah, int pitch, const unsigned long long* num, unsigned long long* pn) {
    const int nt = static_cast<int>(blockDim.x);
    for (int e = threadIdx.x; e < aw * ah; e += nt) {
        const int y = e / aw, x = e - y * aw;
        pn[y * pitch + x] = num[e];
    }
}

// Temporal tile epilogue: den = B x B box sum of the corner weights
// (horizontal pass into scratch, then vertical), and num, as the tile's float
// partials (rows of
// `pitch` floats; pn / pd point at column ax0 & 3 of the tile's first row, so
// that x = 0 mod 4 is 16-byte aligned in every tile). Called by every thread
// of the block after the accumulation's barrier; scratch holds
// (ah - B + 1) * aw floats.
template <int B>
__device__ inline void partials_out_float(int aw, int ah, int pitch, const unsigned long long* num,
                                    const unsigned long long* corner, float* scratch, float* pn, float* pd) {
    const int cw = aw - B + 1, ch = ah - B + 1;
    const int nt = static_cast<int>(blockDim.x);
    if (!pd) {  // numerator only (the weights went to the frame's corner plane)
        const float inv = 1.f / static_cast<float>(aw);
        for (int e = threadIdx.x; e < aw * ah; e += nt) {
            const int y = div_small(e, inv), x = e - y * aw;
            pn[y * pitch + x] =
                static_cast<float>(static_cast<double>(static_cast<long long>(num[e])) * (1.0 / 4294967296.0));
        }
        return;
    }
    // Horizontal: a thread slides the B-wide window over 8 outputs of a row
    // (exact int64 sums, so the order of the adds does not matter).
    const int segs = (aw + 7) >> 3;
    for (int e = threadIdx.x; e < ch * segs; e += nt) {
        const int y = e / segs, x0 = (e - y * segs) * 8;
        const unsigned long long* row = corner + y * cw;
        unsigned long long w[B + 7];  // corners x0 - B + 1 .. x0 + 7
#pragma unroll
        for (int i = 0; i < B + 7; ++i) {
            const int cx = x0 - B + 1 + i;
            w[i] = (cx >= 0 && cx < cw) ? row[cx] : 0ull;
        }
        unsigned long long sum = 0;
#pragma unroll
        for (int i = 0; i < B - 1; ++i) sum += w[i];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            sum += w[B - 1 + j];
            if (x0 + j < aw)
                scratch[y * aw + x0 + j] =
                    static_cast<float>(static_cast<double>(static_cast<long long>(sum)) * (1.0 / 4294967296.0));
            sum -= w[j];
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < aw * ah; e += nt) {
        const int y = e / aw, x = e - (e / aw) * aw;
        float d = 0.f;
#pragma unroll
        for (int i = 0; i < B; ++i) {
            const int cy = y - i;
            if (cy >= 0 && cy < ch) d += scratch[cy * aw + x];
        }
        pn[y * pitch + x] = static_cast<float>(static_cast<double>(static_cast<long long>(num[e])) * (1.0 / 4294967296.0));
        pd[y * pitch + x] = d;
    }
}

__device__ inline void tile_partials(const FilterJob& jb, int tile, int ax0, const unsigned long long* num) {
    const size_t base = static_cast<size_t>(tile) * jb.tiles.pitch * jb.tiles.ah + (ax0 & 3);
    partials_out(jb.tiles.aw, jb.tiles.ah, jb.tiles.pitch, num, jb.part_num + base);
}

// Tile path: numerator sums of a tile of groups in LDS, then exact partials;
// each group's weight to gweight. LDS: num [ah][aw] int64 | per-wave cubes.
template <int B, bool WIENER>
__global__ __launch_bounds__(256) void filter_tile_kernel(FilterTable tab) {
    extern __shared__ __align__(16) unsigned long long acc[];
    constexpr int A = B * B;
    constexpr int PS = A + 1;
    const int lb = xcd_block();
    const FilterJob& jb = tab.job[find_job(tab, lb)];
    const TileGeom& tg = jb.tiles;
    const int tile = lb - jb.wg_begin;  // partials index
    const int tx = (tile + jb.tile0) % tg.ntx, ty = (tile + jb.tile0) / tg.ntx;
    const int aw = tg.aw, ah = tg.ah;
    const int ax0 = tg.ax0(tx, jb.width, B, jb.grid.step, jb.range);
    const int ay0 = tg.ay0(ty, jb.height, B, jb.grid.step, jb.range);
    unsigned long long* num = acc;
    float* scratch = reinterpret_cast<float*>(acc + aw * ah);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    for (int e = threadIdx.x; e < aw * ah; e += 256) acc[e] = 0ull;
    __syncthreads();

    const int G = jb.group;
    const int cube_floats = G * PS * (WIENER ? 2 : 1);
    float* cube = scratch + wave * cube_floats;
    float* rc = cube + G * PS;
    const int i_begin = tx * tg.tw, j_begin = ty * tg.th;
    const int ni = min(tg.tw, jb.grid.nx - i_begin), nj = min(tg.th, jb.grid.ny - j_begin);
    for (int g = wave; g < ni * nj; g += 4) {
        const int gj = g / ni, gi = g - gj * ni;
        const int rid = (j_begin + gj - jb.grid.row0) * jb.grid.nx + i_begin + gi;
        const int k = jb.counts[rid];
        const MatchRec* rec = jb.matches + static_cast<size_t>(rid) * G;
        const float w = filter_group_wave<B, WIENER>(jb, rec, k, cube, rc, lane);
        const unsigned long long wfix = to_fixed(w);
        for (int j = 0; j < k; ++j) {
            const int lx = rec[j].x - ax0, ly = rec[j].y - ay0;
            for (int e = lane; e < A; e += 64) {
                const int py = e / B, px = e - (e / B) * B;
                lds_add(num + (ly + py) * aw + lx + px, to_fixed(w * cube[j * PS + e]));
            }
        }
        if (lane == 0) jb.gweight[rid] = wfix;
        wave_sync();
    }
    __syncthreads();
    tile_partials(jb, tile, ax0, num);
}

// ---------------------------------------------------------------------------
// Block-8 group filter in registers (G in {8, 16, 32}). One wave per group;
// three layouts of the G x 8 x 8 cube over the 64 lanes, with LDS transposes
// between them (per-wave buffer T, address g*72 + row*9 + col):
//   rows    lane (gb, y): rows y of patches g = gb + 8m, 8 samples over x
//   columns lane (gb, kx): columns kx of the same patches, 8 samples over y
//   group   lane (ky, kx): coefficient (ky, kx) of all G patches
// Row DCT, column DCT and the group-axis Haar + shrink are then lane-local.
// ---------------------------------------------------------------------------
inline constexpr int kTs = 72;  // patch stride in the transpose buffer
inline constexpr int kTr = 9;   // row stride

// 8-point orthonormal DCT-II (forward) or its transpose, DCT-III (inverse),
// by the even/odd split of the definition X_k = a_k sum_n x_n cos(pi (2n+1) k / 16):
// X_{2m} is the 4-point transform of x_n + x_{7-n} (split once more into
// sums and differences), X_{2m+1} the 4 x 4 cosine matrix times
// x_n - x_{7-n}; the inverse runs the same steps transposed. 36 operations
// instead of 64 multiply-adds; the constants are cos(j pi / 16) / 2 and
// 1 / sqrt(8) rounded from double.
template <bool INVERSE>
__device__ inline void dct8(float v[8]) {
    constexpr float k0 = 0.353553391f;  // 1/sqrt(8) = cos(4 pi/16) / 2
    constexpr float c1 = 0.490392640f, c2 = 0.461939766f, c3 = 0.415734806f;
    constexpr float c5 = 0.277785117f, c6 = 0.191341716f, c7 = 0.0975451610f;
    if (!INVERSE) {
        const float a0 = v[0] + v[7], a1 = v[1] + v[6], a2 = v[2] + v[5], a3 = v[3] + v[4];
        const float b0 = v[0] - v[7], b1 = v[1] - v[6], b2 = v[2] - v[5], b3 = v[3] - v[4];
        const float e0 = a0 + a3, e1 = a1 + a2, d0 = a0 - a3, d1 = a1 - a2;
        v[0] = k0 * (e0 + e1);
        v[4] = k0 * (e0 - e1);
        v[2] = fmaf(c2, d0, c6 * d1);
        v[6] = fmaf(c6, d0, -c2 * d1);
        v[1] = fmaf(c1, b0, fmaf(c3, b1, fmaf(c5, b2, c7 * b3)));
        v[3] = fmaf(c3, b0, fmaf(-c7, b1, fmaf(-c1, b2, -c5 * b3)));
        v[5] = fmaf(c5, b0, fmaf(-c1, b1, fmaf(c7, b2, c3 * b3)));
        v[7] = fmaf(c7, b0, fmaf(-c5, b1, fmaf(c3, b2, -c1 * b3)));
    } else {
        const float s = k0 * (v[0] + v[4]), t = k0 * (v[0] - v[4]);
        const float p = fmaf(c2, v[2], c6 * v[6]), q = fmaf(c6, v[2], -c2 * v[6]);
        const float e0 = s + p, e3 = s - p, e1 = t + q, e2 = t - q;
        const float o0 = fmaf(c1, v[1], fmaf(c3, v[3], fmaf(c5, v[5], c7 * v[7])));
        const float o1 = fmaf(c3, v[1], fmaf(-c7, v[3], fmaf(-c1, v[5], -c5 * v[7])));
        const float o2 = fmaf(c5, v[1], fmaf(-c1, v[3], fmaf(c7, v[5], c3 * v[7])));
        const float o3 = fmaf(c7, v[1], fmaf(-c5, v[3], fmaf(c3, v[5], -c1 * v[7])));
        v[0] = e0 + o0;
        v[7] = e0 - o0;
        v[1] = e1 + o1;
        v[6] = e1 - o1;
        v[2] = e2 + o2;
        v[5] = e2 - o2;
        v[3] = e3 + o3;
        v[4] = e3 - o3;
    }
}

// rows (or columns) layout -> the transposed layout within each patch.
template <int M>
__device__ inline void transpose_rc(float (&v)[M][8], float* T, int lane) {
    const int gb = lane >> 3, q = lane & 7;
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int i = 0; i < 8; ++i) T[(gb + 8 * m) * kTs + q * kTr + i] = v[m][i];
    wave_sync();
#pragma unroll
    for (int m = 0; m < M; ++m)
#pragma unroll
        for (int i = 0; i < 8; ++i) v[m][i] = T[(gb + 8 * m) * kTs + i * kTr + q];
    wave_sync();
}

// columns layout (lane (gb, kx) holds ky = 0..7) -> group layout.
template <int G>
__device__ inline void columns_to_group(float (&v)[G / 8][8], float (&c)[G], float* T, int lane) {
    const int gb = lane >> 3, kx = lane & 7;
#pragma unroll
    for (int m = 0; m < G / 8; ++m)
#pragma unroll
        for (int ky = 0; ky < 8; ++ky) T[(gb + 8 * m) * kTs + ky * kTr + kx] = v[m][ky];
    wave_sync();
    const int ky = lane >> 3;
#pragma unroll
    for (int g = 0; g < G; ++g) c[g] = T[g * kTs + ky * kTr + kx];
    wave_sync();
}

template <int G>
__device__ inline void group_to_columns(float (&c)[G], float (&v)[G / 8][8], float* T, int lane) {
    const int ky = lane >> 3, kx = lane & 7;
#pragma unroll
    for (int g = 0; g < G; ++g) T[g * kTs + ky * kTr + kx] = c[g];
    wave_sync();
    const int gb = lane >> 3;
#pragma unroll
    for (int m = 0; m < G / 8; ++m)
#pragma unroll
        for (int k = 0; k < 8; ++k) v[m][k] = T[(gb + 8 * m) * kTs + k * kTr + kx];
    wave_sync();
}

template <int G>
__device__ inline void haar_forward_reg(float (&c)[G]) {
#pragma unroll
    for (int h = 1; h < G; h <<= 1)
#pragma unroll
        for (int i = 0; i < G; i += 2 * h) {
            const float a = c[i], b = c[i + h];
            c[i] = a + b;
            c[i + h] = a - b;
        }
#pragma unroll
    for (int j = 0; j < G; ++j) c[j] *= haar_scale(G, j);
}

template <int G>
__device__ inline void haar_inverse_reg(float (&c)[G]) {
#pragma unroll
    for (int j = 0; j < G; ++j) c[j] *= haar_scale(G, j);
#pragma unroll
    for (int h = G >> 1; h >= 1; h >>= 1)
#pragma unroll
        for (int i = 0; i < G; i += 2 * h) {
            const float a = c[i], b = c[i + h];
            c[i] = a + b;
            c[i + h] = a - b;
        }
}

// Forward: rows (spatial) -> group-layout 3-D coefficients.
template <int G>
__device__ inline void forward_b8(float (&v)[G / 8][8], float (&c)[G], float* T, int lane) {
#pragma unroll
    for (int m = 0; m < G / 8; ++m) dct8<false>(v[m]);
    transpose_rc<G / 8>(v, T, lane);
#pragma unroll
    for (int m = 0; m < G / 8; ++m) dct8<false>(v[m]);
    columns_to_group<G>(v, c, T, lane);
    haar_forward_reg<G>(c);
}

// Gathers the rows this lane owns (zero beyond k).
template <int G>
__device__ inline void gather_rows_b8(const float* plane, int stride, const MatchRec* rec, int k, int lane,
                                      float (&v)[G / 8][8]) {
    const int gb = lane >> 3, y = lane & 7;
#pragma unroll
    for (int m = 0; m < G / 8; ++m) {
        const int g = gb + 8 * m;
        if (g < k) {
            const float* p = plane + static_cast<size_t>(rec[g].y + y) * stride + rec[g].x;
#pragma unroll
            for (int x = 0; x < 8; ++x) v[m][x] = p[x];
        } else {
#pragma unroll
            for (int x = 0; x < 8; ++x) v[m][x] = 0.f;
        }
    }
}

// Tile kernel for block 8: LDS = num [ah][aw] int64 | match records of the
// tile | per-wave transpose buffers.
template <int G, bool WIENER, int MAXW>
__global__ __launch_bounds__(64 * MAXW) void filter_tile_b8_kernel(FilterTable tab) {
    extern __shared__ __align__(16) unsigned long long acc[];
    constexpr int B = 8;
    constexpr int M = G / 8;
    const int lb = xcd_block();
    const FilterJob& jb = tab.job[find_job(tab, lb)];
    const TileGeom& tg = jb.tiles;
    const int tile = lb - jb.wg_begin;  // partials index
    const int tx = (tile + jb.tile0) % tg.ntx, ty = (tile + jb.tile0) / tg.ntx;
    const int aw = tg.aw, ah = tg.ah;
    const int ax0 = tg.ax0(tx, jb.width, B, jb.grid.step, jb.range);
    const int ay0 = tg.ay0(ty, jb.height, B, jb.grid.step, jb.range);
    const int i_begin = tx * tg.tw, j_begin = ty * tg.th;
    const int ni = min(tg.tw, jb.grid.nx - i_begin), nj = min(tg.th, jb.grid.ny - j_begin);
    const int ngroups = ni * nj;
    unsigned long long* num = acc;
    MatchRec* recs = reinterpret_cast<MatchRec*>(acc + aw * ah);
    int* cnt = reinterpret_cast<int*>(recs + tg.tw * tg.th * G);
    float* scratch = reinterpret_cast<float*>(cnt + ((tg.tw * tg.th + 3) & ~3));
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int nt = static_cast<int>(blockDim.x), waves = nt >> 6;
    float* T = scratch + wave * (G * kTs);
    for (int e = threadIdx.x; e < aw * ah; e += nt) acc[e] = 0ull;
    // The tile's match records and counts, row by row of the grid.
    for (int e = threadIdx.x; e < ngroups * G; e += nt) {
        const int g = e / G, j = e - g * G;
        const int gj = g / ni, gi = g - gj * ni;
        const int rid = (j_begin + gj - jb.grid.row0) * jb.grid.nx + i_begin + gi;
        recs[e] = jb.matches[static_cast<size_t>(rid) * G + j];
    }
    for (int g = threadIdx.x; g < ngroups; g += nt) {
        const int gj = g / ni, gi = g - gj * ni;
        cnt[g] = jb.counts[(j_begin + gj - jb.grid.row0) * jb.grid.nx + i_begin + gi];
    }
    __syncthreads();

    const float thr = 2.7f * jb.sigma;  // include/nss/params.hpp:46 kBmHardLambda
    const float sig2 = jb.sigma * jb.sigma;
    float v[M][8], vr[M][8];
    int g = wave;
    if (g < ngroups) {
        gather_rows_b8<G>(jb.src, jb.stride, recs + g * G, cnt[g], lane, v);
        if constexpr (WIENER) gather_rows_b8<G>(jb.wref, jb.wref_stride, recs + g * G, cnt[g], lane, vr);
    }
    for (; g < ngroups; g += waves) {
        const int k = cnt[g];
        const MatchRec* rec = recs + g * G;
        float c[G];
        float r[G];
        forward_b8<G>(v, c, T, lane);
        if constexpr (WIENER) forward_b8<G>(vr, r, T, lane);
        // Prefetch the next group's patches while this one is filtered.
        const int gn = g + waves;
        if (gn < ngroups) {
            gather_rows_b8<G>(jb.src, jb.stride, recs + gn * G, cnt[gn], lane, v);
            if constexpr (WIENER) gather_rows_b8<G>(jb.wref, jb.wref_stride, recs + gn * G, cnt[gn], lane, vr);
        }
        int kept = 0;
        float w2 = 0.f;
        if constexpr (WIENER) w2 = wiener_shrink<G>(c, r, sig2, lane);
#pragma unroll
        for (int j = 0; j < G; ++j) {
            if constexpr (!WIENER) {
                if (!(lane == 0 && j == 0) && fabsf(c[j]) < thr)
                    c[j] = 0.f;
                else
                    ++kept;
            }
        }
        haar_inverse_reg<G>(c);
        float u[M][8];
        group_to_columns<G>(c, u, T, lane);
#pragma unroll
        for (int m = 0; m < M; ++m) dct8<true>(u[m]);
        transpose_rc<M>(u, T, lane);
#pragma unroll
        for (int m = 0; m < M; ++m) dct8<true>(u[m]);
        float w;
        if constexpr (WIENER) {
            w = 1.f / fmaxf(wave_sum_f32(w2), 1e-12f);
        } else {
            w = 1.f / static_cast<float>(max(wave_sum_i32(kept), 1));
        }
        const int gb = lane >> 3, y = lane & 7;
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const int p = gb + 8 * m;
            if (p < k) {
                const int lx = rec[p].x - ax0, ly = rec[p].y - ay0;
                unsigned long long* row = num + (ly + y) * aw + lx;
                float wu[8];
#pragma unroll
                for (int x = 0; x < 8; ++x) wu[x] = w * u[m][x];
                unsigned long long fx[8];
                to_fixed_n<8>(wu, fx);
#pragma unroll
                for (int x = 0; x < 8; ++x) lds_add(row + x, fx[x]);
            }
        }
        if (lane == 0) {
            const int gj = g / ni, gi = g - gj * ni;
            jb.gweight[(j_begin + gj - jb.grid.row0) * jb.grid.nx + i_begin + gi] = to_fixed(w);
        }
    }
    __syncthreads();
    tile_partials(jb, tile, ax0, num);
}

// ---------------------------------------------------------------------------
// Block-8 group filter on MFMA (groups of 8 or 16), in bf16x3 or fp16 with
// FP32 accumulation. One wave filters a unit of 16 patches (two groups of 8
// or one of 16):
//   2-D DCT   four patches at a time as a 16 x 16 tile Q = [[P0, P1], [P2, P3]]
//             (pixel rows 8 pr + y, columns 8 pc + x): Z = bd(D) (Q bd(D^T))
//             with bd(M) = diag(M, M), two 16x16x16 products per tile; the
//             first product reads Q from memory in the A layout, its C-layout
//             output is the B operand of the second.
//   Haar      coefficient-major through LDS, then per 16 coefficients one
//             16x16x16 product with the exact +-1 butterfly matrix (block
//             diagonal for two groups of 8), scaled in FP32 to the
//             orthonormal transform.
//   shrink    hard threshold or Wiener in FP32 on the product's output.
//   inverse   the same steps reversed: Haar^T product, LDS back to the tile
//             layout, bd(D^T) (Z bd(D)).
// bf16x3 splits each operand v = hi + lo (both bf16, round to nearest even)
// and sums lo*hi + hi*lo + hi*hi; fp16 scales each group's pixels by a power
// of two to max |x| in [0.5, 1) (exact, undone in FP32) before rounding.
// Matching, weights and the fixed-point aggregation are those of the FP32
// kernels. MFMA 16x16x16 operand layouts (lane l, j = 0..3):
//   A[i][k]: i = l % 16, k = 4 (l / 16) + j;  B[k][n] and C[k][n]: n = l % 16,
//   k = 4 (l / 16) + j. So A(M) holds the entries of B(M^T).
// ---------------------------------------------------------------------------
typedef _Float16 h16x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

inline constexpr int kFormBf16x3 = 1;
inline constexpr int kFormF16 = 2;

template <int FORM>
struct Operand;
template <>
struct Operand<kFormBf16x3> {
    s16x4 hi, lo;
};
template <>
struct Operand<kFormF16> {
    h16x4 v;
};

typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 b16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 h16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Two values rounded to nearest even into one dword (v_cvt_pk_bf16_f32 /
// v_cvt_pk_f16_f32).
__device__ inline uint32_t pack_bf16(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, b16x2));
}
__device__ inline uint32_t pack_f16(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, h16x2));
}

// bf16x3 keeps the rounding residual as the lo part; the hi values are read
// back from the packed bits (low half << 16, high half masked).
template <int FORM>
__device__ inline Operand<FORM> operand(f32x4 v) {
    Operand<FORM> o;
    if constexpr (FORM == kFormBf16x3) {
        const uint32_t h0 = pack_bf16(v[0], v[1]), h1 = pack_bf16(v[2], v[3]);
        const uint32_t l0 = pack_bf16(v[0] - __uint_as_float(h0 << 16), v[1] - __uint_as_float(h0 & 0xffff0000u));
        const uint32_t l1 = pack_bf16(v[2] - __uint_as_float(h1 << 16), v[3] - __uint_as_float(h1 & 0xffff0000u));
        o.hi = __builtin_bit_cast(s16x4, u32x2{h0, h1});
        o.lo = __builtin_bit_cast(s16x4, u32x2{l0, l1});
    } else {
        o.v = __builtin_bit_cast(h16x4, u32x2{pack_f16(v[0], v[1]), pack_f16(v[2], v[3])});
    }
    return o;
}

// acc + a b (bf16x3 drops lo * lo only).
template <int FORM>
__device__ inline f32x4 mma(const Operand<FORM>& a, const Operand<FORM>& b, f32x4 acc) {
    if constexpr (FORM == kFormBf16x3) {
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a.lo, b.hi, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a.hi, b.lo, acc, 0, 0, 0);
        return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a.hi, b.hi, acc, 0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_16x16x16f16(a.v, b.v, acc, 0, 0, 0);
    }
}

// a b for an A operand that is exact in the operand type (a.lo = 0).
template <int FORM>
__device__ inline f32x4 mma_exact_a(const Operand<FORM>& a, const Operand<FORM>& b) {
    const f32x4 z = {0.f, 0.f, 0.f, 0.f};
    if constexpr (FORM == kFormBf16x3) {
        const f32x4 t = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a.hi, b.lo, z, 0, 0, 0);
        return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a.hi, b.hi, t, 0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_16x16x16f16(a.v, b.v, z, 0, 0, 0);
    }
}

// Lane's A-operand entries of bd(D) (transposed = false) or bd(D^T).
__device__ inline f32x4 dct_bd_entries(bool transposed, int lane) {
    const float* d = c_dct + dct_offset<8>();
    const int i = lane & 15;
    f32x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int k = 4 * (lane >> 4) + j;
        v[j] = (i >> 3) != (k >> 3) ? 0.f : transposed ? d[(k & 7) * 8 + (i & 7)] : d[(i & 7) * 8 + (k & 7)];
    }
    return v;
}

// Entry (j, g) of the unnormalised in-place Haar butterfly matrix: row 0 sums
// all samples; row j > 0 with lowest set bit h is the sum over [j - h, j)
// minus the sum over [j, j + h) (the level-h difference haar_forward writes
// to position j).
__device__ inline float haar_entry(int j, int g) {
    if (j == 0) return 1.f;
    const int h = j & -j;
    return (g >= j - h && g < j) ? 1.f : (g >= j && g < j + h) ? -1.f : 0.f;
}

// Lane's A-operand entries of the unit's Haar matrix (block diagonal for two
// groups of 8) or of its transpose.
template <int G>
__device__ inline f32x4 haar_unit_entries(bool transposed, int lane) {
    const int i = lane & 15;
    f32x4 v;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int k = 4 * (lane >> 4) + j;
        const int r = transposed ? k : i, c = transposed ? i : k;
        v[j] = (G == 8 && (r >> 3) != (c >> 3)) ? 0.f : haar_entry(r & (G - 1), c & (G - 1));
    }
    return v;
}

// Coefficient-major transpose buffer of one wave: 64 coefficients x 16
// patches (dwords) at a pitch of 20, patch quads permuted per coefficient
// (XOR by 4 ((coef >> 4) & 3)), so that the b32 scatters / gathers and the
// b128 accesses below are at most 2-way bank conflicts.
inline constexpr int kMfmaBuf = 64 * 20;

__device__ inline int mfma_slot(int coef, int patch) { return coef * 20 + (patch ^ (4 * ((coef >> 4) & 3))); }

// Forward 3-D transform of a unit. x[q] = lane's pixels of tile q in the A
// layout, already scaled. Out: raw Haar products out[t][j] = coefficient
// 16 t + (lane & 15) of Haar row 4 (lane >> 4) + j (not yet normalised).
// fp16: dlo holds the DCT matrix's fp16 rounding residual, so the matrix
// enters as hi + lo and only the data operand is rounded.
template <int FORM>
__device__ inline void forward_unit(const f32x4 (&x)[4], const Operand<FORM>& dct, const Operand<FORM>& dlo,
                                    const Operand<FORM>& haar, float* T, int lane, f32x4 (&out)[4]) {
    const f32x4 z0 = {0.f, 0.f, 0.f, 0.f};
    const int h = (lane >> 4) & 1, kx = lane & 7, pc = (lane >> 3) & 1, pr = lane >> 5;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const Operand<FORM> xq = operand<FORM>(x[q]);
        f32x4 y = mma<FORM>(xq, dct, z0);  // Q bd(D^T)
        if constexpr (FORM == kFormF16) y = mma<FORM>(xq, dlo, y);
        const Operand<FORM> yq = operand<FORM>(y);
        f32x4 z = mma<FORM>(dct, yq, z0);  // bd(D) Q bd(D^T)
        if constexpr (FORM == kFormF16) z = mma<FORM>(dlo, yq, z);
#pragma unroll
        for (int j = 0; j < 4; ++j) T[mfma_slot(8 * (4 * h + j) + kx, 4 * q + 2 * pr + pc)] = z[j];
    }
    wave_sync();
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const f32x4 c = *reinterpret_cast<const f32x4*>(T + mfma_slot(16 * t + (lane & 15), 4 * (lane >> 4)));
        out[t] = mma_exact_a<FORM>(haar, operand<FORM>(c));
    }
    wave_sync();
}

// Inverse of a unit: c[t] = Haar-domain coefficients (layout of forward_unit's
// output, in the operand scale and before the butterfly factors are undone).
// Out: xo[q][j] = pixel (y = 4 ((lane >> 4) & 1) + j, x = lane & 7) of patch
// 4 q + 2 (lane >> 5) + ((lane >> 3) & 1).
template <int FORM>
__device__ inline void inverse_unit(const f32x4 (&c)[4], const Operand<FORM>& dctt, const Operand<FORM>& dtlo,
                                    const Operand<FORM>& haart, float* T, int lane, f32x4 (&xo)[4]) {
    const f32x4 z0 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 4; ++t) {
        const f32x4 u = mma_exact_a<FORM>(haart, operand<FORM>(c[t]));
        *reinterpret_cast<f32x4*>(T + mfma_slot(16 * t + (lane & 15), 4 * (lane >> 4))) = u;
    }
    wave_sync();
    const int ky = lane & 7, pr = (lane >> 3) & 1, pc = lane >> 5, kx0 = 4 * ((lane >> 4) & 1);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        f32x4 z;
#pragma unroll
        for (int j = 0; j < 4; ++j) z[j] = T[mfma_slot(8 * ky + kx0 + j, 4 * q + 2 * pr + pc)];
        const Operand<FORM> zq = operand<FORM>(z);
        f32x4 v = mma<FORM>(zq, dctt, z0);  // Z bd(D)
        if constexpr (FORM == kFormF16) v = mma<FORM>(zq, dtlo, v);
        const Operand<FORM> vq = operand<FORM>(v);
        xo[q] = mma<FORM>(dctt, vq, z0);  // bd(D^T) Z bd(D)
        if constexpr (FORM == kFormF16) xo[q] = mma<FORM>(dtlo, vq, xo[q]);
    }
    wave_sync();
}

// Lane's pixels of a unit in the A layout (zero for patches beyond a group's
// count or groups beyond the tile): tile q, patch 4 q + 2 ((lane >> 3) & 1) +
// (lane >> 5), row lane & 7, columns 4 ((lane >> 4) & 1) + j. Patch positions
// as x | y << 16.
template <int G>
__device__ inline void load_unit(const float* plane, int stride, const uint32_t* pos, const int* cnt, int ngroups,
                                 int unit, int lane, f32x4 (&x)[4]) {
    const int pr = (lane >> 3) & 1, pc = lane >> 5, y = lane & 7, x0 = 4 * ((lane >> 4) & 1);
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int p = 4 * q + 2 * pr + pc;
        const int g = G == 8 ? 2 * unit + (p >> 3) : unit, idx = p & (G - 1);
        if (g < ngroups && idx < cnt[g]) {
            const uint32_t xy = pos[g * G + idx];
            const float* src = plane + static_cast<size_t>((xy >> 16) + y) * stride + (xy & 0xffffu) + x0;
#pragma unroll
            for (int j = 0; j < 4; ++j) x[q][j] = src[j];
        } else {
            x[q] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
}

// Power-of-two scale taking max |x| of a group to [0.5, 1); 1 for a zero or
// non-finite maximum.
__device__ inline float group_scale(float m) {
    if (!(m > 0.f) || !(m <= 3.4e38f)) return 1.f;
    return ldexpf(1.f, -__builtin_amdgcn_frexp_expf(m));
}

// The fp16 rounding residual of four values (the lo half of a split operand).
__device__ inline f32x4 f16_residual(f32x4 v) {
    const h16x4 h = __builtin_convertvector(v, h16x4);
    return v - __builtin_convertvector(h, f32x4);
}

// sum over g < k of the unnormalised Haar butterfly entry (j, g): the Haar
// coefficient of a constant over the k real patches of a group, before the
// orthonormal factor (row 0 sums k; a difference row j with lowest set bit h
// the part of [j - h, j) below k minus the part of [j, j + h) below k).
__device__ inline int haar_row_count(int j, int k) {
    if (j == 0) return k;
    const int h = j & -j;
    const int plus = min(max(min(j, k) - (j - h), 0), h);
    const int minus = min(max(min(j + h, k) - j, 0), h);
    return plus - minus;
}

// MFMA forms: each group's pixels are centred on their mean mu over the
// group's real patches (padding patches stay zero) and scaled by a power of
// two taking max |x - mu| to [0.5, 1) (fp16's range; exact, undone in FP32),
// so the low-precision operands carry the texture and the noise, not the
// group's level; the level's contribution (2-D DC coefficients only) is added
// back in FP32. m = max |x - mu| (unscaled). Groups: q >> 1 for two groups
// of 8, one group of 16.
template <int G>
__device__ inline void unit_centre(f32x4 (&x)[4], const int* cnt, int ngroups, int unit, int lane, float (&mu)[2],
                                   float (&s)[2], float (&m)[2]) {
    const int pr = (lane >> 3) & 1, pc = lane >> 5;
    bool real[4];
    float sum[2] = {0.f, 0.f};
    int k[2] = {0, 0};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int p = 4 * q + 2 * pr + pc;
        const int g = G == 8 ? 2 * unit + (p >> 3) : unit, idx = p & (G - 1);
        real[q] = g < ngroups && idx < cnt[g];
        if (real[q]) sum[G == 8 ? q >> 1 : 0] += (x[q][0] + x[q][1]) + (x[q][2] + x[q][3]);
    }
#pragma unroll
    for (int gs = 0; gs < (G == 8 ? 2 : 1); ++gs) {
        const int g = G == 8 ? 2 * unit + gs : unit;
        k[gs] = g < ngroups ? cnt[g] : 0;
        const float tot = wave_sum_dpp(sum[gs]);
        mu[gs] = k[gs] > 0 ? tot / static_cast<float>(64 * k[gs]) : 0.f;
    }
    if constexpr (G == 16) mu[1] = mu[0];
    float mx[2] = {0.f, 0.f};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int gs = G == 8 ? q >> 1 : 0;
        if (real[q]) x[q] -= mu[gs];
#pragma unroll
        for (int j = 0; j < 4; ++j) mx[gs] = fmaxf(mx[gs], fabsf(x[q][j]));
    }
    m[0] = wave_max_dpp(mx[0]);
    m[1] = G == 8 ? wave_max_dpp(mx[1]) : m[0];
    s[0] = group_scale(m[0]);
    s[1] = group_scale(m[1]);
#pragma unroll
    for (int q = 0; q < 4; ++q) x[q] *= s[G == 8 ? q >> 1 : 0];
}

// FP32 value, in data units, of coefficient ci = 8 u + v (u along y) of Haar
// row jr of unit group gs, from the lane-held centred and scaled pixels xc
// (A layout) and the DCT table d (LDS): sum over the group's patches p of
// haar(jr, p) D[u][y] D[v][x] xc_p[y][x], times the Haar factor and 1 / s,
// plus the centre's share corr. Every argument but xc, d and lane is
// wave-uniform; every lane returns the value.
template <int G>
__device__ inline float exact_coef(const f32x4 (&xc)[4], const float* d, int ci, int jr, int gs, float inv_s,
                                   float corr, int lane) {
    const int u = ci >> 3, v = ci & 7;
    const float dy = d[u * 8 + (lane & 7)];
    const f32x4 dx = *reinterpret_cast<const f32x4*>(d + v * 8 + 4 * ((lane >> 4) & 1));
    float acc = 0.f;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        if (G == 8 && (q >> 1) != gs) continue;
        const int p = 4 * q + 2 * ((lane >> 3) & 1) + (lane >> 5);
        const float r = fmaf(dx[3], xc[q][3], fmaf(dx[2], xc[q][2], fmaf(dx[1], xc[q][1], dx[0] * xc[q][0])));
        acc = fmaf(haar_entry(jr, p & (G - 1)) * dy, r, acc);
    }
    return fmaf(wave_sum_dpp(acc) * haar_scale(G, jr), inv_s, corr);
}

// A hard-threshold decision of an MFMA form is re-made in FP32 when the
// coefficient lies within band * max |x - mu| of the threshold. fp16: the
// measured error of a coefficient stays below 5.2 * 2^-11 max |x - mu|
// over two million coefficients of sigma-20 groups (the data rounding, 2^-12
// relative, carried through the orthonormal transforms; the DCT matrix
// enters split hi + lo), band 6 * 2^-11. bf16x3: each operand is hi + lo
// with a residual near 2^-17 relative, band 8 * 2^-16.
template <int FORM>
__device__ constexpr float redecide_band() {
    return FORM == kFormF16 ? 6.f * (1.f / 2048.f) : 8.f * (1.f / 65536.f);
}

template <int G, bool WIENER, int FORM>
__global__ __launch_bounds__(256) void filter_tile_mfma_kernel(FilterTable tab) {
    extern __shared__ __align__(16) unsigned long long acc[];
    constexpr int B = 8;
    static_assert(G == 8 || G == 16, "units of 16 patches");
    const int lb = xcd_block();
    const FilterJob& jb = tab.job[find_job(tab, lb)];
    const TileGeom& tg = jb.tiles;
    const int tile = lb - jb.wg_begin;  // partials index
    const int tx = (tile + jb.tile0) % tg.ntx, ty = (tile + jb.tile0) / tg.ntx;
    const int aw = tg.aw, ah = tg.ah;
    const int ax0 = tg.ax0(tx, jb.width, B, jb.grid.step, jb.range);
    const int ay0 = tg.ay0(ty, jb.height, B, jb.grid.step, jb.range);
    const int i_begin = tx * tg.tw, j_begin = ty * tg.th;
    const int ni = min(tg.tw, jb.grid.nx - i_begin), nj = min(tg.th, jb.grid.ny - j_begin);
    const int ngroups = ni * nj;
    const int nunits = G == 8 ? (ngroups + 1) / 2 : ngroups;
    unsigned long long* num = acc;
    // Patch positions (x | y << 16) and counts of the tile's groups, then the
    // transpose buffers, 16-byte aligned.
    uint32_t* recs = reinterpret_cast<uint32_t*>(acc + ((aw * ah + 1) & ~1));
    int* cnt = reinterpret_cast<int*>(recs + ((tg.tw * tg.th * G + 3) & ~3));
    float* scratch = reinterpret_cast<float*>(cnt + ((tg.tw * tg.th + 3) & ~3));
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    float* T = scratch + wave * kMfmaBuf;
    for (int e = threadIdx.x; e < aw * ah; e += 256) acc[e] = 0ull;
    for (int e = threadIdx.x; e < ngroups * G; e += 256) {
        const int g = e / G, j = e - g * G;
        const int gj = g / ni, gi = g - gj * ni;
        const MatchRec r =
            jb.matches[static_cast<size_t>((j_begin + gj - jb.grid.row0) * jb.grid.nx + i_begin + gi) * G + j];
        recs[e] = static_cast<uint32_t>(r.x) | (static_cast<uint32_t>(r.y) << 16);
    }
    for (int g = threadIdx.x; g < ngroups; g += 256) {
        const int gj = g / ni, gi = g - gj * ni;
        cnt[g] = jb.counts[(j_begin + gj - jb.grid.row0) * jb.grid.nx + i_begin + gi];
    }
    __syncthreads();

    const f32x4 de = dct_bd_entries(false, lane), dte = dct_bd_entries(true, lane);
    const Operand<FORM> dct = operand<FORM>(de);
    const Operand<FORM> dctt = operand<FORM>(dte);
    const Operand<FORM> dlo = operand<FORM>(FORM == kFormF16 ? f16_residual(de) : de);
    const Operand<FORM> dtlo = operand<FORM>(FORM == kFormF16 ? f16_residual(dte) : dte);
    const Operand<FORM> haar = operand<FORM>(haar_unit_entries<G>(false, lane));
    const Operand<FORM> haart = operand<FORM>(haar_unit_entries<G>(true, lane));
    // The DCT table for the FP32 re-decisions of the hard threshold.
    float* dtab = scratch + 4 * kMfmaBuf;
    if (!WIENER && threadIdx.x < 64) dtab[threadIdx.x] = c_dct[dct_offset<8>() + threadIdx.x];
    const float thr = 2.7f * jb.sigma;  // include/nss/params.hpp:46 kBmHardLambda
    const float sig2 = jb.sigma * jb.sigma;
    // Haar rows of this lane in the coefficient layout: 4 (lane >> 4) + j; for
    // two groups of 8 the group is lane >> 5.
    const int hgroup = G == 8 ? lane >> 5 : 0;
    float hs[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) hs[j] = haar_scale(G, (4 * (lane >> 4) + j) & (G - 1));
    if (!WIENER) __syncthreads();

    f32x4 x[4], xr[4];
    int u = wave;
    if (u < nunits) {
        load_unit<G>(jb.src, jb.stride, recs, cnt, ngroups, u, lane, x);
        if constexpr (WIENER) load_unit<G>(jb.wref, jb.wref_stride, recs, cnt, ngroups, u, lane, xr);
    }
    for (; u < nunits; u += 4) {
        float s[2], sr[2], mu[2], mur[2], mx[2], mxr[2];
        unit_centre<G>(x, cnt, ngroups, u, lane, mu, s, mx);
        f32x4 c[4], r[4];
        forward_unit<FORM>(x, dct, dlo, haar, T, lane, c);
        if constexpr (WIENER) {
            unit_centre<G>(xr, cnt, ngroups, u, lane, mur, sr, mxr);
            forward_unit<FORM>(xr, dct, dlo, haar, T, lane, r);
        }
        // Hard threshold: the centred, scaled pixels, kept for the FP32
        // re-decisions after the next unit's loads replace x.
        f32x4 xc[4];
        if constexpr (!WIENER) {
#pragma unroll
            for (int q = 0; q < 4; ++q) xc[q] = x[q];
        }
        const int un = u + 4;
        if (un < nunits) {
            load_unit<G>(jb.src, jb.stride, recs, cnt, ngroups, un, lane, x);
            if constexpr (WIENER) load_unit<G>(jb.wref, jb.wref_stride, recs, cnt, ngroups, un, lane, xr);
        }
        // The centres' share of each 2-D DC coefficient (coefficient 0 of
        // every Haar row; zero on the other lanes).
        float corr[4] = {0.f, 0.f, 0.f, 0.f}, corr_r[4] = {0.f, 0.f, 0.f, 0.f};
        {
            if ((lane & 15) == 0) {
                const int g = G == 8 ? 2 * u + hgroup : u;
                const int k = g < ngroups ? cnt[g] : 0;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float e = hs[j] * static_cast<float>(haar_row_count((4 * (lane >> 4) + j) & (G - 1), k)) * 8.f;
                    corr[j] = e * mu[hgroup];
                    corr_r[j] = e * mur[hgroup];
                }
            }
        }
        // Shrink in FP32 on the orthonormal coefficients of the unscaled data.
        const float inv_s = 1.f / s[hgroup];
        float vv[4][4];
        bool band[4][4];
        float w2 = 0.f;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const bool dc = t == 0 && (lane & 15) == 0 && ((4 * (lane >> 4) + j) & (G - 1)) == 0;
                const float cj = t == 0 ? corr[j] : 0.f;
                float v = fmaf(c[t][j] * hs[j], inv_s, cj);
                band[t][j] = false;
                if constexpr (WIENER) {
                    const float rv = fmaf(r[t][j] * hs[j], 1.f / sr[hgroup], t == 0 ? corr_r[j] : 0.f);
                    float w = 1.f;
                    if (!dc) {
                        const float r2 = rv * rv;
                        const float den = r2 + sig2;
                        w = den > 0.f ? r2 / den : 0.f;
                    }
                    v *= w;
                    w2 = fmaf(w, w, w2);
                } else {
                    band[t][j] = !dc && fabsf(fabsf(v) - thr) <= redecide_band<FORM>() * mx[hgroup];
                }
                vv[t][j] = v;
            }
        bool any_band = false;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) any_band |= band[t][j];
        if (!WIENER && __ballot(any_band)) {
            // Coefficients whose MFMA value cannot decide the threshold: their
            // FP32 value, one coefficient at a time by the whole wave.
#pragma unroll
            for (int t = 0; t < 4; ++t)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    unsigned long long pend = __ballot(band[t][j]);
                    while (pend) {
                        const int L = __builtin_ctzll(pend);
                        pend &= pend - 1;
                        const int gs = G == 8 ? L >> 5 : 0;
                        const float cl = t == 0 ? __shfl(corr[j], L, 64) : 0.f;
                        const float e = exact_coef<G>(xc, dtab, 16 * t + (L & 15), (4 * (L >> 4) + j) & (G - 1), gs,
                                                      1.f / s[gs], cl, lane);
                        if (lane == L) vv[t][j] = e;
                    }
                }
        }
        int kept = 0;
#pragma unroll
        for (int t = 0; t < 4; ++t)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                float v = vv[t][j];
                if constexpr (!WIENER) {
                    const bool dc = t == 0 && (lane & 15) == 0 && ((4 * (lane >> 4) + j) & (G - 1)) == 0;
                    if (!dc && fabsf(v) < thr)
                        v = 0.f;
                    else
                        ++kept;
                }
                // back to the operand scale without the centre's share,
                // butterfly factor applied again (the inverse orthonormal
                // Haar is H^T diag(factors))
                c[t][j] = (v - (t == 0 ? corr[j] : 0.f)) * hs[j] * s[hgroup];
            }
        float wg[2];
        if constexpr (WIENER) {
            float sum = w2;
#pragma unroll
            for (int off = 16; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, 64);
            if constexpr (G == 16) sum += __shfl_xor(sum, 32, 64);
            wg[0] = 1.f / fmaxf(__shfl(sum, 0, 64), 1e-12f);
            wg[1] = 1.f / fmaxf(__shfl(sum, 32, 64), 1e-12f);
        } else {
            int sum = kept;
#pragma unroll
            for (int off = 16; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, 64);
            if constexpr (G == 16) sum += __shfl_xor(sum, 32, 64);
            wg[0] = 1.f / static_cast<float>(max(__shfl(sum, 0, 64), 1));
            wg[1] = 1.f / static_cast<float>(max(__shfl(sum, 32, 64), 1));
        }
        f32x4 xo[4];
        inverse_unit<FORM>(c, dctt, dtlo, haart, T, lane, xo);
        const int pr = lane >> 5, pc = (lane >> 3) & 1, px = lane & 7, y0 = 4 * ((lane >> 4) & 1);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int p = 4 * q + 2 * pr + pc;
            const int g = G == 8 ? 2 * u + (p >> 3) : u, idx = p & (G - 1);
            const int gsel = G == 8 ? (q >> 1) : 0;
            if (g < ngroups && idx < cnt[g]) {
                const uint32_t xy = recs[g * G + idx];
                const int lx = static_cast<int>(xy & 0xffffu) - ax0, ly = static_cast<int>(xy >> 16) - ay0;
                const float w = wg[gsel];
                const float wq = w / s[gsel];
                const float wm = w * mu[gsel];  // the centre, added back
                unsigned long long* cell = num + (ly + y0) * aw + lx + px;
                float wx[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) wx[j] = fmaf(wq, xo[q][j], wm);
                unsigned long long fx[4];
                to_fixed_n<4>(wx, fx);
#pragma unroll
                for (int j = 0; j < 4; ++j) lds_add(cell + j * aw, fx[j]);
            }
        }
        // the unit's group weights (two groups of 8 or one of 16)
        if (lane < (G == 8 ? 2 : 1)) {
            const int g = G == 8 ? 2 * u + lane : u;
            if (g < ngroups) {
                const int gj = g / ni, gi = g - gj * ni;
                jb.gweight[(j_begin + gj - jb.grid.row0) * jb.grid.nx + i_begin + gi] = to_fixed(lane ? wg[1] : wg[0]);
            }
        }
    }
    __syncthreads();
    tile_partials(jb, tile, ax0, num);
}

// Atomic path: one wave per group, frame-sized fixed-point sums (den at the
// patch corner).
template <int B, bool WIENER>
__device__ inline void atomic_group(const FilterJob& jb, int g, float* cube, int lane) {
    constexpr int A = B * B;
    constexpr int PS = A + 1;
    const int G = jb.group;
    const int k = jb.counts[g];
    const MatchRec* rec = jb.matches + static_cast<size_t>(g) * G;
    float* rc = cube + G * PS;
    const float weight = filter_group_wave<B, WIENER>(jb, rec, k, cube, rc, lane);
    const unsigned long long wfix = to_fixed(weight);
    for (int j = 0; j < k; ++j) {
        const int mx = rec[j].x, my = rec[j].y;
        for (int e = lane; e < A; e += 64) {
            const int py = e / B, px = e - (e / B) * B;
            atomicAdd(jb.num + static_cast<size_t>(my + py) * jb.width + mx + px, to_fixed(weight * cube[j * PS + e]));
        }
        if (lane == 0) atomicAdd(jb.den + static_cast<size_t>(my) * jb.width + mx, wfix);
    }
}

template <int B, bool WIENER>
__global__ __launch_bounds__(64) void filter_atomic_kernel(FilterTable tab) {
    extern __shared__ __align__(16) float lds_cube[];
    const int lane = threadIdx.x;
    if (tab.cube) {
        // Cubes beyond the LDS: workgroup b takes groups b, b + gridDim.x, ...
        // with its own cube in global memory (the same arithmetic; a wave's
        // global stores and loads stay in order on its CU).
        const FilterJob& last = tab.job[tab.n - 1];
        const int total = last.wg_begin + last.nref;
        float* cube = tab.cube + static_cast<size_t>(blockIdx.x) * tab.cube_floats;
        for (int gi = blockIdx.x; gi < total; gi += gridDim.x) {
            const FilterJob& jb = tab.job[find_job(tab, gi)];
            atomic_group<B, WIENER>(jb, gi - jb.wg_begin, cube, lane);
            wave_sync();
        }
        return;
    }
    const int lb = xcd_block();
    const FilterJob& jb = tab.job[find_job(tab, lb)];
    const int g = lb - jb.wg_begin;
    if (g >= jb.nref) return;
    atomic_group<B, WIENER>(jb, g, lds_cube, lane);
}

// ---------------------------------------------------------------------------
// Temporal: predictive search (src/cpu/bm/matcher.hpp:319-373) and the
// group filter with per-slot sources and accumulators.
// ---------------------------------------------------------------------------
__device__ inline unsigned long long pack_pos(int t, int y, int x) {
    return (static_cast<unsigned long long>(t) << 26) | (static_cast<unsigned long long>(y) << 13) |
           static_cast<unsigned long long>(x);
}

// One wave per reference. The spatial matches (slot radius) seed the search:
// per direction, layer dt scores the union of (2 ps_range + 1)^2 windows
// around the previous layer's winners (every union position once), keeps its
// min(ps_num, G) smallest (dist, y, x), and those feed the global G-1
// smallest (dist, t, y, x) with the spatial matches. Layer 1's centres are
// the first ps_num spatial matches. When the layer's windows fit the staging
// buffer, their pixels are copied to LDS once and each lane scores three
// horizontally adjacent candidates from one register row per block row
// (same sums, same order as scoring from the frame).
// LDS: reference patch | layer chunk keys | best, next best | centres | merged
// | staged windows.
template <int B>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(6))) void predictive_kernel(PredTable tab) {
    extern __shared__ __align__(16) unsigned char smem[];
    const int lane = threadIdx.x;
    // XCD-contiguous references: neighbours share their frames' rows in L2.
    const int lb = xcd_block();
    const PredJob& jb = tab.job[find_job(tab, lb)];
    const int ref = lb - jb.wg_begin;
    if (ref >= jb.nref) return;
    const int G = jb.group;
    const Slots& sl = jb.slots;
    const int t0 = sl.radius;
    MatchRec* rec = jb.recs + static_cast<size_t>(ref) * G;
    const int n = jb.counts[ref];
    const int cx = rec[0].x, cy = rec[0].y;
    float* refp = reinterpret_cast<float*>(smem);
    unsigned long long* cand = reinterpret_cast<unsigned long long*>(refp + ((B * B + 3) & ~3));
    unsigned long long* best = reinterpret_cast<unsigned long long*>(cand + tab.chunk);
    unsigned long long* nbest = best + kMaxGroup;
    int* centers = reinterpret_cast<int*>(nbest + kMaxGroup);
    unsigned long long* merged = reinterpret_cast<unsigned long long*>(centers + kMaxGroup);
    float* region = reinterpret_cast<float*>(smem + tab.region_offset);
    {
        const float* p0 = jb.match.frame(sl.frame(t0));
        for (int e = lane; e < B * B; e += 64) refp[e] = p0[static_cast<size_t>(cy + e / B) * jb.stride + cx + e % B];
    }
    for (int i = lane; i < n - 1; i += 64)
        merged[i] = (static_cast<unsigned long long>(rec[1 + i].dist) << 32) | pack_pos(t0, rec[1 + i].y, rec[1 + i].x);
    int nm = n - 1;
    const int vb = sl.valid_begin(), ve = sl.valid_end();
    const int kl = min(jb.ps_num, G);
    const int seeds = min(n, jb.ps_num);
    const int ps = jb.ps_range;
    const int maxx = jb.width - B, maxy = jb.height - B;
    __syncthreads();
    for (int sign = -1; sign <= 1; sign += 2) {
        if (lane < seeds) centers[lane] = (rec[lane].y << 13) | rec[lane].x;
        int nc = seeds;
        __syncthreads();
        for (int dt = 1; dt <= sl.radius; ++dt) {
            const int t = t0 + sign * dt;
            if (t < vb || t >= ve) break;
            const float* pt = jb.match.frame(sl.frame(t));
            // The union of the centres' (2 ps + 1)^2 windows (clamped to the
            // plane), enumerated window by window: a cell belongs to the first
            // window that contains it, so every union position is scored once.
            const int W = 2 * ps + 1, WW = W * W;
            const int cells = nc * WW;
            auto ssd = [&](const float* base, int stride) {
                float acc = 0.f;
                for (int py = 0; py < B; ++py) {
                    const float* row = base + py * stride;
#pragma unroll
                    for (int px = 0; px < B; ++px) {
                        const float d = refp[py * B + px] - row[px];
                        acc = fmaf(d, d, acc);
                    }
                }
                return acc;
            };
            auto member_of = [&](int w, int y, int x) {
                bool m = y >= 0 && y <= maxy && x >= 0 && x <= maxx;
                for (int q = 0; q < w && m; ++q) {
                    const int cq = centers[q];
                    m = !(abs(y - (cq >> 13)) <= ps && abs(x - (cq & 8191)) <= ps);
                }
                return m;
            };
            const int R = W + B - 1, P = pred_region_pitch(W, B), SW = (W + 2) / 3;
            const bool staged = cells <= tab.chunk && nc * R * P <= tab.region;
            // A layer of up to 64 strips keeps its keys in registers, three a
            // lane: the winners come from wave minima instead of passes over
            // the keys in LDS (1080p YUV420, two windows of 9 x 9: 142 -> 126
            // us per launch, with the strips' divisions by reciprocals).
            bool held = false;
            unsigned long long strip[3] = {~0ull, ~0ull, ~0ull};
            if (staged) {
                // Window w's pixels (rows y_w - ps .., columns x_w - ps ..) at
                // region[w R P + j P + i]. Columns from R on and pixels off the
                // plane are read only for discarded candidates (positions off
                // the plane are not members; a member's patch lies in rows and
                // columns below R), so the loads leave them as they are.
                // Lanes cover 64 / P rows of P columns per step (P <= 64), or
                // one row in steps of 64 columns.
                const int rows_per = P <= 64 ? 64 / P : 1;
                const int lr = P <= 64 ? div_small(lane, __builtin_amdgcn_rcpf(static_cast<float>(P))) : 0;
                const int li = P <= 64 ? lane - lr * P : lane;
                for (int w = 0; w < nc; ++w) {
                    const int cw = centers[w];
                    const int y0 = (cw >> 13) - ps, x0 = (cw & 8191) - ps;
                    float* dst = region + w * (R * P);
                    if (lr >= rows_per) continue;
                    if (P <= 64 && R <= 8 * rows_per) {
                        // one column per lane, up to 8 rows, each load
                        // straight to LDS (global_load_lds: lane l's word at
                        // the wave-uniform address dst + q rows_per P + 4 l,
                        // which is row j = lr + q rows_per, column li);
                        // the barrier below waits for them
#pragma unroll
                        for (int q = 0; q < 8; ++q) {
                            const int j = lr + q * rows_per, y = y0 + j, x = x0 + li;
                            if (j < R && li < R && y >= 0 && y < jb.height && x >= 0 && x < jb.width)
                                __builtin_amdgcn_global_load_lds(
                                    (const __attribute__((address_space(1))) void*)(pt + static_cast<size_t>(y) * jb.stride + x),
                                    (__attribute__((address_space(3))) void*)(dst + q * rows_per * P), 4, 0, 0);
                        }
                        continue;
                    }
                    // the same loads for any pitch: lane l's word at
                    // dst + j P + i = (dst + j P + i - l) + 4 l, the base
                    // alike for every lane of a step
                    for (int j = lr; j < R; j += rows_per)
                        for (int i = li; i < P; i += (P <= 64 ? P : 64)) {
                            const int y = y0 + j, x = x0 + i;
                            if (i < R && y >= 0 && y < jb.height && x >= 0 && x < jb.width)
                                __builtin_amdgcn_global_load_lds(
                                    (const __attribute__((address_space(1))) void*)(pt + static_cast<size_t>(y) * jb.stride + x),
                                    (__attribute__((address_space(3))) void*)(dst + j * P + i - lane), 4, 0, 0);
                        }
                }
                __syncthreads();
                const int strips = nc * W * SW;
                held = strips <= 64;
                const float inv_ws = __builtin_amdgcn_rcpf(static_cast<float>(W * SW));
                const float inv_s = __builtin_amdgcn_rcpf(static_cast<float>(SW));
                for (int sidx = lane; sidx < strips; sidx += 64) {
                    // (below 2^20 strips: exact from the hardware reciprocals)
                    const int w = div_small(sidx, inv_ws), o = sidx - w * (W * SW);
                    const int dy = div_small(o, inv_s), dx0 = 3 * (o - dy * SW);
                    const float* rb = region + w * (R * P) + dy * P + dx0;
                    float a0 = 0.f, a1 = 0.f, a2 = 0.f;
#pragma unroll 1
                    for (int py = 0; py < B; ++py) {
                        float v[B + 2];
#pragma unroll
                        for (int q = 0; q < B + 2; ++q) v[q] = rb[py * P + q];
#pragma unroll
                        for (int px = 0; px < B; ++px) {
                            const float rv = refp[py * B + px];
                            const float d0 = rv - v[px], d1 = rv - v[px + 1], d2 = rv - v[px + 2];
                            a0 = fmaf(d0, d0, a0);
                            a1 = fmaf(d1, d1, a1);
                            a2 = fmaf(d2, d2, a2);
                        }
                    }
                    const int cw = centers[w];
                    const int y = (cw >> 13) - ps + dy;
#pragma unroll
                    for (int q = 0; q < 3; ++q) {
                        const int dx = dx0 + q;
                        if (dx < W) {
                            const int x = (cw & 8191) - ps + dx;
                            const float a = q == 0 ? a0 : q == 1 ? a1 : a2;
                            const unsigned long long key =
                                member_of(w, y, x)
                                    ? (static_cast<unsigned long long>(dist_key(a)) << 32) | pack_pos(0, y, x)
                                    : ~0ull;
                            if (held)
                                strip[q] = key;
                            else
                                cand[w * WW + dy * W + dx] = key;
                        }
                    }
                }
            }
            int nb = 0;
            for (; held && nb < kl; ++nb) {
                const unsigned long long m = min(strip[0], min(strip[1], strip[2]));
                const uint32_t d = static_cast<uint32_t>(m >> 32), at = static_cast<uint32_t>(m);
                const uint32_t mn = wave_min_u32_dpp(d);
                if (mn == kTaken) break;  // no member left
                const unsigned long long who = __builtin_amdgcn_ballot_w64(d == mn);
                uint32_t first = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(at), __builtin_ctzll(who)));
                if ((who & (who - 1u)) != 0) first = wave_min_u32_dpp(d == mn ? at : ~0u);  // equal distances
                const unsigned long long win = (static_cast<unsigned long long>(mn) << 32) | first;
#pragma unroll
                for (int q = 0; q < 3; ++q) strip[q] = strip[q] == win ? ~0ull : strip[q];
                if (lane == 0) best[nb] = win;
            }
            if (held) __syncthreads();
            for (int base = 0; base < cells && !held; base += tab.chunk) {
                const int cnt = min(tab.chunk, cells - base);
                for (int c = lane; c < cnt && !staged; c += 64) {
                    const int cell = base + c;
                    const int w = cell / WW, o = cell - w * WW;
                    const int dy = o / W;
                    const int cw = centers[w];
                    const int y = (cw >> 13) - ps + dy, x = (cw & 8191) - ps + (o - dy * W);
                    unsigned long long key = ~0ull;
                    if (member_of(w, y, x))
                        key = (static_cast<unsigned long long>(dist_key(ssd(pt + static_cast<size_t>(y) * jb.stride + x,
                                                                            jb.stride)))
                               << 32) |
                              pack_pos(0, y, x);
                    cand[c] = key;
                }
                __syncthreads();
                // The chunk's candidates and the running best: the kl smallest
                // keys (unique: one per position), each taken by its owner lane.
                int nn = 0;
                for (int k = 0; k < kl; ++k) {
                    unsigned long long m = ~0ull, mb = ~0ull;
                    int mi = 0, bi = 0;
                    for (int c = lane; c < cnt; c += 64)
                        if (cand[c] < m) {
                            m = cand[c];
                            mi = c;
                        }
                    for (int i = lane; i < nb; i += 64)
                        if (best[i] < mb) {
                            mb = best[i];
                            bi = i;
                        }
                    const unsigned long long mine = m < mb ? m : mb;
                    const unsigned long long win = wave_min_u64(mine);
                    if (win == ~0ull) break;
                    if (mine == win) {
                        if (m < mb)
                            cand[mi] = ~0ull;
                        else
                            best[bi] = ~0ull;
                    }
                    if (lane == 0) nbest[nn] = win;
                    ++nn;
                    __syncthreads();
                }
                for (int i = lane; i < nn; i += 64) best[i] = nbest[i];
                nb = nn;
                __syncthreads();
            }
            // Layer winners (ascending): into the merged list, and the next centres.
            for (int i = lane; i < nb; i += 64) {
                const unsigned long long b = best[i];
                merged[nm + i] = (b & 0xffffffff00000000ull) | pack_pos(t, static_cast<int>((b >> 13) & 8191),
                                                                       static_cast<int>(b & 8191));
                centers[i] = static_cast<int>(b & 0x3ffffff);
            }
            nm += nb;
            nc = nb;
            __syncthreads();
            if (nc == 0) break;
        }
    }
    // The G-1 smallest merged keys in ascending order: keys are unique (one
    // per (t, y, x)), so each key's rank is the count of smaller keys.
    const int K = min(G - 1, nm);
    for (int i = lane; i < nm; i += 64) {
        const unsigned long long m = merged[i];
        int rank = 0;
        for (int j = 0; j < nm; ++j) rank += merged[j] < m ? 1 : 0;
        if (rank < K)
            rec[1 + rank] = MatchRec{static_cast<int>(m & 8191), static_cast<int>((m >> 13) & 8191),
                                     static_cast<int>((m >> 26) & 63), static_cast<uint32_t>(m >> 32)};
    }
    if (lane == 0) jb.counts[ref] = 1 + K;
}

// One wave per group: patches from their slots' frames, sums into the
// accumulators of those frames.
template <int B, bool WIENER>
__device__ inline void temporal_group(const TFilterJob& jb, int g, float* cube, int lane) {
    constexpr int A = B * B;
    constexpr int PS = A + 1;
    const int G = jb.group;
    const int k = jb.counts[g];
    const MatchRec* rec = jb.matches + static_cast<size_t>(g) * G;
    float* rc = cube + G * PS;
    gather_group_wave<B, WIENER>(
        rec, k, G, jb.stride, jb.wref_stride, [&](int t) { return jb.src.frame(jb.slots.frame(t)); },
        [&](int t) { return jb.wref.frame(jb.slots.frame(t)); }, cube, rc, lane);
    const float weight = transform_group_wave<B, WIENER>(G, jb.sigma, cube, rc, lane);
    const unsigned long long wfix = to_fixed(weight);
    const size_t plane = static_cast<size_t>(jb.width) * jb.height;
    for (int j = 0; j < k; ++j) {
        const int mx = rec[j].x, my = rec[j].y;
        const size_t slot = static_cast<size_t>(jb.slots.frame(rec[j].t) % jb.acc_ring) * plane;
        unsigned long long* num = jb.num + slot;
        for (int e = lane; e < A; e += 64) {
            const int py = e / B, px = e - (e / B) * B;
            atomicAdd(num + static_cast<size_t>(my + py) * jb.width + mx + px, to_fixed(weight * cube[j * PS + e]));
        }
        if (lane == 0) atomicAdd(jb.den + slot + static_cast<size_t>(my) * jb.width + mx, wfix);
    }
}

template <int B, bool WIENER>
__global__ __launch_bounds__(64) void filter_temporal_kernel(TFilterTable tab) {
    extern __shared__ __align__(16) float lds_cube[];
    const int lane = threadIdx.x;
    if (tab.cube) {
        // Cubes beyond the LDS, as in filter_atomic_kernel.
        const TFilterJob& last = tab.job[tab.n - 1];
        const int total = last.wg_begin + last.nref;
        float* cube = tab.cube + static_cast<size_t>(blockIdx.x) * tab.cube_floats;
        for (int gi = blockIdx.x; gi < total; gi += gridDim.x) {
            const TFilterJob& jb = tab.job[find_job(tab, gi)];
            temporal_group<B, WIENER>(jb, gi - jb.wg_begin, cube, lane);
            wave_sync();
        }
        return;
    }
    const int lb = xcd_block();
    const TFilterJob& jb = tab.job[find_job(tab, lb)];
    const int g = lb - jb.wg_begin;
    if (g >= jb.nref) return;
    temporal_group<B, WIENER>(jb, g, lds_cube, lane);
}

// Block 8, G in {8, 16, 32}: four groups per workgroup, a wave per group with
// the cube in registers (the spatial register kernel's transforms); patches
// from their slot's frame, device-scope int64 atomics into the sums of that
// frame (den at the patch corner).
template <int G, bool WIENER>
__global__ __launch_bounds__(256) void filter_temporal_b8_kernel(TFilterTable tab) {
    extern __shared__ __align__(16) float tbuf[];
    constexpr int M = G / 8;
    const int lb = xcd_block();
    const TFilterJob& jb = tab.job[find_job(tab, lb)];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int g = (lb - jb.wg_begin) * 4 + wave;
    if (g >= jb.nref) return;  // whole wave; no workgroup barrier below
    float* T = tbuf + wave * (G * kTs);
    const int k = jb.counts[g];
    const MatchRec* rec = jb.matches + static_cast<size_t>(g) * G;
    const int gb = lane >> 3, y = lane & 7;
    float v[M][8], vr[M][8];
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int p = gb + 8 * m;
        if (p < k) {
            const MatchRec r = rec[p];
            const int f = jb.slots.frame(r.t);
            const size_t o = static_cast<size_t>(r.y + y) * jb.stride + r.x;
            const float* sp = jb.src.frame(f) + o;
#pragma unroll
            for (int x = 0; x < 8; ++x) v[m][x] = sp[x];
            if constexpr (WIENER) {
                const float* wp = jb.wref.frame(f) + static_cast<size_t>(r.y + y) * jb.wref_stride + r.x;
#pragma unroll
                for (int x = 0; x < 8; ++x) vr[m][x] = wp[x];
            }
        } else {
#pragma unroll
            for (int x = 0; x < 8; ++x) v[m][x] = vr[m][x] = 0.f;
        }
    }
    float c[G], r[G];
    forward_b8<G>(v, c, T, lane);
    if constexpr (WIENER) forward_b8<G>(vr, r, T, lane);
    const float thr = 2.7f * jb.sigma;  // include/nss/params.hpp:46 kBmHardLambda
    const float sig2 = jb.sigma * jb.sigma;
    int kept = 0;
    float w2 = 0.f;
    if constexpr (WIENER) w2 = wiener_shrink<G>(c, r, sig2, lane);
#pragma unroll
    for (int j = 0; j < G; ++j) {
        if constexpr (!WIENER) {
            if (!(lane == 0 && j == 0) && fabsf(c[j]) < thr)
                c[j] = 0.f;
            else
                ++kept;
        }
    }
    haar_inverse_reg<G>(c);
    float u[M][8];
    group_to_columns<G>(c, u, T, lane);
#pragma unroll
    for (int m = 0; m < M; ++m) dct8<true>(u[m]);
    transpose_rc<M>(u, T, lane);
#pragma unroll
    for (int m = 0; m < M; ++m) dct8<true>(u[m]);
    float w;
    if constexpr (WIENER) {
        w = 1.f / fmaxf(wave_sum_f32(w2), 1e-12f);
    } else {
        w = 1.f / static_cast<float>(max(wave_sum_i32(kept), 1));
    }
    const unsigned long long wfix = to_fixed(w);
    const size_t plane = static_cast<size_t>(jb.width) * jb.height;
#pragma unroll
    for (int m = 0; m < M; ++m) {
        const int p = gb + 8 * m;
        if (p < k) {
            const MatchRec rr = rec[p];
            const size_t slot = static_cast<size_t>(jb.slots.frame(rr.t) % jb.acc_ring) * plane;
            unsigned long long* row = jb.num + slot + static_cast<size_t>(rr.y + y) * jb.width + rr.x;
#pragma unroll
            for (int x = 0; x < 8; ++x) atomicAdd(row + x, to_fixed(w * u[m][x]));
            if (y == 0) atomicAdd(jb.den + slot + static_cast<size_t>(rr.y) * jb.width + rr.x, wfix);
        }
    }
}

// Temporal tile path, block 8, G in {8, 16, 32}: 8 waves per workgroup (16 at
// groups of 8 where the slots leave one workgroup per CU), a wave per group with
// the register cube; every slot's contributions go into that slot's LDS sums
// (apron = the slot's reach around the tile), then out as the centre's float
// partials, slot by slot. The LDS (well over half a CU's)
// leaves one workgroup per CU, so the kernel is persistent: workgroup L (in
// XCD-contiguous order) filters tiles [L T / n, (L + 1) T / n) of the T tiles,
// and while one tile's partials are written it loads the next tile's records
// and each wave's first patches; within a tile, a wave loads its next
// group's patches while the current one is filtered.
// LDS: match records | counts | per slot num [ah][aw] and corners [ch][cw]
// (int64) | per-wave transpose buffers (also the box sum).
inline constexpr int kTTileWaves = 8;

struct SlotLds {
    int off;       // int64 offset of the slot's num (corners follow)
    int ax0, ay0;  // apron origin
    int aw, ah;
};

struct TileAt {
    int job, tile, tx, ty, i_begin, j_begin, ni, ngroups;
};

__device__ inline TileAt ttile_at(const TTileTable& tab, int lt) {
    TileAt a;
    a.job = find_job(tab, lt);
    const TTileJob& jb = tab.job[a.job];
    const TileGeom& tg = jb.tiles[0];
    a.tile = lt - jb.wg_begin;
    a.tx = a.tile % tg.ntx;
    a.ty = a.tile / tg.ntx;
    a.i_begin = a.tx * tg.tw;
    a.j_begin = a.ty * tg.th;
    a.ni = min(tg.tw, jb.grid.nx - a.i_begin);
    a.ngroups = a.ni * min(tg.th, jb.grid.ny - a.j_begin);
    return a;
}

// This lane's rows (patch gb + 8 m, row y) of a group with k patches, from
// their slots' frames (zero beyond k); the Wiener reference rows too.
template <int G, bool WIENER>
__device__ inline void ttile_gather(const TTileJob& jb, const MatchRec* rec, int k, int gb, int y,
                                    float (&v)[G / 8][8], float (&vr)[G / 8][8]) {
#pragma unroll
    for (int m = 0; m < G / 8; ++m) {
        const int p = gb + 8 * m;
        if (p < k) {
            const MatchRec r = rec[p];
            const int f = jb.slots.frame(r.t);
            const float* sp = jb.src.frame(f) + static_cast<size_t>(r.y + y) * jb.stride + r.x;
#pragma unroll
            for (int x = 0; x < 8; ++x) v[m][x] = sp[x];
            if constexpr (WIENER) {
                const float* wp = jb.wref.frame(f) + static_cast<size_t>(r.y + y) * jb.wref_stride + r.x;
#pragma unroll
                for (int x = 0; x < 8; ++x) vr[m][x] = wp[x];
            }
        } else {
#pragma unroll
            for (int x = 0; x < 8; ++x) {
                v[m][x] = 0.f;
                if constexpr (WIENER) vr[m][x] = 0.f;
            }
        }
    }
}

template <int G, bool WIENER>
__global__ __launch_bounds__(G == 8 ? 1024 : 512) void filter_temporal_tile_kernel(TTileTable tab, int total_tiles) {
    extern __shared__ __align__(16) unsigned long long smem64[];
    constexpr int B = 8;
    constexpr int M = G / 8;
    const int L = xcd_block(), nb = static_cast<int>(gridDim.x);
    const int lo = static_cast<int>(static_cast<long long>(L) * total_tiles / nb);
    const int hi = static_cast<int>(static_cast<long long>(L + 1) * total_tiles / nb);
    if (lo >= hi) return;
    // Groups per tile (one tile shape per launch; tw * th * G <= 512, one
    // record per thread at most).
    const int cap = tab.job[0].tiles[0].tw * tab.job[0].tiles[0].th;
    MatchRec* recs = reinterpret_cast<MatchRec*>(smem64);
    int* cnt = reinterpret_cast<int*>(recs + cap * G);
    unsigned long long* acc = reinterpret_cast<unsigned long long*>(cnt + ((cap + 3) & ~3));
    __shared__ SlotLds sl[kMaxTileSlots];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int nt = static_cast<int>(blockDim.x), waves = nt >> 6;
    const int gb = lane >> 3, y = lane & 7;

    // Thread e's record (e < ngroups G) and count (e < ngroups) of tile a,
    // as four record words and the count.
    struct Fetched {
        int x, y, t;
        uint32_t dist;
        int count;
    };
    auto fetch = [&](const TileAt& a) {
        const int e = threadIdx.x;
        const TTileJob& jb = tab.job[a.job];
        Fetched f{0, 0, 0, 0u, 0};
        if (e < a.ngroups * G) {
            const int g = e / G, j = e - g * G;
            const int gj = g / a.ni, gi = g - gj * a.ni;
            const MatchRec r = jb.matches[static_cast<size_t>((a.j_begin + gj) * jb.grid.nx + a.i_begin + gi) * G + j];
            f.x = r.x;
            f.y = r.y;
            f.t = r.t;
            f.dist = r.dist;
        }
        if (e < a.ngroups) {
            const int gj = e / a.ni, gi = e - gj * a.ni;
            f.count = jb.counts[(a.j_begin + gj) * jb.grid.nx + a.i_begin + gi];
        }
        return f;
    };
    auto publish = [&](const TileAt& a, const Fetched& f) {
        const int e = threadIdx.x;
        if (e < a.ngroups * G) recs[e] = MatchRec{f.x, f.y, f.t, f.dist};
        if (e < a.ngroups) cnt[e] = f.count;
    };
    auto gather = [&](const TileAt& a, int g, float (&v)[M][8], float (&vr)[M][8]) {
        ttile_gather<G, WIENER>(tab.job[a.job], recs + g * G, cnt[g], gb, y, v, vr);
    };

    TileAt cur = ttile_at(tab, lo);
    publish(cur, fetch(cur));
    __syncthreads();
    float v[M][8], vr[M][8];
    if (wave < cur.ngroups) gather(cur, wave, v, vr);
    for (int lt = lo; lt < hi; ++lt) {
        const TTileJob& jb = tab.job[cur.job];
        const int ns = jb.nslots;
        // per slot: the numerator sums, then (den partials only) the corner sums
        const int cs = jb.corners ? 0 : 1;
        int total = 0;
        for (int t = 0; t < ns; ++t) {
            const TileGeom& g = jb.tiles[t];
            total += g.aw * g.ah + cs * (g.aw - B + 1) * (g.ah - B + 1);
        }
        if (static_cast<int>(threadIdx.x) < ns) {
            const int t = static_cast<int>(threadIdx.x);
            int o = 0;
            for (int q = 0; q < t; ++q)
                o += jb.tiles[q].aw * jb.tiles[q].ah + cs * (jb.tiles[q].aw - B + 1) * (jb.tiles[q].ah - B + 1);
            const TileGeom& g = jb.tiles[t];
            sl[t] = SlotLds{o, g.ax0(cur.tx, jb.width, B, jb.grid.step, jb.range[t]),
                            g.ay0(cur.ty, jb.height, B, jb.grid.step, jb.range[t]), g.aw, g.ah};
        }
        float* scratch = reinterpret_cast<float*>(acc + ((total + 1) & ~1));
        float* T = scratch + wave * (G * kTs);
        for (int e = threadIdx.x; e < total; e += nt) acc[e] = 0ull;
        __syncthreads();

        const float thr = 2.7f * jb.sigma;  // include/nss/params.hpp:46 kBmHardLambda
        const float sig2 = jb.sigma * jb.sigma;
        for (int g = wave; g < cur.ngroups; g += waves) {
            const int k = cnt[g];
            const MatchRec* rec = recs + g * G;
            float c[G], r[G];
            forward_b8<G>(v, c, T, lane);
            if constexpr (WIENER) forward_b8<G>(vr, r, T, lane);
            if (g + waves < cur.ngroups) gather(cur, g + waves, v, vr);
            int kept = 0;
            float w2 = 0.f;
            if constexpr (WIENER) w2 = wiener_shrink<G>(c, r, sig2, lane);
#pragma unroll
            for (int j = 0; j < G; ++j) {
                if constexpr (!WIENER) {
                    if (!(lane == 0 && j == 0) && fabsf(c[j]) < thr)
                        c[j] = 0.f;
                    else
                        ++kept;
                }
            }
            haar_inverse_reg<G>(c);
            float u[M][8];
            group_to_columns<G>(c, u, T, lane);
#pragma unroll
            for (int m = 0; m < M; ++m) dct8<true>(u[m]);
            transpose_rc<M>(u, T, lane);
#pragma unroll
            for (int m = 0; m < M; ++m) dct8<true>(u[m]);
            float w;
            if constexpr (WIENER) {
                w = 1.f / fmaxf(wave_sum_f32(w2), 1e-12f);
            } else {
                w = 1.f / static_cast<float>(max(wave_sum_i32(kept), 1));
            }
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const int p = gb + 8 * m;
                if (p < k) {
                    const MatchRec rr = rec[p];
                    const SlotLds q = sl[rr.t];
                    const int lx = rr.x - q.ax0, ly = rr.y - q.ay0;
                    // The predictive search keeps every slot-t match within the
                    // slot's reach; a patch outside the apron is dropped rather
                    // than written out of bounds.
                    if (lx >= 0 && ly >= 0 && lx <= q.aw - B && ly <= q.ah - B) {
                        unsigned long long* row = acc + q.off + (ly + y) * q.aw + lx;
                        float wu[8];
#pragma unroll
                        for (int x = 0; x < 8; ++x) wu[x] = w * u[m][x];
                        unsigned long long fx[8];
                        to_fixed_n<8>(wu, fx);
#pragma unroll
                        for (int x = 0; x < 8; ++x) lds_add(row + x, fx[x]);
                        if (y == 0) {
                            if (jb.corners)
                                atomicAdd(jb.corners +
                                              static_cast<size_t>(jb.slots.frame(rr.t) % jb.acc_ring) * jb.width *
                                                  jb.height +
                                              static_cast<size_t>(rr.y) * jb.width + rr.x,
                                          to_fixed(w));
                            else
                                lds_add(acc + q.off + q.aw * q.ah + ly * (q.aw - B + 1) + lx, to_fixed(w));
                        }
                    }
                }
            }
        }
        __syncthreads();
        // The next tile's records: loaded now, stored once the first slot's
        // partials are out (the records area is idle until then).
        const bool more = lt + 1 < hi;
        const TileAt nxt = more ? ttile_at(tab, lt + 1) : cur;
        const Fetched nf = more ? fetch(nxt) : Fetched{0, 0, 0, 0u, 0};
        for (int t = 0; t < ns; ++t) {
            const SlotLds q = sl[t];
            const TileGeom& g = jb.tiles[t];
            const size_t area = static_cast<size_t>(g.pitch) * g.ah;
            float* pn = jb.part + jb.slot_off[t] + static_cast<size_t>(cur.tile) * area + (q.ax0 & 3);
            float* pd = jb.corners ? nullptr : pn + static_cast<size_t>(g.ntx) * g.nty * area;
            partials_out_float<B>(q.aw, q.ah, g.pitch, acc + q.off, acc + q.off + q.aw * q.ah, scratch, pn, pd);
            if (t == 0 && more) publish(nxt, nf);
            __syncthreads();
            if (t == 0 && more && wave < nxt.ngroups) gather(nxt, wave, v, vr);
        }
        cur = nxt;
    }
}

// Temporal finish: frame n from the partials of every centre that reaches
// it (sources in ascending centre order), 64 x 16 pixels per block, four per
// thread, as finish_tiles_kernel.
__global__ __launch_bounds__(256) void finish_temporal_tiles_kernel(TFinishTable tab) {
    extern __shared__ __align__(16) unsigned long long tsm[];
    const int lb = xcd_block();
    const TFinishJob& jb = tab.job[find_job(tab, lb)];
    const int t = lb - jb.wg_begin;
    const int bx0 = (t % jb.tiles_x) * 64, by0 = (t / jb.tiles_x) * 16;
    const int x0 = bx0 + (threadIdx.x & 15) * 4;
    const int y = by0 + (threadIdx.x >> 4);
    const int B = jb.block, s = jb.step;
    long long dw[4] = {0, 0, 0, 0};
    if (jb.corners) {
        // den: the B x B box sum of the frame's corner plane (corners
        // (x - B + 1 .. x, y - B + 1 .. y)), staged in LDS, exact
        const int CW = 64 + B - 1, CH = 16 + B - 1;
        const int cx0 = bx0 - B + 1, cy0 = by0 - B + 1;
        unsigned long long* ct = tsm;            // [CH][CW]
        unsigned long long* hs = tsm + CH * CW;  // [CH][64]
        // eight loads per thread in flight before their stores
        for (int e0 = threadIdx.x; e0 < CH * CW; e0 += 8 * 256) {
            unsigned long long v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int e = e0 + 256 * u;
                const int r = e / CW, c = e - r * CW;
                const int py = cy0 + r, px = cx0 + c;
                v[u] = e < CH * CW && py >= 0 && px >= 0 && py < jb.height && px < jb.width
                           ? jb.corners[static_cast<size_t>(py) * jb.width + px]
                           : 0ull;
            }
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (e0 + 256 * u < CH * CW) ct[e0 + 256 * u] = v[u];
        }
        __syncthreads();
        for (int e = threadIdx.x; e < CH * 64; e += 256) {
            const int row = e >> 6, x = e & 63;
            const unsigned long long* cr = ct + row * CW + x;
            unsigned long long sum = 0;
            for (int b = 0; b < B; ++b) sum += cr[b];
            hs[e] = sum;
        }
        __syncthreads();
        unsigned long long* den = ct;  // [16][64]
        for (int e = threadIdx.x; e < 16 * 64; e += 256) {
            const unsigned long long* hc = hs + e;
            unsigned long long sum = 0;
            for (int a = 0; a < B; ++a) sum += hc[a * 64];
            den[e] = sum;
        }
        __syncthreads();
        const unsigned long long* dr = den + (y - by0) * 64 + (x0 - bx0);
#pragma unroll
        for (int q = 0; q < 4; ++q) dw[q] = static_cast<long long>(dr[q]);
    }
    if (x0 >= jb.width || y >= jb.height) return;
    const int xr = min(x0 + 3, jb.width - 1);
    f32x4 n = {0.f, 0.f, 0.f, 0.f}, d = {0.f, 0.f, 0.f, 0.f};
    for (int q = 0; q < jb.nsrc; ++q) {
        const TSource& src = jb.src[q];
        const TileGeom& tg = src.tiles;
        const int r = src.range;
        int txh = min(tg.ntx - 1, (xr + r) / (tg.tw * s));
        while (txh + 1 < tg.ntx && tg.ax0(txh + 1, jb.width, B, s, r) <= xr) ++txh;
        int tyh = min(tg.nty - 1, (y + r) / (tg.th * s));
        while (tyh + 1 < tg.nty && tg.ay0(tyh + 1, jb.height, B, s, r) <= y) ++tyh;
        const size_t area = static_cast<size_t>(tg.pitch) * tg.ah;
        for (int ty = tyh; ty >= 0; --ty) {
            const int oy = y - tg.ay0(ty, jb.height, B, s, r);
            if (oy >= tg.ah) break;
            for (int tx = txh; tx >= 0; --tx) {
                const int ax0 = tg.ax0(tx, jb.width, B, s, r);
                if (ax0 + tg.aw <= x0) break;
                const size_t o = (static_cast<size_t>(ty) * tg.ntx + tx) * area + static_cast<size_t>(oy) * tg.pitch +
                                 (x0 - ax0 + (ax0 & 3));
                const f32x4 pn = *reinterpret_cast<const f32x4*>(src.num + o);
                const f32x4 pd = jb.corners ? f32x4{0.f, 0.f, 0.f, 0.f} : *reinterpret_cast<const f32x4*>(src.den + o);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const bool in = static_cast<unsigned>(x0 + i - ax0) < static_cast<unsigned>(tg.aw);
                    n[i] += in ? pn[i] : 0.f;
                    d[i] += in ? pd[i] : 0.f;
                }
            }
        }
    }
    if (jb.corners)
#pragma unroll
        for (int i = 0; i < 4; ++i) d[i] = static_cast<float>(static_cast<double>(dw[i]) * (1.0 / 4294967296.0));
    float* dst = jb.dst + static_cast<size_t>(y) * jb.width;
    const float* fb = jb.fallback + static_cast<size_t>(y) * jb.width;
#pragma unroll
    for (int i = 0; i < 4; ++i)
        if (x0 + i < jb.width) dst[x0 + i] = d[i] > 1e-12f ? n[i] / d[i] : fb[x0 + i];
}

// ---------------------------------------------------------------------------
// Finish (src/cpu/bm/agg.cpp:17-42 AggFinish): dst = den > 1e-12 ? num/den : src.
// ---------------------------------------------------------------------------

// Tile path: 64 x 16 pixels per block, four consecutive pixels of a row per
// thread; per pixel, the partials of every tile whose rectangle covers it
// (tiles in descending (ty, tx) order), read as aligned vectors per tile for
// the four pixels. EXACT: the spatial path's int64 numerator partials, summed
// exactly, and the weights from the records: every patch of a reference
// whose window reaches the block adds its group's weight (gweight) at its
// top-left corner in an LDS corner tile, which is box-summed B x B; then one
// conversion and num / den in double rounded to float (the atomic path's
// formula, finish_corner_kernel). Otherwise the temporal slot partials
// (floats) in slice mode.
template <bool EXACT, int PX>
__global__ __launch_bounds__(1024 / PX) void finish_tiles_kernel(FinishTable tab) {
    extern __shared__ __align__(16) unsigned long long fsm[];
    // XCD-contiguous blocks: neighbouring blocks read the same tile partial
    // lines through one L2.
    const int lb = xcd_block();
    constexpr int nt = 1024 / PX;
    constexpr int U = PX == 1 ? 4 : 2;  // tiles' partials in flight
    const FinishJob& jb = tab.job[find_job(tab, lb)];
    const int t = lb - jb.wg_begin;
    const int bx0 = (t % jb.tiles_x) * 64, by0 = jb.py0 + (t / jb.tiles_x) * 16;
    const int x0 = bx0 + (threadIdx.x & (64 / PX - 1)) * PX;
    const int y = by0 + threadIdx.x / (64 / PX);
    const int B = jb.block, s = jb.step, r = jb.range;
    long long dw[PX] = {};  // EXACT: the weights' sums
    if constexpr (EXACT) {
        const int CW = 64 + B - 1, CH = 16 + B - 1;
        const int cx0 = bx0 - B + 1, cy0 = by0 - B + 1;  // corner tile origin
        unsigned long long* ct = fsm;                     // [CH][CW] corner weights
        unsigned long long* hs = fsm + CH * CW;           // [CH][64] horizontal B-wide sums
        for (int e = threadIdx.x; e < CH * CW; e += nt) ct[e] = 0ull;
        __syncthreads();
        // The references whose windows (reference +- range, clamped) reach
        // the corner tile, of the grid rows the records hold.
        const Grid& g = jb.grid;
        const int lx = cx0 - r, ux = bx0 + 63 + r, ly = cy0 - r, uy = by0 + 15 + r;
        const int i_lo = min(max(lx, 0) / s, g.nx - 1);
        const int i_hi = jb.width - B <= ux ? g.nx - 1 : min(g.nx - 1, ux / s);
        const int a_lo = max(max(ly, 0) / s, g.row0);
        const int a_hi = min(jb.height - B <= uy ? g.row0 + g.ny - 1 : uy / s, g.row0 + g.ny - 1);
        const int ni = i_hi - i_lo + 1, nj = a_hi - a_lo + 1;
        const int G = jb.group;
        const int pairs = ni > 0 && nj > 0 ? ni * nj * G : 0;
        // four (reference, record) pairs per thread and step, every load of
        // them issued before any is used (a reference holds G records; the
        // ones at or beyond its count are read and not used)
        for (int e0 = threadIdx.x; e0 < pairs; e0 += 4 * nt) {
            int cnt[4], kk[4], ox[4], oy[4];
            unsigned long long wgt[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int e = min(e0 + nt * u, pairs - 1);
                const int ref = e / G, k = e - ref * G;
                const int rj = ref / ni, ri = ref - rj * ni;
                const int rid = (a_lo - g.row0 + rj) * g.nx + i_lo + ri;
                cnt[u] = jb.counts[rid];
                const MatchRec m = jb.matches[static_cast<size_t>(rid) * G + k];
                wgt[u] = jb.gweight[rid];
                kk[u] = e0 + nt * u < pairs ? k : G;
                ox[u] = m.x - cx0;
                oy[u] = m.y - cy0;
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (kk[u] < cnt[u] && static_cast<unsigned>(ox[u]) < static_cast<unsigned>(CW) &&
                    static_cast<unsigned>(oy[u]) < static_cast<unsigned>(CH))
                    lds_add(ct + oy[u] * CW + ox[u], wgt[u]);
        }
        __syncthreads();
        // hs[row][x] = sum of ct[row][x .. x + B - 1], then the B-high sums
        // into the corner tile's area, den[yr][x]: a wave's lanes take 64
        // consecutive x of one row (bank-conflict-free reads and writes)
        for (int e = threadIdx.x; e < CH * 64; e += nt) {
            const int row = e >> 6, x = e & 63;
            const unsigned long long* cr = ct + row * CW + x;
            unsigned long long sum = 0;
            for (int b = 0; b < B; ++b) sum += cr[b];
            hs[e] = sum;
        }
        __syncthreads();
        unsigned long long* den = ct;  // [16][64]
        for (int e = threadIdx.x; e < 16 * 64; e += nt) {
            const unsigned long long* hc = hs + e;
            unsigned long long sum = 0;
            for (int a = 0; a < B; ++a) sum += hc[a * 64];
            den[e] = sum;
        }
        __syncthreads();
        // the weight at (x, y): corners (x - B + 1 .. x, y - B + 1 .. y)
        const unsigned long long* dr = den + (y - by0) * 64 + (x0 - bx0);
#pragma unroll
        for (int q = 0; q < PX; ++q) dw[q] = static_cast<long long>(dr[q]);
    }
    if (x0 >= jb.width || y >= jb.height) return;
    const TileGeom& tg = jb.tiles;
    const int xr = min(x0 + PX - 1, jb.width - 1);
    int txh = min(tg.ntx - 1, (xr + r) / (tg.tw * s));
    while (txh + 1 < tg.ntx && tg.ax0(txh + 1, jb.width, B, s, r) <= xr) ++txh;
    int tyh = min(tg.nty - 1, (y + r) / (tg.th * s));
    while (tyh + 1 < tg.nty && tg.ay0(tyh + 1, jb.height, B, s, r) <= y) ++tyh;
    // a batch of tile rows: only its tiles, at partials index ty - ty0
    const bool batch = EXACT && jb.acc_num;
    const int ty_lo = batch ? jb.ty0 : 0;
    if (batch) tyh = min(tyh, jb.ty1 - 1);
    using Acc = typename std::conditional<EXACT, long long, float>::type;
    Acc n[PX] = {}, d[PX] = {};
    const size_t area = static_cast<size_t>(tg.pitch) * tg.ah;
    // The covering tiles are the rectangle [tyl, tyh] x [txl, txh]; walked
    // in descending (ty, tx) order, U tiles' partials are loaded before any is
    // added, so their memory latencies overlap (four at a time with four pixels
    // each need 106 VGPRs and ran slower).
    int tyl = tyh + 1;
    while (tyl - 1 >= ty_lo && y - tg.ay0(tyl - 1, jb.height, B, s, r) < tg.ah) --tyl;
    int txl = txh + 1;
    while (txl - 1 >= 0 && tg.ax0(txl - 1, jb.width, B, s, r) + tg.aw > x0) --txl;
    const int nx = txh - txl + 1;
    const int count = tyl <= tyh ? (tyh - tyl + 1) * nx : 0;
    for (int k0 = 0; k0 < count; k0 += U) {
        Acc pn[U][PX], pd[U][PX];
        int lo[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int k = k0 + u;
            lo[u] = x0 + PX;  // no pixel inside
#pragma unroll
            for (int i = 0; i < PX; ++i) pn[u][i] = pd[u][i] = Acc(0);
            if (k < count) {
                const int ty = tyh - k / nx, tx = txh - k % nx;
                const int oy = y - tg.ay0(ty, jb.height, B, s, r);
                const int ax0 = tg.ax0(tx, jb.width, B, s, r);
                lo[u] = ax0;
                // column of x0: a multiple of PX in [0, pitch - PX]
                const size_t o = (static_cast<size_t>(ty - ty_lo) * tg.ntx + tx) * area +
                                 static_cast<size_t>(oy) * tg.pitch + (x0 - ax0 + (ax0 & 3));
                if constexpr (EXACT && PX == 1) {
                    pn[u][0] = static_cast<long long>(jb.exact_num[o]);
                } else if constexpr (EXACT) {
                    const longlong2* qn =
                        static_cast<const longlong2*>(__builtin_assume_aligned(jb.exact_num + o, 32));
                    const longlong2 n0 = qn[0], n1 = qn[1];
                    pn[u][0] = n0.x, pn[u][1] = n0.y, pn[u][2] = n1.x, pn[u][3] = n1.y;
                } else {
                    const f32x4 vn = *reinterpret_cast<const f32x4*>(jb.part_num + o);
                    const f32x4 vd = *reinterpret_cast<const f32x4*>(jb.part_den + o);
#pragma unroll
                    for (int i = 0; i < PX; ++i) pn[u][i] = vn[i], pd[u][i] = vd[i];
                }
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < PX; ++i) {
                const bool in = k0 + u < count && static_cast<unsigned>(x0 + i - lo[u]) < static_cast<unsigned>(tg.aw);
                n[i] += in ? pn[u][i] : Acc(0);
                d[i] += in ? pd[u][i] : Acc(0);
            }
    }
    if constexpr (EXACT) {
#pragma unroll
        for (int i = 0; i < PX; ++i) d[i] = dw[i];
        if (batch) {
            long long* an = jb.acc_num + static_cast<size_t>(y) * jb.width;
            long long* ad = jb.acc_den + static_cast<size_t>(y) * jb.width;
#pragma unroll
            for (int i = 0; i < PX; ++i)
                if (x0 + i < jb.width) {
                    an[x0 + i] += n[i];
                    ad[x0 + i] += d[i];
                }
            return;
        }
    }
    float* dst = jb.dst + static_cast<size_t>(y) * jb.dstride;
    if (jb.dst_den) {
        float* dd = jb.dst_den + static_cast<size_t>(y) * jb.dstride;
#pragma unroll
        for (int i = 0; i < PX; ++i)
            if (x0 + i < jb.width) {
                if constexpr (EXACT) {
                    dst[x0 + i] = static_cast<float>(static_cast<double>(n[i]) * (1.0 / 4294967296.0));
                    dd[x0 + i] = static_cast<float>(static_cast<double>(d[i]) * (1.0 / 4294967296.0));
                } else {
                    dst[x0 + i] = n[i];
                    dd[x0 + i] = d[i];
                }
            }
        return;
    }
    const float* src = jb.src + static_cast<size_t>(y) * jb.sstride;
#pragma unroll
    for (int i = 0; i < PX; ++i)
        if (x0 + i < jb.width) {
            if constexpr (EXACT)
                dst[x0 + i] = d[i] > 0 ? static_cast<float>(static_cast<double>(n[i]) / static_cast<double>(d[i]))
                                       : src[x0 + i];
            else
                dst[x0 + i] = d[i] > 1e-12f ? n[i] / d[i] : src[x0 + i];
        }
}

// Atomic path: den kept at each patch's top-left corner, box-summed here.
template <int B>
__global__ __launch_bounds__(256) void finish_corner_kernel(FinishTable tab) {
    constexpr int T = 16;
    constexpr int TS = T + B - 1;
    __shared__ unsigned long long corner[TS * TS];
    __shared__ unsigned long long colsum[T * TS];
    const int lb = xcd_block();
    const FinishJob& jb = tab.job[find_job(tab, lb)];
    const int tile = lb - jb.wg_begin;
    const int x0 = (tile % jb.tiles_x) * T, y0 = (tile / jb.tiles_x) * T;
    const int tid = threadIdx.x;
    for (int e = tid; e < TS * TS; e += 256) {
        const int yy = e / TS, xx = e - (e / TS) * TS;
        const int gy = y0 - (B - 1) + yy, gx = x0 - (B - 1) + xx;
        corner[e] = (gy >= 0 && gx >= 0 && gy < jb.height && gx < jb.width)
                        ? jb.den[static_cast<size_t>(gy) * jb.width + gx]
                        : 0ull;
    }
    __syncthreads();
    for (int e = tid; e < T * TS; e += 256) {
        const int oy = e / TS, xx = e - (e / TS) * TS;
        unsigned long long s = 0;
#pragma unroll
        for (int i = 0; i < B; ++i) s += corner[(oy + i) * TS + xx];
        colsum[e] = s;
    }
    __syncthreads();
    const int oy = tid / T, ox = tid % T;
    const int y = y0 + oy, x = x0 + ox;
    if (y < jb.height && x < jb.width) {
        unsigned long long d = 0;
#pragma unroll
        for (int i = 0; i < B; ++i) d += colsum[oy * TS + ox + i];
        const long long n = static_cast<long long>(jb.num[static_cast<size_t>(y) * jb.width + x]);
        const long long dd = static_cast<long long>(d);
        if (jb.dst_den) {
            jb.dst[static_cast<size_t>(y) * jb.dstride + x] =
                static_cast<float>(static_cast<double>(n) * (1.0 / 4294967296.0));
            jb.dst_den[static_cast<size_t>(y) * jb.dstride + x] =
                static_cast<float>(static_cast<double>(dd) * (1.0 / 4294967296.0));
            return;
        }
        jb.dst[static_cast<size_t>(y) * jb.dstride + x] =
            dd > 0 ? static_cast<float>(static_cast<double>(n) / static_cast<double>(dd))
                   : jb.src[static_cast<size_t>(y) * jb.sstride + x];
    }
}

// The output from frame-sized exact sums with the den per pixel (the
// memory-limited plan's tile buckets, whose batches added their partials
// into acc_num / acc_den): the division of finish_tiles_kernel. 64 x 4
// pixels per block.
__global__ __launch_bounds__(256) void finish_sums_kernel(FinishTable tab) {
    const int lb = xcd_block();
    const FinishJob& jb = tab.job[find_job(tab, lb)];
    const int t = lb - jb.wg_begin;
    const int x = (t % jb.tiles_x) * 64 + (threadIdx.x & 63);
    const int y = (t / jb.tiles_x) * 4 + (threadIdx.x >> 6);
    if (x >= jb.width || y >= jb.height) return;
    const size_t o = static_cast<size_t>(y) * jb.width + x;
    const long long n = jb.acc_num[o], d = jb.acc_den[o];
    jb.dst[static_cast<size_t>(y) * jb.dstride + x] =
        d > 0 ? static_cast<float>(static_cast<double>(n) / static_cast<double>(d))
              : jb.src[static_cast<size_t>(y) * jb.sstride + x];
}

// nss.VAggregate's reduction of one plane (src/cpu/bm/agg.cpp:159-201
// vaggregate_target): sum(num) / sum(den) over the contributions in their
// order, the source where sum(den) <= 1e-12. 64 x 4 pixels per block.
__global__ __launch_bounds__(256) void vaggregate_kernel(VAggJob jb) {
    const int x = blockIdx.x * 64 + (threadIdx.x & 63);
    const int y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= jb.width || y >= jb.height) return;
    float n = 0.f, d = 0.f;
    for (int k = 0; k < jb.count; ++k) {
        const size_t o = static_cast<size_t>(y) * jb.stride[k] + x;
        n += jb.num[k][o];
        d += jb.den[k][o];
    }
    jb.dst[static_cast<size_t>(y) * jb.dstride + x] =
        d > 1e-12f ? n / d : jb.src[static_cast<size_t>(y) * jb.sstride + x];
}

hipError_t launch_vaggregate(const VAggJob& jb, hipStream_t s) {
    if (launch_fault()) return hipErrorLaunchFailure;
    const dim3 grid((jb.width + 63) / 64, (jb.height + 3) / 4);
    vaggregate_kernel<<<grid, 256, 0, s>>>(jb);
    return hipGetLastError();
}

__global__ __launch_bounds__(256) void zero_kernel(ZeroTable tab) {
    const ZeroJob& jb = tab.job[find_job(tab, static_cast<int>(blockIdx.x))];
    const long long base = static_cast<long long>(static_cast<int>(blockIdx.x) - jb.wg_begin) * 1024;
    for (int i = threadIdx.x; i < 1024; i += 256) {
        const long long o = base + i;
        if (o < jb.count) jb.p[o] = 0ull;
    }
}

// ---------------------------------------------------------------------------
// WNNM: weighted nuclear-norm shrinkage of each group (src/cpu/wnnm/shrink.cpp:13-49,
// src/cpu/finishers.hpp:12-36, src/cpu/common/sv_shrink.cpp:9-24). The group
// matrix A has m = B^2 rows and k matched patches as columns, optionally
// centred row by row. Its spectrum comes from the k x k Gram matrix
// A^T A = V diag(s^2) V^T by cyclic Jacobi in round-robin order: every round
// rotates N/2 disjoint index pairs, so the whole N x N matrix updates at once,
// one entry per lane and step. The shrunk group is X = A V diag(s'/s) V^T
// (the product src/cpu/batch.cpp:490-520 forms), added back to the centre.
// ---------------------------------------------------------------------------
inline constexpr int kWnnmSweeps = 16;
// A pair rotates while |g_pq| > tol sqrt(g_pp g_qq) (src/cpu/wnnm/numerics.hpp:10)
// and |g_pq| is above FP32 rounding noise of the matrix, floor * trace: a
// rotation leaves g_pq at a few ulps of the largest entries, which the
// relative test alone can keep seeing for a pair of a large and a tiny
// eigenvalue. An off-diagonal at the floor moves the eigenvalues by about
// g_pq^2 / gap.
inline constexpr float kWnnmTol = 1e-6f;
inline constexpr float kWnnmFloor = 0x1p-21f;

// Round r of the round-robin pairing of the first n indices (n even):
// n - 1 is paired with r, and i with (2r - i) mod (n - 1) otherwise; over
// r = 0 .. n - 2 every pair meets once. Indices from n on pair with
// themselves. The schedule depends on the group's own column count only, so
// a group gives the same bits whatever size it is padded to.
__device__ inline int rr_partner(int i, int r, int n) {
    if (i >= n) return i;
    if (i == n - 1) return r;
    if (i == r) return n - 1;
    int j = 2 * r - i;
    if (j < 0) j += n - 1;
    else if (j >= n - 1) j -= n - 1;
    return j;
}

// One wave per reference. N = 8, 16 or 32 >= group; indices k .. N - 1 are
// zero columns that never rotate. LDS: A (N columns of m + 1) | Gram, later
// the shrink operator W (N x N + 1) | V (N x N + 1) | per-index rotation
// coefficients, diagonal steps (later the singular values) and gains.
template <int N, bool NCSR>
__device__ __forceinline__ void gram_group_body(const WnnmTable& tab) {
    extern __shared__ __align__(16) float wn[];
    constexpr int GP = N + 1;
    constexpr int E = N * N / 64;
    constexpr int LOG_N = N == 8 ? 3 : N == 16 ? 4 : 5;
    const int lane = threadIdx.x;
    const int lb = xcd_block();
    const WnnmJob& jb = tab.job[find_job(tab, lb)];
    const int g = lb - jb.wg_begin;
    if (g >= jb.nref) return;
    const int k = min(jb.counts[g], N);
    if (k <= 0) return;
    const int B = jb.block, m = B * B, P = m + 1;
    const MatchRec* rec = jb.matches + static_cast<size_t>(g) * jb.group;
    float* A = wn;
    float* G = A + N * P;
    float* V = G + N * GP;
    float* cself = V + N * GP;
    float* cpart = cself + N;
    float* tstep = cpart + N;
    float* gain = tstep + N;

    // The lane's pixels e = lane + 64 q of a patch (m <= 256).
    int soff[4], noff[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int e = lane + 64 * q, ey = e / B, ex = e - ey * B;
        soff[q] = ey * jb.stride + ex;
        noff[q] = ey * jb.width + ex;
    }
    for (int j = 0; j < N; ++j) {
        if (j < k) {
            const float* plane = jb.temporal ? jb.ring.frame(jb.slots.frame(rec[j].t)) : jb.src;
            const float* base = plane + static_cast<size_t>(rec[j].y) * jb.stride + rec[j].x;
            float v[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) v[q] = lane + 64 * q < m ? base[soff[q]] : 0.f;
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (lane + 64 * q < m) A[j * P + lane + 64 * q] = v[q];
        } else {
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (lane + 64 * q < m) A[j * P + lane + 64 * q] = 0.f;
        }
    }
    // Row centring (src/cpu/common/group_center.cpp:15-58): the mean of each
    // pixel over the k patches, subtracted; only the lane's own rows.
    float mean[4] = {0.f, 0.f, 0.f, 0.f};
    if (jb.residual) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int e = lane + 64 * q;
            if (e < m) {
                float sum = 0.f;
                for (int j = 0; j < k; ++j) sum += A[j * P + e];
                mean[q] = sum / static_cast<float>(k);
                for (int j = 0; j < k; ++j) A[j * P + e] -= mean[q];
            }
        }
    }
    __syncthreads();

    // Gram matrix and V = I. G[a][b] and G[b][a] take the same fmaf chain,
    // so the matrix starts exactly symmetric.
#pragma unroll
    for (int t = 0; t < E; ++t) {
        const int idx = lane + 64 * t, a = idx >> LOG_N, b = idx & (N - 1);
        float acc = 0.f;
        if (a < k && b < k)
            for (int r = 0; r < m; ++r) acc = fmaf(A[a * P + r], A[b * P + r], acc);
        G[a * GP + b] = acc;
        V[a * GP + b] = a == b ? 1.f : 0.f;
    }
    __syncthreads();
    float trace = 0.f;
    for (int j = 0; j < k; ++j) trace += G[j * GP + j];
    const float floor_abs = kWnnmFloor * trace;

    const int ke = k + (k & 1);  // the schedule's size: k rounded up to even
    if constexpr (N == 8) {
        // One entry per lane, in registers: lane (a, b) = 8a + b holds G[a][b]
        // and V[a][b]; the same rotations as the LDS form below, with the
        // neighbours' entries read across lanes (ds_bpermute) and no barriers.
        // Each lane forms its row index's rotation; column b's is row b's.
        const int a = lane >> 3, b = lane & 7;
        float g = G[a * GP + b], v = a == b ? 1.f : 0.f;
        for (int sweep = 0; sweep < kWnnmSweeps; ++sweep) {
            bool rotated = false;
            for (int r = 0; r < ke - 1; ++r) {
                const int pa = rr_partner(a, r, ke), pb = rr_partner(b, r, ke);
                const int p0 = min(a, pa), q0 = max(a, pa);
                const float app = __shfl(g, p0 * 9, 64), aqq = __shfl(g, q0 * 9, 64);
                const float apq = __shfl(g, p0 * 8 + q0, 64);
                float c = 1.f, sn = 0.f, tn = 0.f;
                bool rot = false;
                if (q0 < k && fabsf(apq) > floor_abs && apq * apq > kWnnmTol * kWnnmTol * fabsf(app * aqq)) {
                    const float delta = (aqq - app) * 0.5f;
                    const float root = __builtin_amdgcn_sqrtf(fmaf(delta, delta, apq * apq));
                    tn = apq * __builtin_amdgcn_rcpf(delta + copysignf(root, delta));
                    c = __builtin_amdgcn_rsqf(fmaf(tn, tn, 1.f));
                    sn = tn * c;
                    rot = true;
                }
                if (!__any(rot)) continue;
                rotated = true;
                const float ca = c, sa = a == p0 ? -sn : sn, ta = a == p0 ? -tn : tn;
                const float cb = __shfl(ca, b * 8, 64), sb = __shfl(sa, b * 8, 64);
                const float g_apb = __shfl(g, a * 8 + pb, 64), v_apb = __shfl(v, a * 8 + pb, 64);
                const float g_pab = __shfl(g, pa * 8 + b, 64), g_papb = __shfl(g, pa * 8 + pb, 64);
                const float vgen = ca * fmaf(cb, g, sb * g_apb) + sa * fmaf(cb, g_pab, sb * g_papb);
                const float vdiag = fmaf(ta, g_apb, g);  // at a == b, pb == pa
                const float vpair = sa != 0.f ? 0.f : g;
                const float gn = a == b ? vdiag : (b == pa ? vpair : vgen);
                v = fmaf(cb, v, sb * v_apb);
                g = gn;
            }
            if (!rotated) break;
        }
        G[a * GP + b] = g;
        V[a * GP + b] = v;
        __syncthreads();
    } else {
    for (int sweep = 0; sweep < kWnnmSweeps; ++sweep) {
        bool rotated = false;
        for (int r = 0; r < ke - 1; ++r) {
            // Rotation of pair (p, q), p < q, zeroing g_pq: J = [c s; -s c],
            // G' = J^T G J, V' = V J, t = tan(theta) the smaller root of
            // t^2 + 2 zeta t - 1 = 0 with zeta = (g_qq - g_pp) / (2 g_pq).
            bool rot = false;
            if (lane < N) {
                const int i = lane, o = rr_partner(i, r, ke);
                const int p0 = min(i, o), q0 = max(i, o);
                float c = 1.f, sn = 0.f, tn = 0.f;
                if (q0 < k) {
                    const float app = G[p0 * GP + p0], aqq = G[q0 * GP + q0], apq = G[p0 * GP + q0];
                    // |g_pq| > tol sqrt(g_pp g_qq), squared. Gram entries of
                    // plane values stay far from overflow in the squares, so
                    // the tangent needs no scaling; v_rcp / v_sqrt (1 ulp)
                    // keep the rotation orthogonal to a few ulps.
                    if (fabsf(apq) > floor_abs && apq * apq > kWnnmTol * kWnnmTol * fabsf(app * aqq)) {
                        const float delta = (aqq - app) * 0.5f;
                        const float root = __builtin_amdgcn_sqrtf(fmaf(delta, delta, apq * apq));
                        tn = apq * __builtin_amdgcn_rcpf(delta + copysignf(root, delta));
                        c = __builtin_amdgcn_rsqf(fmaf(tn, tn, 1.f));
                        sn = tn * c;
                        rot = true;
                    }
                }
                cself[i] = c;
                cpart[i] = i == p0 ? -sn : sn;
                tstep[i] = i == p0 ? -tn : tn;
                rotated |= rot;
            }
            __syncthreads();
            // A round where no pair rotates leaves G and V as they are; the
            // next round's coefficients overwrite these unread.
            if (!__any(rot)) continue;
            float ng[E], nv[E];
            // A lane's entries share their column (64 is a multiple of N).
            const int b = lane & (N - 1), pb = rr_partner(b, r, ke);
            const float cb = cself[b], sb = cpart[b];
#pragma unroll
            for (int t = 0; t < E; ++t) {
                const int a = (lane + 64 * t) >> LOG_N;
                const int pa = rr_partner(a, r, ke);
                const float ca = cself[a], sa = cpart[a];
                const float gab = G[a * GP + b];
                // Selected, not branched: the three cases share the wave.
                const float vgen =
                    ca * fmaf(cb, gab, sb * G[a * GP + pb]) + sa * fmaf(cb, G[pa * GP + b], sb * G[pa * GP + pb]);
                const float vdiag = fmaf(tstep[a], G[a * GP + pa], gab);
                const float vpair = sa != 0.f ? 0.f : gab;
                ng[t] = a == b ? vdiag : (b == pa ? vpair : vgen);
                nv[t] = fmaf(cb, V[a * GP + b], sb * V[a * GP + pb]);
            }
            __syncthreads();
#pragma unroll
            for (int t = 0; t < E; ++t) {
                const int a = (lane + 64 * t) >> LOG_N;
                G[a * GP + b] = ng[t];
                V[a * GP + b] = nv[t];
            }
            __syncthreads();
        }
        if (!__any(rotated)) break;
    }
    }

    // Spectrum: s_j and its place in descending order (ties by index).
    if (lane < N) tstep[lane] = lane < k ? sqrtf(fmaxf(G[lane * GP + lane], 0.f)) : 0.f;
    if constexpr (NCSR) {
        // Column weights exp(-dist / h), h = max(2 m sigma^2, 1e-12), the
        // reference column at distance 0 (src/cpu/ncsr/centralize.cpp:60-88).
        const float sg = jb.sigma;
        const float h = fmaxf(2.f * static_cast<float>(m) * sg * sg, 1e-12f);
        if (lane < N) cpart[lane] = lane < k ? expf(-(lane > 0 ? __uint_as_float(rec[lane].dist) : 0.f) / h) : 0.f;
    }
    __syncthreads();
    int place = 0;
    if (lane < k) {
        const float sj = tstep[lane];
        for (int i = 0; i < k; ++i) {
            const float si = tstep[i];
            place += (si > sj || (si == sj && i < lane)) ? 1 : 0;
        }
    }
    const int rank = min(m, k);
    int kept = 0;
    if constexpr (NCSR) {
        // Code row i of the centred group's PCA, b_ij = s_i V[j][i]: its
        // weighted mean beta, the second moment over the k columns about it,
        // tau = 2 sqrt(2) sigma^2 / (sqrt(moment / k) + 1e-12), the row
        // soft-thresholded about beta (src/cpu/finishers.hpp:53-80,
        // src/cpu/ncsr/centralize.cpp:90-141), kept for the rank largest
        // values with s > 0 and stored over s_i: C[i][j]. The Gram area is
        // free (the spectrum is in tstep).
        const float sg = jb.sigma;
        float wsum = 0.f;
        for (int j = 0; j < k; ++j) wsum += cpart[j];
        const bool unit = !(wsum > 0.f);
        const float inverse = 1.f / (unit ? static_cast<float>(k) : wsum);
        if (lane < k) {
            const int i = lane;
            const float si = tstep[i];
            if (!(sg > 0.f)) {
                for (int j = 0; j < k; ++j) G[i * GP + j] = V[j * GP + i];
            } else if (place < rank && si > 0.f) {
                float beta = 0.f;
                for (int j = 0; j < k; ++j) beta = fmaf(unit ? 1.f : cpart[j], si * V[j * GP + i], beta);
                beta *= inverse;
                float moment = 0.f;
                for (int j = 0; j < k; ++j) {
                    const float e = si * V[j * GP + i] - beta;
                    moment = fmaf(e, e, moment);
                }
                const float tau = 2.8284271247461903f * sg * sg / (sqrtf(moment / static_cast<float>(k)) + 1e-12f);
                const float inv_s = 1.f / si;
                for (int j = 0; j < k; ++j) {
                    const float d = si * V[j * GP + i] - beta, a = fabsf(d);
                    G[i * GP + j] = ((a > tau ? copysignf(a - tau, d) : 0.f) + beta) * inv_s;
                }
            } else {
                for (int j = 0; j < k; ++j) G[i * GP + j] = 0.f;
            }
        }
        __syncthreads();
        // M = V C (M[a][b] = sum_i V[a][i] C[i][b]), then over the Gram area.
        float mv[E];
#pragma unroll
        for (int t = 0; t < E; ++t) {
            const int idx = lane + 64 * t, a = idx >> LOG_N, b = idx & (N - 1);
            float w = 0.f;
            if (a < k && b < k)
                for (int i = 0; i < k; ++i) w = fmaf(V[a * GP + i], G[i * GP + b], w);
            mv[t] = w;
        }
        __syncthreads();
#pragma unroll
        for (int t = 0; t < E; ++t) {
            const int idx = lane + 64 * t;
            G[(idx >> LOG_N) * GP + (idx & (N - 1))] = mv[t];
        }
        __syncthreads();
    } else {
        // Places below `start` stay; later ones shrink to
        // (s + sqrt(s^2 - c)) / 2 while s^2 > c, with c = 8 sqrt(2k) sigma^2.
        bool keep = false;
        float gj = 0.f;
        if (lane < k) {
            const float sj = tstep[lane];
            const int start = min(jb.residual ? 0 : 1, rank);
            const float constant = 8.f * sqrtf(2.f * static_cast<float>(k)) * jb.sigma * jb.sigma;
            if (place < start) {
                gj = 1.f;
                keep = true;
            } else if (place < rank) {
                const float tmp = sj * sj - constant;
                if (tmp > 0.f) {
                    gj = ((sj + sqrtf(tmp)) * 0.5f) / sj;
                    keep = true;
                }
            }
        }
        if (lane < N) gain[lane] = gj;
        kept = static_cast<int>(__popcll(__ballot(keep)));
        __syncthreads();
        // W = V diag(gain) V^T over the Gram area (G is no longer read).
#pragma unroll
        for (int t = 0; t < E; ++t) {
            const int idx = lane + 64 * t, a = idx >> LOG_N, b = idx & (N - 1);
            float w = 0.f;
            if (a < k && b < k)
                for (int i = 0; i < k; ++i) w = fmaf(V[a * GP + i] * gain[i], V[b * GP + i], w);
            G[a * GP + b] = w;
        }
        __syncthreads();
    }

    // X = A W (A M for NCSR) plus the centre, weighted into the sums: WNNM
    // 1 / kept when adaptive and kept > 0, else 1 (src/cuda/wnnm/kernels.cu:84-105);
    // NCSR 1.
    const float wt = !NCSR && jb.adaptive && kept > 0 ? 1.f / static_cast<float>(kept) : 1.f;
    const unsigned long long wfix = to_fixed(wt);
    for (int j = 0; j < k; ++j) {
        const size_t slice = jb.temporal ? static_cast<size_t>(rec[j].t) * jb.sum_slot : 0;
        unsigned long long* cell = jb.num + slice + static_cast<size_t>(rec[j].y) * jb.width + rec[j].x;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int e = lane + 64 * q;
            if (e < m) {
                float x = 0.f;
                for (int i = 0; i < k; ++i) x = fmaf(A[i * P + e], G[i * GP + j], x);
                atomicAdd(cell + noff[q], to_fixed(wt * (x + mean[q])));
            }
        }
        if (lane == 0) atomicAdd(jb.den + slice + static_cast<size_t>(rec[j].y) * jb.width + rec[j].x, wfix);
    }
}

template <int N>
__global__ __launch_bounds__(64) void wnnm_group_kernel(WnnmTable tab) {
    gram_group_body<N, false>(tab);
}

// NCSR on the same eigenbasis (src/cuda/ncsr/kernels.cu:48-190): the rows
// are always centred and the shrink works on the code rows.
template <int N>
__global__ __launch_bounds__(64) void ncsr_group_kernel(WnnmTable tab) {
    gram_group_body<N, true>(tab);
}

// ---------------------------------------------------------------------------
// Spatial planes of full groups of 8 or 16 blocks of 8 (m = 64, k = N): the
// arithmetic of gram_group_body, operation for operation (the outputs keep
// their bits), 64 / N groups to a wave, in registers and on the matrix cores,
// and the sums of a tile of references in LDS.
//   unit     16 columns: one group of 16, or two of 8 (column c of group
//            c >> 3). Four units per wave.
//   MFMA     v_mfma_f32_16x16x4_f32 sums its four products as a chain of
//            fused multiply-adds in index order (checked bit for bit against
//            fmaf chains), so the Gram matrix, the column sums of the
//            centring, W = V diag(g) V^T (NCSR: V C) and X = A W are MFMAs
//            with the results of the scalar loops. At N = 8 a product over
//            columns sums each group's columns (steps s of group s >> 1) in an
//            accumulator of its own: a neighbour's infinity or NaN stays there.
//   pixels   lane (kq, n) = 16 kq + n holds pixel 16 t + n of column 4 s + kq:
//            the B operand of X, and row 4 kq + s of its result is made
//            column 4 s + kq, so the sums' cells are the gather's. The Gram
//            operands (column on n, pixel 4 s + kq) go through LDS. X gathers
//            the pixels again (they are in L1 / L2): holding 64 registers of
//            them through the rounds would halve the waves per SIMD.
//   Jacobi   lane i of a group holds row i of G and V, the diagonal apart. A
//            round's pairs are static, so the column rotations are register
//            operations with the pair's coefficients broadcast (DPP
//            row_newbcast, or a swizzle at N = 8); the row rotations read the
//            partner's row (ds_bpermute). No barriers and no LDS addressing.
//   sums     the tile's int64 numerators in LDS and one weight per group, as
//            filter_tile_b8_kernel writes them for finish_tiles_kernel. With
//            device atomics the kernel is bound by them whatever computes the
//            groups (77 G/s: 218 us for the 16.6 M of 32 400 groups of 8).
// Measured on a 1080p plane (MI355X; gram_group_body with its atomics before):
// groups of 8, step 8 (32 400): 215 -> 59 us, NCSR 225 -> 67 us; groups of 16,
// step 4 (128 855): 3 732 -> 984 us. There VALU issue in the rounds bounds it: 17
// k instructions per wave, 1.04 of the two a CU can issue per cycle, 19 % of the
// wave cycles waiting. The smaller launch holds four waves per SIMD and waits a
// third of its cycles. The selects' masks
// take all scalar registers at groups of 16: 25 (NCSR 26) of them spill, and the
// WNNM kernel keeps 36 bytes of scratch per lane.
// ---------------------------------------------------------------------------

// rr_partner for a full group.
template <int N>
__host__ __device__ constexpr int rr_pair(int i, int r) {
    if (i == N - 1) return r;
    if (i == r) return N - 1;
    return (2 * r - i + N - 1) % (N - 1);
}

// v of lane P of the caller's group of N lanes.
template <int N, int P>
__device__ __forceinline__ float group_lane_f32(float v) {
    if constexpr (N == 16)
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + P, 0xf, 0xf, true));
    else
        return __int_as_float(__builtin_amdgcn_ds_swizzle(__float_as_int(v), 0x18 | (P << 5)));
}

// Round R of a sweep over the lanes' rows g, v and diagonal d; oi the lane's
// row, lane4 and partner4 its lane and its partner's, times four. False, and nothing changed,
// when no pair of the wave rotates.
template <int N, int R>
__device__ __forceinline__ bool jacobi_round(float (&g)[N], float (&v)[N], float& d, int oi, int lane4, int partner4,
                                             float floor_abs) {
    auto from_partner = [&](float x) {
        return __int_as_float(__builtin_amdgcn_ds_bpermute(partner4, __float_as_int(x)));
    };
    float own = g[rr_pair<N>(0, R)];  // G[i][partner]
#pragma unroll
    for (int j = 1; j < N; ++j) own = oi == j ? g[rr_pair<N>(j, R)] : own;
    const float dp = from_partner(d), other = from_partner(own);
    // the lane of the smaller index is p (g_pp, g_pq), the other q
    const bool low = lane4 < partner4;
    const float apq = low ? own : other, app = low ? d : dp, aqq = low ? dp : d;
    const float apq2 = apq * apq;
    const bool rot = fabsf(apq) > floor_abs && apq2 > kWnnmTol * kWnnmTol * fabsf(app * aqq);
    if (!__any(rot)) return false;
    const float delta = (aqq - app) * 0.5f;
    const float root = __builtin_amdgcn_sqrtf(fmaf(delta, delta, apq2));
    float tn = apq * __builtin_amdgcn_rcpf(delta + copysignf(root, delta));
    float c = __builtin_amdgcn_rsqf(fmaf(tn, tn, 1.f));
    float sn = tn * c;
    c = rot ? c : 1.f;
    sn = rot ? sn : 0.f;
    tn = rot ? tn : 0.f;
    const float sa = low ? -sn : sn, ta = low ? -tn : tn;
    float t[N];
    static_for<N>([&](auto pc) {
        constexpr int p = decltype(pc)::value, q = rr_pair<N>(p, R);
        if constexpr (p < q) {
            const float cb = group_lane_f32<N, p>(c), sb = group_lane_f32<N, p>(sa);
            const float g0 = g[p], g1 = g[q], v0 = v[p], v1 = v[q];
            t[p] = fmaf(cb, g0, sb * g1);
            t[q] = fmaf(cb, g1, -(sb * g0));
            v[p] = fmaf(cb, v0, sb * v1);
            v[q] = fmaf(cb, v1, -(sb * v0));
        }
    });
    const float pair = sa != 0.f ? 0.f : own;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        const float x = fmaf(c, t[j], sa * from_partner(t[j]));
        g[j] = oi == rr_pair<N>(j, R) ? pair : x;
    }
    d = fmaf(ta, own, d);
    return true;
}

// Floats of a wave's scratch: the unit matrices, a unit's half columns (NCSR:
// the code rows of all units) and two vectors.
inline constexpr int kGramP = 17;   // pitch of a unit's matrices
inline constexpr int kGramPx = 44;  // pitch of a half column's 32 pixels: both operand reads spread over the banks
inline constexpr int kGramMat = 4 * 16 * kGramP;
inline constexpr int kGramScratch = 2 * kGramMat + 128;

// One workgroup of four waves per tile of at most 4 (64 / N) references. LDS:
// the waves' scratch, then (over it) the tile's numerator sums.
template <int N, bool NCSR>
__global__ __launch_bounds__(256, 4) void gram_group_tile_kernel(WnnmTable tab) {
    extern __shared__ __align__(16) unsigned long long acc[];
    constexpr int GW = 64 / N;   // groups of a wave
    constexpr int HN = 16 / N;   // groups of a unit
    constexpr int P = kGramP, PX = kGramPx;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, n = lane & 15, kq = lane >> 4;
    const int lb = xcd_block();
    const WnnmJob& jb = tab.job[find_job(tab, lb)];
    const TileGeom& tg = jb.tiles;
    const int tile = lb - jb.wg_begin, tx = tile % tg.ntx, ty = tile / tg.ntx;
    const int aw = tg.aw, ah = tg.ah;
    const int ax0 = tg.ax0(tx, jb.width, 8, jb.grid.step, jb.range);
    const int ay0 = tg.ay0(ty, jb.height, 8, jb.grid.step, jb.range);
    const int i_begin = tx * tg.tw, j_begin = ty * tg.th;
    const int ni = min(tg.tw, jb.grid.nx - i_begin), ngroups = ni * min(tg.th, jb.grid.ny - j_begin);
    const int g0 = wave * GW;
    float* mat = reinterpret_cast<float*>(acc) + wave * kGramScratch;  // Gram, then V, then W
    float* px = mat + kGramMat;
    float* vec = px + kGramMat;
    float* vec2 = vec + 64;
    // Group (of the tile) of column c of unit u; groups past the tile's last
    // repeat it and add nothing.
    auto group_of = [&](int u, int c) { return g0 + u * HN + c / N; };
    auto ref_of = [&](int g) {
        const int q = min(g, ngroups - 1), gj = q / ni;
        return (j_begin + gj) * jb.grid.nx + i_begin + (q - gj * ni);
    };
    auto record = [&](int u, int c) {
        return jb.matches[static_cast<size_t>(ref_of(group_of(u, c))) * N + c % N];
    };
    // Pixel 16 t + n of columns 4 s + kq of a unit.
    auto gather = [&](const MatchRec (&rec)[4], float (&b)[4][4]) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const float* p = jb.src + static_cast<size_t>(rec[s].y + (n >> 3)) * jb.stride + rec[s].x + (n & 7);
#pragma unroll
            for (int t = 0; t < 4; ++t) b[t][s] = p[static_cast<size_t>(2 * t) * jb.stride];
        }
    };
    // Row centring (src/cpu/common/group_center.cpp:15-58) of one pixel tile:
    // a row of ones times the columns sums them in order (every row of the
    // result is alike); the means (0 without centring) are subtracted.
    auto centre = [&](float (&b)[4], float (&mu)[HN]) {
#pragma unroll
        for (int h = 0; h < HN; ++h) mu[h] = 0.f;
        if (!jb.residual) return;
        f32x4 sum[HN];
#pragma unroll
        for (int h = 0; h < HN; ++h) sum[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < 4; ++s)
            sum[4 * s / N] = __builtin_amdgcn_mfma_f32_16x16x4f32(1.f, b[s], sum[4 * s / N], 0, 0, 0);
#pragma unroll
        for (int h = 0; h < HN; ++h) mu[h] = sum[h][0] * (1.f / N);
#pragma unroll
        for (int s = 0; s < 4; ++s) b[s] -= mu[4 * s / N];
    };

    float wt = 1.f;    // of the lane's group
    float wv[4][4];    // W's A operand: rows 4 s + kq, column orow
    const int orow = 4 * (n & 3) + (n >> 2);
    if (g0 < ngroups) {
        {
            MatchRec rec[4][4];
            float b[4][4][4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int s = 0; s < 4; ++s) rec[u][s] = record(u, 4 * s + kq);
#pragma unroll
            for (int u = 0; u < 4; ++u) gather(rec[u], b[u]);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                f32x4 gram = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int half = 0; half < 2; ++half) {
#pragma unroll
                    for (int t = 0; t < 2; ++t) {
                        float mu[HN];
                        centre(b[u][2 * half + t], mu);
#pragma unroll
                        for (int s = 0; s < 4; ++s) px[(4 * s + kq) * PX + 16 * t + n] = b[u][2 * half + t][s];
                    }
                    wave_sync();
#pragma unroll
                    for (int s = 0; s < 8; ++s) {
                        const float x = px[n * PX + 4 * s + kq];
                        gram = __builtin_amdgcn_mfma_f32_16x16x4f32(x, x, gram, 0, 0, 0);
                    }
                    wave_sync();
                }
#pragma unroll
                for (int j = 0; j < 4; ++j) mat[u * 16 * P + (4 * kq + j) * P + n] = gram[j];
            }
            wave_sync();
        }

        // Jacobi: lane = (group, row).
        const int oi = lane & (N - 1), base = lane & ~(N - 1);
        float* row = mat + lane / 16 * (16 * P) + (lane & 15) * P + (lane & 15 & ~(N - 1));
        float d = 0.f;
        {
            float g[N], v[N];
            float trace = 0.f;
#pragma unroll
            for (int j = 0; j < N; ++j) {
                g[j] = row[j];
                v[j] = oi == j ? 1.f : 0.f;
                d = oi == j ? g[j] : d;
            }
            static_for<N>([&](auto jc) { trace += group_lane_f32<N, decltype(jc)::value>(d); });
            const float floor_abs = kWnnmFloor * trace;
            // A group whose trace is not finite never rotates; where a
            // neighbour in the wave does, its rows are put back below.
            const bool frozen = !(fabsf(floor_abs) < __builtin_inff());
            const float d0 = d;
            uint32_t partners[(N + 2) / 4];
#pragma unroll
            for (int r = 0; r < N - 1; ++r) {
                const uint32_t at = static_cast<uint32_t>(base | rr_partner(oi, r, N)) << (8 * (r & 3));
                partners[r >> 2] = (r & 3) == 0 ? at : partners[r >> 2] | at;
            }
            for (int sweep = 0; sweep < kWnnmSweeps; ++sweep) {
                bool rotated = false;
                static_for<N - 1>([&](auto rc) {
                    constexpr int r = decltype(rc)::value;
                    const int partner4 = static_cast<int>((partners[r >> 2] >> (8 * (r & 3))) & 63u) << 2;
                    rotated |= jacobi_round<N, r>(g, v, d, oi, lane << 2, partner4, floor_abs);
                });
                if (!rotated) break;
            }
            d = frozen ? d0 : d;
#pragma unroll
            for (int j = 0; j < N; ++j) row[j] = frozen ? (oi == j ? 1.f : 0.f) : v[j];
        }

        // Spectrum: s_j, lane = eigenvalue.
        const float sj = sqrtf(fmaxf(d, 0.f));
        vec[lane] = sj;
        // sums over the unit's indices l = 4 s + kq, a group's steps apart;
        // the rows 4 kq + j of the result from their own group's sums
        auto product = [&](auto left, auto right) {
            f32x4 sum[HN];
#pragma unroll
            for (int h = 0; h < HN; ++h) sum[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < 4; ++s)
                sum[4 * s / N] =
                    __builtin_amdgcn_mfma_f32_16x16x4f32(left(4 * s + kq), right(4 * s + kq), sum[4 * s / N], 0, 0, 0);
            f32x4 out = sum[0];
            if constexpr (HN == 2)
#pragma unroll
                for (int j = 0; j < 4; ++j) out[j] = kq >= 2 ? sum[1][j] : sum[0][j];
            return out;
        };
        if constexpr (NCSR) {
            // beta is rounded before it is added, as there
#pragma clang fp contract(off)
            // The code rows of gram_group_body, C[i][j] over s_i, into px.
            const float sg = jb.sigma;
            const float h = fmaxf(2.f * 64.f * sg * sg, 1e-12f);
            vec2[lane] = expf(-(oi > 0 ? __uint_as_float(record(lane >> 4, lane & 15).dist) : 0.f) / h);
            wave_sync();
            float wsum = 0.f;
#pragma unroll
            for (int j = 0; j < N; ++j) wsum += vec2[base + j];
            const bool unit = !(wsum > 0.f);
            const float inverse = 1.f / (unit ? static_cast<float>(N) : wsum);
            const float* vcol = mat + lane / 16 * (16 * P) + (lane & 15 & ~(N - 1)) * P + (lane & 15);
            float code[N], beta = 0.f, moment = 0.f;
#pragma unroll
            for (int j = 0; j < N; ++j) {
                code[j] = vcol[j * P];
                beta = fmaf(unit ? 1.f : vec2[base + j], sj * code[j], beta);
            }
            beta *= inverse;
#pragma unroll
            for (int j = 0; j < N; ++j) {
                const float e = fmaf(sj, code[j], -beta);
                moment = fmaf(e, e, moment);
            }
            const float tau = 2.8284271247461903f * sg * sg / (sqrtf(moment / static_cast<float>(N)) + 1e-12f);
            const float inv_s = 1.f / sj;
            float* crow = px + lane / 16 * (16 * P) + (lane & 15) * P + (lane & 15 & ~(N - 1));
#pragma unroll
            for (int j = 0; j < N; ++j) {
                const float e = fmaf(sj, code[j], -beta), ae = fabsf(e);
                const float x = ((ae > tau ? copysignf(ae - tau, e) : 0.f) + beta) * inv_s;
                crow[j] = !(sg > 0.f) ? code[j] : sj > 0.f ? x : 0.f;
            }
            wave_sync();
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float* vu = mat + u * 16 * P + n * P;
                const float* cu = px + u * 16 * P + n;
                const f32x4 m = product([&](int l) { return vu[l]; }, [&](int l) { return cu[l * P]; });
                wave_sync();
#pragma unroll
                for (int j = 0; j < 4; ++j) mat[u * 16 * P + (4 * kq + j) * P + n] = m[j];
            }
        } else {
            // Gains of gram_group_body; only the first place matters there.
            wave_sync();
            bool keep = false;
            float gj = 0.f;
            if (!jb.residual) {
                int place = 0;
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    const float si = vec[base + i];
                    place += (si > sj || (si == sj && i < oi)) ? 1 : 0;
                }
                keep = place == 0;
                gj = keep ? 1.f : 0.f;
            }
            const float constant = 8.f * sqrtf(2.f * static_cast<float>(N)) * jb.sigma * jb.sigma;
            const float tmp = fmaf(sj, sj, -constant);
            if (!keep && tmp > 0.f) {
                gj = ((sj + sqrtf(tmp)) * 0.5f) / sj;
                keep = true;
            }
            const int kept = __popc(static_cast<uint32_t>(__ballot(keep) >> base) & ((1u << N) - 1u));
            wt = jb.adaptive && kept > 0 ? 1.f / static_cast<float>(kept) : 1.f;
            vec2[lane] = gj;
            wave_sync();
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float* vu = mat + u * 16 * P + n * P;
                const float* gu = vec2 + u * 16;
                const f32x4 w = product([&](int l) { return vu[l] * gu[l]; }, [&](int l) { return vu[l]; });
                wave_sync();
#pragma unroll
                for (int j = 0; j < 4; ++j) mat[u * 16 * P + (4 * kq + j) * P + n] = w[j];
            }
        }
        wave_sync();
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int s = 0; s < 4; ++s) wv[u][s] = mat[u * 16 * P + (4 * s + kq) * P + orow];
        if (oi == 0 && g0 + lane / N < ngroups) jb.gweight[ref_of(g0 + lane / N)] = to_fixed(wt);
    }
    __syncthreads();
    for (int e = threadIdx.x; e < aw * ah; e += 256) acc[e] = 0ull;
    __syncthreads();

    // X[c][e] = sum_i W[i][c] A[i][e] plus the centre: row 4 kq + j of the
    // result is column c = 4 j + kq.
    if (g0 < ngroups) {
        MatchRec rec[4][4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int s = 0; s < 4; ++s) rec[u][s] = record(u, 4 * s + kq);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            float b[4][4];
            gather(rec[u], b);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                f32x4 x[HN];
                float mu[HN];
                centre(b[t], mu);
#pragma unroll
                for (int h = 0; h < HN; ++h) x[h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < 4; ++s)
                    x[4 * s / N] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[u][s], b[t][s], x[4 * s / N], 0, 0, 0);
                float wx[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) wx[j] = lane_f32(wt, N * (u * HN + 4 * j / N)) * (x[4 * j / N][j] + mu[4 * j / N]);
                unsigned long long fx[4];
                to_fixed_n<4>(wx, fx);
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int h = 4 * j / N;
                    unsigned long long* cell = acc + (rec[u][j].y - ay0 + 2 * t + (n >> 3)) * aw + rec[u][j].x - ax0 + (n & 7);
                    if (g0 + u * HN + h < ngroups) lds_add(cell, fx[j]);
                }
            }
        }
    }
    __syncthreads();
    partials_out(aw, ah, tg.pitch, acc, jb.part_num + static_cast<size_t>(tile) * tg.pitch * ah + (ax0 & 3));
}

// NCSR rounds after the first: est += delta (noisy - est)
// (src/cpu/common/iter_regularize.cpp:15-39). 64 x 4 pixels per block.
__global__ __launch_bounds__(256) void regularize_kernel(float* est, int est_stride, const float* noisy,
                                                         int noisy_stride, int width, int height, float delta) {
    const int x = blockIdx.x * 64 + (threadIdx.x & 63);
    const int y = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (x >= width || y >= height) return;
    float* e = est + static_cast<size_t>(y) * est_stride + x;
    const float n = noisy[static_cast<size_t>(y) * noisy_stride + x];
    *e = fmaf(delta, n - *e, *e);
}

// ---------------------------------------------------------------------------
// Host-side sizing and launchers.
// ---------------------------------------------------------------------------

size_t match_wave_lds_bytes(int block, int range, bool stage) {
    const int w = 2 * range + 1;
    const size_t cand = static_cast<size_t>(w) * w * 4;
    if (!stage) return cand;
    const size_t reg = static_cast<size_t>(w + block - 1) * (w + block - 1);
    return ((reg + 3) & ~static_cast<size_t>(3)) * 4 + cand;
}

static int mm_list(int group) { return group > 16 ? 192 : 128; }
inline constexpr size_t kMmStagedLds = 40 * 1024;

// LDS words of the MFMA matcher for `list` candidates per reference: the fp16
// region (the exact keys over it), the exchange and lists, counters, and with
// `staged` the FP32 region. Plans ask for every block size: unions wider than
// the pitch table (steps above 8 only) get a size that no LDS holds.
static size_t mm_lds_words(int step, int range, size_t list, bool staged) {
    // the union of a 4 x 4 block's windows spans at most 3 step + 2 range + 1
    // candidate columns and rows
    const int span = 3 * step + 2 * range + 1;
    const int nt = (span + 15) >> 4;
    if (nt > kMmTiles) return size_t{1} << 20;
    const size_t reg = (std::max(static_cast<size_t>(span + 7) * static_cast<size_t>(h_mm_pitch.of[nt]), 16 * list) + 3) & ~static_cast<size_t>(3);
    return reg + 8 * list + kMmCounters +
           (staged ? static_cast<size_t>(span + 7) * mm_pitch32(nt) : 0);
}

// Regions staged in FP32 as well: those that leave four workgroups per CU.
static bool mm_staged(int step, int range, size_t list) {
    return mm_lds_words(step, range, list, true) * 4 <= kMmStagedLds;
}

size_t match_mfma_lds_bytes(int step, int range, int group) {
    const size_t list = static_cast<size_t>(mm_list(group));
    return mm_lds_words(step, range, list, mm_staged(step, range, list)) * 4;
}

bool match_mfma_fits(int block, int group, int step, int range, int width, int height) {
    return block == 8 && group >= 1 && group <= 32 && width >= 8 && height >= 8 &&
           match_mfma_lds_bytes(step, range, group) <= 160 * 1024;
}

int match_workgroups(int kind, const Grid& g) {
    if (kind == 3) return ((g.nx + 3) >> 2) * ((g.ny + 3) >> 2);
    if (kind == 2) return g.ny * ((g.nx + kRunRefs - 1) / kRunRefs);
    return g.nx * g.ny;
}

// LDS of the run matcher in a layout: NT = 1 or kRunMidTiles (keys in
// registers; the window keys and the gathered keys both over the region) or
// 0 (the window keys after the region, the gathered keys over it, or after
// the window keys when the region is smaller).
static size_t run_lds_layout(int block, int step, int range, int nt) {
    const size_t w = 2 * static_cast<size_t>(range) + 1;
    const size_t region = static_cast<size_t>(run_region_floats(block, step, range)) * 4;
    const size_t keys = kRunRefs * w * w * 4;
    const size_t gather = kRunRefs * static_cast<size_t>(nt == kRunMidTiles ? kRunMidGather : kRunGather) * 8;
    return nt > 0 ? std::max(region, keys + gather) : region + keys + (region < gather ? gather : 0);
}

// The layout a job of this range takes alone.
static int run_layout(int range) { return run_keys_in_regs(range) ? 1 : run_keys_mid(range) ? kRunMidTiles : 0; }

size_t match_run_lds_bytes(int block, int step, int range) {
    return run_lds_layout(block, step, range, run_layout(range));
}

size_t filter_atomic_lds_bytes(int block, int group, bool wiener) {
    return static_cast<size_t>(group) * (block * block + 1) * 4 * (wiener ? 2 : 1);
}

size_t filter_tile_b8_lds_bytes(int group, const TileGeom& t) {
    const size_t aw = t.aw, ah = t.ah;
    const size_t acc = aw * ah * 8;
    const size_t recs = static_cast<size_t>(t.tw) * t.th * group * sizeof(MatchRec) +
                        ((static_cast<size_t>(t.tw) * t.th + 3) & ~static_cast<size_t>(3)) * 4;
    const size_t tbuf = 4 * static_cast<size_t>(group) * kTs * 4;
    return acc + recs + tbuf;
}

size_t filter_tile_mfma_lds_bytes(int group, const TileGeom& t) {
    const size_t aw = t.aw, ah = t.ah;
    const size_t acc = ((aw * ah + 1) & ~static_cast<size_t>(1)) * 8;
    const size_t recs = ((static_cast<size_t>(t.tw) * t.th * group + 3) & ~static_cast<size_t>(3)) * 4 +
                        ((static_cast<size_t>(t.tw) * t.th + 3) & ~static_cast<size_t>(3)) * 4;
    const size_t tbuf = 4 * static_cast<size_t>(kMfmaBuf) * 4 + 64 * 4;  // + the fp16 form's DCT table
    return acc + recs + tbuf;
}

size_t filter_tile_lds_bytes(int block, int group, bool wiener, const TileGeom& t) {
    const size_t aw = t.aw, ah = t.ah;
    const size_t acc = aw * ah * 8;
    return acc + 4 * filter_atomic_lds_bytes(block, group, wiener);
}

template <typename K>
static void allow_lds(K kernel, size_t lds) {
    if (lds > 65536)
        (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                                  static_cast<int>(lds));
}

template <int B>
static hipError_t launch_match_b(const MatchTable& t, int total_wg, size_t lds, int kind, hipStream_t s) {
    if (kind == 3) {
        if constexpr (B == 8) {
            // One list length for the whole launch (the largest group's) and
            // one staging form, so the LDS is sized here for every job.
            int gmax = 0;
            for (int j = 0; j < t.n; ++j) gmax = std::max(gmax, t.job[j].group);
            const size_t list = static_cast<size_t>(mm_list(gmax));
            bool staged = true;
            for (int j = 0; j < t.n; ++j) staged &= mm_staged(t.job[j].grid.step, t.job[j].range, list);
            lds = 0;
            for (int j = 0; j < t.n; ++j)
                lds = std::max(lds, mm_lds_words(t.job[j].grid.step, t.job[j].range, list, staged) * 4);
            if (lds > 160 * 1024) return hipErrorInvalidValue;
            auto launch = [&](auto kernel) {
                allow_lds(kernel, lds);
                kernel<<<total_wg, 256, lds, s>>>(t);
            };
            if (list == 192)
                staged ? launch(&match_mfma_kernel<192, true>) : launch(&match_mfma_kernel<192, false>);
            else
                staged ? launch(&match_mfma_kernel<128, true>) : launch(&match_mfma_kernel<128, false>);
        } else {
            return hipErrorInvalidValue;
        }
    } else if (kind == 2) {
        if constexpr (B <= 12) {
            // the layout every job's window takes (the one of the largest
            // range); the LDS for the layout launched
            int nt = 1;
            for (int j = 0; j < t.n; ++j) {
                const int l = run_layout(t.job[j].range);
                nt = nt == 0 || l == 0 ? 0 : std::max(nt, l);
            }
            lds = 0;
            for (int j = 0; j < t.n; ++j)
                lds = std::max(lds, run_lds_layout(B, t.job[j].grid.step, t.job[j].range, nt));
            if (nt == 1) {
                allow_lds(&match_run_kernel<B, true>, lds);
                match_run_kernel<B, true><<<total_wg, 256, lds, s>>>(t);
            } else if (nt == kRunMidTiles) {
                allow_lds(&match_run_mid_kernel<B>, lds);
                match_run_mid_kernel<B><<<total_wg, 256, lds, s>>>(t);
            } else {
                allow_lds(&match_run_kernel<B, false>, lds);
                match_run_kernel<B, false><<<total_wg, 256, lds, s>>>(t);
            }
        } else {
            return hipErrorInvalidValue;
        }
    } else if (kind == 1) {
        allow_lds(&match_wave_kernel<B, true>, lds);
        match_wave_kernel<B, true><<<total_wg, 64, lds, s>>>(t);
    } else {
        allow_lds(&match_wave_kernel<B, false>, lds);
        match_wave_kernel<B, false><<<total_wg, 64, lds, s>>>(t);
    }
    return hipGetLastError();
}

// Block sizes outside the BM3D set (the group filters take any block from 1
// to 16): the wave matcher only, window in LDS (kind 1) or from global (0).
template <int B>
static hipError_t launch_match_wave(const MatchTable& t, int total_wg, size_t lds, int kind, hipStream_t s) {
    if (kind == 1) {
        allow_lds(&match_wave_kernel<B, true>, lds);
        match_wave_kernel<B, true><<<total_wg, 64, lds, s>>>(t);
    } else if (kind == 0) {
        allow_lds(&match_wave_kernel<B, false>, lds);
        match_wave_kernel<B, false><<<total_wg, 64, lds, s>>>(t);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// kind: 3 MFMA matcher (B = 8), 2 run matcher, 1 wave matcher with the
// window in LDS, 0 from global.
hipError_t launch_match(int block, const MatchTable& t, int total_wg, size_t lds, int kind, hipStream_t s) {
    if (launch_fault()) return hipErrorLaunchFailure;
    switch (block) {
        case 3: return launch_match_wave<3>(t, total_wg, lds, kind, s);
        case 5: return launch_match_wave<5>(t, total_wg, lds, kind, s);
        case 6: return launch_match_wave<6>(t, total_wg, lds, kind, s);
        case 7: return launch_match_wave<7>(t, total_wg, lds, kind, s);
        case 9: return launch_match_wave<9>(t, total_wg, lds, kind, s);
        case 10: return launch_match_wave<10>(t, total_wg, lds, kind, s);
        case 11: return launch_match_wave<11>(t, total_wg, lds, kind, s);
        case 13: return launch_match_wave<13>(t, total_wg, lds, kind, s);
        case 14: return launch_match_wave<14>(t, total_wg, lds, kind, s);
        case 15: return launch_match_wave<15>(t, total_wg, lds, kind, s);
        case 1: return launch_match_b<1>(t, total_wg, lds, kind, s);
        case 2: return launch_match_b<2>(t, total_wg, lds, kind, s);
        case 4: return launch_match_b<4>(t, total_wg, lds, kind, s);
        case 8: return launch_match_b<8>(t, total_wg, lds, kind, s);
        case 12: return launch_match_b<12>(t, total_wg, lds, kind, s);
        case 16: return launch_match_b<16>(t, total_wg, lds, kind, s);
        case 32: return launch_match_b<32>(t, total_wg, lds, kind, s);
        default: return hipErrorInvalidValue;
    }
}

template <int B>
static hipError_t launch_filter_b(const FilterTable& t, int total_wg, size_t lds, bool wiener, bool tiles,
                                  hipStream_t s) {
    if (tiles) {
        if (wiener) {
            allow_lds(&filter_tile_kernel<B, true>, lds);
            filter_tile_kernel<B, true><<<total_wg, 256, lds, s>>>(t);
        } else {
            allow_lds(&filter_tile_kernel<B, false>, lds);
            filter_tile_kernel<B, false><<<total_wg, 256, lds, s>>>(t);
        }
    } else {
        // a table with global cubes runs kCubeSlots workgroups (no LDS cube)
        const int grid = t.cube ? std::min(total_wg, t.cube_slots) : total_wg;
        if (t.cube) lds = 0;
        if (wiener) {
            allow_lds(&filter_atomic_kernel<B, true>, lds);
            filter_atomic_kernel<B, true><<<grid, 64, lds, s>>>(t);
        } else {
            allow_lds(&filter_atomic_kernel<B, false>, lds);
            filter_atomic_kernel<B, false><<<grid, 64, lds, s>>>(t);
        }
    }
    return hipGetLastError();
}

// A launch of up to 256 workgroups has a CU for each: 16 waves share a filter
// tile's groups, and the finish takes one pixel per thread. 128 x 96 YUV420,
// group 8: hard 10.8 -> 7.1 us, Wiener 12.5 -> 8.4; finish of 256 x 256 at step
// 3, group 16: 22.7 -> 19.6. Above that four waves serve the Wiener stage
// (1080p YUV420 57.3 us against 60.8 with eight: its registers leave the fifth
// to eighth wave of a SIMD out), and eight the hard stage where they put a
// fifth more waves on a CU than workgroups of four do, or where the tiles fill
// the device no more than twice. Eight against four, 1080p, group 8: step 8, range 9
// 28.4 us against 29.3, range 24 47.1 / 55.3, step 6, range 24 61.6 / 78.8; RGB,
// step 3, range 7 (28 waves to 32) 397 / 374; group 16: step 3, range 24 309 /
// 398, but range 12 (16 waves either way) 271 / 255. Each form is compiled for
// its own size: one bound of 1024 threads for all of them took group 16's hard
// kernel from 71 to 86 registers (RGB, step 3, range 4: 711 -> 790 us).
inline constexpr int kFinishAloneBlocks = 256;
inline constexpr int kFilterAloneTiles = 256;

template <int G>
static hipError_t launch_filter_b8(const FilterTable& t, int total_wg, size_t lds, bool wiener, hipStream_t s) {
    int waves = 4;  // what lds holds transpose buffers for
    if (G <= 16) {
        const size_t each = static_cast<size_t>(G) * kTs * 4;
        int groups = 1;
        for (int j = 0; j < t.n; ++j) groups = std::max(groups, t.job[j].tiles.tw * t.job[j].tiles.th);
        // waves of a CU with workgroups of w (LDS comes in units of 1280 bytes;
        // group 16's registers hold 24)
        const auto per_cu = [&](int w) {
            const size_t units = (lds + (w - 4) * each + 1279) / 1280;
            return std::min(G <= 8 ? 32 : 24, w * static_cast<int>(128 / units));
        };
        const bool eight = !wiener && (5 * per_cu(8) >= 6 * per_cu(4) || total_wg <= 2 * 64 * per_cu(4));
        const int want = total_wg <= kFilterAloneTiles ? 16 : eight ? 8 : 4;
        while (2 * waves <= want && waves < groups && lds + waves * each <= (want == 16 ? 160 : 80) * 1024) {
            lds += waves * each;
            waves *= 2;
        }
    }
    const auto launch = [&](auto kernel) {
        allow_lds(kernel, lds);
        kernel<<<total_wg, 64 * waves, lds, s>>>(t);
        return hipGetLastError();
    };
    if constexpr (G <= 16) {
        if (wiener && waves > 4) return launch(&filter_tile_b8_kernel<G, true, 16>);
        if (!wiener && waves > 8) return launch(&filter_tile_b8_kernel<G, false, 16>);
        if (!wiener && waves > 4) return launch(&filter_tile_b8_kernel<G, false, 8>);
    }
    return wiener ? launch(&filter_tile_b8_kernel<G, true, 4>) : launch(&filter_tile_b8_kernel<G, false, 4>);
}

template <int G, int FORM>
static hipError_t launch_filter_mfma(const FilterTable& t, int total_wg, size_t lds, bool wiener, hipStream_t s) {
    if (wiener) {
        allow_lds(&filter_tile_mfma_kernel<G, true, FORM>, lds);
        filter_tile_mfma_kernel<G, true, FORM><<<total_wg, 256, lds, s>>>(t);
    } else {
        allow_lds(&filter_tile_mfma_kernel<G, false, FORM>, lds);
        filter_tile_mfma_kernel<G, false, FORM><<<total_wg, 256, lds, s>>>(t);
    }
    return hipGetLastError();
}

// fast_group: 8, 16 or 32 selects the block-8 register kernel (tile path);
// form 1 (bf16x3) or 2 (fp16) with fast_group 8 or 16 the MFMA kernel.
hipError_t launch_filter(int block, const FilterTable& t, int total_wg, size_t lds, bool wiener, bool tiles,
                         int fast_group, int form, hipStream_t s) {
    if (launch_fault()) return hipErrorLaunchFailure;
    if (tiles && block == 8 && form) {
        if (fast_group == 8) return form == 1 ? launch_filter_mfma<8, kFormBf16x3>(t, total_wg, lds, wiener, s)
                                              : launch_filter_mfma<8, kFormF16>(t, total_wg, lds, wiener, s);
        if (fast_group == 16) return form == 1 ? launch_filter_mfma<16, kFormBf16x3>(t, total_wg, lds, wiener, s)
                                               : launch_filter_mfma<16, kFormF16>(t, total_wg, lds, wiener, s);
        return hipErrorInvalidValue;
    }
    if (tiles && block == 8 && fast_group) {
        switch (fast_group) {
            case 8: return launch_filter_b8<8>(t, total_wg, lds, wiener, s);
            case 16: return launch_filter_b8<16>(t, total_wg, lds, wiener, s);
            case 32: return launch_filter_b8<32>(t, total_wg, lds, wiener, s);
            default: return hipErrorInvalidValue;
        }
    }
    switch (block) {
        case 1: return launch_filter_b<1>(t, total_wg, lds, wiener, tiles, s);
        case 2: return launch_filter_b<2>(t, total_wg, lds, wiener, tiles, s);
        case 4: return launch_filter_b<4>(t, total_wg, lds, wiener, tiles, s);
        case 8: return launch_filter_b<8>(t, total_wg, lds, wiener, tiles, s);
        case 12: return launch_filter_b<12>(t, total_wg, lds, wiener, tiles, s);
        case 16: return launch_filter_b<16>(t, total_wg, lds, wiener, tiles, s);
        case 32: return launch_filter_b<32>(t, total_wg, lds, wiener, tiles, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_finish_sums(const FinishTable& t, int total_wg, hipStream_t s) {
    if (launch_fault()) return hipErrorLaunchFailure;
    finish_sums_kernel<<<total_wg, 256, 0, s>>>(t);
    return hipGetLastError();
}

size_t finish_tiles_lds_bytes(int block) {
    const size_t ch = 16 + block - 1, cw = 64 + block - 1;
    return (ch * cw + ch * 64) * 8;
}

hipError_t launch_finish(int block, const FinishTable& t, int total_wg, bool tiles, hipStream_t s) {
    if (launch_fault()) return hipErrorLaunchFailure;
    if (tiles) {
        if (t.n && t.job[0].exact_num) {
            // the corner tile and its horizontal sums of the largest block
            int bmax = 1;
            for (int k = 0; k < t.n; ++k) bmax = std::max(bmax, t.job[k].block);
            const size_t lds = finish_tiles_lds_bytes(bmax);
            if (total_wg <= kFinishAloneBlocks) {
                allow_lds(&finish_tiles_kernel<true, 1>, lds);
                finish_tiles_kernel<true, 1><<<total_wg, 1024, lds, s>>>(t);
            } else {
                allow_lds(&finish_tiles_kernel<true, 4>, lds);
                finish_tiles_kernel<true, 4><<<total_wg, 256, lds, s>>>(t);
            }
        } else {
            finish_tiles_kernel<false, 4><<<total_wg, 256, 0, s>>>(t);
        }
        return hipGetLastError();
    }
    switch (block) {
        case 1: finish_corner_kernel<1><<<total_wg, 256, 0, s>>>(t); break;
        case 2: finish_corner_kernel<2><<<total_wg, 256, 0, s>>>(t); break;
        case 4: finish_corner_kernel<4><<<total_wg, 256, 0, s>>>(t); break;
        case 8: finish_corner_kernel<8><<<total_wg, 256, 0, s>>>(t); break;
        case 12: finish_corner_kernel<12><<<total_wg, 256, 0, s>>>(t); break;
        case 16: finish_corner_kernel<16><<<total_wg, 256, 0, s>>>(t); break;
        case 32: finish_corner_kernel<32><<<total_wg, 256, 0, s>>>(t); break;
        case 3: finish_corner_kernel<3><<<total_wg, 256, 0, s>>>(t); break;
        case 5: finish_corner_kernel<5><<<total_wg, 256, 0, s>>>(t); break;
        case 6: finish_corner_kernel<6><<<total_wg, 256, 0, s>>>(t); break;
        case 7: finish_corner_kernel<7><<<total_wg, 256, 0, s>>>(t); break;
        case 9: finish_corner_kernel<9><<<total_wg, 256, 0, s>>>(t); break;
        case 10: finish_corner_kernel<10><<<total_wg, 256, 0, s>>>(t); break;
        case 11: finish_corner_kernel<11><<<total_wg, 256, 0, s>>>(t); break;
        case 13: finish_corner_kernel<13><<<total_wg, 256, 0, s>>>(t); break;
        case 14: finish_corner_kernel<14><<<total_wg, 256, 0, s>>>(t); break;
        case 15: finish_corner_kernel<15><<<total_wg, 256, 0, s>>>(t); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_zero(const ZeroTable& t, int total_wg, hipStream_t s) {
    if (launch_fault()) return hipErrorLaunchFailure;
    zero_kernel<<<total_wg, 256, 0, s>>>(t);
    return hipGetLastError();
}

size_t predictive_table_lds(int block, PredTable& t, int radius) {
    // Candidate keys: one pass for a layer's union when it fits kPredChunk.
    // Merged candidates: (G - 1) spatial + min(ps_num, G) per layer and direction.
    int chunk = 64, region = 0;
    size_t merged = 0;
    for (int j = 0; j < t.n; ++j) {
        const PredJob& p = t.job[j];
        const int kl = std::min(p.ps_num, p.group);
        const int w = 2 * p.ps_range + 1, cells = kl * w * w;
        chunk = std::max(chunk, std::min(kPredChunk, (cells + 63) / 64 * 64));
        merged = std::max(merged, static_cast<size_t>(p.group - 1 + 2 * radius * kl));
        const int need = kl * (w + block - 1) * pred_region_pitch(w, block);
        if (cells <= kPredChunk && need <= kPredRegionCap) region = std::max(region, need);
    }
    const size_t head = ((static_cast<size_t>(block) * block + 3) & ~static_cast<size_t>(3)) * 4 + chunk * 8 +
                        2 * kMaxGroup * 8 + kMaxGroup * 4 + merged * 8;
    t.chunk = chunk;
    t.region = region;
    t.region_offset = static_cast<int>((head + 15) & ~static_cast<size_t>(15));
    return t.region_offset + static_cast<size_t>(region) * 4;
}

hipError_t launch_predictive(int block, const PredTable& t, int total_wg, size_t lds, hipStream_t s) {
    if (launch_fault()) return hipErrorLaunchFailure;
    switch (block) {
        case 1: allow_lds(&predictive_kernel<1>, lds); predictive_kernel<1><<<total_wg, 64, lds, s>>>(t); break;
        case 2: allow_lds(&predictive_kernel<2>, lds); predictive_kernel<2><<<total_wg, 64, lds, s>>>(t); break;
        case 4: allow_lds(&predictive_kernel<4>, lds); predictive_kernel<4><<<total_wg, 64, lds, s>>>(t); break;
        case 8: allow_lds(&predictive_kernel<8>, lds); predictive_kernel<8><<<total_wg, 64, lds, s>>>(t); break;
        case 12: allow_lds(&predictive_kernel<12>, lds); predictive_kernel<12><<<total_wg, 64, lds, s>>>(t); break;
        case 16: allow_lds(&predictive_kernel<16>, lds); predictive_kernel<16><<<total_wg, 64, lds, s>>>(t); break;
        case 32: allow_lds(&predictive_kernel<32>, lds); predictive_kernel<32><<<total_wg, 64, lds, s>>>(t); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int B>
static hipError_t launch_tfilter_b(const TFilterTable& t, int total_wg, size_t lds, bool wiener, hipStream_t s) {
    const int grid = t.cube ? std::min(total_wg, t.cube_slots) : total_wg;
    if (t.cube) lds = 0;
    if (wiener) {
        allow_lds(&filter_temporal_kernel<B, true>, lds);
        filter_temporal_kernel<B, true><<<grid, 64, lds, s>>>(t);
    } else {
        allow_lds(&filter_temporal_kernel<B, false>, lds);
        filter_temporal_kernel<B, false><<<grid, 64, lds, s>>>(t);
    }
    return hipGetLastError();
}

size_t filter_temporal_b8_lds_bytes(int group) { return 4 * static_cast<size_t>(group) * kTs * 4; }

// Dynamic LDS of filter_temporal_tile_kernel for per-slot geometries g[0..ns).
size_t filter_temporal_tile_lds_bytes(int group, const TileGeom* g, int ns, bool corner_planes) {
    size_t acc = 0, boxsum = 0;
    for (int t = 0; t < ns; ++t) {
        acc += static_cast<size_t>(g[t].aw) * g[t].ah;
        if (corner_planes) continue;  // no corner sums, no den box sum
        acc += static_cast<size_t>(g[t].aw - 7) * (g[t].ah - 7);
        boxsum = std::max(boxsum, static_cast<size_t>(g[t].ah - 7) * g[t].aw * 4);
    }
    acc = ((acc + 1) & ~static_cast<size_t>(1)) * 8;
    const size_t recs = static_cast<size_t>(g[0].tw) * g[0].th * group * sizeof(MatchRec) +
                        ((static_cast<size_t>(g[0].tw) * g[0].th + 3) & ~static_cast<size_t>(3)) * 4;
    const size_t tbuf = static_cast<size_t>(kTTileWaves) * group * kTs * 4;
    return recs + acc + std::max(tbuf, boxsum);
}

// Persistent grid: as many workgroups as the device holds at once (at most
// one per tile).
template <int G, typename Kernel>
static hipError_t launch_persistent_ttile(Kernel k, const TTileTable& t, int tiles, size_t lds, hipStream_t s) {
    allow_lds(k, lds);
    int dev = 0, cus = 0, per_cu = 0, threads = 64 * kTTileWaves;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
    if (e == hipSuccess) e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k, threads, lds);
    if (e != hipSuccess) return e;
    // Slots that leave room for one workgroup only: 16 waves share its tiles
    // (two per SIMD were a third of the VALU's rate; 1080p YUV420, radius 1,
    // group 8: hard 126 -> 102 us, Wiener 183 -> 169 us per launch; groups of
    // 16 would spill at 128 registers).
    const size_t more = static_cast<size_t>(kTTileWaves) * G * kTs * 4;
    if (G == 8 && per_cu <= 1 && lds + more <= 160 * 1024) {
        lds += more;
        threads *= 2;
        allow_lds(k, lds);
    }
    const int grid = std::max(1, std::min(tiles, std::max(cus, 1) * std::max(per_cu, 1)));
    k<<<grid, threads, lds, s>>>(t, tiles);
    return hipGetLastError();
}

template <int G>
static hipError_t launch_ttile(const TTileTable& t, int tiles, size_t lds, bool wiener, hipStream_t s) {
    if (t.job[0].tiles[0].tw * t.job[0].tiles[0].th * G > 512) return hipErrorInvalidValue;
    return wiener ? launch_persistent_ttile<G>(&filter_temporal_tile_kernel<G, true>, t, tiles, lds, s)
                  : launch_persistent_ttile<G>(&filter_temporal_tile_kernel<G, false>, t, tiles, lds, s);
}

hipError_t launch_filter_temporal_tiles(int group, const TTileTable& t, int total_wg, size_t lds, bool wiener,
                                        hipStream_t s) {
    if (launch_fault()) return hipErrorLaunchFailure;
    switch (group) {
        case 8: return launch_ttile<8>(t, total_wg, lds, wiener, s);
        case 16: return launch_ttile<16>(t, total_wg, lds, wiener, s);
        case 32: return launch_ttile<32>(t, total_wg, lds, wiener, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_finish_temporal_tiles(const TFinishTable& t, int total_wg, hipStream_t s) {
    if (launch_fault()) return hipErrorLaunchFailure;
    // the corner tile and its horizontal sums when the weights come from corner planes
    int bmax = 0;
    for (int k = 0; k < t.n; ++k)
        if (t.job[k].corners) bmax = std::max(bmax, t.job[k].block);
    const size_t lds = bmax ? finish_tiles_lds_bytes(bmax) : 0;
    if (lds) {
        allow_lds(&finish_temporal_tiles_kernel, lds);
        finish_temporal_tiles_kernel<<<total_wg, 256, lds, s>>>(t);
        return hipGetLastError();
    }
    finish_temporal_tiles_kernel<<<total_wg, 256, 0, s>>>(t);
    return hipGetLastError();
}

template <int G>
static hipError_t launch_tfilter_b8(const TFilterTable& t, int total_wg, size_t lds, bool wiener, hipStream_t s) {
    if (wiener) {
        allow_lds(&filter_temporal_b8_kernel<G, true>, lds);
        filter_temporal_b8_kernel<G, true><<<total_wg, 256, lds, s>>>(t);
    } else {
        allow_lds(&filter_temporal_b8_kernel<G, false>, lds);
        filter_temporal_b8_kernel<G, false><<<total_wg, 256, lds, s>>>(t);
    }
    return hipGetLastError();
}

// fast_group 8, 16 or 32 (block 8): four groups per workgroup, register cube.
hipError_t launch_filter_temporal(int block, const TFilterTable& t, int total_wg, size_t lds, bool wiener,
                                  int fast_group, hipStream_t s) {
    if (launch_fault()) return hipErrorLaunchFailure;
    if (block == 8 && fast_group) {
        switch (fast_group) {
            case 8: return launch_tfilter_b8<8>(t, total_wg, lds, wiener, s);
            case 16: return launch_tfilter_b8<16>(t, total_wg, lds, wiener, s);
            case 32: return launch_tfilter_b8<32>(t, total_wg, lds, wiener, s);
            default: return hipErrorInvalidValue;
        }
    }
    switch (block) {
        case 1: return launch_tfilter_b<1>(t, total_wg, lds, wiener, s);
        case 2: return launch_tfilter_b<2>(t, total_wg, lds, wiener, s);
        case 4: return launch_tfilter_b<4>(t, total_wg, lds, wiener, s);
        case 8: return launch_tfilter_b<8>(t, total_wg, lds, wiener, s);
        case 12: return launch_tfilter_b<12>(t, total_wg, lds, wiener, s);
        case 16: return launch_tfilter_b<16>(t, total_wg, lds, wiener, s);
        case 32: return launch_tfilter_b<32>(t, total_wg, lds, wiener, s);
        default: return hipErrorInvalidValue;
    }
}

static int wnnm_pad(int group) { return group <= 8 ? 8 : group <= 16 ? 16 : 32; }

size_t wnnm_lds_bytes(int block, int group) {
    const size_t n = wnnm_pad(group), m = static_cast<size_t>(block) * block;
    return 4 * (n * (m + 1) + 2 * n * (n + 1) + 4 * n);
}

hipError_t launch_regularize(float* est, int est_stride, const float* noisy, int noisy_stride, int width, int height,
                             float delta, hipStream_t s) {
    if (launch_fault()) return hipErrorLaunchFailure;
    const dim3 grid((width + 63) / 64, (height + 3) / 4);
    regularize_kernel<<<grid, 256, 0, s>>>(est, est_stride, noisy, noisy_stride, width, height, delta);
    return hipGetLastError();
}

template <int N>
static hipError_t launch_gram_groups(const WnnmTable& t, int total_wg, size_t lds, bool ncsr, hipStream_t s) {
    if (ncsr) {
        allow_lds(&ncsr_group_kernel<N>, lds);
        ncsr_group_kernel<N><<<total_wg, 64, lds, s>>>(t);
    } else {
        allow_lds(&wnnm_group_kernel<N>, lds);
        wnnm_group_kernel<N><<<total_wg, 64, lds, s>>>(t);
    }
    return hipGetLastError();
}

// LDS of gram_group_tile_kernel for a plane whose every reference has a full
// group (the smallest window, a corner's, holds it) in tiles of g; 0 where
// the kernel does not serve the shape.
size_t gram_tile_lds_bytes(int block, int group, int range, int width, int height, const TileGeom& g) {
    if (block != 8 || (group != 8 && group != 16) || g.tw * g.th > 4 * (64 / group)) return 0;
    const long long w = std::min(range, width - block) + 1, h = std::min(range, height - block) + 1;
    if (w * h < group) return 0;
    return std::max(static_cast<size_t>(g.aw) * g.ah * 8, static_cast<size_t>(4 * kGramScratch) * 4);
}

hipError_t launch_wnnm_tiles(const WnnmTable& t, int total_wg, size_t lds, bool ncsr, hipStream_t s) {
    if (launch_fault()) return hipErrorLaunchFailure;
    const int group = t.job[0].group;
    for (int j = 0; j < t.n; ++j) {
        const WnnmJob& q = t.job[j];
        const size_t need = gram_tile_lds_bytes(q.block, q.group, q.range, q.width, q.height, q.tiles);
        if (q.group != group || need == 0 || need > lds || q.temporal) return hipErrorInvalidValue;
    }
    auto launch = [&](auto kernel) {
        allow_lds(kernel, lds);
        kernel<<<total_wg, 256, lds, s>>>(t);
        return hipGetLastError();
    };
    if (group == 8) return ncsr ? launch(&gram_group_tile_kernel<8, true>) : launch(&gram_group_tile_kernel<8, false>);
    return ncsr ? launch(&gram_group_tile_kernel<16, true>) : launch(&gram_group_tile_kernel<16, false>);
}

hipError_t launch_wnnm(const WnnmTable& t, int total_wg, bool ncsr, hipStream_t s) {
    if (launch_fault()) return hipErrorLaunchFailure;
    int gmax = 0, bmax = 0;
    for (int j = 0; j < t.n; ++j) {
        if (t.job[j].group < 1 || t.job[j].group > 32 || t.job[j].block < 1 || t.job[j].block > 16)
            return hipErrorInvalidValue;
        gmax = std::max(gmax, t.job[j].group);
        bmax = std::max(bmax, t.job[j].block);
    }
    const size_t lds = wnnm_lds_bytes(bmax, gmax);
    switch (wnnm_pad(gmax)) {
        case 8: return launch_gram_groups<8>(t, total_wg, lds, ncsr, s);
        case 16: return launch_gram_groups<16>(t, total_wg, lds, ncsr, s);
        default: return launch_gram_groups<32>(t, total_wg, lds, ncsr, s);
    }
}

hipError_t upload_dct_tables(const float* host, size_t count) {
    if (count != sizeof(c_dct) / sizeof(float)) return hipErrorInvalidValue;
    return hipMemcpyToSymbol(HIP_SYMBOL(c_dct), host, sizeof(c_dct), 0, hipMemcpyHostToDevice);
}

}  // namespace nsship
