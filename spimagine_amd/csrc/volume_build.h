// volume_build.h -- a volume's device layout from the uploaded (nz, ny, nx) array: the padded
// copy (volume_sampler.h), the window grid and the brick keys (brick_bounds.h).
#pragma once
#include "volume_sampler.h"

namespace spr {

// 16 bytes of voxels
template <typename T>
struct alignas(16) VoxelUnit {
    static constexpr uint32_t E = 16u / (uint32_t)sizeof(T);
    T v[E];
};

// Minimum and maximum of one 4x4x4 block of padded voxels
template <typename T>
struct BlockBounds {
    T lo, hi;
};

// Padded voxels and their 4x4x4 block bounds in one pass over the source.  A thread takes
// one 16-byte unit column: 4 rows of 4 planes of the padded copy, written as aligned units
// and reduced on the way to one block (4 voxels along x) per 4 elements.  Padded planes
// [4 bz0, 4 (bz0 + gridDim.y)) clipped to nz + 2; src holds source planes from sz0 on.
// blocks: (bz, by, bx) with pitch / 4 blocks a row, or nullptr (no bounds wanted).
//
// Bound by HBM: the source read once and the copy written once.  Before, the copy went
// voxel by voxel (2-byte loads and stores) and a second pass read the copy back one brick
// a thread: 0.36 + 0.37 ms for a 512^3 uint16 volume, 268 MB.
template <typename T>
__global__ __launch_bounds__(256) void k_pad_blocks(const T* __restrict__ src, T* __restrict__ dst,
                                                    int nx, int ny, int nz, uint32_t bz0, int sz0,
                                                    BlockBounds<T>* __restrict__ blocks) {
    using U = VoxelUnit<T>;
    constexpr int E = (int)U::E;
    constexpr bool kBounds = std::is_arithmetic<T>::value;
    const uint32_t pitch = padded_pitch<T>(nx), PY = (uint32_t)ny + 2u, PZ = (uint32_t)nz + 2u;
    const uint32_t units = pitch / (uint32_t)E, nby = win_entries(PY);
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    const uint32_t by = i / units, ux = i - by * units, bz = bz0 + blockIdx.y;
    if (by >= nby) return;
    const int x0 = (int)(ux * (uint32_t)E) - 1;  // source x of the unit's first voxel
    const bool whole = x0 >= 0 && x0 + E <= nx;
    T lo[E], hi[E];
    bool bad[E / 4];
#pragma unroll
    for (int b = 0; b < E / 4; ++b) bad[b] = false;
    bool first = true;
    for (uint32_t k = 0; k < kWinStride; ++k) {
        const uint32_t z = bz * kWinStride + k;
        if (z >= PZ) break;
        const int sz = min(max((int)z - 1, 0), nz - 1) - sz0;
        U u[kWinStride];
#pragma unroll
        for (uint32_t r = 0; r < kWinStride; ++r) {
            const uint32_t y = min(by * kWinStride + r, PY - 1u);
            const int sy = min(max((int)y - 1, 0), ny - 1);
            const T* row = src + ((size_t)sz * ny + sy) * nx;
            if (whole) {
                __builtin_memcpy(&u[r], row + x0, 16);
            } else {
#pragma unroll
                for (int e = 0; e < E; ++e) u[r].v[e] = row[min(max(x0 + e, 0), nx - 1)];
            }
        }
#pragma unroll
        for (uint32_t r = 0; r < kWinStride; ++r) {
            const uint32_t y = by * kWinStride + r;
            if (y < PY)
                *reinterpret_cast<U*>(dst + ((size_t)z * PY + y) * pitch + ux * (uint32_t)E) = u[r];
            if constexpr (kBounds) {  // (a row past the last repeats it: the same bounds)
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const T v = u[r].v[e];
                    if constexpr (std::is_same<T, float>::value) bad[e / 4] = bad[e / 4] || v != v;
                    lo[e] = first || v < lo[e] ? v : lo[e];
                    hi[e] = first || v > hi[e] ? v : hi[e];
                }
                first = false;
            }
        }
    }
    if constexpr (kBounds) {
        if (blocks == nullptr) return;
        BlockBounds<T>* o = blocks + ((size_t)bz * nby + by) * (pitch / 4u) + ux * (uint32_t)(E / 4);
#pragma unroll
        for (int b = 0; b < E / 4; ++b) {
            BlockBounds<T> m{lo[4 * b], hi[4 * b]};
#pragma unroll
            for (int e = 4 * b + 1; e < 4 * b + 4; ++e) {
                m.lo = lo[e] < m.lo ? lo[e] : m.lo;
                m.hi = hi[e] > m.hi ? hi[e] : m.hi;
            }
            if constexpr (std::is_same<T, float>::value)
                if (bad[b]) m = BlockBounds<T>{-INFINITY, INFINITY};
            o[b] = m;
        }
    }
}

// The window grid from the 4x4x4 blocks (window (x, y, z) = blocks x, x+1 / y, y+1 / z, z+1
// that exist), the 8x8x8 brick keys (brick b is window 2b) and the minimum of every brick's
// keys (total: the volume's bounds).  grid.y = window planes; a few workgroups a plane, so
// that few atomics meet in total.  Reads 1/16 of the volume's bytes or less.
template <typename T>
__global__ __launch_bounds__(256) void k_block_windows(const BlockBounds<T>* __restrict__ blocks,
                                                       uint32_t bpitch, uint32_t gx, uint32_t gy,
                                                       uint32_t gz, T* __restrict__ wmax,
                                                       T* __restrict__ wmin, uint32_t nbx,
                                                       uint32_t nby, BrickKey* __restrict__ keys,
                                                       BrickKey* __restrict__ total) {
    __shared__ BrickKey part[4];
    const uint32_t z = blockIdx.y;
    uint32_t kmin = 0xFFFFFFFFu, nkmax = 0xFFFFFFFFu;
    for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < gx * gy; i += gridDim.x * 256u) {
        const uint32_t y = i / gx, x = i - y * gx;
        BlockBounds<T> m = blocks[((size_t)z * gy + y) * bpitch + x];
#pragma unroll
        for (uint32_t c = 1; c < 8; ++c) {
            const uint32_t xx = min(x + (c & 1u), gx - 1u), yy = min(y + ((c >> 1) & 1u), gy - 1u),
                           zz = min(z + (c >> 2), gz - 1u);
            const BlockBounds<T> b = blocks[((size_t)zz * gy + yy) * bpitch + xx];
            m.lo = b.lo < m.lo ? b.lo : m.lo;
            m.hi = b.hi > m.hi ? b.hi : m.hi;
        }
        if (((x | y | z) & 1u) == 0u) {
            BrickKey k{order_key(m.lo), ~order_key(m.hi)};
            if constexpr (std::is_same<T, float>::value)
                if (m.lo == -INFINITY && m.hi == INFINITY) k = BrickKey{0u, 0u};
            keys[((size_t)(z >> 1) * nby + (y >> 1)) * nbx + (x >> 1)] = k;
            kmin = min(kmin, k.kmin);
            nkmax = min(nkmax, k.nkmax);
        }
        if constexpr (std::is_same<T, float>::value) {
            const float g = bound_margin<T>(m.lo, m.hi);
            m.lo = m.lo - g;
            m.hi = m.hi + g;
        }
        const size_t o = ((size_t)z * gy + y) * gx + x;
        wmax[o] = m.hi;
        wmin[o] = m.lo;
    }
    for (int off = 32; off > 0; off >>= 1) {
        kmin = min(kmin, (uint32_t)__shfl_xor((int)kmin, off));
        nkmax = min(nkmax, (uint32_t)__shfl_xor((int)nkmax, off));
    }
    if ((threadIdx.x & 63u) == 0u) part[threadIdx.x >> 6] = BrickKey{kmin, nkmax};
    __syncthreads();
    if (threadIdx.x == 0 && (z & 1u) == 0u) {
        for (int w = 0; w < 4; ++w) {
            kmin = min(kmin, part[w].kmin);
            nkmax = min(nkmax, part[w].nkmax);
        }
        atomicMin(&total->kmin, kmin);
        atomicMin(&total->nkmax, nkmax);
    }
}

// The window grid of a channel pair's padded copy: the maximum of each channel.  First every
// 4x4x4 block (a thread a block, 16-byte rows), then windows of 2x2x2 of them.
__device__ __forceinline__ uint32_t pair_max(uint32_t a, uint32_t b) {
    return max(a & 0xFFFFu, b & 0xFFFFu) | max(a >> 16, b >> 16) << 16;
}
static __global__ __launch_bounds__(256) void k_pair_blocks(const U16Pair* __restrict__ pad,
                                                            int nx, int ny, int nz, uint32_t gx,
                                                            uint32_t gy, uint32_t* __restrict__ blocks) {
    const uint32_t pitch = padded_pitch<U16Pair>(nx), PY = (uint32_t)ny + 2u, PZ = (uint32_t)nz + 2u;
    const uint32_t i = blockIdx.x * 256u + threadIdx.x, by = i / gx, bx = i - by * gx, bz = blockIdx.y;
    if (by >= gy) return;
    uint32_t m = 0;
    for (uint32_t z = 4u * bz; z < min(4u * bz + 4u, PZ); ++z)
#pragma unroll
        for (uint32_t r = 0; r < 4u; ++r) {  // (rows past the last repeat it, voxels past a
            const uint32_t y = min(4u * by + r, PY - 1u);  // row's end the edge voxel)
            const uint4 v = *reinterpret_cast<const uint4*>(pad + ((size_t)z * PY + y) * pitch + 4u * bx);
            m = pair_max(m, pair_max(pair_max(v.x, v.y), pair_max(v.z, v.w)));
        }
    blocks[((size_t)bz * gy + by) * gx + bx] = m;
}
static __global__ __launch_bounds__(256) void k_pair_windows(const uint32_t* __restrict__ blocks,
                                                             uint32_t gx, uint32_t gy, uint32_t gz,
                                                             uint32_t* __restrict__ wmax) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x, y = i / gx, x = i - y * gx, z = blockIdx.y;
    if (y >= gy) return;
    uint32_t m = 0;
#pragma unroll
    for (uint32_t c = 0; c < 8u; ++c)
        m = pair_max(m, blocks[((size_t)min(z + (c >> 2), gz - 1u) * gy + min(y + (c >> 1 & 1u), gy - 1u)) * gx +
                               min(x + (c & 1u), gx - 1u)]);
    wmax[((size_t)z * gy + y) * gx + x] = m;
}

// Share of the windows that a max projection has to sample, measured along kNeedRays x kNeedRays
// rays parallel to each axis, between the voxels: the windows of a ray whose maximum exceeds the
// ray's own (a pair's: in either channel).  One wave a ray; sum[0]: the rays' shares, 16 bits each;
// sum[1], a float: the means of their samples (channel 0), which finite rays have.
//
// Windows alone do not tell: where few voxels are bright or noise is strong a ray seldom meets a
// window's maximum.  Against three quarters of the best window of a column, which was counted
// before, this misjudged half as often by how much the better march would have gained (0.8% of
// the time of frames on average instead of 1.1, batches 1.4 instead of 2.6).
constexpr uint32_t kNeedRays = 16;

__device__ __forceinline__ float2 need_value(float v) { return make_float2(v, 0.0f); }
__device__ __forceinline__ float2 need_value(uint16_t v) { return make_float2((float)v, 0.0f); }
__device__ __forceinline__ float2 need_value(uint8_t v) { return make_float2((float)v, 0.0f); }
__device__ __forceinline__ float2 need_value(U16Pair v) {
    return make_float2((float)(v.bits & 0xFFFFu), (float)(v.bits >> 16));
}

template <typename T>
__global__ __launch_bounds__(64) void k_ray_need(const T* __restrict__ pad, int nx, int ny, int nz,
                                                 const T* __restrict__ wmax, uint32_t gx, uint32_t gy,
                                                 uint32_t gz, uint32_t* __restrict__ sum) {
    const uint32_t n[3] = {(uint32_t)nx, (uint32_t)ny, (uint32_t)nz}, g[3] = {gx, gy, gz};
    const size_t pitch = padded_pitch<T>(nx), stride[3] = {1, pitch, pitch * (n[1] + 2u)};
    const size_t wstride[3] = {1, gx, (size_t)gx * gy};
    const uint32_t a = blockIdx.y, b = a == 0 ? 1u : 0u, c = a == 2 ? 1u : 2u, lane = threadIdx.x;
    const uint32_t rb = blockIdx.x % kNeedRays, rc = blockIdx.x / kNeedRays;
    const uint32_t ib = min(1u + (rb * n[b] + n[b] / 2u) / kNeedRays, n[b]),
                   ic = min(1u + (rc * n[c] + n[c] / 2u) / kNeedRays, n[c]);
    const T* at = pad + ib * stride[b] + ic * stride[c];
    float top = 0.0f, top2 = 0.0f, mean = 0.0f;
    for (uint32_t k = lane; k <= n[a]; k += 64u) {
        float s = 0.0f, s2 = 0.0f;
#pragma unroll
        for (uint32_t j = 0; j < 8u; ++j) {
            const float2 v = need_value(at[(k + (j & 1u)) * stride[a] + (j >> 1 & 1u) * stride[b] + (j >> 2) * stride[c]]);
            s += v.x;
            s2 += v.y;
        }
        mean += 0.125f * s;
        top = fmaxf(top, 0.125f * s);
        top2 = fmaxf(top2, 0.125f * s2);
    }
    for (int o = 32; o > 0; o >>= 1) {
        mean += __shfl_xor(mean, o);
        top = fmaxf(top, __shfl_xor(top, o));
        top2 = fmaxf(top2, __shfl_xor(top2, o));
    }
    const T* w = wmax + (ib >> kWinShift) * wstride[b] + (ic >> kWinShift) * wstride[c];
    uint32_t need = 0;
    for (uint32_t k = lane; k < g[a]; k += 64u) {
        const float2 v = need_value(w[k * wstride[a]]);
        need += v.x > top || v.y > top2 ? 1u : 0u;
    }
    for (int o = 32; o > 0; o >>= 1) need += (uint32_t)__shfl_xor((int)need, o);
    if (lane == 0u) {
        atomicAdd(sum, (need << 16) / g[a]);
        if (fabsf(mean) < __builtin_inff()) atomicAdd((float*)sum + 1, mean / (float)(n[a] + 1u));
    }
}

}  // namespace spr
