// mip_windows.h -- max projection that samples only where a ray's maximum can still rise.
//
// Same result, bit for bit, as k_max_project (volume_kernel.cl:20-185, :190-345 with
// alpha_pow == 0): a maximum does not depend on which samples that cannot change it are
// left out, and every sample taken sits at the reference's running-sum position.
//
// Each ray asks the window grid (brick_bounds.h) for the largest voxel its next GS samples
// can read -- one lookup, ~4 instructions a sample against ~52 for a trilinear sample -- and
// samples a group only when that exceeds its running maximum.  Skipping pays once the
// maxima are high, so a ray first probes the grid along its length and takes the samples
// where the bound is largest.  On 512^3 blob volumes with camera noise 27% of the rays'
// groups are then left; asked per 8x8 rays, as a staged box would be, 44%, and by the
// wave's 32-sample box and 8^3 bricks (mip_staged.h) 94%.
#pragma once
#include "march_choice.h"
#include "mip_staged.h"
#include "ray_sums.h"

namespace spr {

constexpr int kWinGroups = 8;  // groups asked for together

// What a window lookup allows for, as a share of the volume, between a position estimated
// with one fma and the running sum: each addition since the exact position is off by half an
// ulp of the position, 3.0e-8 inside the volume (2e-6 over the at most 64 samples that the max
// projection asks ahead, 2.7e-5 over kIsoAnchor), and 6.0e-8 times how far the box reaches
// where that is past it.
constexpr float kMipMargin = 1e-5f, kIsoMargin = 3e-5f;
__device__ __forceinline__ float window_margin(const RayParams& p, float inside) {
    float reach = 0.0f;  // (uniform)
#pragma unroll
    for (int k = 0; k < 6; ++k) reach = fmaxf(reach, 0.5f + 0.5f * fabsf(p.box[k]));
    return reach <= 1.0f ? inside : 2.0f * reach * inside;
}

// A window's largest voxel, or a pair's of each channel
__device__ __forceinline__ float win_value(float v) { return v; }
__device__ __forceinline__ float win_value(uint16_t v) { return (float)v; }
__device__ __forceinline__ float win_value(uint8_t v) { return (float)v; }
__device__ __forceinline__ float win_value(U16Pair v) { return (float)(v.bits >> 16); }
__device__ __forceinline__ float win_value2(U16Pair v) { return (float)(v.bits & 0xFFFFu); }

// One sample, or a pair's two
struct PairValue {
    float v1, v0;  // channels 1 and 0
};
template <int FILT, typename PV>
__device__ __forceinline__ auto window_sample(const PV& vol, float px, float py, float pz) {
    if constexpr (std::is_same<typename PV::value_type, U16Pair>::value) {
        PairValue r;
        linear_pair(vol, px, py, pz, r.v0, r.v1);
        return r;
    } else {
        return vol.template sample<FILT>(px, py, pz);
    }
}

// One ray's window lookups: the block coordinates of the least corner of group j's samples
// are (wx + j gx, ...), in windows.
template <typename V, int GS>
struct WindowRay {
    using T = typename V::value_type;
    float gx, gy, gz;  // advance of one group
    bool ok;           // a group's corners always lie in the one window

    __device__ __forceinline__ void begin(const V& vol, float dx, float dy, float dz, float mgx,
                                          float mgy, float mgz) {
        const float vx = dx * vol.fnx, vy = dy * vol.fny, vz = dz * vol.fnz;
        gx = (float)GS * 0.25f * vx;
        gy = (float)GS * 0.25f * vy;
        gz = (float)GS * 0.25f * vz;
        const float span = (float)(GS - 1);
        ok = fmaf(span, fabsf(vx), 2.0f * mgx) <= 3.0f && fmaf(span, fabsf(vy), 2.0f * mgy) <= 3.0f &&
             fmaf(span, fabsf(vz), 2.0f * mgz) <= 3.0f;
    }
    // block coordinates of the group whose first sample is at (px, py, pz)
    __device__ __forceinline__ void at(const V& vol, float px, float py, float pz, float mgx,
                                       float mgy, float mgz, float& wx, float& wy,
                                       float& wz) const {
        constexpr float kBack = (float)(GS - 1) / (float)GS;
        wx = fmaf(0.25f, texel<V::kPow2>(px, vol.fnx) + (1.0f - mgx), fminf(kBack * gx, 0.0f));
        wy = fmaf(0.25f, texel<V::kPow2>(py, vol.fny) + (1.0f - mgy), fminf(kBack * gy, 0.0f));
        wz = fmaf(0.25f, texel<V::kPow2>(pz, vol.fnz) + (1.0f - mgz), fminf(kBack * gz, 0.0f));
    }
    // entries of kWinGroups groups, every APART-th from the one `ahead` groups past (px, py, pz)
    template <int APART = 1>
    __device__ __forceinline__ void ask(const V& vol, float px, float py, float pz, float mgx,
                                        float mgy, float mgz, float ahead, const T* plane,
                                        T (&u)[kWinGroups]) const {
        float wx, wy, wz;
        at(vol, px, py, pz, mgx, mgy, mgz, wx, wy, wz);
#pragma unroll
        for (int j = 0; j < kWinGroups; ++j) {
            const float f = ahead + (float)(APART * j);
            u[j] = plane[vol.window(fmaf(f, gx, wx), fmaf(f, gy, wy), fmaf(f, gz, wz))];
        }
    }
    // first sample of the two groups most likely to hold the ray's maximum among `count`
    // samples from (px, py, pz) on: the largest bound among windows two groups apart
    __device__ __forceinline__ int best(const V& vol, float px, float py, float pz,
                                        int count) const {
        constexpr int PS = 2 * GS;
        const int probes = (count + PS - 1) / PS;
        // a probed window reaches two voxels either side of the two groups' middle
        const float sx = 2.0f * gx, sy = 2.0f * gy, sz = 2.0f * gz;
        const float bx = fmaf(0.25f, texel<V::kPow2>(px, vol.fnx) - 1.0f, gx),
                    by = fmaf(0.25f, texel<V::kPow2>(py, vol.fny) - 1.0f, gy),
                    bz = fmaf(0.25f, texel<V::kPow2>(pz, vol.fnz) - 1.0f, gz);
        float top_u = -1.0f;
        int at = 0;
        for (int i = 0; i < probes; i += 16) {
            T v[16];
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const float f = (float)min(i + k, probes - 1);
                v[k] = vol.win_max[vol.window(fmaf(f, sx, bx), fmaf(f, sy, by), fmaf(f, sz, bz))];
            }
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const float u = win_value(v[k]);
                at = u > top_u ? min(i + k, probes - 1) : at;
                top_u = fmaxf(top_u, u);
            }
        }
        return max(0, min(at * PS, count - PS));
    }
};

// One 8x8 pixel quarter of a 16x16 tile per workgroup; its kWinSegments waves march a
// segment each of the rays' samples and share the running maxima.  No boxes are staged: a
// wave puts the groups its rays still need into a queue in LDS, and whenever 64 are waiting
// GS neighbouring lanes take one each round, gather its samples from global memory and post
// the maximum to the ray's word, so no lane idles through groups that other rays need.
//
// Bound by the vector-memory path, in cache lines a gather touches: with a lane taking the
// whole group ~40 of 64 lanes touched lines of their own.  1024x1024x512 uint16 -> 1024^2,
// 1536 steps: 1144 us a lane a group, 849 us GS lanes a group; 2048x2048x512 -> 2048^2 5561
// and 4657 us; 64 frames of 1024x1024x256 -> 1024^2 48.0 and 41.6 ms.
constexpr int kWinSegments = 4;
// Waves per SIMD that the registers are held to (five: 96 of them).  Short marches wait on
// one load after another and gain by a fifth wave; groups of four trilinear samples (32 loads
// a lane in flight) and single float ones need the registers.  us with four / five waves,
// 800^2 frames: nearest, 512^3 uint16 200 steps 146 / 111; linear, 256^3 uint16 200 steps
// (2 a group) 197 / 178, 512^3 float 896 steps (4) 568 / 616, 200 steps (1) 251 / 257.
template <typename T, int GS, int FILT>
constexpr int kWinWaves =
    !std::is_same<T, U16Pair>::value &&
            (FILT == 1 || GS == 2 || (GS == 1 && !std::is_same<T, float>::value))
        ? 5
        : 4;
// workgroups of one grid dimension: a launch has fewer than 2^32 threads along it
constexpr uint64_t kWinMaxGroups = (1ull << 32) / (64 * kWinSegments) - 1;

// Samples per group for a step of at most `step` voxels along an axis: as many as one window
// surely holds (WindowRay::ok; rays whose group spans more sample everything).
__host__ inline int windows_group(float step) {
    return 3.0f * step <= 2.9f ? 4 : step <= 2.9f ? 2 : 1;
}

// Whether a frame is gathered (march_choice.h)
__host__ inline bool windows_pay(bool nearest, float need, int nmax, float step, const RayParams& p) {
    const float quarters = 4.0f * (float)p.ntiles;
    return windows_pay(nearest, false, need, nmax, step, quarters) ||
           windows_pay(nearest, false, need, nmax, step, quarters * hit_share(p.invP, p.invM, p.box));
}

// the rays of a workgroup: which lanes have one, sample 0 and step
struct SharedRays {
    float pos[3][64], step[3][64];
    uint64_t act;
    __device__ __forceinline__ void put(uint32_t lane, uint64_t a, float px, float py, float pz,
                                        float dx, float dy, float dz) {
        pos[0][lane] = px;
        pos[1][lane] = py;
        pos[2][lane] = pz;
        step[0][lane] = dx;
        step[1][lane] = dy;
        step[2][lane] = dz;
        if (lane == 0) act = a;
    }
    __device__ __forceinline__ void get(uint32_t lane, float& px, float& py, float& pz, float& dx,
                                        float& dy, float& dz) const {
        px = pos[0][lane];
        py = pos[1][lane];
        pz = pos[2][lane];
        dx = step[0][lane];
        dy = step[1][lane];
        dz = step[2][lane];
    }
};
struct WindowShared {
    float4 item[kWinSegments][128];  // each wave's waiting groups: position, ray (w's bits)
    SharedRays rays;
    uint32_t top[64];                // the rays' running maxima (bits of floats >= 0); a pair's
    uint32_t top2[64];               // channel 1 in top, channel 0 in top2
};

// Samples of n >= 1 waiting groups, GS neighbouring lanes a group: batch b's lane takes sample
// lane % GS of item b 64 / GS + lane / GS, at the position the reference's running sum gives
// it (the lanes past the last item repeat it).  post(b, value, item's word).
//
// The samples of a group lie on one ray within ~3 voxels, so GS lanes mostly share the cache
// lines that a lane taking the whole group would ask for one after the other.
template <int FILT, int GS, typename PV, typename F>
__device__ __forceinline__ void gather_groups(const PV& vol, const float4* item, uint32_t n,
                                              uint32_t lane, const SharedRays& rays, F&& post) {
    constexpr uint32_t IPB = 64u / GS;
    float on[GS];  // on[k]: 1 in the lanes past sample k
#pragma unroll
    for (int k = 0; k < GS; ++k) on[k] = (int)(lane % GS) > k ? 1.0f : 0.0f;
    auto value = [&](uint32_t b, uint32_t& w) {
        const float4 it = item[min(b * IPB + lane / GS, n - 1u)];
        w = __float_as_uint(it.w);
        const uint32_t ray = w & 63u;
        float qx = it.x, qy = it.y, qz = it.z;
        const float ex = rays.step[0][ray], ey = rays.step[1][ray], ez = rays.step[2][ray];
#pragma unroll
        for (int k = 0; k + 1 < GS; ++k) {  // (fma(e, 1, q) is q + e, rounded once)
            qx = fmaf(ex, on[k], qx);
            qy = fmaf(ey, on[k], qy);
            qz = fmaf(ez, on[k], qz);
        }
        return window_sample<FILT>(vol, qx, qy, qz);
    };
    if (n == 64u) {
        decltype(window_sample<FILT>(vol, 0.0f, 0.0f, 0.0f)) v[GS];
        uint32_t w[GS];
#pragma unroll
        for (int b = 0; b < GS; ++b) v[b] = value((uint32_t)b, w[b]);
#pragma unroll
        for (int b = 0; b < GS; ++b) post((uint32_t)b, v[b], w[b]);
    } else {
#pragma unroll 1
        for (uint32_t b = 0; b * IPB < n; ++b) {
            uint32_t w;
            const auto v = value(b, w);
            post(b, v, w);
        }
    }
}

// the larger of a value and its neighbour's, 1 or 2 lanes away within each four
template <int AWAY>
__device__ __forceinline__ float max_quad(float v) {
    constexpr int perm = AWAY == 1 ? 0xB1 : 0x4E;  // quad_perm [1,0,3,2], [2,3,0,1]
    return fmaxf(v, __uint_as_float(__builtin_amdgcn_mov_dpp(__float_as_uint(v), perm, 0xF, 0xF, true)));
}

template <typename T, bool POW2, int GS, bool WIDE, int FILT>
__device__ __forceinline__ void mip_windows_rays(const PaddedVolume<T, POW2, WIDE>& vol,
                                                 const RayParams& p, uint32_t x, uint32_t y,
                                                 bool inside, float* __restrict__ out,
                                                 float* __restrict__ alpha, WindowShared& sh) {
    using PV = PaddedVolume<T, POW2, WIDE>;
    constexpr bool kShort = !std::is_same<T, float>::value;
    constexpr bool kPair = std::is_same<T, U16Pair>::value;  // out: two planes of W x H
    static_assert(!kPair || (FILT == 0 && !WIDE), "pairs: linear filter, volumes below 4 GiB");
    constexpr int BS = kWinGroups * GS;
    const uint32_t lane = threadIdx.x & 63u, seg = threadIdx.x >> 6;
    // one wave sets the rays up (~300 instructions, most of them divisions)
    float px = 0.5f, py = 0.5f, pz = 0.5f, dx = 0.0f, dy = 0.0f, dz = 0.0f, tnear = 0.0f;
    if (seg == 0) {
        const bool hits = inside && staged_ray_pos(p, x, y, px, py, pz, dx, dy, dz, tnear);
        if (inside && !hits) {
            out[x + p.W * y] = 0.0f;
            alpha[x + p.W * y] = kShort ? 0.0f : -1.0f;
            if constexpr (kPair) out[x + p.W * y + p.W * p.H] = 0.0f;
        }
        const uint64_t act = __ballot(hits);
        if (act != 0) shadow_first_active(act, hits, px, py, pz, dx, dy, dz);
        sh.rays.put(lane, act, px, py, pz, dx, dy, dz);
        sh.top[lane] = 0u;
        sh.top2[lane] = 0u;
    }
    __syncthreads();
    const bool active = (sh.rays.act >> lane & 1u) != 0;
    if (sh.rays.act == 0) return;  // uniform over the workgroup
    if (seg != 0) sh.rays.get(lane, px, py, pz, dx, dy, dz);
    float4* const item = sh.item[seg];
    const int total = (p.nouter + 1) * kLoopUnroll;
    const int per = ((total + BS - 1) / BS + kWinSegments - 1) / kWinSegments * BS;
    const int s0 = min((int)seg * per, total);
    const int count = min(per, total - s0);
    px = sum_n(px, dx, (uint32_t)s0);
    py = sum_n(py, dy, (uint32_t)s0);
    pz = sum_n(pz, dz, (uint32_t)s0);
    const float mg = window_margin(p, kMipMargin);
    const float mgx = mg * vol.fnx + 0.01f, mgy = mg * vol.fny + 0.01f, mgz = mg * vol.fnz + 0.01f;
    Opacity op;  // (unused)
    WindowRay<PV, GS> win;
    win.begin(vol, dx, dy, dz, mgx, mgy, mgz);
    T cur[kWinGroups], nxt[kWinGroups];
    if (count > 0) {
        win.ask(vol, px, py, pz, mgx, mgy, mgz, 0.0f, vol.win_max, cur);
        const int first = win.best(vol, px, py, pz, count);
        float qx = sum_n(px, dx, (uint32_t)first), qy = sum_n(py, dy, (uint32_t)first),
              qz = sum_n(pz, dz, (uint32_t)first), c = 0.0f;
        if constexpr (kPair) {
            float c2 = 0.0f;
            staged_sample_global_pair<PV, 2 * GS>(vol, qx, qy, qz, dx, dy, dz, c2, c);
            if (c2 > 0.0f) atomicMax(&sh.top2[lane], __float_as_uint(c2));
        } else {
            staged_sample_global<PV, 2 * GS, false, FILT>(vol, qx, qy, qz, dx, dy, dz, c, op);
        }
        if (c > 0.0f) atomicMax(&sh.top[lane], __float_as_uint(c));
    }
    __syncthreads();
    uint32_t waiting = 0;  // items in the queue (uniform)
    // n items from the queue's end, one a lane
    auto take = [&](uint32_t n) {
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        waiting -= n;
        auto raise = [&](uint32_t* word, float v) {
            float c = fmaxf(v, 0.0f);
            if constexpr (GS >= 2) c = max_quad<1>(c);
            if constexpr (GS >= 4) c = max_quad<2>(c);
            if (lane % GS == 0 && c > 0.0f) atomicMax(word, __float_as_uint(c));
        };
        gather_groups<FILT, GS>(vol, item + waiting, n, lane, sh.rays,
                                [&](uint32_t, auto v, uint32_t ray) {
                                    if constexpr (kPair) {
                                        raise(&sh.top[ray], v.v1);
                                        raise(&sh.top2[ray], v.v0);
                                    } else {
                                        raise(&sh.top[ray], v);
                                    }
                                });
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    for (int s = 0; s < count; s += BS) {
        if (s + BS < count)
            win.ask(vol, px, py, pz, mgx, mgy, mgz, (float)kWinGroups, vol.win_max, nxt);
        // (other waves may raise it meanwhile: a stale value only asks for more groups)
        auto now = [](const uint32_t* word) {
            return __uint_as_float(
                __hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP));
        };
        const float col = now(&sh.top[lane]), col2 = kPair ? now(&sh.top2[lane]) : 0.0f;
#pragma unroll
        for (int j = 0; j < kWinGroups; ++j) {
            bool rises = win_value(cur[j]) > col;
            if constexpr (kPair) rises = rises || win_value2(cur[j]) > col2;
            const bool need = active && s + j * GS < count && (!win.ok || rises);
            const uint64_t m = __ballot(need);
            if (need)
                item[waiting + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] =
                    float4{px, py, pz, __uint_as_float(lane)};
            waiting += (uint32_t)__popcll(m);
            if (waiting >= 64u) take(64u);
#pragma unroll
            for (int k = 0; k < GS; ++k) {
                px = px + dx;
                py = py + dy;
                pz = pz + dz;
            }
            cur[j] = nxt[j];
        }
    }
    if (waiting) take(waiting);
    __syncthreads();
    if (active && seg == 0) {
        const float col = __uint_as_float(sh.top[lane]);
        if constexpr (kPair) {
            staged_ray_end<kShort>(p, x + p.W * y, __uint_as_float(sh.top2[lane]), tnear, out, alpha);
            staged_plane_end(p, x + p.W * y + p.W * p.H, col, out);
        } else {
            staged_ray_end<kShort>(p, x + p.W * y, col, tnear, out, alpha);
        }
    }
}

template <typename T, bool POW2, int GS, bool WIDE, int FILT>
__global__ __launch_bounds__(64 * kWinSegments, (kWinWaves<T, GS, FILT>)) void k_mip_windows(
    PaddedVolume<T, POW2, WIDE> vol, RayParams p, float* __restrict__ out, float* __restrict__ alpha) {
    static_assert(FILT == 0 || !WIDE, "nearest: volumes below 4 GiB");
    __shared__ WindowShared sh;
    if (gate_closed(p)) return;  // uniform over the launch
    uint32_t x = 0, y = 0;
    const bool inside = wave_tile_pixel(p, blockIdx.x, &x, &y);
    mip_windows_rays<T, POW2, GS, WIDE, FILT>(vol, p, x, y, inside, out, alpha, sh);
}

// The frames of a batch (many volumes x poses, or frames of their own sizes and settings)
// the same way, one launch.  Uniform batches: grid.y = job.  Mixed ones: job k's first
// workgroup in jobs[k].first[0].  A workgroup per quarter instead of persistent ones
// claiming tiles: the workgroups are short and hold 10 KB of LDS, so the next ones fill in.
// gates: nullptr, or one device word per frame (0: the frame is left untouched).
template <typename T, bool POW2, int GS, int FILT>
__global__ __launch_bounds__(64 * kWinSegments, (kWinWaves<T, GS, FILT>)) void k_mip_windows_batch(
    const BatchJob* __restrict__ jobs, RayParams shared, uint32_t njobs, bool mixed,
    const uint32_t* __restrict__ gates) {
    __shared__ WindowShared sh;
    uint32_t jid = blockIdx.y, b = blockIdx.x;
    if (mixed) {
        jid = batch_job_of(jobs, njobs, 0, b);
        b -= jobs[jid].first[0];
    }
    if (gates != nullptr && gates[jid] == 0u) return;  // uniform: a closed frame
    const BatchJob& j = jobs[jid];
    RayParams p = shared;
    batch_params(p, j, mixed);
    uint32_t x = 0, y = 0;
    const bool inside = wave_tile_pixel(p, b, &x, &y);
    mip_windows_rays<T, POW2, GS, false, FILT>(job_volume<T, POW2>(j), p, x, y, inside, j.out, j.alpha,
                                               sh);
}

// Iso-surface march by the window grid (iso_kernel.cl:83-131, k_iso_surface): sample 0 sets a
// ray's side, the first later sample on the other side is the crossing.  A group is sampled
// only when its window reaches the other side of the iso value.  The four waves of an 8x8
// quarter take every fourth group each, so they move front to back together and stop together;
// waiting groups are queued and gathered 64 at a time as above, a crossing is posted as the
// least sample index, and no group past a posted one is queued: rays that cross at once (white
// noise, 256^3 float, 800^2, 200 steps) take 259 us, 284 with every fourth run of eight groups
// a wave and crossings looked up once a run, 250 staged.  Noise that reaches the iso value now and then
// all along the rays stays 5-20% slower than staged: no window falls away.  The refinement, the
// gradient and the shading then run per ray (iso_finish).
//
// Bound by VALU (65% busy; address units 40%): ~5 instructions a sample in windows on one
// side, the rest in groups near surfaces, their exact positions and the finish.  512^3
// uint16 -> 1024^2, 896 steps: frame 467 us (487 with runs of groups a wave, 511
// with a lane taking a whole group; march of the frame 412 us before that, 828 us staged with 8^3
// brick tests of a wave's box).
struct IsoWindowShared {
    float4 item[kWinSegments][128];  // position; w's bits: ray | side << 6 | first sample << 7
    SharedRays rays;
    uint64_t above;    // the rays that start above the iso value
    uint32_t hit[64];  // the rays' least crossing sample (~0: none)
};
// Waves per SIMD that the registers are held to (1: none).  The finish of a ray is one wave's work,
// so the workgroups resident count: left alone trilinear uint8 frames take 139 registers (1200^2
// frames of 128^3 white noise, 112 steps, 550 us, held to five 450; 512x512x256 blobs, 768 steps 561 /
// 520).  The others take 100 to 112 and gain nothing on average (300 frames of 48 to 1,024 voxels an
// axis drawn at random 1.7% slower held to five, those of few rays 2%).
template <typename T, int FILT>
constexpr int kIsoWaves = std::is_same<T, uint8_t>::value && FILT == 0 ? 5 : 1;
constexpr uint32_t kIsoAnchor = 900;  // samples that a lookup may lie past an exact position
constexpr int kIsoWindowMaxSteps = 1 << 24;

template <typename T, bool POW2, int GS, bool WIDE, int FILT>
__global__ __launch_bounds__(64 * kWinSegments, (kIsoWaves<T, FILT>)) void k_iso_windows(
    PaddedVolume<T, POW2, WIDE> vol, RayParams p, float* __restrict__ out, float* __restrict__ alpha,
    float* __restrict__ depth, float* __restrict__ normals) {
    using PV = PaddedVolume<T, POW2, WIDE>;
    static_assert(FILT == 0 || !WIDE, "nearest: volumes below 4 GiB");
    constexpr uint32_t NS = kWinSegments * GS, RS = kWinGroups * NS;  // samples from one of a wave's
                                                                     // groups, runs to the next
    __shared__ IsoWindowShared sh;
    const uint32_t lane = threadIdx.x & 63u, seg = threadIdx.x >> 6;
    uint32_t x = 0, y = 0;
    const bool inside = wave_tile_pixel(p, blockIdx.x, &x, &y);
    const uint32_t o = x + p.W * y;
    F4 orig = mk4(0, 0, 0, 0), direc = mk4(0, 0, 0, 0), pos0 = mk4(0.5f, 0.5f, 0.5f, 0.0f),
       delta = mk4(0, 0, 0, 0);
    float tnear = 0.0f, tfar = 0.0f, dt = 0.0f;
    float px = 0.5f, py = 0.5f, pz = 0.5f, dx = 0.0f, dy = 0.0f, dz = 0.0f;
    if (seg == 0) {  // one wave sets the rays up and takes sample 0
        bool hits = false;
        if (inside) {
            ray_setup(p.invP, p.invM, x, y, p.W, p.H, &orig, &direc);
            hits = intersect_box(orig, direc, p.box, &tnear, &tfar);
            if (hits) {
                if (tnear < 0.0f) tnear = 0.0f;
                dt = 1.0f * (tfar - tnear) / ((float)p.max_steps - 1.0f);
                delta = scl4(0.5f * dt, direc);
                pos0 = scl4(0.5f, add4(mk4(1.0f + orig.x, 1.0f + orig.y, 1.0f + orig.z,
                                           1.0f + orig.w),
                                       scl4(tnear, direc)));
                px = pos0.x;
                py = pos0.y;
                pz = pos0.z;
                dx = delta.x;
                dy = delta.y;
                dz = delta.z;
            } else {
                iso_miss(o, out, alpha, depth, normals);
            }
        }
        const uint64_t act = __ballot(hits);
        if (act != 0) shadow_first_active(act, hits, px, py, pz, dx, dy, dz);
        sh.rays.put(lane, act, px, py, pz, dx, dy, dz);
        sh.hit[lane] = 0xFFFFFFFFu;
        const uint64_t above =
            act != 0 ? __ballot(vol.template sample<FILT>(px, py, pz) > p.iso_val) : 0;
        if (lane == 0) sh.above = above;
    }
    __syncthreads();
    if (sh.rays.act == 0) return;  // uniform over the workgroup
    const bool active = (sh.rays.act >> lane & 1u) != 0;
    const bool gt = (sh.above >> lane & 1u) != 0;  // the ray's side
    if (seg != 0) sh.rays.get(lane, px, py, pz, dx, dy, dz);
    const float mg = window_margin(p, kIsoMargin);
    const float mgx = mg * vol.fnx + 0.01f, mgy = mg * vol.fny + 0.01f, mgz = mg * vol.fnz + 0.01f;
    WindowRay<PV, GS> win;
    win.begin(vol, dx, dy, dz, mgx, mgy, mgz);
    const T* const plane = gt ? vol.win_min : vol.win_max;
    float4* const item = sh.item[seg];
    uint32_t waiting = 0;  // items in the queue (uniform)
    auto take = [&](uint32_t n) {
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        waiting -= n;
        gather_groups<FILT, GS>(vol, item + waiting, n, lane, sh.rays,
                                [&](uint32_t, float v, uint32_t w) {
                                    const uint32_t k = (w >> 7) + lane % GS;
                                    if ((v > p.iso_val) != ((w >> 6 & 1u) != 0) &&
                                        k < (uint32_t)p.max_steps)
                                        atomicMin(&sh.hit[w & 63u], k);
                                });
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    const uint32_t nsteps = (uint32_t)p.max_steps;
    // (px, py, pz): the exact position of sample ka, a whole number of groups from k0 and at
    // most kIsoAnchor samples before the last one asked for; a run without waiting groups
    // moves only k0
    uint32_t k0 = seg * (uint32_t)GS, ka = 0;
    auto ask = [&](uint32_t k, T (&u)[kWinGroups]) {
        win.template ask<kWinSegments>(vol, px, py, pz, mgx, mgy, mgz, (float)((int)(k - ka) / GS), plane, u);
    };
    auto anchor = [&](uint32_t k) {
        px = sum_n(px, dx, k - ka);
        py = sum_n(py, dy, k - ka);
        pz = sum_n(pz, dz, k - ka);
        ka = k;
    };
    T cur[kWinGroups], nxt[kWinGroups];
    ask(k0, cur);
    for (; k0 < nsteps; k0 += RS) {
        const uint32_t hit = min(nsteps, __hip_atomic_load(&sh.hit[lane], __ATOMIC_RELAXED,
                                                           __HIP_MEMORY_SCOPE_WORKGROUP));
        if (__ballot(active && k0 < hit) == 0) break;  // every ray has crossed before
        if (k0 + 2u * RS > ka + kIsoAnchor) anchor(k0);
        ask(k0 + RS, nxt);
        uint32_t mask = 0, any = 0;  // groups that may cross: this ray's, some ray's (uniform)
#pragma unroll
        for (int j = 0; j < kWinGroups; ++j) {
            const uint32_t k = k0 + (uint32_t)(j * NS);
            const bool need = active && k < hit && (!win.ok || ((float)cur[j] > p.iso_val) != gt);
            mask |= need ? 1u << j : 0u;
            any |= __ballot(need) != 0 ? 1u << j : 0u;
            cur[j] = nxt[j];
        }
        if (any == 0) continue;
        const uint32_t first = (uint32_t)__builtin_ctz(any);
        anchor(k0 + first * NS);
        float qx = px, qy = py, qz = pz;
        for (uint32_t j = first; any >> j != 0u; ++j) {
            if (any >> j & 1u) {
                // (not past a crossing that the groups before have shown)
                const bool need = (mask >> j & 1u) != 0 &&
                                  k0 + j * NS <
                                      __hip_atomic_load(&sh.hit[lane], __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_WORKGROUP);
                const uint64_t m = __ballot(need);
                if (need)
                    item[waiting + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] =
                        float4{qx, qy, qz,
                               __uint_as_float(lane | (gt ? 64u : 0u) | (k0 + j * NS) << 7)};
                waiting += (uint32_t)__popcll(m);
                if (waiting >= 64u) take(64u);
            }
#pragma unroll
            for (uint32_t k = 0; k < NS; ++k) {
                qx = qx + dx;
                qy = qy + dy;
                qz = qz + dz;
            }
        }
        if (waiting) take(waiting);  // (a crossing found now saves the groups behind it)
    }
    __syncthreads();
    if (!active || seg != 0) return;
    const uint32_t hit = sh.hit[lane];
    if (hit == 0xFFFFFFFFu) {
        iso_miss(o, out, alpha, depth, normals);
        return;
    }
    iso_finish<FILT>(vol, p, o, tnear, dt, delta, pos0, (int)hit, gt ? 1 : 0, direc, out, alpha,
                     depth, normals);
}

}  // namespace spr
