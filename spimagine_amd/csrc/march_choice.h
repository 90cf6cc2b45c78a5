// march_choice.h -- which march a frame or a batch takes (host).
#pragma once
#include <math.h>

namespace spr {

// Whether frames are gathered group by group (k_mip_windows) instead of staged box by box, or
// read sample by sample from the persistent queues (batches with the nearest filter).
// need: the volume's share of windows to sample (k_ray_need); step: voxels a sample; hits: 8x8
// pixel quarters of all frames whose rays hit the volume.  True for fewer hits where it is for more.
//
// A gathered trilinear sample costs ~1.5 times a staged one at a fine step, so most groups have
// to fall away there.  From 1.5 voxels a step on a staged box holds few samples of many voxels.
// Few quarters leave the GPU (2,048 of its waves) idle unless their rays' segments are marched
// side by side, and leave a persistent launch's workgroups without tiles.  A nearest sample is
// one load, cheaper than its share of a staged box unless rays are short and leave little to
// skip; the queues' are as cheap as a lookup while neighbouring rays share the lines of a volume
// that the caches hold.  In volumes of few voxels (nmax, the largest dimension) most of a march
// is its set-up and first samples.
//
// The lines by hits: over 1,200 frames and batches of 48^3 to 1024^2 x 512 voxels drawn at random,
// seen whole and in part, the march chosen takes 1-3% more than the better one (26% with all
// quarters counted for the hit ones, 1.02 to 1.07 with every frame gathered).  us staged / gathered:
//   frames 150x150x147 uint16 (need 0.35), 200 steps, 150 hits of 748 quarters 105 / 28; 643x287x108
//     (0.62), 278 of 5,940 132 / 78; 87x85x147 white noise, 15,700 hits 107 / 182
//   nearest, 446x450x309 shell (0.57), 3,022 hits 126 / 92; 172x61x89 spots in noise, 9,700 41 / 57
//   batches 57x131x368 texture (0.36), 5,429 hits of 34,860 779 / 360; 120x464x357 noisy spots, 1,852
//     779 / 1264; nearest 140x210x242 shell (0.61), 108,000 1318 / 2680; 72x96x212 (0.37), 813 236 / 50
//
// Beyond those each line lies below the smallest need at which one of 15 kinds of volume (blobs in
// noise of 0.5 to 30% of their height, spots in noise, textures, white noise, sparse voxels,
// labels, a shell; 112 to 512 voxels, uint16 and float) ran more than 3-6% slower gathered:
//   linear, from 224 voxels: 0.55 at coarse steps: shell (need 0.57), 384^3, 1000^2, 200 steps 281 / 340;
//     0.35 and 0.23 (from 320) at fine ones: float texture (0.39) 256^3, 1000^2, 448 steps 366 / 425,
//     512^3 (0.26), 768 steps 571 / 617, gained below: blobs (0.13) 571 / 520, batches of it 0.65
//   192^3: 0.4 and 0.27: texture (0.43), 24 x 500^2, 112 steps 1447 / 1620; float blobs (0.29), 1000^2,
//     336 steps 282 / 330; 112^3 and 128^3: 0.3: texture (0.34), 6 x 800^2, 200 steps 950 / 1130
//   nearest, from 224 voxels: 0.55; 192^3: 0.4: texture (0.43), 1000^2, 200 steps 124 / 141; smaller:
//     labels (0.10), 1000^2, 112 steps 86 / 95
//   nearest batches of 20,000: shell (0.57) 384^3, 6 x 800^2 911 / 966; texture (0.39) 256^3, 448 steps
//     1010 / 1050; labels (0.10) 128^3, 24 x 500^2, 112 steps 22% slower, blobs (0.15) 256^3, 200 steps
//     604 / 713
inline bool windows_pay(bool nearest, bool batch, float need, int nmax, float step, float hits) {
    if (hits < (nearest ? (batch ? 8000.0f : nmax >= 190 ? 6000.0f : 1500.0f)
                : batch ? 1500.0f
                : need < 0.9f ? (step >= 2.0f ? 3000.0f : 700.0f) : (step >= 2.0f ? 1500.0f : 500.0f)))
        return true;
    if (hits < (batch ? (nearest ? 12000.0f : 6000.0f) : 1000.0f) && need < (batch ? 0.7f : 0.6f))
        return true;
    if (nearest && batch && hits >= 20000.0f)
        return nmax >= 320 ? need < 0.5f : nmax >= 224 && step < 1.0f && need < 0.35f;
    if (nearest && nmax < 160 && !batch && hits >= 4000.0f) return false;
    if (nearest) return need < (nmax >= 160 && nmax < 224 && !batch ? 0.4f : 0.55f);
    const bool coarse = step >= 1.5f;
    if (nmax < 160) return need < 0.3f;
    if (nmax < 224) return need < (coarse ? 0.4f : 0.27f);
    return need < (coarse ? 0.55f : nmax < 320 ? 0.35f : 0.23f);
}

// The share of a frame's rays that hit its box: of 8x8 spread over the frame, set up as ray_setup
// does (a box behind the camera is hit too, as by the march).  ~1 us, asked only where the answer
// can change the march.
inline float hit_share(const float* invP, const float* invM, const float* box) {
    int hit = 0;
    for (int k = 0; k < 64; ++k) {
        const float u = ((float)(k & 7) - 3.5f) * 0.25f, v = ((float)(k >> 3) - 3.5f) * 0.25f;
        float f[4], b[4], near = -__builtin_inff(), far = __builtin_inff();
        for (int r = 0; r < 4; ++r) {
            const float at = invP[4 * r] * u + invP[4 * r + 1] * v + invP[4 * r + 3];
            f[r] = at - invP[4 * r + 2];
            b[r] = at + invP[4 * r + 2];
        }
        for (int r = 0; r < 3; ++r) {
            f[r] /= f[3];
            b[r] = b[r] / b[3] - f[r];
        }
        for (int r = 0; r < 3; ++r) {
            const float* m = invM + 4 * r;
            const float o = m[0] * f[0] + m[1] * f[1] + m[2] * f[2] + m[3],
                        d = 1.0f / (m[0] * b[0] + m[1] * b[1] + m[2] * b[2]);
            const float t0 = (box[2 * r] - o) * d, t1 = (box[2 * r + 1] - o) * d;
            near = fmaxf(near, fminf(t0, t1));
            far = fminf(far, fmaxf(t0, t1));
        }
        hit += near < far ? 1 : 0;
    }
    return (float)hit / 64.0f;
}

}  // namespace spr
