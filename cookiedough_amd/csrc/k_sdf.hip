// k_sdf.hip -- sphere tracer of the synthetic SDF scene.
//
// Structure of the reference tracers (RenderSpikeyMap_2x2_Distant,
// code/shadertoy.cpp:525-598): `for (step = 0; march > eps && step < max;
// ++step) { hit = o + d*total; march = sdf(hit); total += march; }` (plus a
// far clip), shading wherever the march stopped, ExpFog, a vLerp4 towards
// the fog colour with alpha, GammaAdj and ToPixel4 packing
// (code/shadertoy-util.h:62,136-146,186-190,237-241).
//
// The march, the hit point and the central-difference normal are FP32.
// Shading (Lambert, albedo, fog blend, gamma) is FP32 for CKD_SHADE_FP32 and
// packed FP16 (two channels per register, FP32 for the fog exponent and
// the final 255 scale) for CKD_SHADE_FP16.
//
// A 256-lane block renders a 16x16 tile as four 8x8 wave tiles, so the
// lanes of a wave march neighbouring rays.
#include "ckd_internal.h"
#include "ckd_pixel.h"
#include "ckd_jobs.h"

#include <algorithm>
#include <cmath>
#include <type_traits>


namespace {

// output pixels in the global address space
typedef __attribute__((address_space(1))) uint32_t global_px;

typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));

// v_sqrt_f32 (1 ulp) for the distance field; the default sqrtf is the
// correctly rounded multi-instruction sequence
CKD_DEV float fsqrt(float x) { return __builtin_amdgcn_sqrtf(x); }

struct SdfCam {
    float o[3], f[3], r[3], u[3];
};

CKD_DEV uint32_t to_chan(float c)
{
    // _mm_cvtps_epi32 (round to nearest even) of 255*c, max 0, saturate
    const float v = rintf(255.f * c);
    return v > 0.f ? (v < 255.f ? (uint32_t)v : 255u) : 0u;
}

// total: the ray's length; nl2: the normal's squared length (it is not yet of
// unit length); ndl: its product with the light's direction
template <bool kHalf>
CKD_DEV uint32_t shade_lit(const ckd_sdf_scene &sc, float total, float nl2, float ndl, int id)
{
    const float t3 = total * total * total;
    if (!kHalf) {
        const float nl = fsqrt(nl2);
        const float inl = nl > 0.f ? 1.f / nl : 0.f;
        float diff = ndl * inl;
        diff = diff > 0.f ? diff : 0.f;
        const float lit = sc.ambient + (1.f - sc.ambient) * diff;
        const float fog = 1.f - expf(-sc.fogDensity * t3);
        uint32_t px = 0;
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const float base = sc.albedo[id][c] * lit;
            const float col = base + fog * (sc.fogColor[c] - base);
            const float g = col > 0.f ? expf(sc.gamma * logf(col)) : 0.f;
            px |= to_chan(g) << (8 * c);
        }
        const float ga = fog > 0.f ? expf(sc.gamma * logf(fog)) : 0.f;
        return px | (to_chan(ga) << 24);
    } else {
        // the normalisation scale and the dot product with the light stay
        // FP32 (rsqrt of a sum of squares of small differences); albedo,
        // lighting, fog blend and gamma run on packed halves
        const float inl = nl2 > 0.f ? rsqrtf(nl2) : 0.f;
        const float diffF = ndl * inl;
        const h2 diff = h2((_Float16)(diffF > 0.f ? diffF : 0.f));
        const h2 amb = h2((_Float16)sc.ambient);
        const h2 lit = (h2((_Float16)1.f) - amb) * diff + amb;
        const _Float16 fogE = __builtin_elementwise_exp2((_Float16)(-sc.fogDensity * t3 * 1.44269504f));
        const h2 fog = h2((_Float16)1.f - fogE);
        const h2 albBG = {(_Float16)sc.albedo[id][0], (_Float16)sc.albedo[id][1]};
        const h2 albRA = {(_Float16)sc.albedo[id][2], (_Float16)0.f};
        const h2 fogBG = {(_Float16)sc.fogColor[0], (_Float16)sc.fogColor[1]};
        const h2 fogRA = {(_Float16)sc.fogColor[2], (_Float16)1.f};
        const h2 baseBG = albBG * lit, baseRA = albRA * lit;
        const h2 cBG = fog * (fogBG - baseBG) + baseBG;
        const h2 cRA = fog * (fogRA - baseRA) + baseRA;
        const h2 g = h2((_Float16)sc.gamma);
        const h2 tiny = h2((_Float16)6.1e-5f);
        // c^gamma = exp2(gamma*log2(c)); c == 0 stays 0
        h2 pBG = __builtin_elementwise_exp2(g * __builtin_elementwise_log2(__builtin_elementwise_max(cBG, tiny)));
        h2 pRA = __builtin_elementwise_exp2(g * __builtin_elementwise_log2(__builtin_elementwise_max(cRA, tiny)));
        const float b = cBG.x > (_Float16)0.f ? (float)pBG.x : 0.f;
        const float gg = cBG.y > (_Float16)0.f ? (float)pBG.y : 0.f;
        const float r = cRA.x > (_Float16)0.f ? (float)pRA.x : 0.f;
        const float a = cRA.y > (_Float16)0.f ? (float)pRA.y : 0.f;
        return to_chan(b) | (to_chan(gg) << 8) | (to_chan(r) << 16) | (to_chan(a) << 24);
    }
}

CKD_DEV void count_steps(unsigned long long *stepCount, int steps)
{
    if (!stepCount) return;
    unsigned long long s = (unsigned long long)steps;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) atomicAdd(stepCount, s);
}

// ---- persistent batched tracer ------------------------------------------
//
// One launch renders every SDF request of a batch.  Each wave pulls square
// pixel chunks (sdf_chunk_side) from global queues (one atomic per chunk).
// At its start it finds the spheres that can be the nearest surface anywhere
// on the chunk's rays (chunk_spheres); the march evaluates only those.  Inside
// a chunk
// the wave keeps its 64 lanes busy: lanes whose ray has finished are
// refilled with the chunk's next pixels (ballot + mbcnt ranks), so a
// long-marching ray no longer holds 63 idle lanes.  Finished rays are
// pushed to a per-wave LDS queue and shaded 64 at a time, so shading also
// runs with full waves.
//
// The march evaluates |o + t*d - c|^2 about the ray's closest approach to
// each centre: with m = d.(o-c) and w = (o-c) - m*d (the centre's offset
// perpendicular to the ray, |w| about the radius near a silhouette),
// |o + t*d - c|^2 = (t + m)^2 + |w|^2 for a unit d.  Per sphere and step
// that is an add, an FMA, a square root, a subtract and a min.  Both
// per-ray constants carry absolute errors of order 1e-6, as the direct
// form |p - c|^2 does; the expanded t^2 + t*B + |o-c|^2 cancels terms of
// several hundred and is off by up to 1e-4 near a surface, which decides
// hit or miss for rays that pass within that much of the 1e-3 threshold
// and moves rays that run out of steps.

struct ShadeEntry {
    uint32_t job, xy; // xy = x | y << 16 (W <= 4096, H <= 2160)
    float tHit, total;
    // the ray's direction as its set-up computed it: shading reads it rather
    // than computing it again from the job's camera
    float dx, dy, dz, pad;
};

constexpr int kQueueCap = 128;
constexpr int kWavesPerBlock = 4;

CKD_DEV uint32_t lane_id() { return __lane_id(); }

// the lane's bit of the wave mask m ? a : b: one v_cndmask that reads m from
// SGPRs (a select on a bool the compiler rebuilds from the mask costs it
// three compares again)
CKD_DEV float sel_lane(uint64_t m, float a, float b)
{
    float r;
    asm("v_cndmask_b32_e64 %0, %1, %2, %3" : "=v"(r) : "v"(b), "v"(a), "s"(m));
    return r;
}
// a + the lane's bit of m: one v_addc with m as the carry in
CKD_DEV int add_lane(uint64_t m, int a)
{
    int r;
    uint64_t carry;
    asm("v_addc_co_u32_e64 %0, %1, %2, 0, %3" : "=v"(r), "=s"(carry) : "v"(a), "s"(m));
    return r;
}

// v_cmp into a wave mask (LLVM predicates: 2 ordered >, 4 ordered <, 40
// signed <); a __ballot of a bool made of several compares costs a
// v_cndmask and a v_cmp more
constexpr int kCmpGt = 2, kCmpLt = 4, kCmpSlt = 40;

// a zero the compiler cannot see through: indexing LDS tables with it keeps
// their loads inside the loop instead of hoisting every table entry into
// registers for the whole kernel
CKD_DEV uint32_t opaque_zero()
{
    uint32_t z;
    asm volatile("s_mov_b32 %0, 0" : "=s"(z));
    return z;
}

// lane k's value, in a scalar register
CKD_DEV float lane_f(float v, int k) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), k)); }

// a wave-uniform float kept in a scalar register
CKD_DEV float uniform_f(float v)
{
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// a / b rounded to nearest, from rb = 1 / b rounded to nearest: Markstein's
// correction of the quotient estimate a * rb (within an ulp) by the residual
// a - b * (a * rb), which the FMA gives exactly.  For the integers |a| <= 4096 and
// 1 <= b <= 2160 of a batch it equals the IEEE quotient bit for bit (every pair:
// tests/test_sdf_setup_arith.py); larger single frames only cull by it.
CKD_DEV float div_rn(float a, float b, float rb)
{
    const float q = a * rb;
    return fmaf(fmaf(-b, q, a), rb, q);
}

// direction of pixel (x, y) through the camera basis; invH = 1 / H rounded
// to nearest
CKD_DEV void ray_dir(const float *cam, uint32_t W, uint32_t H, float invH, uint32_t x, uint32_t y,
                     float &dx, float &dy, float &dz)
{
    const float fH = (float)H;
    const float u = div_rn(2.f * (float)x - (float)W, fH, invH);
    const float v = div_rn(fH - 2.f * (float)y, fH, invH);
    dx = cam[3] + u * cam[6] + v * cam[9];
    dy = cam[4] + u * cam[7] + v * cam[10];
    dz = cam[5] + u * cam[8] + v * cam[11];
    const float il = __builtin_amdgcn_rsqf(dx * dx + dy * dy + dz * dz);
    dx *= il;
    dy *= il;
    dz *= il;
}

// shading of one finished ray: hit point, central-difference normal with
// the six offsets taken from one |p-c|^2 per sphere
// (|p +- h e_k - c|^2 = q + h^2 +- 2 h (p-c)_k), argmin id, Lambert, fog,
// gamma, pack
// Where the spheres' bounding sphere (centre C, radius R) is farther from
// the hit point p than the ground by more than 2h (an offset of h moves a
// sphere's distance by at most h) plus the rounding margin, every sphere
// term of the six offsets and of the argmin exceeds the ground's: the
// minima are the ground's values and the id is the ground's, exactly as the
// loop over the spheres gives them.  The loop runs only when some lane of
// the wave needs it.
template <bool kHalf, int kMaxSph>
CKD_DEV uint32_t shade_hit(const ckd_sdf_scene &sc, const float *cam, float dx, float dy, float dz,
                           float tHit, float total, const f4 &bound, uint32_t &evaluated)
{
    const float hx = cam[0] + dx * tHit, hy = cam[1] + dy * tHit, hz = cam[2] + dz * tHit;
    const float h = 1e-3f, hh = h * h, h2 = 2.f * h;
    const float pl = hy - sc.groundY;
    float mxp = pl, mxm = pl, myp = pl + h, mym = pl - h, mzp = pl, mzm = pl;
    float best = pl;
    int id = sc.nSpheres;
    const float bx = hx - bound.x, by = hy - bound.y, bz = hz - bound.z;
    const float db = fsqrt(bx * bx + by * by + bz * bz) - bound.w;
    const bool near = db < fmaf(fabsf(pl), 1e-3f, pl + (2.f * h + 1e-3f));
    const bool loop = __ballot(near) != 0;
    evaluated += loop ? 1u : 0u;
    if (loop)
#pragma unroll 4
    for (int i = 0; i < kMaxSph; ++i) {
        if (i < sc.nSpheres) {
            const float ex = hx - sc.sphere[i][0], ey = hy - sc.sphere[i][1], ez = hz - sc.sphere[i][2];
            const float r = sc.sphere[i][3];
            const float q = ex * ex + ey * ey + ez * ez;
            const float qh = q + hh;
            const float c = fsqrt(q) - r;
            if (c < best) {
                best = c;
                id = i;
            }
            mxp = fminf(mxp, fsqrt(qh + h2 * ex) - r);
            mxm = fminf(mxm, fsqrt(qh - h2 * ex) - r);
            myp = fminf(myp, fsqrt(qh + h2 * ey) - r);
            mym = fminf(mym, fsqrt(qh - h2 * ey) - r);
            mzp = fminf(mzp, fsqrt(qh + h2 * ez) - r);
            mzm = fminf(mzm, fsqrt(qh - h2 * ez) - r);
        }
    }
    const float nx = mxp - mxm, ny = myp - mym, nz = mzp - mzm;
    return shade_lit<kHalf>(sc, total, nx * nx + ny * ny + nz * nz,
                            nx * sc.light[0] + ny * sc.light[1] + nz * sc.light[2], id);
}

// far above the rounding of distances in a scene of that scale, |b|^2 = bb from
// the camera to the bounding sphere's centre
CKD_DEV float cull_margin(float bb, float R) { return fmaf(1e-4f, fsqrt(bb) + R, 1e-3f); }

// The stretch (tNear, tFar) of a ray outside which no sphere can be nearer than
// the ground.  Every sphere lies inside the bounding sphere (centre C, radius
// R; b = o - C), so each one's distance is at least |p - C| - R; where that is
// at least the ground's distance g plus a margin the ground is the minimum.
// With p = o + t d and g = og + t dy that is
//   (t + m)^2 + |b|^2 - m^2 >= (a + c t)^2,  m = d.b,
//   a = 1.001 og + R + margin,  c = 1.001 dy,
// (or a + c t < 0, where it holds anyway): true outside the roots of
//   (1 - c^2) t^2 + 2 (m - a c) t + |b|^2 - a^2.
// The margin, 1e-3 + 1e-4 (|b| + R) + 1e-3 g, is far above the rounding of the
// roots and of either side (about 1e-6 of the scene's scale), also where the
// discriminant nearly vanishes: a wrong sign there moves the test by less than
// the margin.  g < 0 beyond that is met only at the first step of a camera
// below the ground: such rays, and near-vertical ones (1 - c^2 small), get the
// whole line.  Against evaluating the bound at every step this takes 4 VALU of
// a step's 14 (64 frames of 1280x720: 1459 -> 1390 us).
// spread: bound of |d' - d| over the rays d' the stretch has to hold for (their
// points at t lie within t * spread of the ray's, which moves either side of
// the test by that much).
CKD_DEV void near_interval(float bx, float by, float bz, float R, float og, float dx, float dy, float dz,
                           float spread, float &tNear, float &tFar)
{
    const float bb = bx * bx + by * by + bz * bz;
    const float m = dx * bx + dy * by + dz * bz;
    const float a = fmaf(1.001f, og, R + cull_margin(bb, R)), c = fmaf(1.001f, dy, 2.002f * spread);
    const float A = fmaf(-c, c, 1.f), B = fmaf(-a, c, m);
    const float disc = fmaf(B, B, -A * (bb - a * a));
    const float s = fsqrt(fmaxf(disc, 0.f)), inv = __builtin_amdgcn_rcpf(A);
    tNear = (-B - s) * inv;
    tFar = (-B + s) * inv;
    if (disc < 0.f || tFar < 0.f) tNear = INFINITY;
    if (!(A > 0.01f) || !(og > 0.f) || !(disc < INFINITY)) {
        tNear = -INFINITY;
        tFar = INFINITY;
    }
}

// lanes that must be idle before a wave refills them (checked every
// kStepsPerRefill march steps)
constexpr int kRefillMinIdle = 32;

// The spheres that can be the nearest surface to some point of a chunk's rays,
// as a bit mask.  The chunk's rays stay within t * spread of its central ray
// (d; spread bounds |d' - d| over the chunk).  The stretch of it that can be
// near any sphere is cut into 64 pieces, one per lane: every point of a ray in
// the piece lies within rho of the piece's middle q, and a distance changes by
// no more than the way moved.  The nearest surface at such a point is at most
// m + rho away, m the scene's distance at q, so a sphere whose distance at q
// exceeds m + 2 rho (and the rounding margin) is not the nearest anywhere in
// the piece.  One that no piece needs can be left out of the chunk's minimum,
// which stays the same to the bit.  64 frames of 1280x720 with 8 spheres: 1213
// -> 1101 us; 24 of 2560x1440 with 32: 5273 -> 2962 us.
CKD_DEV uint32_t chunk_spheres(const ckd_sdf_scene &sc, const float *cam, const f4 &bound, float bx, float by, float bz,
                               float dx, float dy, float dz, float spread, uint32_t lane, uint32_t all,
                               float slack)
{
    const float og = cam[1] - sc.groundY, bb = bx * bx + by * by + bz * bz;
    float t0, t1;
    near_interval(bx, by, bz, bound.w, og, dx, dy, dz, spread, t0, t1);
    t0 = fmaxf(t0, 0.f);
    t1 = fminf(t1, sc.tMax);
    if (__builtin_amdgcn_readfirstlane(t0 >= t1)) return 0;
    if (__builtin_amdgcn_readfirstlane(!(t1 < 1e6f))) return all;
    const float h = (t1 - t0) * (1.f / 64.f), t = fmaf((float)lane + 0.5f, h, t0);
    const float rho = fmaf(t + h, spread, 0.5f * h);
    const float qx = fmaf(t, dx, cam[0]), qy = fmaf(t, dy, cam[1]), qz = fmaf(t, dz, cam[2]);
    auto distance = [&](int i) {
        const float ex = qx - sc.sphere[i][0], ey = qy - sc.sphere[i][1], ez = qz - sc.sphere[i][2];
        return fsqrt(ex * ex + ey * ey + ez * ez) - sc.sphere[i][3];
    };
    float m = qy - sc.groundY;
#pragma unroll 4
    for (int i = 0; i < sc.nSpheres; ++i) m = fminf(m, distance(i));
    const float reach = fmaf(2.002f, rho, m) + cull_margin(bb, bound.w) + 1e-3f * fabsf(m) + slack;
    uint32_t keep = 0;
#pragma unroll 1
    for (int i = 0; i < sc.nSpheres; ++i) keep |= __ballot(!(distance(i) > reach)) ? 1u << i : 0u;
    return keep;
}

// what coordinates near the camera's lose by rounding (of the point, and of the
// differences from it), generously
CKD_DEV float origin_slack(const float *o) { return 2e-6f * (fabsf(o[0]) + fabsf(o[1]) + fabsf(o[2])); }

// chunk_spheres of the rays of w x h pixels at (x0, y0): the corners' and the
// centre's rays (lanes 0-3 and the others) give the spread, as long as they lie
// within 60 degrees.  slack widens the distances by what points beside the rays
// need.
CKD_DEV uint32_t tile_spheres(const ckd_sdf_scene &sc, const float *cam, const f4 &bound, uint32_t W, uint32_t H,
                              float invH, uint32_t x0, uint32_t y0, uint32_t w, uint32_t h, uint32_t lane, uint32_t all,
                              float slack)
{
    const uint32_t x = x0 + (lane < 4 ? (lane & 1) * (w - 1) : w >> 1);
    const uint32_t y = y0 + (lane < 4 ? (lane >> 1) * (h - 1) : h >> 1);
    float ex, ey, ez;
    ray_dir(cam, W, H, invH, x, y, ex, ey, ez);
    const float mx = lane_f(ex, 4), my = lane_f(ey, 4), mz = lane_f(ez, 4);
    const float vx = ex - mx, vy = ey - my, vz = ez - mz, v2 = vx * vx + vy * vy + vz * vz;
    if (__ballot(!(v2 < 1.f))) return all;
    const float far2 = fmaxf(fmaxf(lane_f(v2, 0), lane_f(v2, 1)), fmaxf(lane_f(v2, 2), lane_f(v2, 3)));
    const float spread = fmaf(1.01f, fsqrt(far2), 1e-5f);
    return chunk_spheres(sc, cam, bound, cam[0] - bound.x, cam[1] - bound.y, cam[2] - bound.z, mx, my, mz, spread, lane,
                         all, slack + origin_slack(cam));
}

template <bool kHalf, int kMaxSph, int kStepsPerRefill>
__global__ __launch_bounds__(256, kMaxSph > 8 ? 4 : 5) void k_sdf_persistent(uint32_t *__restrict__ queueCounter,
                                                        uint32_t totalChunks,
                                                        const SdfJob *__restrict__ jobs, int nJobs,
                                                        const ckd_sdf_scene sc,
                                                        unsigned long long *__restrict__ stepCount,
                                                        uint32_t kChunkSide, uint32_t fixedChunks, uint32_t nQueues, bool own, f4 bound,
                                                        unsigned long long *__restrict__ work)
{
    __shared__ ShadeEntry queue[kWavesPerBlock][kQueueCap];
    // the radii, read every step with broadcast LDS loads instead of
    // occupying kMaxSph scalar registers
    __shared__ f4 sphR[kWavesPerBlock][kMaxSph / 4]; // {r_4k .. r_4k+3}
    // o - c_i of the chunk's camera, read when a lane starts a ray
    __shared__ f4 sphOC[kWavesPerBlock][kMaxSph];
    __shared__ uint32_t drained; // a wave of the block found the queue empty
    if (threadIdx.x == 0) drained = 0;
    __syncthreads();
    const uint32_t lane = lane_id();
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    ShadeEntry *q = queue[wave];
    int qn = 0; // entries waiting in this wave's queue (uniform)

    // chunk state (uniform)
    int job = -1;
    uint32_t next = 0, end = 0, cx0 = 0, cy0 = 0, tilesX = 1, tilesM = 1u << 20;
    float invH = 1.f;
    float cam[12];
    uint32_t W = 0, H = 0;
    int sphGroups = 0; // the chunk's spheres (chunk_spheres), in groups of four

    // ray state (per lane)
    bool active = false;
    uint32_t xy = 0; // the ray's pixel, x | y << 16
    // The ray's last march step evaluated the field at tHit and found d; its
    // distance total is t = tHit + d, which is how the step formed it, so t
    // is recomputed from the two instead of kept.  A new ray has tHit = -1
    // and d = 1, so that t = 0; a lane without a ray has tHit = inf, so that t
    // = inf ends every march.
    float d = 1.f, tHit = INFINITY, dx = 0.f, dy = 0.f, dz = 0.f;
    int steps = 0;
    // d.(o-c_i) and |w_i|^2 of the lane's ray for the chunk's first spheres; the
    // few chunks with more compute theirs where they need them
    constexpr int kRegGroups = kMaxSph / 4 < 4 ? kMaxSph / 4 : 4;
    float M[4 * kRegGroups], E2[4 * kRegGroups];
    auto about_ray = [&](const f4 &oc, float &m, float &e2) {
        m = dx * oc.x + dy * oc.y + dz * oc.z;
        const float wx = fmaf(-m, dx, oc.x);
        const float wy = fmaf(-m, dy, oc.y);
        const float wz = fmaf(-m, dz, oc.z);
        e2 = wx * wx + wy * wy + wz * wz;
    };
    float tNear = INFINITY, tFar = 0.f; // the ray needs the spheres for t between them only
    float bx = 0.f, by = 0.f, bz = 0.f; // o - C of the chunk's camera (uniform)
    unsigned long long mySteps = 0;
    // lane march steps of the wave that evaluated the spheres (uniform), and
    // shaded pixels of this lane that did
    unsigned long long evalSteps = 0;
    uint32_t evalShades = 0;

    while (true) {
        // refill finished lanes from the current chunk, once half the wave
        // is idle: a refill runs the new rays' set-up for the whole wave, so
        // it pays to refill many lanes at once (a wave whose lanes are all
        // idle always refills)
        const uint64_t idle = __ballot(!active);
        if (idle && next < end && __popcll(idle) >= kRefillMinIdle) {
            const uint32_t rank = __popcll(idle & ((1ull << lane) - 1));
            if (!active) {
                // the chunk's 8x8 tiles one after the other (rays of a tile
                // march alike), row by row; tile / tilesX as (tile * ceil(2^20
                // / tilesX)) >> 20, exact for tile < 4096 and tilesX <= 64
                const uint32_t k = next + rank, tile = k >> 6;
                const uint32_t ty = __umul24(tile, tilesM) >> 20;
                const uint32_t x = cx0 + 8 * (tile - __umul24(ty, tilesX)) + (k & 7), y = cy0 + 8 * ty + ((k >> 3) & 7);
                if (k < end && x < W && y < H) {
                    xy = x | (y << 16);
                    ray_dir(cam, W, H, invH, x, y, dx, dy, dz);
                    near_interval(bx, by, bz, bound.w, cam[1] - sc.groundY, dx, dy, dz, 0.f, tNear, tFar);
                    if (__any(tNear < tFar)) {
                        const uint32_t z = opaque_zero();
#pragma unroll
                        for (int g = 0; g < kRegGroups; ++g) {
                            if (g >= sphGroups) break;
#pragma unroll
                            for (int i = 4 * g; i < 4 * g + 4; ++i) about_ray(sphOC[wave][i + z], M[i], E2[i]);
                        }
                    } else {
                        // no ray of this refill needs a sphere: where the rest
                        // of the wave makes them run the loop, none is near
#pragma unroll
                        for (int i = 0; i < 4 * kRegGroups; ++i) E2[i] = 1e30f;
                    }
                    d = 1.f;
                    tHit = -1.f;
                    steps = 0;
                    active = true;
                }
            }
            next = min(end, next + (uint32_t)__popcll(idle));
        }
        if (!__any(active)) {
            // a refill may have met only pixels past the image's edge
            if (next < end) continue;
            // chunk drained: take the next one.  The first fixedChunks belong
            // to the launch's waves; the others are dealt to the queues in
            // turn, a block draining its own.  Atomics on one counter queue up
            // at 11 ns each (64 frames of 1280x720 in 16x16 chunks took 2.6 ms
            // of them, 1.2 ms with eight counters 256 bytes apart), so a wave
            // that finds the queue empty also tells its block.
            uint32_t c = 0;
            if (own) {
                c = blockIdx.x * kWavesPerBlock + wave;
                own = false;
            } else {
                if (fixedChunks >= totalChunks || *(volatile uint32_t *)&drained) break;
                const uint32_t queue = blockIdx.x & (nQueues - 1);
                if (lane == 0) c = atomicAdd(queueCounter + kSdfQueueStride * queue, 1u);
                c = fixedChunks + __builtin_amdgcn_readfirstlane(c) * nQueues + queue;
            }
            if (c >= totalChunks) {
                if (lane == 0) *(volatile uint32_t *)&drained = 1u;
                break;
            }
            job = ckd_find_job(jobs, nJobs, c, &SdfJob::chunkBase);
            const SdfJob &J = jobs[job];
            W = J.W;
            H = J.H;
            invH = uniform_f(J.invH);
#pragma unroll
            for (int k = 0; k < 12; ++k) cam[k] = uniform_f(J.cam[k]);
            const uint32_t local = c - J.chunkBase;
            cx0 = (local % J.chunksX) * kChunkSide;
            cy0 = (local / J.chunksX) * kChunkSide;
            tilesX = (min((uint32_t)kChunkSide, W - cx0) + 7) / 8;
            tilesM = ((1u << 20) + tilesX - 1) / tilesX;
            next = 0;
            end = 64 * tilesX * ((min((uint32_t)kChunkSide, H - cy0) + 7) / 8);
            bx = cam[0] - bound.x;
            by = cam[1] - bound.y;
            bz = cam[2] - bound.z;
            uint32_t keep = sc.nSpheres >= 32 ? 0xffffffffu : (1u << sc.nSpheres) - 1u;
            if (kChunkSide > 8)
                keep = tile_spheres(sc, cam, bound, W, H, invH, cx0, cy0, min((uint32_t)kChunkSide, W - cx0),
                                    min((uint32_t)kChunkSide, H - cy0), lane, keep, 0.f);
            // lane i stages sphere i, those kept packed to the front; the last
            // group of four is filled up with a neutral sphere whose distance
            // is never the minimum (a centre 1e15 away, radius 0)
            sphGroups = (__popc(keep) + 3) / 4;
            if (lane < (uint32_t)kMaxSph) {
                reinterpret_cast<float *>(&sphR[wave][lane >> 2])[lane & 3] = 0.f;
                sphOC[wave][lane] = f4{1e15f, 0.f, 0.f, 0.f};
            }
            __builtin_amdgcn_wave_barrier();
            if (lane < (uint32_t)kMaxSph && (keep >> lane & 1u)) {
                const uint32_t slot = __popc(keep & ((1u << lane) - 1u));
                reinterpret_cast<float *>(&sphR[wave][slot >> 2])[slot & 3] = sc.sphere[lane][3];
                sphOC[wave][slot] = f4{cam[0] - sc.sphere[lane][0], cam[1] - sc.sphere[lane][1],
                                       cam[2] - sc.sphere[lane][2], 0.f};
            }
            __builtin_amdgcn_wave_barrier();
            continue;
        }
        // march a few steps; the lanes' conditions are wave masks in SGPRs.  A
        // block whose lanes cannot reach the step limit does without its test.
        const float oyg = cam[1] - sc.groundY;
        auto step = [&](auto limitTag) {
            const float t = tHit + d;
            uint64_t marchM = __builtin_amdgcn_fcmpf(d, sc.eps, kCmpGt) & __builtin_amdgcn_fcmpf(t, sc.tMax, kCmpLt);
            if constexpr (decltype(limitTag)::value) marchM &= __builtin_amdgcn_sicmp(steps, sc.maxSteps, kCmpSlt);
            float dist = fmaf(t, dy, oyg);
            // the spheres are evaluated only when some marching lane may need
            // them (near_interval); elsewhere the ground's distance is the
            // minimum, exactly as the loop would give it
            const uint64_t nearM =
                __builtin_amdgcn_fcmpf(t, tNear, kCmpGt) & __builtin_amdgcn_fcmpf(t, tFar, kCmpLt);
            if (marchM & nearM) {
                evalSteps += (uint32_t)__popcll(marchM);
                const uint32_t z = opaque_zero();
#pragma unroll
                for (int i = 0; i < kRegGroups; ++i) {
                    if (i >= sphGroups) break;
                    const f4 r = sphR[wave][i + z];
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const float u = t + M[4 * i + j];
                        dist = fminf(dist, fsqrt(fmaf(u, u, E2[4 * i + j])) - r[j]);
                    }
                }
                if constexpr (kMaxSph / 4 > kRegGroups) {
#pragma unroll 1
                    for (int i = kRegGroups; i < sphGroups; ++i) {
                        const f4 r = sphR[wave][i];
#pragma unroll
                        for (int j = 0; j < 4; ++j) {
                            float m, e2;
                            about_ray(sphOC[wave][4 * i + j], m, e2);
                            const float u = t + m;
                            dist = fminf(dist, fsqrt(fmaf(u, u, e2)) - r[j]);
                        }
                    }
                }
            }
            tHit = sel_lane(marchM, t, tHit);
            d = sel_lane(marchM, dist, d);
            steps = add_lane(marchM, steps);
        };
        if (__ballot(active && steps > sc.maxSteps - kStepsPerRefill) == 0) {
#pragma unroll
            for (int k = 0; k < kStepsPerRefill; ++k) step(std::false_type{});
        } else {
#pragma unroll 1
            for (int k = 0; k < kStepsPerRefill; ++k) step(std::true_type{});
        }
        const float t = tHit + d;
        // retire finished rays into the shade queue
        const bool fin = active && !(d > sc.eps && steps < sc.maxSteps && t < sc.tMax);
        const uint64_t finMask = __ballot(fin);
        if (finMask) {
            if (fin) {
                const uint32_t slot = qn + __popcll(finMask & ((1ull << lane) - 1));
                // a ray that took no step shades at its origin
                q[slot] = ShadeEntry{(uint32_t)job, xy, steps ? tHit : 0.f, t, dx, dy, dz, 0.f};
                mySteps += (unsigned long long)steps;
                active = false;
                tHit = INFINITY;
            }
            qn += __popcll(finMask);
            __builtin_amdgcn_wave_barrier();
            if (qn >= 64) {
                // shade 64 queued hits with the whole wave
                const ShadeEntry e = q[qn - 64 + lane];
                const SdfJob &J = jobs[e.job];
                const uint32_t x = e.xy & 0xffffu, y = e.xy >> 16;
                const float ex = e.dx, ey = e.dy, ez = e.dz;
                // a global store (the job's pointer would make a flat one,
                // whose completion the next LDS reads would wait for)
                ((global_px *)J.dst)[__umul24(y, J.W) + x] = shade_hit<kHalf, kMaxSph>(sc, J.cam, ex, ey, ez, e.tHit, e.total, bound, evalShades);
                qn -= 64;
                __builtin_amdgcn_wave_barrier();
            }
        }
    }
    // leftover hits
    __builtin_amdgcn_wave_barrier();
    if ((int)lane < qn) {
        const ShadeEntry e = q[lane];
        const SdfJob &J = jobs[e.job];
        const uint32_t x = e.xy & 0xffffu, y = e.xy >> 16;
        const float ex = e.dx, ey = e.dy, ez = e.dz;
        ((global_px *)J.dst)[__umul24(y, J.W) + x] = shade_hit<kHalf, kMaxSph>(sc, J.cam, ex, ey, ez, e.tHit, e.total, bound, evalShades);
    }
    if (stepCount) {
        unsigned long long s = mySteps;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
        if (lane == 0) atomicAdd(stepCount, s);
    }
    if (work) {
        unsigned long long b = evalShades;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) b += __shfl_xor(b, o, 64);
        if (lane == 0) {
            atomicAdd(work, evalSteps);
            atomicAdd(work + 1, b);
        }
    }
}

// ---- one frame per launch ----------------------------------------------------
//
// A 256-lane block renders a 16x16 tile as four 8x8 wave tiles.  The march
// evaluates the distance field directly, |p - c| - r, over the spheres that
// can be the nearest surface to some point of the tile's rays (tile_spheres,
// with 4h of slack for the normal's probes), and only on the steps where a
// lane is on the stretch of its ray that can be near any sphere
// (near_interval): the minimum is the full one to the bit.  The march is VALU
// bound (a square root and 8 more a sphere and step).  A 1280x720 frame with 8
// spheres: 65 -> 39 us with the lists and the stretch, 34 with a list's spheres four
// at a time (one at a time past the last eight, as a plain loop has them, 7 spheres
// of a 320x180 frame took 45 us, 32 now; without lists 33).
constexpr float kProbe = 1e-3f; // the normal's offset h
constexpr int kFewSpheres = 6;

// kFew: few spheres in a frame of few tiles, where a ray's chain of steps is all
// there is: every sphere on every step, from scalar registers.  cull: whether the
// tile leaves spheres out (otherwise it keeps all).  Which is taken, and the times
// either side of the lines: launch_sdf.
template <bool kHalf, bool kFew>
__global__ __launch_bounds__(256) void k_sdf(uint32_t *__restrict__ dst, unsigned W, unsigned H, float invH,
                                             const ckd_sdf_scene sc, const SdfCam cam, f4 bound, bool cull,
                                             unsigned long long *__restrict__ stepCount)
{
    __shared__ f4 spheres[32]; // the tile's: centre, radius
    __shared__ uint32_t kept;  // their mask
    const unsigned lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const unsigned x0 = blockIdx.x * 16, y0 = blockIdx.y * 16;
    if (!kFew && wave == 0) {
        const float c12[12] = {cam.o[0], cam.o[1], cam.o[2], cam.f[0], cam.f[1], cam.f[2],
                               cam.r[0], cam.r[1], cam.r[2], cam.u[0], cam.u[1], cam.u[2]};
        const uint32_t all = sc.nSpheres >= 32 ? 0xffffffffu : (1u << sc.nSpheres) - 1u;
        const uint32_t keep = cull ? tile_spheres(sc, c12, bound, W, H, invH, x0, y0, min(16u, W - x0),
                                                  min(16u, H - y0), lane, all, 4.f * kProbe)
                                   : all;
        if (lane < 32 && (keep >> lane & 1u))
            spheres[__popc(keep & ((1u << lane) - 1u))] =
                f4{sc.sphere[lane][0], sc.sphere[lane][1], sc.sphere[lane][2], sc.sphere[lane][3]};
        if (lane == 0) kept = keep;
    }
    if (!kFew) __syncthreads();
    const uint32_t keep = kFew ? (1u << sc.nSpheres) - 1u : __builtin_amdgcn_readfirstlane(kept);
    const int n = kFew ? sc.nSpheres : __popc(keep);
    const unsigned x = x0 + (wave & 1) * 8 + (lane & 7), y = y0 + (wave >> 1) * 8 + (lane >> 3);
    int step = 0;
    if (x < W && y < H) {
        const float fH = (float)H;
        const float u = (2.f * (float)x - (float)W) / fH;
        const float v = (fH - 2.f * (float)y) / fH;
        float dx = cam.f[0] + u * cam.r[0] + v * cam.u[0];
        float dy = cam.f[1] + u * cam.r[1] + v * cam.u[1];
        float dz = cam.f[2] + u * cam.r[2] + v * cam.u[2];
        const float il = __builtin_amdgcn_rsqf(fmaf(dz, dz, fmaf(dy, dy, dx * dx)));
        dx *= il;
        dy *= il;
        dz *= il;
        float tNear = -INFINITY, tFar = INFINITY;
        if (!kFew)
            near_interval(cam.o[0] - bound.x, cam.o[1] - bound.y, cam.o[2] - bound.z, bound.w + 4.f * kProbe + origin_slack(cam.o),
                      cam.o[1] - sc.groundY, dx, dy, dz, 0.f, tNear, tFar);
        // distance of sphere i of the tile's from (px, py, pz)
        auto distance = [&](int i, float px, float py, float pz) {
            const f4 c = kFew ? f4{sc.sphere[i][0], sc.sphere[i][1], sc.sphere[i][2], sc.sphere[i][3]} : spheres[i];
            const float ex = px - c.x, ey = py - c.y, ez = pz - c.z;
            return fsqrt(fmaf(ez, ez, fmaf(ex, ex, ey * ey))) - c.w;
        };
        float hx = cam.o[0], hy = cam.o[1], hz = cam.o[2];
        float d = 1.f, total = 0.f, tHit = 0.f;
        for (; d > sc.eps && step < sc.maxSteps && total < sc.tMax; ++step) {
            hx = cam.o[0] + dx * total;
            hy = cam.o[1] + dy * total;
            hz = cam.o[2] + dz * total;
            d = hy - sc.groundY;
            if (kFew) {
#pragma unroll
                for (int i = 0; i < kFewSpheres; ++i) {
                    if (i >= n) break;
                    d = fminf(d, distance(i, hx, hy, hz));
                }
            } else if (__ballot(total > tNear && total < tFar)) {
                // four at a time, then two and one: a list's latency is its groups'
                int i = 0;
                auto next = [&](auto count) {
#pragma unroll
                    for (int k = 0; k < decltype(count)::value; ++k) d = fminf(d, distance(i + k, hx, hy, hz));
                    i += decltype(count)::value;
                };
                while (i + 4 <= n) next(std::integral_constant<int, 4>{});
                if (n & 2) next(std::integral_constant<int, 2>{});
                if (n & 1) next(std::integral_constant<int, 1>{});
            }
            tHit = total;
            total += d;
        }
        // the normal's probes and the nearest surface (the first of equals)
        const float h = kProbe;
        int id = sc.nSpheres;
        float p[6] = {hy - sc.groundY, hy - sc.groundY, hy + h - sc.groundY, hy - h - sc.groundY,
                      hy - sc.groundY, hy - sc.groundY};
        if (kFew || __ballot(tHit > tNear && tHit < tFar)) {
            float best = hy - sc.groundY;
            uint32_t rest = keep;
            for (int i = 0; i < n; ++i) {
                const int original = __builtin_ctz(rest);
                rest &= rest - 1;
                const float l = distance(i, hx, hy, hz);
                if (l < best) {
                    best = l;
                    id = original;
                }
                p[0] = fminf(p[0], distance(i, hx + h, hy, hz));
                p[1] = fminf(p[1], distance(i, hx - h, hy, hz));
                p[2] = fminf(p[2], distance(i, hx, hy + h, hz));
                p[3] = fminf(p[3], distance(i, hx, hy - h, hz));
                p[4] = fminf(p[4], distance(i, hx, hy, hz + h));
                p[5] = fminf(p[5], distance(i, hx, hy, hz - h));
            }
        }
        const float nx = p[0] - p[1], ny = p[2] - p[3], nz = p[4] - p[5];
        const float nl2 = fmaf(nz, nz, fmaf(nx, nx, ny * ny));
        const float ndl = fmaf(nz, sc.light[2], fmaf(nx, sc.light[0], ny * sc.light[1]));
        dst[(size_t)y * W + x] = shade_lit<kHalf>(sc, total, nl2, ndl, id);
    }
    count_steps(stepCount, step);
}

ckd_status validate_scene(const ckd_sdf_scene *sc)
{
    CKD_REQUIRE(sc != nullptr, "sdf: null scene");
    CKD_REQUIRE(sc->nSpheres >= 0 && sc->nSpheres <= 32, "sdf: nSpheres %d outside 0..32",
                sc->nSpheres);
    CKD_REQUIRE(sc->maxSteps >= 1 && sc->maxSteps <= 1024, "sdf: maxSteps %d outside 1..1024",
                sc->maxSteps);
    return CKD_OK;
}

} // namespace

namespace ckd {

// A sphere containing every sphere of the scene: centre the centroid of the
// centres, radius the largest |c_i - C| + r_i, in double and rounded up.  A
// scene without spheres gets one far away (every step skips it).  Marches that
// only end below a surface (a negative eps) may run backwards: they get an
// infinite one, which skips nothing.
f4 bounding_sphere(const ckd_sdf_scene &sc)
{
    if (sc.nSpheres <= 0) return f4{1e15f, 0.f, 0.f, 0.f};
    double cx = 0, cy = 0, cz = 0;
    for (int i = 0; i < sc.nSpheres; ++i) {
        cx += sc.sphere[i][0];
        cy += sc.sphere[i][1];
        cz += sc.sphere[i][2];
    }
    cx /= sc.nSpheres;
    cy /= sc.nSpheres;
    cz /= sc.nSpheres;
    const float fx = (float)cx, fy = (float)cy, fz = (float)cz;
    double R = 0;
    for (int i = 0; i < sc.nSpheres; ++i) {
        const double ex = sc.sphere[i][0] - (double)fx, ey = sc.sphere[i][1] - (double)fy,
                     ez = sc.sphere[i][2] - (double)fz;
        R = std::max(R, std::sqrt(ex * ex + ey * ey + ez * ez) + (double)sc.sphere[i][3]);
    }
    return f4{fx, fy, fz, sc.eps < 0.f ? INFINITY : std::nextafter((float)R, 3.4e38f)};
}

ckd_status launch_sdf(ckd_ctx *ctx, uint32_t *dst, unsigned W, unsigned H,
                      const ckd_sdf_scene &sc, const float *cam12, int shading,
                      unsigned long long *stepCount)
{
    SdfCam cam;
    for (int i = 0; i < 3; ++i) {
        cam.o[i] = cam12[i];
        cam.f[i] = cam12[3 + i];
        cam.r[i] = cam12[6 + i];
        cam.u[i] = cam12[9 + i];
    }
    dim3 grid(ckd_div_up(W, 16), ckd_div_up(H, 16));
    const float invH = 1.0f / (float)H;
    const f4 bound = bounding_sphere(sc);
    KernelTimer kt(ctx, CKD_KT_SDF_PLAIN);
    // Frames of few tiles wait for one ray's chain.  All spheres on every step, and
    // tiles that keep all, against tiles that cull (us): 320x200 with 1 sphere 9.1 /
    // 13.2 / 13.7, 4: 14.8 / 19.7 / 20.1, 8: - / 29.5 / 31.8, 32: - / 99 / 92; 960x540 with
    // 4: 21.0 / 22.4 / 23.3, 6: 29.3 / 29.2 / 29.8, 8: - / 31.9 / 33.4, 16: - / 54 / 44;
    // 1280x720 with 1: 16.0 / 17.1 / 17.4, 4: 32.8 / 25.8 / 25.2, 8: - / 38 / 34; 2560x1440
    // with 1: 50 / 42 / 46, 8: - / 88 / 71.
    const uint64_t work = (uint64_t)grid.x * grid.y * (unsigned)sc.nSpheres;
    const bool few = sc.nSpheres <= kFewSpheres && work < 10000, cull = work >= 24000 || sc.nSpheres > 16;
    auto launch = [&](auto half, auto fewSpheres) {
        k_sdf<decltype(half)::value, decltype(fewSpheres)::value>
            <<<grid, 256, 0, ctx->stream>>>(dst, W, H, invH, sc, cam, bound, cull, stepCount);
    };
    using Yes = std::true_type;
    using No = std::false_type;
    if (shading == CKD_SHADE_FP16)
        few ? launch(Yes{}, Yes{}) : launch(Yes{}, No{});
    else
        few ? launch(No{}, Yes{}) : launch(No{}, No{});
    return check_launch("sdf");
}

// blocks of one persistent kernel variant that fit on a CU at once
template <bool kHalf, int kMaxSph>
int persistent_blocks_per_cu(int steps)
{
    int n = 0;
    hipError_t e;
    if (steps <= 1)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_sdf_persistent<kHalf, kMaxSph, 1>, 256, 0);
    else if (steps == 2)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_sdf_persistent<kHalf, kMaxSph, 2>, 256, 0);
    else if (steps == 4)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_sdf_persistent<kHalf, kMaxSph, 4>, 256, 0);
    else if (steps == 8)
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_sdf_persistent<kHalf, kMaxSph, 8>, 256, 0);
    else
        e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k_sdf_persistent<kHalf, kMaxSph, 16>, 256, 0);
    return e == hipSuccess ? n : 0;
}

template <bool kHalf, int kMaxSph>
void launch_persistent_steps(int steps, unsigned blocks, hipStream_t st, uint32_t *queueCounter,
                             uint32_t totalChunks, const SdfJob *jobs, int nJobs,
                             const ckd_sdf_scene &sc, unsigned long long *stepCount, uint32_t chunk,
                             uint32_t fixedChunks, uint32_t nQueues, bool own, f4 bound, unsigned long long *work)
{
    if (steps <= 1)
        k_sdf_persistent<kHalf, kMaxSph, 1><<<blocks, 256, 0, st>>>(queueCounter, totalChunks, jobs, nJobs, sc, stepCount, chunk, fixedChunks, nQueues, own, bound, work);
    else if (steps == 2)
        k_sdf_persistent<kHalf, kMaxSph, 2><<<blocks, 256, 0, st>>>(queueCounter, totalChunks, jobs, nJobs, sc, stepCount, chunk, fixedChunks, nQueues, own, bound, work);
    else if (steps == 4)
        k_sdf_persistent<kHalf, kMaxSph, 4><<<blocks, 256, 0, st>>>(queueCounter, totalChunks, jobs, nJobs, sc, stepCount, chunk, fixedChunks, nQueues, own, bound, work);
    else if (steps == 8)
        k_sdf_persistent<kHalf, kMaxSph, 8><<<blocks, 256, 0, st>>>(queueCounter, totalChunks, jobs, nJobs, sc, stepCount, chunk, fixedChunks, nQueues, own, bound, work);
    else
        k_sdf_persistent<kHalf, kMaxSph, 16><<<blocks, 256, 0, st>>>(queueCounter, totalChunks, jobs, nJobs, sc, stepCount, chunk, fixedChunks, nQueues, own, bound, work);
}

// The side of the batch's chunks, at most the tuned one.  Small chunks spread a
// small batch over the chip (at least as many chunks as resident waves); large
// ones refill lanes longer and find the chunk's spheres less often (8x8 ones
// not at all, which a scene of many spheres pays for).  Measured, us, sides 8,
// 16, 32: 8 spheres 1280x720, 1 frame 44, 60, 148; 4 frames 124, 113, 182; 16
// frames 466, 311, 359; 32 frames 935, 590, 614; 64 frames 1830, 1122, 1101; 32
// spheres 2560x1440, 2 frames -, 338, 567; 24 frames -, 3056, 2962.
uint32_t sdf_chunk_side(int tuned, size_t pixels, int nSpheres)
{
    const uint32_t side = pixels <= 2u << 20 && nSpheres <= 8 ? 8 : pixels <= 32u << 20 ? 16 : 32;
    return std::min(side, (uint32_t)tuned);
}

ckd_status launch_sdf_persistent(ckd_ctx *ctx, uint32_t *queueCounter, uint32_t totalChunks, uint32_t chunk,
                                 const SdfJob *jobs, int nJobs, const ckd_sdf_scene &sc,
                                 int shading, unsigned long long *stepCount, bool helper, bool alone)
{
    if (totalChunks == 0) return CKD_OK;
    const bool big = sc.nSpheres > 8;
    const int steps = ctx->tuning.sdfStepsPerRefill;
    // persistent: sdfBlocksPerCU 4-wave blocks per CU; surplus blocks find
    // the queue empty and exit.  A helper launch (the batch's second stream,
    // once its voxel and tunnel work is done) adds the blocks that fill each
    // CU up to the kernel's occupancy and drains the same queue.  A batch
    // with nothing beside the march (alone) gets that occupancy: the tuned
    // count leaves room for work that is not there.
    int perCU = ctx->tuning.sdfBlocksPerCU;
    const int fit = shading == CKD_SHADE_FP16
                        ? (big ? persistent_blocks_per_cu<true, 32>(steps) : persistent_blocks_per_cu<true, 8>(steps))
                        : (big ? persistent_blocks_per_cu<false, 32>(steps) : persistent_blocks_per_cu<false, 8>(steps));
    if (helper) {
        perCU = fit - perCU;
        if (perCU <= 0) return CKD_OK;
    } else if (alone && fit > 0) {
        perCU = fit;
    }
    unsigned blocks = (unsigned)ctx->cuCount * (unsigned)perCU;
    const unsigned useful = (totalChunks + kWavesPerBlock - 1) / kWavesPerBlock;
    if (blocks > useful) blocks = useful;
    if (blocks == 0) blocks = 1;
    // with nothing beside the march every block is resident: each wave's first
    // chunk is its own
    const bool own = alone;
    // a queue needs a block of the main launch to drain it
    const uint32_t nQueues = blocks >= kSdfQueues ? kSdfQueues : 1;
    const uint32_t fixedChunks = alone ? std::min(totalChunks, (uint32_t)(blocks * kWavesPerBlock)) : 0u;
    // only the main launch is timed: it spans the whole march of the batch
    const f4 bound = bounding_sphere(sc);
    KernelTimer kt(ctx, helper ? -1 : CKD_KT_SDF_PERSISTENT);
    if (shading == CKD_SHADE_FP16) {
        if (big) launch_persistent_steps<true, 32>(steps, blocks, ctx->stream, queueCounter, totalChunks, jobs, nJobs, sc, stepCount, chunk, fixedChunks, nQueues, own, bound, ctx->sdfWork);
        else launch_persistent_steps<true, 8>(steps, blocks, ctx->stream, queueCounter, totalChunks, jobs, nJobs, sc, stepCount, chunk, fixedChunks, nQueues, own, bound, ctx->sdfWork);
    } else {
        if (big) launch_persistent_steps<false, 32>(steps, blocks, ctx->stream, queueCounter, totalChunks, jobs, nJobs, sc, stepCount, chunk, fixedChunks, nQueues, own, bound, ctx->sdfWork);
        else launch_persistent_steps<false, 8>(steps, blocks, ctx->stream, queueCounter, totalChunks, jobs, nJobs, sc, stepCount, chunk, fixedChunks, nQueues, own, bound, ctx->sdfWork);
    }
    return check_launch("sdf persistent");
}

} // namespace ckd

extern "C" {

ckd_status ckd_sdf_work_counter(ckd_ctx *ctx, unsigned long long *counters)
{
    CKD_REQUIRE_CTX(ctx);
    ctx->sdfWork = counters;
    return CKD_OK;
}

ckd_status ckd_sdf_render(ckd_ctx *ctx, uint32_t *dst, unsigned W, unsigned H,
                          const ckd_sdf_scene *scene, const float *cam, int shading,
                          unsigned long long *stepCount)
{
    CKD_REQUIRE(dst && cam, "ckd_sdf_render: null buffer");
    CKD_REQUIRE(W > 0 && H > 0 && W <= 16384 && H <= 16384, "ckd_sdf_render: bad size %ux%u", W, H);
    CKD_REQUIRE(shading == CKD_SHADE_FP32 || shading == CKD_SHADE_FP16,
                "ckd_sdf_render: unknown shading mode %d", shading);
    ckd_status s = validate_scene(scene);
    if (s != CKD_OK) return s;
    CKD_REQUIRE_CTX(ctx);
    return ckd::launch_sdf(ctx, dst, W, H, *scene, cam, shading, stepCount);
}

} // extern "C"
