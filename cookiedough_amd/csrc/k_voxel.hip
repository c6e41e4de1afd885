// k_voxel.hip -- voxel landscape columns (code/landscape.cpp) and the
// tunnelscape rows (code/tunnelscape.cpp).
//
// Both march the reference's 512 front-to-back steps per column (row for
// tunnelscape) and draw the visible spans with the exact cspanISSE16
// arithmetic.  The highest row drawn so far, the only value that carries from
// step to step, is a prefix minimum, so the steps are spread over the lanes
// of a block (landscape) or a wave (tunnelscape).  The memset32 of the fog
// colour is fused: after the march the part of a column no span reached is
// filled, so each pixel is written exactly once.
#include "ckd_internal.h"
#include "ckd_pixel.h"
#include "ckd_jobs.h"

#include <algorithm>
#include <cstring>

namespace {

constexpr unsigned kMapAnd = 1023, kMapShift = 10, kRayLength = 512;
// span lengths with a divisor of their own: 65536 / n is 0 from 65537 on
constexpr unsigned kSpanDivs = 65538;

struct LsFrame {
    float X1, Y1, viewCos, viewSin;
    int mapTilt; // already scaled to H rows
};

// frames per launch, their parameters passed by value: 160 keeps the
// kernel's arguments inside the 4 KiB limit
constexpr int kLsFramesPerLaunch = 160;

struct LsLaunch {
    float rayY, colScale, halfW;
    int mapScale;
    LsFrame f[kLsFramesPerLaunch];
};
static_assert(sizeof(LsLaunch) + 128 <= 4096, "the kernel's arguments fit 4 KiB");

// exact floor(num/den) for num < 2^24 and 0 < den < 2^24 with a quotient
// below 2^22: num * rcp(den) is then within 0.5 of num/den, so the estimate
// floor(num * rcp(den) - 0.5) is the quotient or one less, and one upward
// correction fixes it.  q*den stays below 2^25, so the 24-bit multiply (full
// rate; the 32-bit one is quarter rate) is exact.  tests/test_voxel_arith.py
// sweeps it over every span length and every (num, den) of ts_height, with the
// reciprocal rounded to nearest and one ulp off either way.
CKD_DEV uint32_t udiv24(uint32_t num, uint32_t den)
{
    // qf > -0.5: converting through a signed int truncates it to 0 there
    const float qf = __builtin_fmaf((float)num, __builtin_amdgcn_rcpf((float)den), -0.5f);
    const uint32_t q = (uint32_t)(int32_t)qf;
    return q + (num - ckd_mul_u24(q, den) >= den ? 1u : 0u);
}

// Per-column ray set-up of vscape (code/landscape.cpp:164-190) and
// voxel::vrot2D / vnorm2D (code/voxel-shared.h:8-24) in FP32 with no
// contraction and correctly rounded division and square root, so the
// integer ray parameters equal the host's bit for bit.
#pragma clang fp contract(off)
CKD_DEV void ls_setup(float rayY, float colScale, float halfW, float X1, float Y1, float viewCos,
                      float viewSin, unsigned iRay, int &dX, int &dY, int &fpFishMul)
{
    const float rayX = colScale * ((float)iRay - halfW);
    const float rotRayX = viewCos * rayX - viewSin * rayY;
    const float rotRayY = viewSin * rayX + viewCos * rayY;
    const float X2 = X1 + rotRayX;
    const float Y2 = Y1 + rotRayY;
    float fdX = X2 - X1;
    float fdY = Y2 - Y1;
    if (fabsf(fdX + fdY) > 1.1920928955078125e-07f) {
        const float length = 1.f / sqrtf(fdX * fdX + fdY * fdY);
        fdX *= length;
        fdY *= length;
    }
    const float fishMul = rayY / sqrtf(rotRayX * rotRayX + rotRayY * rotRayY);
    dX = (int)(fdX * 256.f);
    dY = (int)(fdY * 256.f);
    fpFishMul = (int)(fabsf(fishMul) * 256.f);
}
#pragma clang fp contract(on)

// frame pixels in the global address space (a job table's pointer would
// make flat stores, whose completion the fog table's scalar loads would
// wait for)
typedef __attribute__((address_space(1))) uint32_t global_u32;

// the 2x2 texel quads of the landscape maps: quadH[i] holds the heights of
// texels (u,v), (u+1,v), (u,v+1), (u+1,v+1) (indices wrapped into the map) in
// its bytes 0..3, quadC[i] their colours, for i = v*1024 + u
__global__ __launch_bounds__(256) void k_ls_quads(const uint8_t *__restrict__ hmap,
                                                  const uint32_t *__restrict__ cmap,
                                                  uint32_t *__restrict__ quadH,
                                                  uint4 *__restrict__ quadC)
{
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i >= (kMapAnd + 1) * (kMapAnd + 1)) return;
    const unsigned u = i & kMapAnd, v = i >> kMapShift;
    const unsigned u1 = (u + 1) & kMapAnd, v1 = ((v + 1) & kMapAnd) << kMapShift;
    const unsigned v0 = v << kMapShift;
    quadH[i] = (uint32_t)hmap[u + v0] | ((uint32_t)hmap[u1 + v0] << 8) |
               ((uint32_t)hmap[u + v1] << 16) | ((uint32_t)hmap[u1 + v1] << 24);
    quadC[i] = make_uint4(cmap[u + v0], cmap[u1 + v0], cmap[u + v1], cmap[u1 + v1]);
}

// the fog table as the colour blend subtracts it, fog[k]'s B,R and G,A in the
// high bytes of 16-bit lanes, and floor(65536 / n) mod 2^16 for a span of n
// rows (0 for n = 0 and beyond 65535: nothing there reads its high bit)
__global__ __launch_bounds__(256) void k_ls_tables(const uint32_t *__restrict__ fog, uint2 *__restrict__ fogLanes,
                                                   uint16_t *__restrict__ spanDiv)
{
    const unsigned i = blockIdx.x * 256 + threadIdx.x;
    if (i < 256) fogLanes[i] = make_uint2((fog[i] << 8) & 0xff00ff00u, fog[i] & 0xff00ff00u);
    if (i < kSpanDivs) spanDiv[i] = i ? (uint16_t)(65536u / i) : (uint16_t)0;
}

// ---- vscape_ray (code/landscape.cpp:56-107) over a block ---------------------
//
// A column's 512 steps depend on each other only through the highest row
// drawn so far, a running minimum.  A block takes kCols columns, thread
// (segment, column) kSteps consecutive steps of one of them:
//   1  the projected rows of its steps: heights only
//   2  a prefix minimum over the segments gives every step the row D drawn
//      before it; the steps that draw (row < D) go packed into a list in LDS
//   3  one lane per listed span: its two colours, its set-up, its pixels
//   4  the rows no span reached take the fog colour
// One lane per column, the form before, left a 1280-column frame 20 waves on
// 1024 SIMDs and fetched and blended a colour at every step; about 30% of the
// steps draw (155 of 512 at 1280x720), the rest are hidden behind nearer ones.
// What bounds it: VALU issue, 4 cycles an instruction; 27 for a step's row, 10
// for its place in the list, about 105 for a span and 12 for each of its
// pixels.  Measured, one lane per column -> now: 1 frame of 1280x720 172 -> 8.5
// us, 30 of 1366x768 184 -> 73 us, 90 of them 289 -> 198 us, 150 of 1280x720
// 391 -> 289 us.
//
// The list is ordered by (wave, step of the run, lane), so that neighbouring
// lanes take the same step of neighbouring columns: their texels share cache
// lines and their pixels rows.  Blocks that follow one another go to one XCD
// (ls_block_of): the parts of a 128-byte line that neighbouring blocks write
// then meet in its L2 (150 frames 329 -> 296 us).
template <int kCols, int kSteps> constexpr int kLsThreads = kCols * (int)kRayLength / kSteps;

// list entries per column: frames of the bench's landscape draw 140 to 170
// spans a column.  A block with more goes through its list in rounds.
constexpr int kLsListPerCol = 192;

// a drawn span: step i of column c, rows [hgt, D), length rows to the row of
// step i - 1.  hgt < D <= H <= 2160; length < 2^20 (a projected row is below
// 23071 * W >> 8 plus the tilt)
CKD_DEV uint2 ls_span(uint32_t c, uint32_t i, int hgt, int D, int prev)
{
    return make_uint2((uint32_t)hgt | ((uint32_t)D << 12) | (c << 24), i | ((uint32_t)(prev - hgt) << 9));
}

// the projected row of a step (code/landscape.cpp:76-86) from a height quad
// h4 holding (u,v), (u+1,v), (u,v+1), (u+1,v+1) in bytes 0..3: bsamp8
// (code/bilinear.h:34-53), both horizontal lerps in the 16-bit lanes of (h0,h2)
// and (h1,h3), the vertical one a dot product; then ((255 - h) << 16) / den *
// mapScale >> 8 plus the tilt (tilt8 = 256 * tilt).  den = fish * (step + 1) <=
// 2^17 as a float; fish >= 8 keeps the quotient below 2^22, so that num *
// rcp(den) is within 0.5 of num / den, the estimate truncated is the quotient
// or one less and one upward correction fixes it; the remainder, an integer
// below 2^18, is exact from one FMA.  tests/test_voxel_arith.py sweeps every
// (num, den) with den = fish * (step + 1) and fish >= 4, the reciprocal rounded
// to nearest and one ulp off either way.
CKD_DEV int ls_row(uint32_t h4, uint32_t x, uint32_t y, float denF, uint32_t mapScale, uint32_t tilt8)
{
    // both lanes fu, then 256 - fu
    const ckd_u16x2 f = ckd_u16x2_of(ckd_perm(0u, x, 0x0c000c00u)), nf = (unsigned short)256 - f;
    const ckd_u16x2 s = ckd_lerp2x(ckd_u16x2_of(ckd_perm(0u, h4, 0x0c020c00u)),
                                   ckd_u16x2_of(ckd_perm(0u, h4, 0x0c030c01u)), nf, f);
    // lanes (256 - fv, fv) = fv * 65535 + 256
    const ckd_u16x2 g = ckd_u16x2_of(__umul24(y & 0xffu, 0xffffu) + 256u);
    const uint32_t sum = __builtin_amdgcn_udot2(s, g, 0u, false);
    // (255 - (sum >> 8)) << 16, exact in FP32
    const float num = __builtin_fmaf((float)((sum >> 8) & 0xffu), -65536.f, 16711680.f);
    const float q = truncf(__builtin_fmaf(num, __builtin_amdgcn_rcpf(denF), -0.5f));
    const uint32_t n = (uint32_t)(int32_t)q + (__builtin_fmaf(-q, denF, num) >= denF ? 1u : 0u);
    return (int)(__umul24(n, mapScale) + tilt8) >> 8;
}

// bsamp32_16 (code/bilinear.h:58-83) of a texel quad at (x, y) followed by
// _mm_subs_epu16 of the fog colour (code/landscape.cpp:83), channels in the
// 16-bit lanes of br and ga.  The fog (f, k_ls_tables) is subtracted before
// the blend's last >> 8: v - 256 * fog, saturated at 0, then >> 8 is
// max((v >> 8) - fog, 0).
CKD_DEV void ls_color(const uint4 &q, uint32_t x, uint32_t y, uint2 f, ckd_u16x2 &br, ckd_u16x2 &ga)
{
    const uint32_t M = 0x00ff00ffu;
    const ckd_u16x2 u = ckd_u16x2_of(ckd_perm(0u, x, 0x0c000c00u)), v = ckd_u16x2_of(ckd_perm(0u, y, 0x0c000c00u));
    const ckd_u16x2 nu = (unsigned short)256 - u, nv = (unsigned short)256 - v;
    const ckd_u16x2 b = ckd_lerp2x(ckd_u16x2_of(q.x & M), ckd_u16x2_of(q.y & M), nu, u) * nv +
                        ckd_lerp2x(ckd_u16x2_of(q.z & M), ckd_u16x2_of(q.w & M), nu, u) * v;
    const ckd_u16x2 g = ckd_lerp2x(ckd_u16x2_of(ckd_odd_bytes(q.x)), ckd_u16x2_of(ckd_odd_bytes(q.y)), nu, u) * nv +
                        ckd_lerp2x(ckd_u16x2_of(ckd_odd_bytes(q.z)), ckd_u16x2_of(ckd_odd_bytes(q.w)), nu, u) * v;
    br = __builtin_elementwise_sub_sat(b, ckd_u16x2_of(f.x)) >> (unsigned short)8;
    ga = __builtin_elementwise_sub_sat(g, ckd_u16x2_of(f.y)) >> (unsigned short)8;
}

// int16 lane kHi of a times the low int16 of b, plus c
template <bool kHi> CKD_DEV uint32_t ls_mad16(uint32_t a, uint32_t b, uint32_t c)
{
    uint32_t r;
    if constexpr (kHi)
        asm("v_mad_i32_i16 %0, %1, %2, %3 op_sel:[1,0,0,0]" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    else
        asm("v_mad_i32_i16 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
template <bool kHi> CKD_DEV uint32_t ls_mul16(uint32_t a, uint32_t b)
{
    uint32_t r;
    if constexpr (kHi)
        asm("v_mad_i32_i16 %0, %1, %2, 0 op_sel:[1,0,0,0]" : "=v"(r) : "v"(a), "v"(b));
    else
        asm("v_mad_i32_i16 %0, %1, %2, 0" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

// ckd_span_setup_drawn from colours in 16-bit lanes (A the span's first, B
// its last), the low 16 bits of the divisor and the pre-step length: the
// deltas as two packed subtracts, each product with the divisor or the
// pre-step (their low 16 bits, signed) one v_mad_i32_i16
CKD_DEV void ls_span_setup(CkdSpan &s, ckd_u16x2 Abr, ckd_u16x2 Aga, ckd_u16x2 Bbr, ckd_u16x2 Bga,
                           uint32_t divisor, uint32_t pre)
{
    const uint32_t m = ckd_mul_u24_v(divisor, pre);
    const uint32_t br = ckd_u32_of(Bbr - Abr), ga = ckd_u32_of(Bga - Aga);
    const uint32_t a = ckd_u32_of(Abr), g = ckd_u32_of(Aga);
    s.step[0] = ls_mul16<false>(br, divisor);
    s.step[1] = ls_mul16<false>(ga, divisor);
    s.step[2] = ls_mul16<true>(br, divisor);
    s.step[3] = ls_mul16<true>(ga, divisor);
    s.acc[0] = ls_mad16<false>(br, m, a << 16);
    s.acc[1] = g << 16;
    s.acc[2] = ls_mad16<true>(br, m, a & 0xffff0000u);
    s.acc[3] = g & 0xffff0000u;
}

// the parameters every column of a frame shares
struct LsView {
    unsigned W, H;
    float rayY, colScale, halfW;
    int mapScale;
    LsFrame f;
};

struct LsMaps {
    const uint32_t *quadH;
    const uint4 *quadC;
    const uint2 *fogLanes;
    const uint16_t *spanDiv;
    uint32_t sky; // fog[0]
};

template <int kCols, int kSteps>
CKD_DEV void ls_block(global_u32 *__restrict__ dst, const LsView &V, const LsMaps &M, unsigned col0)
{
    constexpr int kThreads = kLsThreads<kCols, kSteps>, kWaves = kThreads / 64;
    static_assert(kThreads % 64 == 0 && kThreads <= 1024 && kCols <= 32, "whole waves of whole step runs");
    constexpr int kBatch = kSteps < 8 ? kSteps : 8, kList = kCols * kLsListPerCol;
    const unsigned W = V.W, H = V.H;
    __shared__ uint2 spans[kList];
    __shared__ int rayDX[kCols], rayDY[kCols], rayFish[kCols], top[kCols];
    __shared__ int waveMin[kWaves][kCols], waveLast[kWaves][kCols];
    __shared__ uint32_t waveCount[kWaves];
    __shared__ uint2 fogS[kRayLength / 2];
    const unsigned t = threadIdx.x, lane = t & 63;
    const unsigned wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const unsigned c = t % kCols, seg = t / kCols;
    const bool valid = col0 + c < W;
    for (unsigned k = t; k < kRayLength / 2; k += kThreads) fogS[k] = M.fogLanes[k];
    if (t < kCols) {
        int dX, dY, fish;
        ls_setup(V.rayY, V.colScale, V.halfW, V.f.X1, V.f.Y1, V.f.viewCos, V.f.viewSin, min(col0 + t, W - 1), dX,
                 dY, fish);
        rayDX[t] = dX;
        rayDY[t] = dY;
        rayFish[t] = fish;
    }
    __syncthreads();
    const int X0 = (int)(V.f.X1 * 256.f), Y0 = (int)(V.f.Y1 * 256.f);

    // 1: the rows of steps seg * kSteps .. + kSteps - 1 (positions wrap as the
    // march's running additions do; |dX|, |dY| <= 256)
    int row[kSteps];
    {
        const int dX = rayDX[c], dY = rayDY[c];
        const float fish = (float)rayFish[c];
        const int first = (int)(seg * kSteps);
        uint32_t x = (uint32_t)X0 + (uint32_t)__mul24(dX, first), y = (uint32_t)Y0 + (uint32_t)__mul24(dY, first);
        float den = fish * (float)first;
        const uint32_t tilt8 = (uint32_t)V.f.mapTilt << 8;
#pragma unroll
        for (int s0 = 0; s0 < kSteps; s0 += kBatch) {
            uint32_t h4[kBatch], xs[kBatch], ys[kBatch];
#pragma unroll
            for (int s = 0; s < kBatch; ++s) {
                x += (uint32_t)dX;
                y += (uint32_t)dY;
                xs[s] = x;
                ys[s] = y;
                const uint32_t at = ((y << 4) & (kMapAnd << (kMapShift + 2))) | ((x >> 6) & (kMapAnd << 2));
                h4[s] = *(const uint32_t *)((const char *)M.quadH + at);
            }
#pragma unroll
            for (int s = 0; s < kBatch; ++s) {
                den += fish;
                row[s0 + s] = ls_row(h4[s], xs[s], ys[s], den, (uint32_t)V.mapScale, tilt8);
            }
        }
    }

    // 2: the row drawn before each step
    int lo = row[0];
#pragma unroll
    for (int s = 1; s < kSteps; ++s) lo = min(lo, row[s]);
#pragma unroll
    for (unsigned o = kCols; o < 64; o <<= 1) {
        const int v = __shfl_up(lo, o, 64);
        if (lane >= o) lo = min(lo, v);
    }
    if (lane >= 64 - kCols) {
        waveMin[wave][c] = lo;
        waveLast[wave][c] = row[kSteps - 1];
    }
    int D = __shfl_up(lo, kCols, 64), prev = __shfl_up(row[kSteps - 1], kCols, 64);
    __syncthreads();
    if (lane < kCols) {
        D = (int)H;
        prev = wave ? waveLast[wave - 1][c] : (int)H;
    }
    D = min(D, (int)H);
    for (unsigned w = 0; w < wave; ++w) D = min(D, waveMin[w][c]);
    // a column past the right edge draws nothing
    const int D0 = valid ? D : INT_MIN;
    D = D0;
    uint32_t n = 0;
#pragma unroll
    for (int s = 0; s < kSteps; ++s) {
        n += (uint32_t)__popcll(__ballot(row[s] < D));
        D = min(D, row[s]);
    }
    if (seg == kRayLength / kSteps - 1) top[c] = D;
    if (lane == 0) waveCount[wave] = n;
    __syncthreads();
    uint32_t base0 = 0, total = 0;
#pragma unroll
    for (unsigned w = 0; w < kWaves; ++w) {
        const uint32_t k = __builtin_amdgcn_readfirstlane(waveCount[w]);
        base0 += w < wave ? k : 0u;
        total += k;
    }

    // 4: the rows above every span
    if (valid) {
        const int rows = top[c];
        for (int y = (int)seg; y < rows; y += kThreads / kCols) dst[(size_t)y * W + col0 + c] = M.sky;
    }

    // the spans kList at a time (nearly always one round)
    for (uint32_t r0 = 0; r0 < total; r0 += kList) {
        if (r0) __syncthreads();
        D = D0;
        uint32_t base = base0 - r0;
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            const bool vis = row[s] < D;
            const uint64_t m = __ballot(vis);
            const uint32_t at = base + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0));
            if (vis && at < (uint32_t)kList)
                spans[at] = ls_span(c, seg * kSteps + s, row[s], D, s ? row[s - 1] : prev);
            base += (uint32_t)__popcll(m);
            D = min(D, row[s]);
        }
        __syncthreads();

        // 3: the spans
        const uint32_t cnt = min(total - r0, (uint32_t)kList);
        for (uint32_t k = t; k < cnt; k += kThreads) {
            const uint2 e = spans[k];
            const uint32_t hgt = e.x & 0xfffu, drawn = (e.x >> 12) & 0xfffu, sc = e.x >> 24;
            const uint32_t i = e.y & 0x1ffu, length = e.y >> 9;
            const int dX = rayDX[sc], dY = rayDY[sc];
            // the positions of steps i - 1 and i; before step 0 the colour is
            // the unfogged texel under the origin
            const uint32_t px = (uint32_t)X0 + (uint32_t)__mul24(dX, (int)i),
                           py = (uint32_t)Y0 + (uint32_t)__mul24(dY, (int)i);
            const uint32_t x = px + (uint32_t)dX, y = py + (uint32_t)dY;
            auto quad = [&M](uint32_t X, uint32_t Y) {
                const uint32_t at = ((Y << 6) & (kMapAnd << (kMapShift + 4))) | ((X >> 4) & (kMapAnd << 4));
                return *(const uint4 *)((const char *)M.quadC + at);
            };
            const uint4 q0 = quad(px, py), q1 = quad(x, y);
            const uint2 f0 = fogS[i ? (i - 1) >> 1 : 0], f1 = fogS[i >> 1];
            const uint32_t divisor = M.spanDiv[min(length, kSpanDivs - 1)];
            ckd_u16x2 lastBR, lastGA, br, ga;
            ls_color(q0, px, py, f0, lastBR, lastGA);
            if (i == 0) {
                lastBR = ckd_u16x2_of(q0.x & 0x00ff00ffu);
                lastGA = ckd_u16x2_of(ckd_odd_bytes(q0.x));
            }
            ls_color(q1, x, y, f1, br, ga);
            const uint32_t drawLength = drawn - hgt;
            CkdSpan sp;
            ls_span_setup(sp, br, ga, lastBR, lastGA, divisor, length - drawLength);
            // hgt < H <= 2160 and W <= 4096: pixel offsets fit 24 bits
            uint32_t at = ckd_mul_u24(hgt, W) + col0 + sc;
            for (uint32_t j = 0; j < drawLength; ++j) {
                dst[at] = ckd_span_pixel(sp.acc);
                at += W;
#pragma unroll
                for (int ch = 0; ch < 4; ++ch) sp.acc[ch] += sp.step[ch];
            }
        }
    }
}

// the unit a block takes: blocks go to the 8 XCDs in turn, units of one XCD
// follow one another (the grid is units rounded up to a multiple of 8)
CKD_DEV unsigned ls_block_of(unsigned units)
{
    return (blockIdx.x & 7) * ((units + 7) / 8) + (blockIdx.x >> 3);
}
unsigned ls_grid(unsigned units) { return (units + 7) / 8 * 8; }

template <int kCols, int kSteps>
__global__ __launch_bounds__((kLsThreads<kCols, kSteps>)) void k_landscape(uint32_t *__restrict__ dst, unsigned W,
                                                                          unsigned H, LsMaps M, LsLaunch P,
                                                                          unsigned groupsPerFrame, unsigned units)
{
    const unsigned u = ls_block_of(units);
    if (u >= units) return;
    const unsigned f = u / groupsPerFrame, g = u - f * groupsPerFrame;
    const LsView V{W, H, P.rayY, P.colScale, P.halfW, P.mapScale, P.f[f]};
    ls_block<kCols, kSteps>((global_u32 *)(dst + (size_t)f * W * H), V, M, g * kCols);
}

// every voxel request of a batch in one launch: unit -> job by binary search
template <int kCols, int kSteps>
__global__ __launch_bounds__((kLsThreads<kCols, kSteps>)) void k_landscape_jobs(const VoxJob *__restrict__ jobs,
                                                                               int nJobs, LsMaps M, unsigned units)
{
    const unsigned u = ls_block_of(units);
    if (u >= units) return;
    const VoxJob &J = jobs[ckd_find_job(jobs, nJobs, u, &VoxJob::blockBase)];
    const LsView V{J.W, J.H, J.rayY, J.colScale, J.halfW, J.mapScale,
                   LsFrame{J.X1, J.Y1, J.viewCos, J.viewSin, J.mapTilt}};
    ls_block<kCols, kSteps>((global_u32 *)J.dst, V, M, (u - J.blockBase) * kCols);
}

LsMaps ls_maps(const ckd_ctx *ctx)
{
    return LsMaps{ctx->lsQuadH, ctx->lsQuadC, ctx->lsFogLanes, ctx->lsSpanDiv, ctx->lsFog0};
}

// ---- tunnelscape ---------------------------------------------------------

constexpr unsigned kTsAnd = 2047, kTsShift = 11;

// tscape_ray (code/tunnelscape.cpp:44-100), one wave per output row: lane l
// takes steps 8l .. 8l + 7, a prefix minimum over the lanes gives every step
// the height D drawn before it, the steps that draw (height < D) go into a
// list in LDS in step order, then one lane draws one span of it: neighbouring
// lanes read neighbouring texels and write neighbouring pixels.  The caller
// guarantees map heights <= 159, so every height is positive.
// One lane per row, the form before, left a 720-row frame 12 waves; what
// bounds this one is a row's chain of latencies: 1280x720 351 -> 14.8 us.
constexpr int kTsSteps = (int)kRayLength / 64;

// a step's height from its bilinear map height h (code/tunnelscape.cpp:75-84):
// ((159 - h) << 8) / 0.28125 truncated, over the step's number, times 160 >>
// 8, plus 120.  0.28125 is 9/32: the FP32 quotient of the exact 8192 m / 9 (m
// = 159 - h) lies within 1/64 of it and its fraction is a multiple of 1/9, so
// both truncations together are floor(8192 m / (9 n)).  num < 2^21 and den <=
// 4608: the estimate num * rcp(den) - 0.5 truncated is the quotient or one less
// (tests/test_voxel_arith.py: every (m, n)).
CKD_DEV int ts_height(uint32_t h, uint32_t n)
{
    const uint32_t q = udiv24((159u - h) << 13, 9u * n);
    return (int)(__umul24(q, 160u) >> 8) + 120;
}

__global__ __launch_bounds__(64) void k_tunnelscape(uint32_t *__restrict__ dst, unsigned W,
                                                    unsigned H, const uint8_t *__restrict__ hmap,
                                                    const uint32_t *__restrict__ cmap,
                                                    const uint32_t *__restrict__ fog,
                                                    float mapStepX, float fromXAdd, int fpFromY,
                                                    int dX, int dY)
{
    __shared__ uint2 spans[kRayLength];
    const unsigned lane = threadIdx.x, iRay = blockIdx.x;
    global_u32 *row = (global_u32 *)(dst + (size_t)iRay * W);
    uint32_t X0, Y0 = (uint32_t)fpFromY;
    {
#pragma clang fp contract(off)
        const float mapX = (float)iRay * mapStepX;
        const float fromX = mapX + fromXAdd;
        X0 = (uint32_t)(int)(fromX * 256.f);
    }
    // texel indices of the four neighbours of a position
    auto corners = [](uint32_t X, uint32_t Y, uint32_t (&at)[4]) {
        const uint32_t u0 = (X >> 8) & kTsAnd, u1 = ((X >> 8) + 1) & kTsAnd;
        const uint32_t v0 = ((Y >> 8) & kTsAnd) << kTsShift, v1 = (((Y >> 8) + 1) & kTsAnd) << kTsShift;
        at[0] = u0 + v0;
        at[1] = u1 + v0;
        at[2] = u0 + v1;
        at[3] = u1 + v1;
    };

    // the heights of this lane's steps
    const uint32_t first = lane * kTsSteps;
    int height[kTsSteps];
    {
        uint32_t h[kTsSteps][4], x = X0 + (uint32_t)dX * first, y = Y0 + (uint32_t)dY * first;
        uint32_t fu[kTsSteps], fv[kTsSteps];
#pragma unroll
        for (int s = 0; s < kTsSteps; ++s) {
            x += (uint32_t)dX;
            y += (uint32_t)dY;
            fu[s] = x & 0xff;
            fv[s] = y & 0xff;
            uint32_t at[4];
            corners(x, y, at);
#pragma unroll
            for (int k = 0; k < 4; ++k) h[s][k] = hmap[at[k]];
        }
#pragma unroll
        for (int s = 0; s < kTsSteps; ++s)
            height[s] = ts_height(ckd_bilerp8(h[s][0], h[s][1], h[s][2], h[s][3], fu[s], fv[s]), first + s + 1);
    }

    // the height drawn before each step, the spans in step order
    int lo = height[0];
#pragma unroll
    for (int s = 1; s < kTsSteps; ++s) lo = min(lo, height[s]);
#pragma unroll
    for (unsigned o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(lo, o, 64);
        if (lane >= o) lo = min(lo, v);
    }
    int D = __shfl_up(lo, 1, 64), prev = __shfl_up(height[kTsSteps - 1], 1, 64);
    if (lane == 0) D = prev = (int)W;
    D = min(D, (int)W);
    const int top = min(__shfl(lo, 63, 64), (int)W);
    const int D0 = D;
    uint32_t n = 0;
#pragma unroll
    for (int s = 0; s < kTsSteps; ++s) {
        n += height[s] < D ? 1u : 0u;
        D = min(D, height[s]);
    }
    uint32_t at = n;
#pragma unroll
    for (unsigned o = 1; o < 64; o <<= 1) {
        const uint32_t v = __shfl_up(at, o, 64);
        if (lane >= o) at += v;
    }
    const uint32_t total = __shfl(at, 63, 64);
    at -= n;
    D = D0;
#pragma unroll
    for (int s = 0; s < kTsSteps; ++s) {
        if (height[s] < D) {
            // height < D <= 4096; the distance to the previous step's height
            // is below 2^17
            spans[at++] = make_uint2((uint32_t)height[s] | ((uint32_t)D << 12),
                                     (first + s) | ((uint32_t)((s ? height[s - 1] : prev) - height[s]) << 9));
            D = height[s];
        }
    }
    __syncthreads();

    // the spans: pixels W - D .. W - height - 1 of the row
    for (uint32_t k = lane; k < total; k += 64) {
        const uint2 e = spans[k];
        const uint32_t hgt = e.x & 0xfffu, drawn = e.x >> 12, i = e.y & 0x1ffu, length = e.y >> 9;
        // the positions of steps i - 1 and i; before step 0 the colour is the
        // unfogged texel under the origin
        const uint32_t px = X0 + (uint32_t)dX * i, py = Y0 + (uint32_t)dY * i;
        const uint32_t x = px + (uint32_t)dX, y = py + (uint32_t)dY;
        uint32_t a0[4], a1[4], c0[4], c1[4];
        corners(px, py, a0);
        corners(x, y, a1);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            c0[j] = cmap[a0[j]];
            c1[j] = cmap[a1[j]];
        }
        const uint32_t f0 = fog[i ? (i - 1) >> 1 : 0], f1 = fog[i >> 1];
        uint32_t lastColor = ckd_subs_u8x4(ckd_bilerp32(c0[0], c0[1], c0[2], c0[3], px & 0xff, py & 0xff), f0);
        if (i == 0) lastColor = c0[0];
        const uint32_t color = ckd_subs_u8x4(ckd_bilerp32(c1[0], c1[1], c1[2], c1[3], x & 0xff, y & 0xff), f1);
        const uint32_t drawLength = drawn - hgt;
        CkdSpan sp;
        ckd_span_setup_drawn(sp, color, lastColor, length, drawLength, udiv24(65536u, length));
        global_u32 *p = row + (W - drawn);
        for (uint32_t j = 0; j < drawLength; ++j) {
            p[j] = ckd_span_pixel(sp.acc);
#pragma unroll
            for (int c = 0; c < 4; ++c) sp.acc[c] += sp.step[c];
        }
    }
    const uint32_t sky = fog[0];
    for (unsigned x = W - (unsigned)top + lane; x < W; x += 64) row[x] = sky;
}

ckd_status upload(const void *host, size_t bytes, void **dev)
{
    if (*dev) {
        (void)hipFree(*dev);
        *dev = nullptr;
    }
    if (ckd::dev_alloc(dev, bytes) != hipSuccess) {
        *dev = nullptr;
        return ckd::fail(CKD_ENOMEM, "map upload: ckd::dev_alloc(%zu) failed", bytes);
    }
    CKD_HIP(hipMemcpy(*dev, host, bytes, hipMemcpyHostToDevice));
    return CKD_OK;
}

float ls_rayY(unsigned W, unsigned H)
{
#pragma clang fp contract(off)
    const float kPI = 3.1415926535897932384626433832795f;
    const float aspect = (float)H / (float)W;
    const float viewLenScale = aspect * (kPI * 0.1f);
    return 1024.f * viewLenScale;
}

int scale_rows(int v720, unsigned H) { return (int)(((long long)v720 * (long long)H) / 720); }

} // namespace

namespace ckd {

void voxel_job_geometry(VoxJob &J, unsigned W, unsigned H, const ckd_landscape_cam &c)
{
    J.W = W;
    J.H = H;
    J.rayY = ls_rayY(W, H);
    J.colScale = 0.25f * (1280.f / (float)W);
    J.halfW = (float)W * 0.5f;
    J.mapScale = scale_rows(512, H);
    J.X1 = c.X1;
    J.Y1 = c.Y1;
    J.viewCos = c.viewCos;
    J.viewSin = c.viewSin;
    J.mapTilt = scale_rows(c.mapTilt, H);
}

// Columns per block of a launch of `columns` columns in all.  Narrow blocks
// split a small launch finer; wide ones share texels and output lines between
// their columns.  Measured with 4, 8 and 16 columns: 320 columns 5.1, 6.7, 9.2
// us; 1280 8.5, 8.4, 11.8; 2560 14.0, 15.1, 15.2; 12 800 32, 29, 31; 41 000 87,
// 75, 75; 123 000 250, 204, 200; 192 000 395, 312, 294 us.
unsigned voxel_block_cols(size_t columns) { return columns <= 4096 ? 4 : columns <= 49152 ? 8 : 16; }

ckd_status launch_landscape_jobs(ckd_ctx *ctx, const VoxJob *jobs, int nJobs, uint32_t totalBlocks,
                                 unsigned blockCols)
{
    if (totalBlocks == 0) return CKD_OK;
    if (!ctx->lsReady)
        return fail(CKD_ESTATE, "voxel requests need the landscape maps (ckd_landscape_create)");
    KernelTimer kt(ctx, CKD_KT_LANDSCAPE);
    const LsMaps M = ls_maps(ctx);
    const unsigned grid = ls_grid(totalBlocks);
    if (blockCols == 4)
        k_landscape_jobs<4, 4><<<grid, kLsThreads<4, 4>, 0, ctx->stream>>>(jobs, nJobs, M, totalBlocks);
    else if (blockCols == 8)
        k_landscape_jobs<8, 8><<<grid, kLsThreads<8, 8>, 0, ctx->stream>>>(jobs, nJobs, M, totalBlocks);
    else
        k_landscape_jobs<16, 16><<<grid, kLsThreads<16, 16>, 0, ctx->stream>>>(jobs, nJobs, M, totalBlocks);
    return check_launch("landscape jobs");
}

} // namespace ckd

extern "C" {

ckd_status ckd_landscape_create(ckd_ctx *ctx, const uint8_t *heightMap, const uint32_t *colorMap,
                                const uint32_t *fog256)
{
    CKD_REQUIRE(heightMap && colorMap && fog256, "ckd_landscape_create: null map");
    CKD_REQUIRE_CTX(ctx);
    CKD_HIP(hipStreamSynchronize(ctx->stream));
    ctx->lsReady = false; // until every table below is whole
    ckd_status s = upload(heightMap, 1024 * 1024, (void **)&ctx->lsHeight);
    if (s == CKD_OK) s = upload(colorMap, 1024 * 1024 * 4, (void **)&ctx->lsColor);
    if (s == CKD_OK) s = upload(fog256, 256 * 4, (void **)&ctx->lsFog);
    if (s != CKD_OK) return s;
    ctx->lsFog0 = fog256[0];
    constexpr size_t kTexels = 1024 * 1024;
    if ((!ctx->lsQuadH && ckd::dev_alloc(&ctx->lsQuadH, kTexels * 4) != hipSuccess) ||
        (!ctx->lsQuadC && ckd::dev_alloc(&ctx->lsQuadC, kTexels * 16) != hipSuccess))
        return ckd::fail(CKD_ENOMEM, "ckd_landscape_create: hipMalloc of the texel quads failed");
    if ((!ctx->lsFogLanes && ckd::dev_alloc(&ctx->lsFogLanes, 256 * sizeof(uint2)) != hipSuccess) ||
        (!ctx->lsSpanDiv && ckd::dev_alloc(&ctx->lsSpanDiv, kSpanDivs * sizeof(uint16_t)) != hipSuccess))
        return ckd::fail(CKD_ENOMEM, "ckd_landscape_create: hipMalloc of the span tables failed");
    k_ls_tables<<<ckd_div_up(kSpanDivs, 256), 256, 0, ctx->stream>>>(ctx->lsFog, ctx->lsFogLanes, ctx->lsSpanDiv);
    k_ls_quads<<<kTexels / 256, 256, 0, ctx->stream>>>(ctx->lsHeight, ctx->lsColor, ctx->lsQuadH,
                                                       ctx->lsQuadC);
    s = ckd::check_launch("landscape quads and tables");
    if (s != CKD_OK) return s;
    CKD_HIP(hipStreamSynchronize(ctx->stream));
    ctx->lsReady = true;
    return CKD_OK;
}

ckd_status ckd_landscape_draw(ckd_ctx *ctx, uint32_t *dst, unsigned W, unsigned H,
                              const ckd_landscape_cam *cams, unsigned nFrames)
{
    CKD_REQUIRE(dst && cams, "ckd_landscape_draw: null buffer");
    CKD_REQUIRE(W >= 8 && H >= 8 && W <= 4096 && H <= 2160, "ckd_landscape_draw: bad size %ux%u",
                W, H);
    // the edge columns' fpFishMul is at least 8 then (udiv24 needs 4)
    CKD_REQUIRE(W <= 64 * H, "ckd_landscape_draw: %ux%u is wider than 64 times its height", W, H);
    for (unsigned f = 0; f < nFrames; ++f)
        CKD_REQUIRE(cams[f].mapTilt >= 0 && cams[f].mapTilt <= 180,
                    "ckd_landscape_draw: frame %u: mapTilt %d outside 0..180", f, cams[f].mapTilt);
    CKD_REQUIRE_CTX(ctx);
    if (!ctx->lsReady) return ckd::fail(CKD_ESTATE, "ckd_landscape_draw: no maps (ckd_landscape_create)");
    LsLaunch P;
    memset(&P, 0, sizeof(P));
    P.rayY = ls_rayY(W, H);
    P.colScale = 0.25f * (1280.f / (float)W);
    P.halfW = (float)W * 0.5f;
    P.mapScale = scale_rows(512, H);
    for (unsigned f0 = 0; f0 < nFrames; f0 += kLsFramesPerLaunch) {
        const unsigned n = nFrames - f0 < (unsigned)kLsFramesPerLaunch ? nFrames - f0
                                                                       : (unsigned)kLsFramesPerLaunch;
        for (unsigned k = 0; k < n; ++k) {
            const ckd_landscape_cam &c = cams[f0 + k];
            P.f[k] = LsFrame{c.X1, c.Y1, c.viewCos, c.viewSin, scale_rows(c.mapTilt, H)};
        }
        const unsigned cols = ckd::voxel_block_cols((size_t)W * n);
        const unsigned groupsPerFrame = ckd_div_up(W, cols), units = groupsPerFrame * n, grid = ls_grid(units);
        uint32_t *out = dst + (size_t)f0 * W * H;
        ckd::KernelTimer kt(ctx, CKD_KT_LANDSCAPE);
        if (cols == 4)
            k_landscape<4, 4><<<grid, kLsThreads<4, 4>, 0, ctx->stream>>>(out, W, H, ls_maps(ctx), P, groupsPerFrame, units);
        else if (cols == 8)
            k_landscape<8, 8><<<grid, kLsThreads<8, 8>, 0, ctx->stream>>>(out, W, H, ls_maps(ctx), P, groupsPerFrame, units);
        else
            k_landscape<16, 16><<<grid, kLsThreads<16, 16>, 0, ctx->stream>>>(out, W, H, ls_maps(ctx), P, groupsPerFrame, units);
        ckd_status s = ckd::check_launch("landscape");
        if (s != CKD_OK) return s;
    }
    return CKD_OK;
}

ckd_status ckd_tunnelscape_create(ckd_ctx *ctx, const uint8_t *heightMap, const uint32_t *colorMap,
                                  const uint32_t *fog256)
{
    CKD_REQUIRE(heightMap && colorMap && fog256, "ckd_tunnelscape_create: null map");
    for (size_t i = 0; i < 2048u * 2048u; ++i)
        CKD_REQUIRE(heightMap[i] <= 159,
                    "ckd_tunnelscape_create: height %u at %zu > 159 (negative span heights)",
                    heightMap[i], i);
    CKD_REQUIRE_CTX(ctx);
    CKD_HIP(hipStreamSynchronize(ctx->stream));
    ckd_status s = upload(heightMap, 2048 * 2048, (void **)&ctx->tsHeight);
    if (s == CKD_OK) s = upload(colorMap, 2048 * 2048 * 4, (void **)&ctx->tsColor);
    if (s == CKD_OK) s = upload(fog256, 256 * 4, (void **)&ctx->tsFog);
    if (s == CKD_OK) ctx->tsFog0 = fog256[0];
    return s;
}

ckd_status ckd_tunnelscape_rows(ckd_ctx *ctx, uint32_t *dst, unsigned W, unsigned H, float stepU,
                                float stepV, float speed, float time)
{
    CKD_REQUIRE(dst, "ckd_tunnelscape_rows: null buffer");
    CKD_REQUIRE(W >= 8 && H >= 8 && W <= 4096 && H <= 4096, "ckd_tunnelscape_rows: bad size %ux%u",
                W, H);
    CKD_REQUIRE_CTX(ctx);
    if (!ctx->tsHeight || !ctx->tsColor || !ctx->tsFog)
        return ckd::fail(CKD_ESTATE, "ckd_tunnelscape_rows: no maps (ckd_tunnelscape_create)");
    // tscape (code/tunnelscape.cpp:103-118) frame constants, host FP32
    float mapStepX, fromXAdd;
    int dX, dY, fpFromY;
    {
#pragma clang fp contract(off)
        const float kGoldenRatio = 1.61803398875f;
        const float aspect = (float)H / (float)W;
        const float kOneOverAspect = 1.f / aspect;
        mapStepX = 2048.f / (float)(H - 1);
        const float speedMul = sqrtf(stepU * stepU + stepV * stepV) * speed;
        const float fromY = 1024.f + speedMul * time;
        dX = (int)(stepV * 256.f);
        dY = (int)((kOneOverAspect * stepU) * 256.f);
        fpFromY = (int)(fromY * 256.f);
        fromXAdd = stepU * time * kGoldenRatio;
    }
    k_tunnelscape<<<H, 64, 0, ctx->stream>>>(dst, W, H, ctx->tsHeight, ctx->tsColor, ctx->tsFog, mapStepX,
                                             fromXAdd, fpFromY, dX, dY);
    return ckd::check_launch("tunnelscape");
}

} // extern "C"
