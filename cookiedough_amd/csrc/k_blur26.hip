// k_blur26.hip -- the 2026 multi-pass box blur (code/boxblur.cpp).
//
// HorzBlur32 (code/boxblur.cpp:87-212) keeps a running i32 sum per channel
// that adds the lerp term T(j) = p[j] + (((p[j+1]-p[j])*alpha) >> 16) at
// the head and subtracts it at the tail.  Integer addition is associative,
// so the sums of a line's outputs are a prefix sum of what each one adds,
//   S(o) = S0 - T(iSpan) + sum_{o'<=o} (T(o'+iSpan) - T(o'-iSpan-1)),
//   S0   = sum_{j<iSpan} p[j] + ((p[iSpan]*alpha) >> 16),
// with T zero before the line and after T(L).  The reference reads p[L] and
// p[L+1] past every line: the next line's first pixels, or (after the last
// line) two pixels defined here as zero.
// Output: iDiv (mul_epu32 of the low dword, >> 22, hadd of the two halves)
// and v2cISSE32 (code/boxblur.cpp:69-79, code/util.h:152-154).
#include "ckd_internal.h"
#include "ckd_pixel.h"

#include <algorithm>

namespace {

constexpr int kMaxRes = 2048, kMaxRadius = 500, kMaxWaves = 16;

struct B26Params {
    int32_t iSpan, iAlpha;
    uint32_t iScale; // the 10:22 scale
    float halfScale, dScale;
};

// code/boxblur.cpp:98-124, FP32 without contraction
#pragma clang fp contract(off)
void b26_setup(unsigned xRes, float strength, float gain, B26Params &P)
{
    strength *= 0.01f;
    const float r0 = strength * (float)((xRes - 2) / 2);
    const float radius = r0 < (float)kMaxRadius ? r0 : (float)kMaxRadius;
    const unsigned iSpan = (unsigned)radius;
    const float scale = 1.f / ((2.f - gain) * radius + 1.f);
    const float alpha = radius - (float)iSpan;
    P.iSpan = (int32_t)iSpan;
    P.iScale = (uint32_t)(uint64_t)(int64_t)(scale * (float)(1 << 22));
    P.iAlpha = (int32_t)(65536.f * alpha);
    P.halfScale = scale * 0.5f;
    P.dScale = iSpan ? P.halfScale / (float)iSpan : 0.f;
}

// the scale of an output i < iSpan pixels from either end of its line
CKD_DEV uint32_t span_scale(float halfScale, float dScale, int i)
{
    return (uint32_t)((halfScale + (float)i * dScale) * (float)(1 << 22));
}
#pragma clang fp contract(on)

// One launch: `passes` passes over every line, then the store.
struct B26Launch {
    int32_t L, rows, passes;
    int32_t iSpan;
    uint32_t weights, round; // lerp_terms
    uint32_t scale;          // iScale << scaleShift
    int32_t sumShift, scaleShift;
    float halfScale, dScale;
    int32_t colStride, rowStride; // output o of line r: r * colStride + o * rowStride
    int32_t lines, wavesPerLine, haloWaves, blocks;
};

// Four channels' values of at most 16 bits: B and R (even), G and A (odd), each
// two as hi * 65536 + lo.  Such pairs add and subtract as one number, a negative
// lo borrowing from hi.
struct Pairs {
    uint32_t even, odd;
};
CKD_DEV Pairs pairs_of(uint32_t pixel) { return {pixel & 0x00ff00ffu, ckd_perm(0, pixel, 0x0c030c01u)}; }
CKD_DEV int32_t pair_lo(uint32_t v) { return (int32_t)(int16_t)v; }
CKD_DEV int32_t pair_hi(uint32_t v) { return (int32_t)(v + 0x8000u) >> 16; }

// The lerp terms of neighbours a, b:
//   A + (((B - A) * alpha) >> 16) = (A * (65536 - alpha) + B * alpha) >> 16,
// one dot product; alpha = 0 takes weights 65535, 0 and 65535 more, which gives
// A as well (65536 does not fit the weight's 16 bits).
CKD_DEV Pairs lerp_terms(uint32_t a, uint32_t b, uint32_t weights, uint32_t round)
{
    typedef unsigned short us2 __attribute__((ext_vector_type(2)));
    const us2 w = __builtin_bit_cast(us2, weights);
    uint32_t t[4];
#pragma unroll
    for (int c = 0; c < 4; ++c)
        t[c] = __builtin_amdgcn_udot2(__builtin_bit_cast(us2, ckd_perm(b, a, 0x0c040c00u + 0x00010001u * c)), w,
                                      round, false);
    return {ckd_perm(t[2], t[0], 0x0c060c02u), ckd_perm(t[3], t[1], 0x0c060c02u)};
}

template <int kCtrl, int kRows> CKD_DEV int32_t dpp_sum(int32_t v)
{
    return v + __builtin_amdgcn_update_dpp(0, v, kCtrl, kRows, 0xf, false);
}

// sums over the lanes of a row (16) up to each one's, of the rows up to each one
CKD_DEV int32_t row_scan(int32_t v)
{
    v = dpp_sum<0x111, 0xf>(v); // row_shr:1, 2, 4, 8
    v = dpp_sum<0x112, 0xf>(v);
    v = dpp_sum<0x114, 0xf>(v);
    return dpp_sum<0x118, 0xf>(v);
}
CKD_DEV int32_t rows_scan(int32_t v)
{
    return dpp_sum<0x143, 0xc>(dpp_sum<0x142, 0xa>(v)); // row_bcast:15, 31
}

// lo * m + c and hi * m + c of a pair whose lo is not negative
CKD_DEV int32_t mad_lo(uint32_t v, int32_t m, int32_t c)
{
    int32_t r;
    asm("v_mad_i32_i16 %0, %1, %2, %3" : "=v"(r) : "v"(v), "s"(m), "v"(c));
    return r;
}
CKD_DEV int32_t mad_hi(uint32_t v, int32_t m, int32_t c)
{
    int32_t r;
    asm("v_mad_i32_i16 %0, %1, %2, %3 op_sel:[1,0,0,0]" : "=v"(r) : "v"(v), "s"(m), "v"(c));
    return r;
}
// (a * b) >> 32 of a, b of 24 bits with the sign
CKD_DEV uint32_t mul_hi24(int32_t a, uint32_t b)
{
    uint32_t r;
    asm("v_mul_hi_i32_i24 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}

typedef int32_t i4 __attribute__((ext_vector_type(4)));

// Sums of the lanes' pairs up to each lane, B G R A, of values that kPer pixels
// give: over a row as pairs, as long as 16 lanes' fit those.
constexpr uint32_t kBias = 0x1000; // above what a lane's sums go below 0
template <int kPer> CKD_DEV i4 wave_sums(Pairs p)
{
    i4 s;
    if constexpr (16 * kPer * 255 <= 32767) {
        const uint32_t even = row_scan(p.even), odd = row_scan(p.odd);
        s = i4{pair_lo(even), pair_lo(odd), pair_hi(even), pair_hi(odd)};
    } else {
        s = i4{row_scan(pair_lo(p.even)), row_scan(pair_lo(p.odd)), row_scan(pair_hi(p.even)),
               row_scan(pair_hi(p.odd))};
    }
    return i4{rows_scan(s.x), rows_scan(s.y), rows_scan(s.z), rows_scan(s.w)};
}

// A block blurs P.lines lines, P.passes times, a line on P.wavesPerLine waves
// with kPer consecutive pixels on a lane; pixels stay in registers from pass to
// pass.  A pass writes the line's T to LDS with zeros either side, sums
// T(o+iSpan) - T(o-iSpan-1) over the lane, the wave (DPP) and the line's waves,
// and scales.  kPer is odd: lanes that far apart hit all banks.
//
// The reads past a line's end couple the lines: pass q of the block's last line
// needs two pixels of the next line after pass q - 1.  haloWaves more waves carry
// that line's first pixels along (as many as the passes left need: two for one
// pass, iSpan + 1 more for each further one).
//
// A pass is bound by its three barriers' chains and the VALU (half busy): 4.7 us
// of 1920x1080, and 5.7 us for the loads and stores of a launch (3.2 us at the
// copy's rate).  Against a launch a pass with the prefix sums in LDS: 59 -> 20 us
// for three passes along the rows, 63 -> 27 along the columns.
template <int kPer>
__global__ __launch_bounds__(64 * kMaxWaves, kPer <= 7 ? 8 : 6)
void k_b26_lines(uint32_t *__restrict__ out, const uint32_t *__restrict__ in, const B26Launch P)
{
    extern __shared__ Pairs lds[];
    // per wave and channel: the sum of the differences, the share of S0 - T(iSpan)
    __shared__ int32_t totals[4 * kMaxWaves], starts[4 * kMaxWaves];
    __shared__ uint32_t firsts[kMaxWaves + 1], seconds[kMaxWaves + 1]; // pixels 0 and 1 of each wave's
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int perXcd = (P.blocks + 7) >> 3, block = (blockIdx.x & 7) * perXcd + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= perXcd || block >= P.blocks) return;

    const int L = P.L, iSpan = P.iSpan, nw = P.wavesPerLine;
    const int slot = min(wave / nw, P.lines), w = wave - slot * nw, slotWaves = slot < P.lines ? nw : P.haloWaves;
    const int row = block * P.lines + slot;
    const bool halo = slot == P.lines, last = !halo && w == nw - 1;
    const int reach = nw * 64 * kPer, stride = reach + 2 * iSpan + 2;
    const int base = w * 64 * kPer, j0 = base + lane * kPer; // the lane's first pixel
    Pairs *T = lds + slot * stride + iSpan + 1;              // T[0]: of pixel 0

    // zeros either side; the halo's from its last wave on: a lane with its last
    // needed pixels may hold others that read past it, and the lane's sums keep to
    // 16 bits only if all its terms do
    const int held = slotWaves * 64 * kPer; // pixels of the slot's waves
    for (int i = w * 64 + lane; i <= iSpan; i += slotWaves * 64) T[i - iSpan - 1] = {0, 0};
    for (int i = (halo ? held : L + 1) + w * 64 + lane; i <= held + iSpan; i += slotWaves * 64) T[i] = {0, 0};
    if (base > iSpan && lane < 4) starts[4 * wave + lane] = 0;

    // the line's pixels, and the two after it (last wave)
    const int n = L * P.rows, at = row * L + j0;
    uint32_t px[kPer + 1], after0 = 0, after1 = 0;
#pragma unroll
    for (int i = 0; i <= kPer; ++i) {
        const uint32_t v = in[min(at + i, n - 1)];
        px[i] = at + i < n ? v : 0u;
    }
    if (last && row + 1 < P.rows) {
        after0 = in[(row + 1) * L];
        after1 = in[(row + 1) * L + 1];
    }

    const int32_t sumUnit = 1 << P.sumShift;
    const int sumLane = 4 * (wave - w) + lane; // lane 4 v + c: channel c of the line's wave v
    for (int pass = 0;; ++pass) {
        const bool store = pass == P.passes - 1, live = !(halo && store);
        if (live) {
            Pairs t[kPer];
#pragma unroll
            for (int i = 0; i < kPer; ++i) t[i] = lerp_terms(px[i], px[i + 1], P.weights, P.round);
            if (last) {
#pragma unroll
                for (int i = 0; i < kPer; ++i)
                    if (j0 + i < L) T[j0 + i] = t[i];
                if (lane == 0) T[L] = lerp_terms(after0, after1, P.weights, P.round);
            } else {
#pragma unroll
                for (int i = 0; i < kPer; ++i) T[j0 + i] = t[i];
            }
            if (base <= iSpan) {
                Pairs sum = {0, 0}, edgeT = {0, 0};
                uint32_t edge = 0;
#pragma unroll
                for (int i = 0; i < kPer; ++i) {
                    const Pairs p = pairs_of(j0 + i < iSpan ? px[i] : 0u);
                    sum.even += p.even;
                    sum.odd += p.odd;
                    if (j0 + i == iSpan) {
                        edge = px[i];
                        edgeT = t[i];
                    }
                }
                // (p * alpha) >> 16: the term between 0 and p
                const Pairs frac = lerp_terms(0, edge, P.weights & 0xffff0000u, 0);
                sum.even += frac.even - edgeT.even;
                sum.odd += frac.odd - edgeT.odd;
                const i4 s = wave_sums<kPer>(sum);
                if (lane == 63) *reinterpret_cast<i4 *>(starts + 4 * wave) = s;
            }
        }
        __syncthreads();
        // the lane's prefix sums, lo biased to stay positive, and the wave's
        uint32_t even[kPer], odd[kPer];
        i4 upTo;
        if (live) {
            Pairs s = {kBias, kBias};
#pragma unroll
            for (int i = 0; i < kPer; ++i) {
                const Pairs h = T[j0 + i + iSpan], l = T[j0 + i - iSpan - 1];
                even[i] = s.even += h.even - l.even;
                odd[i] = s.odd += h.odd - l.odd;
            }
            upTo = wave_sums<kPer>({s.even - kBias, s.odd - kBias});
            if (lane == 63) *reinterpret_cast<i4 *>(totals + 4 * wave) = upTo;
        }
        __syncthreads();
        if (live) {
            // S0 - T(iSpan) and the sums of the waves before: four waves a row
            int32_t part = 0;
            if (lane < 4 * slotWaves) part = starts[sumLane];
            if (lane < 4 * w) part += totals[sumLane];
            part = dpp_sum<0x118, 0xf>(dpp_sum<0x114, 0xf>(part)); // row_shr:4, 8
            i4 line = {0, 0, 0, 0};
            for (int v = 0; v < slotWaves; v += 4)
#pragma unroll
                for (int c = 0; c < 4; ++c) line[c] += __builtin_amdgcn_readlane(part, 4 * v + 12 + c);
            // less the lane's own, which its prefix sums add again
            i4 before = (upTo + line) << P.sumShift;
            before.x = mad_lo(even[kPer - 1], -sumUnit, before.x);
            before.y = mad_lo(odd[kPer - 1], -sumUnit, before.y);
            before.z = mad_hi(even[kPer - 1], -sumUnit, before.z);
            before.w = mad_hi(odd[kPer - 1], -sumUnit, before.w);
            uint32_t scale[kPer];
#pragma unroll
            for (int i = 0; i < kPer; ++i) scale[i] = P.scale;
            if (base < iSpan || base + 64 * kPer > L - iSpan)
#pragma unroll
                for (int i = 0; i < kPer; ++i) {
                    const int o = j0 + i, fromEnd = o < iSpan ? o : L - 1 - o;
                    if (fromEnd < iSpan) scale[i] = span_scale(P.halfScale, P.dScale, fromEnd) << P.scaleShift;
                }
#pragma unroll
            for (int i = 0; i < kPer; ++i) {
                // a negative sum gives a negative product, which is taken as 0
                const uint32_t b = mul_hi24(mad_lo(even[i], sumUnit, before.x), scale[i]);
                const uint32_t g = mul_hi24(mad_lo(odd[i], sumUnit, before.y), scale[i]);
                const uint32_t r = mul_hi24(mad_hi(even[i], sumUnit, before.z), scale[i]);
                const uint32_t a = mul_hi24(mad_hi(odd[i], sumUnit, before.w), scale[i]);
                px[i] = ckd_perm(ckd_sat_pk_u8(ckd_perm(a, r, 0x05040100u)),
                                 ckd_sat_pk_u8(ckd_perm(g, b, 0x05040100u)), 0x05040100u);
            }
        }
        if (store) break;
        if (row >= P.rows)
#pragma unroll
            for (int i = 0; i < kPer; ++i) px[i] = 0;
        if (lane == 0) {
            firsts[wave] = px[0];
            seconds[wave] = px[1];
        }
        __syncthreads();
        // the pixels after the lane's and after the line's
        const uint32_t next = firsts[wave + 1];
        px[kPer] = __builtin_amdgcn_update_dpp(next, px[0], 0x130, 0xf, 0xf, false); // wave_shl:1
        if (last) {
            after0 = next;
            after1 = seconds[wave + 1];
#pragma unroll
            for (int i = 0; i <= kPer; ++i)
                if (j0 + i == L) px[i] = after0;
        }
    }

    // to LDS, to be stored in the order of the output's addresses
    uint32_t *staged = reinterpret_cast<uint32_t *>(lds);
    if (!halo) {
        uint32_t *stage = staged + slot * reach + j0;
#pragma unroll
        for (int i = 0; i < kPer; ++i) stage[i] = px[i];
    }
    __syncthreads();
    if (P.rowStride == 1) {
        if (!halo && row < P.rows)
            for (int o = w * 64 + lane; o < L; o += nw * 64)
                out[(size_t)row * P.colStride + o] = staged[slot * reach + o];
    } else {
        const int shift = P.lines - 1, g = threadIdx.x & shift; // one or two lines
        const int r = block * P.lines + g;
        if (r < P.rows)
            for (int o = threadIdx.x >> shift; o < L; o += blockDim.x >> shift)
                out[(size_t)r * P.colStride + (size_t)o * P.rowStride] = staged[g * reach + o];
    }
}

__global__ __launch_bounds__(256) void k_transpose(uint32_t *__restrict__ dst,
                                                   const uint32_t *__restrict__ src, int xRes,
                                                   int yRes)
{
    __shared__ uint32_t tile[32][33];
    const int bx = blockIdx.x * 32, by = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
    for (int r = ty; r < 32; r += 8) {
        const int x = bx + tx, y = by + r;
        if (x < xRes && y < yRes) tile[r][tx] = src[(size_t)y * xRes + x];
    }
    __syncthreads();
    for (int r = ty; r < 32; r += 8) {
        const int y = by + tx, x = bx + r; // dst row = x, dst col = y
        if (x < xRes && y < yRes) dst[(size_t)x * yRes + y] = tile[tx][r];
    }
}

// How a launch covers the lines.
//
// per, the pixels of a lane: what a line's waves cost is linear in it (a scan of
// the wave and the exchange, about three pixels' worth), so it follows from how
// the line divides, except where all waves fit the chip at once: then the least,
// for the shortest chain (320x180, 2 passes both ways: 9.7 us with 3, 11.0 with 5).
// Three passes of 1920x1080: along the rows 20.0 us with 5, 21.8 with 7, 24.5 with
// 3; along the columns 28.1 with 9 or 7, 30.9 with 5.
// lines: two a block give a transposed store 8-byte pieces (26.7 us instead of
// 28.1), where there are blocks enough left; otherwise blocks of one line fill
// the chip more evenly (1080 lines: 20.0 us, 22.8 with two).
// passes: as many as a halo of a quarter of its waves allows (three of 1920x1080:
// 20.0 us in one launch, 34.8 in three).
struct B26Shape {
    int per, wavesPerLine, lines, haloWaves, passes;
};

// the lines' T, a margin of iSpan + 1 either side of each
size_t b26_lds(int per, int waves, int lines, int iSpan)
{
    return ((size_t)waves * 64 * per + (size_t)(lines + 1) * (2 * iSpan + 2)) * sizeof(Pairs);
}

B26Shape b26_shape(int L, int rows, int iSpan, int passes, bool transposed)
{
    B26Shape s = {};
    auto line_waves = [L](int per) { return (int)ckd_div_up((unsigned)L, 64u * per); };
    s.per = 3;
    if (rows * line_waves(3) > 2048)
        for (int per = 5; per <= 9; per += 2)
            if (line_waves(per) * (per + 3) < line_waves(s.per) * (s.per + 3)) s.per = per;
    s.wavesPerLine = line_waves(s.per);
    s.lines = transposed && rows >= 1536 && s.wavesPerLine <= 6
                      && b26_lds(s.per, 2 * s.wavesPerLine, 2, iSpan) <= 65536 ? 2 : 1;
    const int most = s.lines * s.wavesPerLine;
    s.passes = 1;
    for (int f = 2; f <= passes; ++f) {
        const int need = (f - 1) * (iSpan + 1) + 1; // pixels of the next line
        const int waves = (int)ckd_div_up((unsigned)need, 64u * s.per);
        if (need > L || waves > (most + 3) / 4 || most + waves > kMaxWaves
            || b26_lds(s.per, most + waves, s.lines, iSpan) > 65536)
            break;
        s.passes = f;
        s.haloWaves = waves;
    }
    return s;
}

template <int kPer>
void launch_lines(ckd_ctx *ctx, uint32_t *out, const uint32_t *in, const B26Launch &P)
{
    const int waves = P.lines * P.wavesPerLine + P.haloWaves;
    const size_t lds = b26_lds(kPer, waves, P.lines, P.iSpan);
    k_b26_lines<kPer><<<(P.blocks + 7) / 8 * 8, 64 * waves, lds, ctx->stream>>>(out, in, P);
}

// HorzBlur32's pass loop (code/boxblur.cpp:126-211) over device buffers
ckd_status horz(ckd_ctx *ctx, uint32_t *pDest, uint32_t *pScratch, const uint32_t *pSrc,
                unsigned xRes, unsigned yRes, unsigned wCol, unsigned wRow, float strength,
                float gain, unsigned numPasses)
{
    B26Params B;
    b26_setup(xRes, strength, gain, B);
    B26Launch P = {};
    P.L = (int)xRes;
    P.rows = (int)yRes;
    P.iSpan = B.iSpan;
    P.weights = B.iAlpha ? (uint32_t)(65536 - B.iAlpha) | (uint32_t)B.iAlpha << 16 : 65535u;
    P.round = B.iAlpha ? 0u : 65535u;
    P.halfScale = B.halfScale;
    P.dScale = B.dScale;
    // (sum * scale) >> 22 as the high half of a product of 24-bit factors with
    // signs, 10 bits shared out between them.  S0 - (T(0) + .. + T(iSpan)), what a
    // sum holds beside its 2 iSpan + 1 terms of at most 255, is below 255 + iSpan +
    // 1: rounding down takes less than 1 off each T.  A scale is at most 2^22 /
    // (iSpan + 1), so the two always fit
    int sumBits = 0;
    while (((2 * B.iSpan + 2) * 255 + B.iSpan + 1) >> sumBits) ++sumBits;
    P.sumShift = std::min(10, 23 - sumBits);
    P.scaleShift = 10 - P.sumShift;
    P.scale = B.iScale << P.scaleShift;

    unsigned launches = 0;
    for (unsigned left = numPasses; left; ++launches)
        left -= (unsigned)b26_shape(P.L, P.rows, P.iSpan, (int)left, wRow != 1).passes;
    const uint32_t *pRead = pSrc;
    if ((launches & 1) == 0) std::swap(pDest, pScratch);
    for (unsigned left = numPasses; left;) {
        const B26Shape shape = b26_shape(P.L, P.rows, P.iSpan, (int)left, wRow != 1);
        left -= (unsigned)shape.passes;
        P.passes = shape.passes;
        P.lines = shape.lines;
        P.wavesPerLine = shape.wavesPerLine;
        P.haloWaves = shape.haloWaves;
        P.blocks = (int)ckd_div_up(yRes, (unsigned)shape.lines);
        P.colStride = left ? (int)xRes : (int)wCol;
        P.rowStride = left ? 1 : (int)wRow;
        switch (shape.per) {
        case 3: launch_lines<3>(ctx, pDest, pRead, P); break;
        case 5: launch_lines<5>(ctx, pDest, pRead, P); break;
        case 7: launch_lines<7>(ctx, pDest, pRead, P); break;
        default: launch_lines<9>(ctx, pDest, pRead, P); break;
        }
        ckd_status s = ckd::check_launch("blur26 pass");
        if (s != CKD_OK) return s;
        pRead = pDest;
        std::swap(pDest, pScratch);
    }
    return CKD_OK;
}

ckd_status ensure_scratch(ckd_ctx *ctx, size_t pixels)
{
    if (ctx->b26Cap >= pixels) return CKD_OK;
    CKD_HIP(hipStreamSynchronize(ctx->stream));
    for (int i = 0; i < 2; ++i) {
        if (ctx->b26Scratch[i]) (void)hipFree(ctx->b26Scratch[i]);
        ctx->b26Scratch[i] = nullptr;
    }
    ctx->b26Cap = 0;
    for (int i = 0; i < 2; ++i)
        if (ckd::dev_alloc(&ctx->b26Scratch[i], pixels * 4) != hipSuccess) {
            ctx->b26Scratch[i] = nullptr;
            return ckd::fail(CKD_ENOMEM, "blur26: scratch allocation failed");
        }
    ctx->b26Cap = pixels;
    return CKD_OK;
}

ckd_status validate(const char *fn, const uint32_t *dst, const uint32_t *src, unsigned xRes,
                    unsigned yRes, float strength, float gain, unsigned passes, bool mult4)
{
    CKD_REQUIRE(dst && src, "%s: null buffer", fn);
    CKD_REQUIRE(dst != src, "%s: dst must differ from src", fn);
    CKD_REQUIRE(xRes >= 4 && yRes >= 4 && xRes <= (unsigned)kMaxRes && yRes <= (unsigned)kMaxRes,
                "%s: size %ux%u outside 4..%d", fn, xRes, yRes, kMaxRes);
    CKD_REQUIRE(!mult4 || ((xRes % 4) == 0 && (yRes % 4) == 0), "%s: sizes must be multiples of 4",
                fn);
    CKD_REQUIRE(strength >= 0.f && strength <= 100.f, "%s: strength %g outside [0,100]", fn,
                (double)strength);
    CKD_REQUIRE(gain >= 0.f && gain <= 1.f, "%s: gain %g outside [0,1]", fn, (double)gain);
    CKD_REQUIRE(passes >= 1 && passes <= 64, "%s: numPasses %u outside 1..64", fn, passes);
    return CKD_OK;
}

} // namespace

extern "C" {

ckd_status ckd_blur26_h(ckd_ctx *ctx, uint32_t *dst, const uint32_t *src, unsigned xRes,
                        unsigned yRes, float strength, float gain, unsigned numPasses)
{
    ckd_status s = validate("ckd_blur26_h", dst, src, xRes, yRes, strength, gain, numPasses, false);
    if (s != CKD_OK) return s;
    CKD_REQUIRE_CTX(ctx);
    s = ensure_scratch(ctx, (size_t)xRes * yRes);
    if (s != CKD_OK) return s;
    return horz(ctx, dst, ctx->b26Scratch[0], src, xRes, yRes, xRes, 1, strength, gain, numPasses);
}

ckd_status ckd_blur26_v(ckd_ctx *ctx, uint32_t *dst, const uint32_t *src, unsigned xRes,
                        unsigned yRes, float strength, float gain, unsigned numPasses)
{
    ckd_status s = validate("ckd_blur26_v", dst, src, xRes, yRes, strength, gain, numPasses, true);
    if (s != CKD_OK) return s;
    CKD_REQUIRE_CTX(ctx);
    s = ensure_scratch(ctx, (size_t)xRes * yRes);
    if (s != CKD_OK) return s;
    dim3 g(ckd_div_up(xRes, 32), ckd_div_up(yRes, 32));
    k_transpose<<<g, 256, 0, ctx->stream>>>(ctx->b26Scratch[1], src, (int)xRes, (int)yRes);
    s = ckd::check_launch("blur26 transpose");
    if (s != CKD_OK) return s;
    return horz(ctx, dst, ctx->b26Scratch[0], ctx->b26Scratch[1], yRes, xRes, 1, xRes, strength,
                gain, numPasses);
}

ckd_status ckd_blur26(ckd_ctx *ctx, uint32_t *dst, const uint32_t *src, unsigned xRes,
                      unsigned yRes, float strength, float gain, unsigned numPasses)
{
    ckd_status s = validate("ckd_blur26", dst, src, xRes, yRes, strength, gain, numPasses, true);
    if (s != CKD_OK) return s;
    CKD_REQUIRE_CTX(ctx);
    s = ensure_scratch(ctx, (size_t)xRes * yRes);
    if (s != CKD_OK) return s;
    s = horz(ctx, ctx->b26Scratch[1], ctx->b26Scratch[0], src, xRes, yRes, 1, yRes, strength, gain,
             numPasses);
    if (s != CKD_OK) return s;
    return horz(ctx, dst, ctx->b26Scratch[0], ctx->b26Scratch[1], yRes, xRes, 1, xRes, strength,
                gain, numPasses);
}

} // extern "C"
