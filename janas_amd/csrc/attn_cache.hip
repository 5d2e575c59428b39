/*
 * attn_cache.hip - the device side of the rules around the KV-cache
 * attention: writing new K/V rows into the cache, preparing the queries,
 * turning cached keys back on a context shift, and putting the attention
 * output into Q8_K blocks for the next product. Each kernel follows the
 * reference's arithmetic operation for operation, so that its bits are the
 * reference's:
 *
 *   rows_kernel    qkv_item (src/llm/model_attn.c:75-146): per (token, head)
 *                  row, the rms norm (model_impl.h:635-644: a double sum of
 *                  squares in order, 1 / sqrtf(mean + eps), x * s * w), the
 *                  NeoX rotation of the first n_rot dimensions
 *                  (model_attn.c:30-39), for values optionally the weightless
 *                  norm (model_attn.c:106-113), then 8 or 16 bits with a scale
 *                  of the row's own (the largest magnitude becomes 127 or
 *                  32767, lrintf), or f16 / f32 as they are.
 *   unrotate       unrotate_row (model.c:263-290): dequantize, rotate back,
 *                  find the largest magnitude anew, requantize.
 *   q8k_kernel     q8k_quantize_ref (quant.c:174-200, q8_32_ref :150-172):
 *                  d = amax / 127, 1 / d, rint, sums of 16 and of 32.
 *
 * A row of whole words of four is 16 lanes, its numbers in registers
 * (rows16_kernel); any other row is one wave: its numbers sit in LDS, the
 * lanes take the elementwise steps and the rotation's pairs, a wave reduction
 * (exact: a maximum) finds the largest magnitude, and lane 0 alone adds the
 * squares in the reference's order - the one step whose rounding depends on
 * order. No multiply-add is fused in this file, as in the reference's build
 * (-ffp-contract=off), but for squares that are exact in double.
 */
#pragma clang fp contract(off)

#include <math.h>
#include <stdint.h>

#include <hip/hip_runtime.h>

#include "attn_kernels.h"
#include "attn_q8k.h"

namespace janas {
namespace {

constexpr int kRowWaves = 4;    /* rows (waves) a workgroup */
constexpr int kMaxHd = 512;

__device__ __forceinline__ float wave_max(float x)
{
#pragma unroll
    for (int o = 32; o > 0; o >>= 1)
        x = fmaxf(x, __shfl_xor(x, o, 64));
    return x;
}

/* 1 / sqrtf(mean of squares + eps), the sum of squares in double in the
   order of the row (model_impl.h:638-641); lane 0 computes, all get it */
__device__ float inv_rms(const float *r, uint32_t n, float eps, uint32_t lane,
                         float *slot)
{
    if (lane == 0) {
        double ss = 0.0;
        for (uint32_t i = 0; i < n; i++)
            ss += (double)r[i] * r[i];
        *slot = 1.0f / sqrtf((float)(ss / n) + eps);
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    return *slot;
}

/* the NeoX rotation of r[0 .. n_rot) by the token's table (model_attn.c:
   30-39), or turned back by it (back: model.c:273-277) */
__device__ void rotate(float *r, uint32_t n_rot, const float *cs,
                       const float *sn, uint32_t lane, bool back)
{
    const uint32_t half = n_rot / 2;
    for (uint32_t i = lane; i < half; i += 64) {
        const float a = r[i], b = r[i + half];
        if (!back) {
            r[i] = a * cs[i] - b * sn[i];
            r[i + half] = a * sn[i] + b * cs[i];
        } else {
            r[i] = a * cs[i] + b * sn[i];
            r[i + half] = b * cs[i] - a * sn[i];
        }
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

/* r[0 .. hd) at 8 or 16 bits (or f16 / f32) into dst, the scale to *z */
__device__ void quantize_row(const float *r, uint32_t hd, int kv, void *dst,
                             float *z, uint32_t lane)
{
    float mx = 0.0f;
    for (uint32_t i = lane; i < hd; i += 64)
        mx = fmaxf(mx, fabsf(r[i]));
    mx = wave_max(mx);
    if (kv == kI8 || kv == kI16) {
        const float top = kv == kI16 ? 32767.0f : 127.0f;
        const float inv = mx > 0.0f ? top / mx : 0.0f;
        if (lane == 0)
            *z = mx / top;
        for (uint32_t i = lane; i < hd; i += 64) {
            const float q = rintf(r[i] * inv);
            if (kv == kI16)
                ((int16_t *)dst)[i] = (int16_t)q;
            else
                ((int8_t *)dst)[i] = (int8_t)q;
        }
    } else if (kv == kF16) {
        for (uint32_t i = lane; i < hd; i += 64)
            ((_Float16 *)dst)[i] = (_Float16)r[i];
    } else {
        for (uint32_t i = lane; i < hd; i += 64)
            ((float *)dst)[i] = r[i];
    }
}

/*
 * Rows of the write (qkv_item's key and value part) and of the query
 * preparation: row id = j * heads + h. For the cache write a row is a key
 * and a value; for queries the query alone, turned in place.
 */
__global__ __launch_bounds__(64 * kRowWaves) void rows_kernel(const RowArgs A)
{
    __shared__ float sK[kRowWaves][kMaxHd], sV[kRowWaves][kMaxHd];
    __shared__ float sS[kRowWaves];
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t id = blockIdx.x * kRowWaves + w;
    if (id >= A.n * A.heads)
        return;
    const uint32_t j = id / A.heads, h = id % A.heads, hd = A.hd;
    const uint32_t half = A.n_rot / 2;
    const float *cs = A.cs + (size_t)j * half, *sn = A.sn + (size_t)j * half;
    float *kr = sK[w], *vr = sV[w];
    const size_t src = (size_t)id * hd;
    for (uint32_t i = lane; i < hd; i += 64)
        kr[i] = A.k[src + i];
    if (A.v)
        for (uint32_t i = lane; i < hd; i += 64)
            vr[i] = A.v[src + i];
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");

    if (A.norm) {
        const float s = inv_rms(kr, hd, A.eps, lane, &sS[w]);
        for (uint32_t i = lane; i < hd; i += 64)
            kr[i] = kr[i] * s * A.norm[i];
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    rotate(kr, A.n_rot, cs, sn, lane, false);
    if (!A.kc) {
        /* the query: in place */
        for (uint32_t i = lane; i < hd; i += 64)
            A.k[src + i] = kr[i];
        return;
    }
    if (A.v_norm) {
        const float s = inv_rms(vr, hd, A.eps, lane, &sS[w]);
        for (uint32_t i = lane; i < hd; i += 64)
            vr[i] = vr[i] * s;
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    const uint32_t p = A.pos0 + j, row = A.ring ? p % A.cap : p;
    const size_t at = (size_t)h * A.cap + row;
    const size_t eb = A.kv == kI8 ? 1 : A.kv == kF32 ? 4 : 2;
    quantize_row(kr, hd, A.kv, (char *)A.kc + at * hd * eb, A.kz ? A.kz + at : nullptr,
                 lane);
    quantize_row(vr, hd, A.kv, (char *)A.vc + at * hd * eb, A.vz ? A.vz + at : nullptr,
                 lane);
}

/* ---- rows of whole 4-number words: 16 lanes a row ---------------------- */

/*
 * The same rows, four a wave: lane c of a row's 16 holds numbers 64 b + 4 c ..
 * + 3 for b < NB (head sizes up to 64 NB), so every access is a word of four
 * numbers and the reductions are DPP steps inside 16 lanes. It takes rows of
 * whole words (head size and half the rotation multiples of 4, every array
 * aligned to its word); the kernels above take the rest.
 *
 * What bounded the wave-a-row kernel was the serial sum of squares: one lane,
 * hd double additions behind LDS reads. One token's 32 query rows of 128 took it
 * 7.2 us and take 4.5 here (two memory round trips and a chain of divisions and
 * a square root); 512 tokens' rows 14.9 us and 5.4 (16.8 MB in and out: 3.6 us
 * at the rate of a large copy).
 */
constexpr int kRowLanes = 16;
constexpr int kRowsWg = 256 / kRowLanes;  /* rows a workgroup */

typedef float f4 __attribute__((ext_vector_type(4)));
typedef int i4 __attribute__((ext_vector_type(4)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef int16_t s4 __attribute__((ext_vector_type(4)));

template <int CTRL> __device__ __forceinline__ float dpp(float x)
{
    return __uint_as_float(
        __builtin_amdgcn_update_dpp(0u, __float_as_uint(x), CTRL, 0xf, 0xf, false));
}
template <int CTRL> __device__ __forceinline__ double dpp(double x)
{
    const uint2 u = __builtin_bit_cast(uint2, x);
    return __builtin_bit_cast(
        double, make_uint2(__builtin_amdgcn_update_dpp(0u, u.x, CTRL, 0xf, 0xf, false),
                           __builtin_amdgcn_update_dpp(0u, u.y, CTRL, 0xf, 0xf, false)));
}
/* over a row's 16 lanes, in every lane: quad_perm [1, 0, 3, 2], [2, 3, 0, 1],
   row_ror 8, row_ror 4. In that order each step adds (or compares) the same
   two numbers in both lanes of a pair, so a sum has the same bits in all 16
   (row_ror 4 first would pair each quad with another one in each) */
__device__ __forceinline__ float max16(float x)
{
    x = fmaxf(x, dpp<0xB1>(x));
    x = fmaxf(x, dpp<0x4E>(x));
    x = fmaxf(x, dpp<0x128>(x));
    return fmaxf(x, dpp<0x124>(x));
}
__device__ __forceinline__ double sum16(double x)
{
    x += dpp<0xB1>(x);
    x += dpp<0x4E>(x);
    x += dpp<0x128>(x);
    return x + dpp<0x124>(x);
}

/*
 * 1 / sqrtf(mean of squares + eps) of the row in r (zeros past hd), the bits
 * of the sum in the order of the row (inv_rms above). The sum is taken as a
 * tree. Every square is exact in double and none is negative, so a sum of hd
 * of them, in any order, is within hd 2^-53 of the exact one, and the two
 * orders within hd 2^-52 of each other; with the division's (here a multiply
 * by 1 / hd's) roundings, mean (1 +- (hd + 2) 2^-51) holds the mean of the
 * row's order. Where both ends round to the same float - all but one row in
 * 2^18 at hd 128 - that float is the mean in the row's order too, since
 * rounding is monotone. Otherwise (and where the row holds a NaN) the row's
 * lanes take the sum again in its order.
 */
template <int NB>
__device__ __forceinline__ float inv_rms16(const f4 *r, uint32_t hd, float eps, double inv_hd)
{
    double ss = 0.0;
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int e = 0; e < 4; e++)
            ss = __builtin_fma((double)r[b][e], (double)r[b][e], ss);
    const double mean = sum16(ss) * inv_hd;
    const double off = mean * ((double)(hd + 2) * 0x1p-51);
    const float lo = (float)(mean - off), hi = (float)(mean + off);
    float m = lo;
    if (__builtin_expect(!(lo == hi), 0)) {
        /* lanes of other rows of the wave may be off here: each of the 16
           lanes of this row is on */
        const uint32_t row0 = threadIdx.x & 48;
        double so = 0.0;
#pragma unroll
        for (int b = 0; b < NB; b++)
            for (uint32_t c = 0; c < kRowLanes && 64 * b + 4 * c < hd; c++)
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const double x = (double)__shfl(r[b][e], row0 + c, 64);
                    so = __builtin_fma(x, x, so);
                }
        m = (float)(so / hd);
    }
    return 1.0f / sqrtf(m + eps);
}

/* the rotation of the row's first 2 half numbers by the token's table, or back:
   through the row's LDS words, since number i's partner i + half may be in
   another lane */
template <int NB, bool BACK>
__device__ __forceinline__ void rotate16(f4 *r, float *lds, uint32_t c, uint32_t hd, uint32_t half,
                                         const f4 *cs, const f4 *sn)
{
    if (half == 0)
        return;
#pragma unroll
    for (int b = 0; b < NB; b++)
        if (64 * b + 4 * c < hd)
            *(f4 *)(lds + 64 * b + 4 * c) = r[b];
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const uint32_t col = 64 * b + 4 * c;
        if (col >= 2 * half || col >= hd)
            continue;
        const bool up = col >= half;
        const f4 o = *(const f4 *)(lds + (up ? col - half : col + half));
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const float x = r[b][e], y = o[e], cc = cs[b][e], ss = sn[b][e];
            if (!BACK)
                r[b][e] = up ? y * ss + x * cc : x * cc - y * ss;
            else
                r[b][e] = up ? x * cc - y * ss : x * cc + y * ss;
        }
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}

/* the lane's words of a token's table: column col's angle is col or
   col - half of it (unused past the rotation) */
template <int NB>
__device__ __forceinline__ void load_table(const float *t, uint32_t c, uint32_t half, f4 *x)
{
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const uint32_t col = 64 * b + 4 * c;
        x[b] = f4{0, 0, 0, 0};
        if (col < 2 * half)
            x[b] = *(const f4 *)(t + (col < half ? col : col - half));
    }
}

/* quantize_row for a row in 16 lanes */
template <int NB, int kv>
__device__ __forceinline__ void put_row16(const f4 *r, uint32_t c, uint32_t hd, void *dst,
                                          float *z)
{
    if constexpr (kv == kI8 || kv == kI16) {
        float mx = 0.0f;
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                mx = fmaxf(mx, fabsf(r[b][e]));
        mx = max16(mx);
        const float top = kv == kI16 ? 32767.0f : 127.0f;
        const float inv = mx > 0.0f ? top / mx : 0.0f;
        if (c == 0)
            *z = mx / top;
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const uint32_t col = 64 * b + 4 * c;
            if (col >= hd)
                continue;
            if (kv == kI16) {
                s4 q;
#pragma unroll
                for (int e = 0; e < 4; e++)
                    q[e] = (int16_t)rintf(r[b][e] * inv);
                *(s4 *)((int16_t *)dst + col) = q;
            } else {
                uint32_t q = 0;
#pragma unroll
                for (int e = 0; e < 4; e++)
                    q |= (uint32_t)(uint8_t)(int8_t)rintf(r[b][e] * inv) << (8 * e);
                *(uint32_t *)((int8_t *)dst + col) = q;
            }
        }
        return;
    }
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const uint32_t col = 64 * b + 4 * c;
        if (col >= hd)
            continue;
        if (kv == kF16) {
            h4 q;
#pragma unroll
            for (int e = 0; e < 4; e++)
                q[e] = (_Float16)r[b][e];
            *(h4 *)((_Float16 *)dst + col) = q;
        } else {
            *(f4 *)((float *)dst + col) = r[b];
        }
    }
}

/* rows_kernel's rows, 16 lanes each; KV the cache's type, or -1: queries (a
   type's test in the kernel was a jump over the others' code, a miss of the
   instruction cache: four layers' decode step 106.7 -> 105.4 us) */
template <int NB, int KV>
__global__ __launch_bounds__(256) void rows16_kernel(const RowArgs A)
{
    __shared__ __attribute__((aligned(16))) float sR[kRowsWg][64 * NB];
    const uint32_t c = threadIdx.x % kRowLanes, w = threadIdx.x / kRowLanes;
    const uint32_t id = blockIdx.x * kRowsWg + w;
    if (id >= A.n * A.heads)
        return;
    const uint32_t j = id / A.heads, h = id % A.heads, hd = A.hd, half = A.n_rot / 2;
    const size_t src = (size_t)id * hd;
    /* everything the row needs, asked for at once */
    f4 k[NB], v[NB], nw[NB], cs[NB], sn[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const uint32_t col = 64 * b + 4 * c;
        k[b] = v[b] = nw[b] = f4{0, 0, 0, 0};
        if (col >= hd)
            continue;
        k[b] = *(const f4 *)(A.k + src + col);
        if (A.v)
            v[b] = *(const f4 *)(A.v + src + col);
        if (A.norm)
            nw[b] = *(const f4 *)(A.norm + col);
    }
    load_table<NB>(A.cs + (size_t)j * half, c, half, cs);
    load_table<NB>(A.sn + (size_t)j * half, c, half, sn);
    if (A.norm) {
        const float s = inv_rms16<NB>(k, hd, A.eps, A.inv_hd);
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                k[b][e] = k[b][e] * s * nw[b][e];
    }
    rotate16<NB, false>(k, sR[w], c, hd, half, cs, sn);
    if constexpr (KV < 0) {
        /* the query: in place */
#pragma unroll
        for (int b = 0; b < NB; b++)
            if (64 * b + 4 * c < hd)
                *(f4 *)(A.k + src + 64 * b + 4 * c) = k[b];
        return;
    }
    if (A.v_norm) {
        const float s = inv_rms16<NB>(v, hd, A.eps, A.inv_hd);
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                v[b][e] = v[b][e] * s;
    }
    const uint32_t p = A.pos0 + j, row = A.ring ? p % A.cap : p;
    const size_t at = (size_t)h * A.cap + row;
    constexpr size_t eb = KV == kI8 ? 1 : KV == kF32 ? 4 : 2;
    put_row16<NB, KV>(k, c, hd, (char *)A.kc + at * hd * eb, A.kz + at);
    put_row16<NB, KV>(v, c, hd, (char *)A.vc + at * hd * eb, A.vz + at);
}

/* four numbers of a cached row as the word they are kept in */
template <int KV> struct Word;
template <> struct Word<kI8> {
    typedef uint32_t Raw;
    __device__ static float at(Raw r, int e) { return (float)(int8_t)(r >> (8 * e)); }
};
template <> struct Word<kI16> {
    typedef uint2 Raw;
    __device__ static float at(Raw r, int e)
    {
        return (float)(int16_t)((e < 2 ? r.x : r.y) >> (16 * (e & 1)));
    }
};

/*
 * shift_kernel's rows, 16 lanes each. A row's lanes take the positions i, i +
 * stride, i + 2 stride .. of those that move, in that order. In place (the
 * copy is the cache itself, stride the shift's distance) that is a chain: each
 * position's row is read, then goes to where the one before it in the chain
 * came from, and no other chain reads or writes either row - so the moved rows
 * need no copy. From a copy the stride is all of them: one row each.
 *
 * Bound by memory where chains are short: 16352 of 32768 int8 positions of
 * 8 x 128 moved in 20.4 us (69 MB, 3.4 TB/s), the call 111 -> 31 us; through
 * four strided copies and a wave a row, a byte a lane, the copies took 20 us,
 * the rows 58 and the allocation most of the rest.
 */
template <int KV, int NB>
__global__ __launch_bounds__(256) void shift16_kernel(const ShiftArgs A)
{
    using W = Word<KV>;
    typedef typename W::Raw Raw;
    __shared__ __attribute__((aligned(16))) float sR[kRowsWg][64 * NB];
    const uint32_t c = threadIdx.x % kRowLanes, w = threadIdx.x / kRowLanes;
    const uint64_t id = (uint64_t)blockIdx.x * kRowsWg + w;
    const uint32_t chains = A.stride < A.count ? A.stride : A.count;
    if (id >= (uint64_t)A.n_kv * chains)
        return;
    const uint32_t h = (uint32_t)(id / chains), hd = A.hd, half = A.n_rot / 2;
    const uint32_t words = hd / 4;
    f4 cs[NB], sn[NB];
    load_table<NB>(A.cs, c, half, cs);
    load_table<NB>(A.sn, c, half, sn);
    for (uint64_t i = id % chains; i < A.count; i += A.stride) {
        const uint32_t p = A.first + (uint32_t)i; /* the position as it was */
        const uint32_t srow = A.ring ? p % A.cap : p - A.copy_first;
        const uint32_t drow = A.ring ? (p - A.drop) % A.cap : p - A.drop;
        const size_t sat = (size_t)h * A.copy_rows + srow;
        const size_t dat = (size_t)h * A.cap + drow;
        Raw k[NB], v[NB];
#pragma unroll
        for (int b = 0; b < NB; b++) {
            k[b] = v[b] = Raw{};
            if (16 * b + c < words) {
                k[b] = ((const Raw *)A.ck)[sat * words + 16 * b + c];
                v[b] = ((const Raw *)A.cv)[sat * words + 16 * b + c];
            }
        }
        const float z = A.ckz[sat], vz = A.cvz[sat];
        /* the value row and its scale move as they are, and the key's when
           there is nothing to turn */
#pragma unroll
        for (int b = 0; b < NB; b++)
            if (16 * b + c < words) {
                ((Raw *)A.v)[dat * words + 16 * b + c] = v[b];
                if (half == 0)
                    ((Raw *)A.k)[dat * words + 16 * b + c] = k[b];
            }
        if (c == 0) {
            A.vz[dat] = vz;
            if (half == 0)
                A.kz[dat] = z;
        }
        if (half == 0)
            continue;
        f4 r[NB];
#pragma unroll
        for (int b = 0; b < NB; b++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                r[b][e] = W::at(k[b], e) * z;
        rotate16<NB, true>(r, sR[w], c, hd, half, cs, sn);
        put_row16<NB, KV>(r, c, hd, (Raw *)A.k + dat * words, A.kz + dat);
    }
}

/*
 * Rows that are not whole words: moved position i of KV head h is read from the copy
 * (rows src_first + i of the copy, mod cap for a ring), written to its new
 * row, and its key turned back by the shift's angles and quantized anew
 * (model.c:304-377; unrotate_row :263-290).
 */
__global__ __launch_bounds__(64 * kRowWaves) void shift_kernel(const ShiftArgs A)
{
    __shared__ float sK[kRowWaves][kMaxHd];
    const uint32_t lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t id = blockIdx.x * kRowWaves + w;
    if (id >= A.n_kv * A.count)
        return;
    const uint32_t h = id / A.count, i = id % A.count;
    const uint32_t p = A.first + i; /* the position as it was */
    const uint32_t srow = A.ring ? p % A.cap : p - A.copy_first;
    const uint32_t drow = A.ring ? (p - A.drop) % A.cap : p - A.drop;
    const uint32_t hd = A.hd;
    const size_t eb = A.kv == kI16 ? 2 : 1, rowb = hd * eb;
    const size_t sat = (size_t)h * A.copy_rows + srow;
    const size_t dat = (size_t)h * A.cap + drow;
    /* the value row and its scale move as they are */
    for (uint32_t b = lane; b < rowb; b += 64)
        ((uint8_t *)A.v)[dat * rowb + b] = ((const uint8_t *)A.cv)[sat * rowb + b];
    float *kr = sK[w];
    const float z = A.ckz[sat];
    for (uint32_t e = lane; e < hd; e += 64) {
        const float x = A.kv == kI16 ? (float)((const int16_t *)A.ck)[sat * hd + e]
                                     : (float)((const int8_t *)A.ck)[sat * hd + e];
        kr[e] = x * z;
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    if (lane == 0)
        A.vz[dat] = A.cvz[sat];
    if (A.n_rot / 2 == 0) {
        /* nothing to turn: the key row and its scale move as they are */
        for (uint32_t b = lane; b < rowb; b += 64)
            ((uint8_t *)A.k)[dat * rowb + b] = ((const uint8_t *)A.ck)[sat * rowb + b];
        if (lane == 0)
            A.kz[dat] = z;
        return;
    }
    rotate(kr, A.n_rot, A.cs, A.sn, lane, true);
    quantize_row(kr, hd, A.kv, (char *)A.k + dat * rowb, A.kz + dat, lane);
}

/*
 * One Q8_K block (256 numbers of a token's output) a workgroup of 256:
 * thread t takes number t (quant.c:174-200).
 */
__global__ __launch_bounds__(256) void q8k_kernel(const Q8kArgs A)
{
    __shared__ Q8kLds S;
    const uint32_t t = threadIdx.x, b = blockIdx.x;
    q8k_block(A.x[(size_t)b * 256 + t], t, A.y + (size_t)b * kQ8kBytes, S);
}

/* one 4-byte word a thread: tensor blockIdx.y, word i of its packed rows */
__global__ __launch_bounds__(256) void refresh_kernel(const RefreshArgs A)
{
    const uint32_t t = blockIdx.y, i = blockIdx.x * 256 + threadIdx.x;
    const uint32_t w = A.words[t], per_head = A.count * w;
    if (i >= A.n_kv * per_head)
        return;
    const uint32_t h = i / per_head, r = (i % per_head) / w, e = i % w;
    const uint32_t row = (A.lo + r) % A.cap;
    A.dst[t][((size_t)h * A.cap + row) * w + e] = A.src[t][i];
}

}  // namespace

hipError_t launch_refresh(const RefreshArgs &a, hipStream_t s)
{
    uint32_t most = 0;
    for (uint32_t t = 0; t < a.n_t; t++)
        most = a.words[t] > most ? a.words[t] : most;
    const uint64_t words = (uint64_t)a.n_kv * a.count * most;
    if (a.n_t == 0 || words == 0)
        return hipSuccess;
    if (a.n_t > 4 || words > 0xFFFFFFFFull)
        return hipErrorInvalidValue;
    hipLaunchKernelGGL(refresh_kernel, dim3((uint32_t)((words + 255) / 256), a.n_t), dim3(256),
                       0, s, a);
    return hipGetLastError();
}

/* whether p holds whole words of `bytes` */
static bool aligned(const void *p, size_t bytes) { return (uintptr_t)p % bytes == 0; }

static size_t elem_size(int kv) { return kv == kI8 ? 1 : kv == kF32 ? 4 : 2; }

template <int KV> static hipError_t rows16(const RowArgs &a, hipStream_t s)
{
    const dim3 grid((a.n * a.heads + kRowsWg - 1) / kRowsWg), block(256);
    if (a.hd <= 64)
        hipLaunchKernelGGL((rows16_kernel<1, KV>), grid, block, 0, s, a);
    else if (a.hd <= 128)
        hipLaunchKernelGGL((rows16_kernel<2, KV>), grid, block, 0, s, a);
    else if (a.hd <= 256)
        hipLaunchKernelGGL((rows16_kernel<4, KV>), grid, block, 0, s, a);
    else
        hipLaunchKernelGGL((rows16_kernel<8, KV>), grid, block, 0, s, a);
    return hipGetLastError();
}

hipError_t launch_rows(const RowArgs &a, hipStream_t s)
{
    const uint32_t rows = a.n * a.heads;
    if (rows == 0)
        return hipSuccess;
    /* rows of whole words of four take 16 lanes each, any number of rows (one
       token's 7.2 -> 4.5 us, 512 tokens' 14.9 -> 5.4 us) */
    const size_t word = 4 * elem_size(a.kv);
    if (a.hd % 4 == 0 && a.n_rot % 8 == 0 && aligned(a.k, 16) && aligned(a.v, 16) &&
        aligned(a.norm, 16) && aligned(a.cs, 16) && aligned(a.sn, 16) && aligned(a.kc, word) &&
        aligned(a.vc, word)) {
        switch (a.kc ? a.kv : -1) {
        case -1:
            return rows16<-1>(a, s);
        case kI8:
            return rows16<kI8>(a, s);
        case kI16:
            return rows16<kI16>(a, s);
        case kF16:
            return rows16<kF16>(a, s);
        case kF32:
            return rows16<kF32>(a, s);
        }
        return hipErrorInvalidValue;
    }
    hipLaunchKernelGGL(rows_kernel, dim3((rows + kRowWaves - 1) / kRowWaves),
                       dim3(64 * kRowWaves), 0, s, a);
    return hipGetLastError();
}

bool shift_words(const ShiftArgs &a)
{
    const size_t word = 4 * elem_size(a.kv);
    return a.hd % 4 == 0 && a.n_rot % 8 == 0 && aligned(a.k, word) && aligned(a.v, word) &&
           aligned(a.ck, word) && aligned(a.cv, word) && aligned(a.cs, 16) && aligned(a.sn, 16);
}

template <int KV> static void shift16(const ShiftArgs &a, hipStream_t s)
{
    const uint64_t rows = (uint64_t)a.n_kv * (a.stride < a.count ? a.stride : a.count);
    const dim3 grid((uint32_t)((rows + kRowsWg - 1) / kRowsWg)), block(256);
    if (a.hd <= 64)
        hipLaunchKernelGGL((shift16_kernel<KV, 1>), grid, block, 0, s, a);
    else if (a.hd <= 128)
        hipLaunchKernelGGL((shift16_kernel<KV, 2>), grid, block, 0, s, a);
    else if (a.hd <= 256)
        hipLaunchKernelGGL((shift16_kernel<KV, 4>), grid, block, 0, s, a);
    else
        hipLaunchKernelGGL((shift16_kernel<KV, 8>), grid, block, 0, s, a);
}

hipError_t launch_shift(const ShiftArgs &a, hipStream_t s)
{
    const uint32_t rows = a.n_kv * a.count;
    if (rows == 0)
        return hipSuccess;
    if (shift_words(a)) {
        if (a.kv == kI16)
            shift16<kI16>(a, s);
        else
            shift16<kI8>(a, s);
        return hipGetLastError();
    }
    if (a.stride < a.count)
        return hipErrorInvalidValue; /* in place: words only */
    hipLaunchKernelGGL(shift_kernel, dim3((rows + kRowWaves - 1) / kRowWaves),
                       dim3(64 * kRowWaves), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_q8k(const Q8kArgs &a, hipStream_t s)
{
    if (a.blocks == 0)
        return hipSuccess;
    hipLaunchKernelGGL(q8k_kernel, dim3(a.blocks), dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace janas
