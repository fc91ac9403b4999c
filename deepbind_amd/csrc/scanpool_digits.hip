// Bulk path of the fused scan + bias + ReLU + region pooling forward: the scan as a product of 4-bit one-hot letters
// with the weights' 6-bit digits on the matrix cores.
//
// Written as a product the scan is Z (positions x filters) = H (positions x 4m) . W (4m x filters), H holding the one-hot
// letters of every position's window. v_mfma_scale_f32_32x32x64_f8f6f4 multiplies 4-bit by 6-bit floats with float32
// accumulation, 64 values of the contraction index per 32 clocks - four times what the bf16 instruction does - and both
// operands are exact in those formats:
//  * H: a letter is 4.0 in its own row, "mean of the four" (N, padding: code 255 and any other non-letter) 1.0 in all
//    four rows, code 254 nothing: the multiples 4, 1 and 0 of a quarter.
//  * W: every filter's weights as 30-bit fixed point numbers against the filter's largest (32^5 .. 32^6 units), written
//    in six digits of -16 .. 16: 1/8 .. 16/8 are exact in the 6-bit format (1 sign, 2 exponent, 3 fraction bits). The
//    instruction's per-lane block scale carries the filter's and the digit's power of two.
// So the products are exact and the float32 accumulator sees the small digits first. What is dropped is below 2^-29 of
// the filter's largest weight; measured against float64 the sums are off by 3.3e-8 (16 taps, normal weights) where
// float32 additions tap by tap are off by 7.6e-8 and through a table of 3-mer sums by 6.2e-8.
//
// A weight far below zero only has to keep its window closed: every window's rectified value is at most
// T = sum over the taps of the largest weight (if positive) + the bias, so a window with a weight below -4.125 T is closed, a
// "mean of the four" (-1.03 T + T) as well. Such weights are no part of the digits, whose unit they would make coarse (and
// with it the sums: an instruction adds to a float32 with the precision of its largest operands, as they would be with a
// first digit in every place): tiles that have them take one more product per 16 taps, -7.5 times a power of two above T in the
// place of every such weight. Filters that fixed point does not express well (an
// infinite or undefined weight, windows that may hold nothing but weights below a 256th to a 512th of the largest) are left to a launch behind
// this one (scanpool_fprop_left_kernel), which does nothing where no tile of filters asks for it.
//
// Mapping: a workgroup of 16 waves (one per CU) owns 32 filters, up to 16 taps one of 12 waves 64 of them; their digits stay in its registers
// (24 taps: 9 instructions' operands, 54 registers a lane). A wave takes a region at a time from the workgroup's counter and walks it
// in tiles of 32 positions. 224 positions' letters at a time become one 16-byte entry per position in the wave's own
// LDS: the one-hot nibbles of the eight letters from there on, which is half of an instruction's operand (lanes 0-31
// take taps 0-7, lanes 32-63 taps 8-15), so a tile costs one or two 16-byte reads per lane. An entry's place is
// q + q / 16: writes (four consecutive entries per lane) and reads are both free of bank conflicts.
//
// Bound: the matrix pipe, and through it the chip's power: an instruction takes its 34 clocks, at 1.5-1.6 GHz under this
// load (2.3 GHz with all operands zero), 22 ns per SIMD. A table of 3-mer sums in LDS (one 4-byte read and add per three
// taps), which this replaced, moved its 248 ns worth of LDS bytes per 32 x 32 tile of 24 taps; nine instructions are 198.
// Measured, table / all digits: max pooling, 100 000 x 500 letters x 1024 filters x 24 taps 12.8 / 10.4 ms (7.35 through half of the
// products, scanpool_digits_max_kernel below); 65 536 x 101 x 256
// filters, 24 taps 0.721 / 0.513, 16 taps 0.552 / 0.380; 20 000 x 500 x 256 x 8 taps 0.491 / 0.261; max + average, 20 000 x
// 30-150 x 384 x 16 taps 0.275 / 0.215 (0.19 now: launch_sets, scanpool_digits_body); with an argmax 65 536 x 101 x 256 x 24 taps 0.867 / 0.616; averages are off by
// 5.6e-8 instead of 1.7e-7 (a tile's sum first, then the tiles').
//
// Reference chain being fused: kangaroo/_ext/corr1ord.py:97-117 -> deepity/std/elemwise.py:162-180,71-82
// -> kangaroo/_ext/poolrgn.py:56-76 (kernels corr1ord.cuh:139-157, poolrgn.cuh:44-79).
#include "dbk_common.h"
#include "scan_common.h"
#include "mfma_common.h"
#include <mutex>
#include <type_traits>

namespace dbk_scanpool_general {
int fprop_left(hipStream_t st, const float* W, const float* bias, size_t m, size_t F, const uint8_t* X, size_t N,
               const uint32_t* R, size_t P, int ptype, float* pooled, uint32_t* argmax, const unsigned* flags);
}

namespace dbk_scanpool_digits {

using dbk_mfma::f32x16_t;
using dbk_scan::TILE_BULK;
using dbk_scan::TILE_CLOSES;
using dbk_scan::TILE_INFINITE;
using dbk_scan::TILE_LEFT;
using dbk_scan::TILE_NOT_FINITE;

typedef int i32x8_t __attribute__((ext_vector_type(8)));

constexpr int FTILE = 32;                     // filters per workgroup: columns of a tile
constexpr int ROWS = 32;                      // positions per tile
constexpr int NDIGIT = 6;                     // digits per weight
constexpr int NTOP = 3;                       // of them, the first ones that find a maximum's place
constexpr int NWAVE = 16;                     // waves per workgroup
constexpr unsigned CHUNK = 224;               // rows whose letters are staged at a time: seven tiles
constexpr unsigned ENTRIES = 304;             // entries of a wave: 256 positions, one entry of padding per 16, what a read past the last tile touches
constexpr unsigned SLOT_BYTES = FTILE * 24;   // one digit of eight taps of all the tile's filters: 32 values of 6 bits per filter
constexpr float CLOSED = -3.0e38f;            // the value of a row outside the region

// the LDS entry of a position: consecutive positions of a lane and of neighbouring lanes fall into different banks
__device__ __forceinline__ unsigned place(unsigned q) { return q + (q >> 4); }

// ---------------------------------------------------------------------------------------------- the weights' digits
// What a call keeps in its scratch, per tile of 32 filters: a flag (TILE_LEFT and its like), the filters'
// exponents, the digits, [8-tap block][digit][filter][24 bytes], to find a maximum's place NTOP digits per weight in
// units of the filter's own (no power of two) with what the scan has to know of them, and the weights that close windows,
// [8-tap block][filter][24 bytes].
struct digit_facts {
    float unit;         // digit NTOP - 1's step; zero where every window's sum is zero, or closed
    float above;        // the most that a window's weights lie above those digits, in units, and some slack
    float lowest;       // weights below only close their windows
    int whole;          // what an open window's weights and the bias come to, times 2^whole, is below 2^30
    unsigned shut;      // block scales of a closing weight: beside all the digits, beside the first ones
};
struct digit_store { unsigned* flags; int* expo; digit_facts* facts; unsigned char *digits, *top, *shut; };
inline size_t tile_bytes(unsigned tb) { return FTILE * (sizeof(int) + sizeof(digit_facts)) + (size_t)tb * (NDIGIT + NTOP + 1) * SLOT_BYTES; }
inline digit_store store_at(unsigned* flags, unsigned char* ws, unsigned ntile, unsigned tb)
{
    digit_store s;
    s.flags = flags;
    s.expo = reinterpret_cast<int*>(ws);
    s.facts = reinterpret_cast<digit_facts*>(s.expo + (size_t)ntile * FTILE);
    s.digits = reinterpret_cast<unsigned char*>(s.facts + (size_t)ntile * FTILE);
    s.top = s.digits + (size_t)ntile * tb * NDIGIT * SLOT_BYTES;
    s.shut = s.top + (size_t)ntile * tb * NTOP * SLOT_BYTES;
    return s;
}

// x, of magnitude up to 32, as ND digits base 32, each the nearest number that the 6-bit format has (in eighths: 0 .. 16, the even
// ones up to 32); what remains, in units of the next digit
template <int ND>
__device__ __forceinline__ void split_digits(float (&x)[4], unsigned char* o)
{
#pragma unroll
    for (int p = 0; p < ND; ++p) {
        unsigned word = 0u;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float d = fabsf(x[c]) <= 16.0f ? rintf(x[c]) : 2.0f * rintf(0.5f * x[c]);
            x[c] = (x[c] - d) * 32.0f;                            // (exact)
            const int i = (int)d;
            const unsigned a = (unsigned)(i < 0 ? -i : i);
            // a / 8 in 1 + 2 + 3 bits: the numbers 0 .. 16 are their own codes (denormal below 8), 18 .. 32 17 .. 24
            word |= ((a <= 16u ? a : 8u + (a >> 1)) | (i < 0 ? 32u : 0u)) << (6 * c);
        }
        unsigned char* q = o + (size_t)p * SLOT_BYTES;
        q[0] = (unsigned char)word; q[1] = (unsigned char)(word >> 8); q[2] = (unsigned char)(word >> 16);
    }
}

__device__ __forceinline__ float power_of_two(int k) { return __uint_as_float((unsigned)(127 + k) << 23); }
__device__ __forceinline__ int exponent_of(float v) { return (int)((__float_as_uint(v) >> 23) & 0xffu) - 127; }

// A workgroup splits one tile's weights, a thread per tap and filter. Latency only (4m x 32 values): with a thread per eight taps, which it
// was, 24 taps took 10 us.
template <int TB>
__global__ __launch_bounds__(256 * TB) void weight_digits_kernel(const float* __restrict__ W, const float* __restrict__ bias, unsigned m, unsigned F,
                                                                 unsigned f0, digit_store out)
{
    constexpr unsigned THREADS = 256 * TB, PARTS = 4 * TB;        // a filter's sums: a part per wave (two taps)
    __shared__ float parts[3][PARTS][FTILE];
    __shared__ unsigned most[4][FTILE], fewest[FTILE];            // maxima of numbers that are not negative, as their bits; a minimum
    __shared__ __align__(16) unsigned char dig[TB * (NDIGIT + NTOP + 1) * SLOT_BYTES];
    __shared__ unsigned tile, closing[FTILE];                     // what is noted of the tile's filters; which of them have closing weights
    const unsigned fl = threadIdx.x & 31u, tap = threadIdx.x >> 5, wave = threadIdx.x >> 6, f = f0 + blockIdx.x * FTILE + fl;
    if (threadIdx.x < FTILE) {
        most[0][fl] = most[1][fl] = most[2][fl] = most[3][fl] = closing[fl] = 0u;
        fewest[fl] = 0x7f000000u;
        tile = TILE_BULK;
    }
    float w[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) w[c] = (tap < m && f < F) ? W[(size_t)(4 * tap + c) * F + f] : 0.0f;
    const float b = f < F ? bias[f] : 0.0f;
    const unsigned bias_bits = __float_as_uint(b) & 0x7fffffffu;      // (the file is compiled without NaN: test the bits)
    bool finite = bias_bits < 0x7f800000u, infinite = false;          // infinite: minus infinity among the weights
    float best = 0.0f;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const unsigned bits = __float_as_uint(w[c]) & 0x7fffffffu;
        finite &= bits < 0x7f800000u || __float_as_uint(w[c]) == 0xff800000u;
        infinite |= bits == 0x7f800000u;
        best = fmaxf(best, w[c]);
    }
    // a filter's sum over its taps: the wave's two first, then the waves' in order
    auto part = [&](int k, float v) { const float two = v + __shfl_xor(v, 32, 64); if ((tap & 1u) == 0u) parts[k][wave][fl] = two; };
    auto sum = [&](int k) { float v = 0.0f; for (unsigned i = 0; i < PARTS; ++i) v += parts[k][i][fl]; return v; };
    part(0, best);
    __syncthreads();
    // ---- what a window and the bias come to at most; the weights that an open window can hold: all but those below -4.125 times that
    const float open = sum(0) + fmaxf(b, 0.0f), lowest = -4.125f * open;
    float largest = 0.0f, smallest = 3.0e38f, finer = 3.0e38f;     // of those: the tap's largest, smallest, smallest that is not zero
    bool closes[4], any_closes = false;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const float v = fabsf(w[c]);
        closes[c] = w[c] < lowest;
        any_closes |= closes[c];
        if (!closes[c]) {
            largest = fmaxf(largest, v);
            smallest = fminf(smallest, v);
            if (v > 0.0f) finer = fminf(finer, v);
        }
    }
    part(1, largest);
    atomicMax(&most[0][fl], __float_as_uint(largest));
    atomicMax(&most[3][fl], __float_as_uint(best));
    if (smallest < 3.0e38f) atomicMax(&most[1][fl], __float_as_uint(smallest));
    if (finer < 1.0e38f) atomicMin(&fewest[fl], __float_as_uint(finer));
    if (any_closes) atomicOr(&closing[fl], 1u);
    if (!finite) atomicMax(&most[2][fl], 1u);
    if (infinite) atomicOr(&tile, TILE_INFINITE);
    __syncthreads();
    const float mid = __uint_as_float(most[0][fl]), size = sum(1);
    const bool any = closing[fl] != 0u;
    // every open window that is not zero holds a weight, or the bias, of this size
    const float least = fmaxf(fmaxf(fabsf(b), __uint_as_float(most[1][fl])), __uint_as_float(fewest[fl]));
    // ---- all the digits: x = w * 2^(3 - e), the largest weight below 16, the others that count below 32
    const bool none = mid == 0.0f && !(any && open > 0.0f);       // every window's sum is zero, or closed with no bias to open it
    const int e_top = exponent_of(__uint_as_float(most[3][fl])), e_mid = exponent_of(mid) - 1;
    int e = mid > 0.0f ? (e_top > e_mid ? e_top : e_mid) : 0;
    // sizes near the type's ends, where a weight's bf16 pieces or a sum may leave it, go with the infinite and undefined ones
    const bool far = most[2][fl] != 0u || bias_bits >= 0x71000000u || !(open < 1.0e30f) || !(mid < 1.0e30f) || (mid != 0.0f && mid < 1.0e-32f);
    // The sums of windows without the largest weights are rounded in the size of those all the same. Where all of a window's weights may be
    // below 2^(e - 8), that is a 256th to a 512th of the largest (a 1024th of negative ones), the tile is left out. Measured, root mean square of the windows' relative error, 8 / 24 taps, two weights
    // for one letter at about that many times the others, letters without it (a float32 sum tap by tap 0.8e-7 / 1.7e-7): once 0.5e-7 / 0.6e-7,
    // 15 times 2.4e-7 / 1.6e-7, 30 4.2e-7 / 3.3e-7, 120 1.9e-7 / 2.5e-7, 240 3.6e-7 / 5.0e-7, 970 1.5e-6 / 1.9e-6, 15 000 2.4e-5 / 3.1e-5. Worst of 600 random sets of
    // weights of fifteen kinds that the digits keep: 8.2e-7 (3 taps, heavy tails), a single window 1.2e-5 (20 taps, large negative weights that do not
    // close; its value a small difference, float32 4e-6).
    const bool bad = far || e < -84 || (!none && open < 1.0e-25f) || (mid > 0.0f && __uint_as_float((unsigned)(127 + e - 8) << 23) > least);
    const unsigned notes = (far ? TILE_NOT_FINITE : bad ? TILE_LEFT : TILE_BULK) | (any ? TILE_CLOSES : TILE_BULK);
    if (tap == 0u && notes != TILE_BULK) atomicOr(&tile, notes);
    if (bad) e = 0;
    // The first ones by themselves: x = w / unit with a window's x at most 240 (so that its sum, in 1/1024, leaves room for a row's
    // number below it: see the scan) and a weight's at most 16.4
    const float scale = __uint_as_float((unsigned)(127 + 3 - e) << 23);
    const float finest = bad || none ? 1.0f : fmaxf(fmaxf(size * (1.0f / 240.0f), mid * (1.0f / 16.4f)), fmaxf(any ? open * 0x1.0p-40f : 0.0f, 1.0e-30f));
    const float per = 1.0f / finest;
    float x[4], y[4];
    unsigned shut = 0u;                                           // 63: -7.5
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        x[c] = bad || closes[c] ? 0.0f : w[c] * scale;
        y[c] = bad || closes[c] ? 0.0f : w[c] * per;
        shut |= closes[c] ? 63u << (6 * c) : 0u;
    }
    const unsigned block = tap >> 3, at = fl * 24u + 3u * (tap & 7u);
    split_digits<NDIGIT>(x, dig + block * NDIGIT * SLOT_BYTES + at);
    split_digits<NTOP>(y, dig + (TB * NDIGIT + block * NTOP) * SLOT_BYTES + at);
    unsigned char* q = dig + (TB * (NDIGIT + NTOP) + block) * SLOT_BYTES + at;
    q[0] = (unsigned char)shut; q[1] = (unsigned char)(shut >> 8); q[2] = (unsigned char)(shut >> 16);
    // the most that the weights exceed the first digits by, in units of the next digit (a letter that counts nothing exceeds nothing)
    part(2, fmaxf(fmaxf(fmaxf(y[0], y[1]), fmaxf(y[2], y[3])), 0.0f));
    __syncthreads();
    const uint2* src = reinterpret_cast<const uint2*>(dig);
    auto give = [&](unsigned char* to, unsigned digits) {
        uint2* dst = reinterpret_cast<uint2*>(to + (size_t)blockIdx.x * (TB * digits * SLOT_BYTES));
        for (unsigned i = threadIdx.x; i < TB * digits * SLOT_BYTES / 8; i += THREADS) dst[i] = src[i];
        src += TB * digits * SLOT_BYTES / 8;
    };
    give(out.digits, NDIGIT);
    give(out.top, NTOP);
    give(out.shut, 1u);
    if (tap == 0u) {
        out.expo[blockIdx.x * FTILE + fl] = e;
        digit_facts k;
        k.unit = none ? 0.0f : finest * (1.0f / 1024.0f);
        // a quarter of a unit for the rounding of a window's sum and of the scaled weights (sums of at most 240 * 1024 units, half a dozen
        // roundings of 2^-24) and of all the digits' (below 1/32), so that a place that is sure is the one that all the digits find. A bias
        // far above the weights makes the value coarse, by 2^-30 of it per tap. (The rows' numbers only raise the second sum.)
        k.above = sum(2) * (1.00001f / 32.0f) + 0.25f + (float)(8 * TB) * 0x1.0p-30f * (open * per * 1024.0f);
        k.lowest = lowest;
        k.whole = open > 0.0f && !bad ? 29 - exponent_of(open) : 0;   // open < 2^(exponent + 1)
        k.shut = open > 0.0f && !bad ? (unsigned)(130 + exponent_of(open)) | (unsigned)(130 + exponent_of(open * per * 1024.0f)) << 8 : 127u | 127u << 8;
        out.facts[blockIdx.x * FTILE + fl] = k;
    }
    if (threadIdx.x == 0) out.flags[blockIdx.x] = tile;
}

// ---------------------------------------------------------------------------------------------- letters
// Four letter codes (bytes) as four 16-bit groups of one-hot nibbles, two registers. 6 is 4.0 and 2 is 1.0 in the 4-bit
// format. The codes' low three bits (0-3 letters, 6: 254, 7: 255) select the byte of an eight-byte table each.
__device__ __forceinline__ uint2 letter_nibbles(unsigned v)
{
    const unsigned sel = v & 0x07070707u;
    const unsigned lo = __builtin_amdgcn_perm(0x22002222u, 0x00006006u, sel), hi = __builtin_amdgcn_perm(0x22002222u, 0x60060000u, sel);
    return make_uint2(__builtin_amdgcn_perm(hi, lo, 0x05010400u), __builtin_amdgcn_perm(hi, lo, 0x07030602u));
}
// nonzero where a byte's upper six bits differ from each other: a code between 4 and 251, which counts as 255
__device__ __forceinline__ unsigned odd_codes(unsigned v) { return (v ^ (v << 1)) & 0xf8f8f8f8u; }
__device__ __forceinline__ unsigned plain_codes(unsigned v)
{
    unsigned r = 0u;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const unsigned c = (v >> (8 * k)) & 0xffu;
        r |= ((c < 4u || c == 254u) ? c : 255u) << (8 * k);
    }
    return r;
}

// B bytes of X from o on, which run past its end: bytes past the end are undefined (they only reach windows that are closed).
// Kept small and out of the way: only a stream's last stretches come here.
template <int B>
__device__ __forceinline__ void load_tail(const uint8_t* __restrict__ X, size_t N, size_t o, unsigned (&v)[B / 4])
{
#pragma unroll
    for (int k = 0; k < B / 4; ++k) v[k] = 0u;
#pragma unroll 1
    for (unsigned i = 0; i < B; ++i) {
        const unsigned c = o + i < N ? X[o + i] : 0u;
#pragma unroll
        for (int k = 0; k < B / 4; ++k) v[k] |= (i >> 2) == (unsigned)k ? c << (8u * (i & 3u)) : 0u;
    }
}

// The twelve letters from position c + 4 * lane on.
__device__ __forceinline__ void load12(const uint8_t* __restrict__ X, size_t N, unsigned c, unsigned lane, unsigned (&v)[3])
{
    const size_t o = (size_t)c + 4u * lane;
    if ((size_t)c + 4u * 63u + 12u <= N) __builtin_memcpy(v, X + o, 12);
    else load_tail<12>(X, N, o, v);
}

// A wave's 256 positions (each lane: its twelve letters) into its entries: the nibbles of eight letters per position.
__device__ __forceinline__ void stage(uint4* entries, unsigned lane, unsigned (&v)[3])
{
    if (__any((odd_codes(v[0]) | odd_codes(v[1]) | odd_codes(v[2])) != 0u)) {
#pragma unroll
        for (int k = 0; k < 3; ++k) v[k] = plain_codes(v[k]);
    }
    const uint2 n0 = letter_nibbles(v[0]), n1 = letter_nibbles(v[1]), n2 = letter_nibbles(v[2]);
    const unsigned p[6] = {n0.x, n0.y, n1.x, n1.y, n2.x, n2.y};
    unsigned q[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) q[k] = __builtin_amdgcn_alignbit(p[k + 1], p[k], 16);
    uint4* dst = entries + place(4u * lane);
    __builtin_amdgcn_wave_barrier();
    dst[0] = make_uint4(p[0], p[1], p[2], p[3]);
    dst[1] = make_uint4(q[0], q[1], q[2], q[3]);
    dst[2] = make_uint4(p[1], p[2], p[3], p[4]);
    dst[3] = make_uint4(q[1], q[2], q[3], q[4]);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The next region of the workgroup's, the same in all lanes.
__device__ __forceinline__ unsigned claim(unsigned* counter, unsigned lane)
{
    unsigned v = 0u;
    if (lane == 0u) v = atomicAdd(counter, 1u);
    return (unsigned)__builtin_amdgcn_readfirstlane((int)v);
}

// Where a lane's operands lie: tile t of a staged stretch reads entries 34 t + these (34 entries per 32 positions). The
// first holds its half wave's block of taps 0-15, the second that of taps 16-31.
template <int TB> __device__ __forceinline__ unsigned first_operand(unsigned col, unsigned h) { return place(col + (TB >= 2 ? 8u * h : 0u)); }
template <int TB> __device__ __forceinline__ unsigned second_operand(unsigned col, unsigned h) { return place(col + 16u + (TB == 4 ? 8u * h : 0u)); }

// Rows from c on that the scan defines, as far as a staged stretch is concerned.
__device__ __forceinline__ unsigned defined_rows(size_t ndef, unsigned c)
{
    return (size_t)c >= ndef ? 0u : (ndef - c < 2 * CHUNK ? (unsigned)(ndef - c) : 2 * CHUNK);
}
// Rows the scan does not define hold the rectified bias: no letter in their windows. Only the stream's last tiles come here;
// the empty statement keeps it a branch (as selects it would be a third of a tile's vector instructions).
__device__ __forceinline__ void close_undefined(uint4& a0, uint4& a1, bool defined)
{
    asm volatile("");
    if (!defined) { a0 = make_uint4(0u, 0u, 0u, 0u); a1 = a0; }
}

// ---------------------------------------------------------------------------------------------- the products
// instructions per tile: two 8-tap blocks (one per half wave) or two digits of one block at a time
template <int TB> struct product_count { static constexpr int N = TB == 1 ? 3 : (TB == 2 ? 6 : (TB == 3 ? 9 : 12)); };

// (operand formats 4: 4-bit, and 2: 6-bit with two exponent bits; a scale is a power of two plus 127)
template <int SEL>
__device__ __forceinline__ f32x16_t product(const uint4& a, const unsigned (&b)[6], const f32x16_t& c, int scale, int one = 125)
{
    const i32x8_t av = {(int)a.x, (int)a.y, (int)a.z, (int)a.w, 0, 0, 0, 0};
    const i32x8_t bv = {(int)b[0], (int)b[1], (int)b[2], (int)b[3], (int)b[4], (int)b[5], 0, 0};
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, bv, c, 4, 2, 0, one, SEL, scale);      // (one = 2^-2: the 4.0 of a letter)
}

// Block scales of a filter of exponent `expo`: digit p counts 2^(expo - 3 - 5 p) and is stored in eighths. s[0] and s[1]: the
// digits one by one; s[2]: pairs of digits 2 j, 2 j + 1 of one block, this half wave's. Byte 2 of s[1]: that of weights that close windows.
// (Below 2^-102 the smallest digits would have none: such weights are nothing beside a bias that is 2^100 times theirs.)
__device__ __forceinline__ void digit_scales(int expo, unsigned shut, unsigned h, int (&s)[3])
{
    const int e = expo > -102 ? expo + 127 : 25, eh = e - 5 * (int)h;
    s[0] = (e & 255) | ((e - 5) & 255) << 8 | ((e - 10) & 255) << 16 | (int)((unsigned)((e - 15) & 255) << 24);
    s[1] = ((e - 20) & 255) | ((e - 25) & 255) << 8 | (int)((shut & 255u) << 16);
    s[2] = (eh & 255) | ((eh - 10) & 255) << 8 | ((eh - 20) & 255) << 16;
}

// which 8-tap block and digit the half wave h holds in operand i of a tile (operands in the order they are multiplied:
// small digits first)
template <int TB> __device__ __forceinline__ void operand_slot(int i, unsigned h, unsigned& block, unsigned& digit)
{
    if (TB == 1) { block = 0u; digit = 2u * (2 - i) + h; }                          // digit pairs (4,5) (2,3) (0,1)
    else if (TB == 2) { block = h; digit = 5 - i; }
    else if (TB == 3) {
        const int j = 2 - i / 3, k = i % 3;                                         // block pair digit 2j + 1, digit 2j, third block's pair
        if (k < 2) { block = h; digit = 2 * j + 1 - k; }
        else { block = 2u; digit = 2u * j + h; }
    } else { block = (i & 1 ? 2u : 0u) + h; digit = 5 - i / 2; }
}

// a lane's operands: column `col` of the weights, the half wave's 32 rows of every product
template <int TB>
__device__ __forceinline__ void load_operands(const unsigned char* digits, unsigned col, unsigned h, unsigned (&B)[product_count<TB>::N][6])
{
#pragma unroll
    for (int i = 0; i < product_count<TB>::N; ++i) {
        unsigned block, digit;
        operand_slot<TB>(i, h, block, digit);
        const uint2* src = reinterpret_cast<const uint2*>(digits + ((block * NDIGIT + digit) * FTILE + col) * 24u);
#pragma unroll
        for (int k = 0; k < 3; ++k) { const uint2 v = src[k]; B[i][2 * k] = v.x; B[i][2 * k + 1] = v.y; }
    }
}

// A tile's products with NT sets of filters, which take turns.
template <int TB, int NT, int I>
__device__ __forceinline__ void products(f32x16_t (&z)[NT], const uint4& a0, const uint4& a1, const unsigned (&B)[NT][product_count<TB>::N][6], const int (&s)[NT][3])
{
    if constexpr (I < product_count<TB>::N) {
#pragma unroll
        for (int q = 0; q < NT; ++q) {
            if constexpr (TB == 1) z[q] = product<2 - I>(a0, B[q][I], z[q], s[q][2]);
            else if constexpr (TB == 2) { constexpr int p = 5 - I; z[q] = product<(p & 3)>(a0, B[q][I], z[q], s[q][p >> 2]); }
            else if constexpr (TB == 3) {
                constexpr int j = 2 - I / 3, k = I % 3, p = 2 * j + 1 - k;
                if constexpr (k < 2) z[q] = product<(p & 3)>(a0, B[q][I], z[q], s[q][p >> 2]);
                else z[q] = product<j>(a1, B[q][I], z[q], s[q][2]);
            } else { constexpr int p = 5 - I / 2; z[q] = product<(p & 3)>(I & 1 ? a1 : a0, B[q][I], z[q], s[q][p >> 2]); }
        }
        products<TB, NT, I + 1>(z, a0, a1, B, s);
    }
}

// The weights that close windows, -7.5 2^scale in the place of each, before anything else is added: nothing at all where the window has
// none of them. `shut`: this half wave's and column's, in LDS, [block][filter][24 bytes], the blocks an even number (the last one may be empty).
template <int TB> constexpr unsigned SHUT_BYTES = (TB <= 2 ? 2 : 4) * SLOT_BYTES;
template <int TB, int SEL>
__device__ __forceinline__ f32x16_t closed_windows(const f32x16_t& z, const uint4& a0, const uint4& a1, const unsigned char* shut, int scale)
{
    f32x16_t r = z;
#pragma unroll
    for (int i = 0; i < (TB <= 2 ? 1 : 2); ++i) {
        unsigned B[6];
        const uint2* src = reinterpret_cast<const uint2*>(shut + 2 * i * SLOT_BYTES);
#pragma unroll
        for (int k = 0; k < 3; ++k) { const uint2 v = src[k]; B[2 * k] = v.x; B[2 * k + 1] = v.y; }
        r = product<SEL>(i == 0 ? a0 : a1, B, r, scale);
    }
    return r;
}
// a tile's from the scratch into LDS, by the whole workgroup
template <int TB>
__device__ __forceinline__ void load_shut(const unsigned char* from, unsigned char* shut, unsigned threads)
{
    for (unsigned i = threadIdx.x; i < SHUT_BYTES<TB> / 4; i += threads)
        reinterpret_cast<unsigned*>(shut)[i] = i < TB * SLOT_BYTES / 4 ? reinterpret_cast<const unsigned*>(from)[i] : 0u;
}

// Whether the launch behind this one takes a tile: it takes tiles of 64 filters, that is pairs.
__device__ __forceinline__ bool left_out(const unsigned* __restrict__ flags, unsigned tile)
{
    return ((flags[tile & ~1u] | flags[tile | 1u]) & (TILE_LEFT | TILE_NOT_FINITE)) != 0u;
}

// a row's rectified sum and bias, both below one half in magnitude where it is not zero: one addition that clamps
__device__ __forceinline__ float open_part(float z, float b) { return __builtin_amdgcn_fmed3f(z + b, 0.0f, 1.0f); }

// Lanes 0-31 of x beside lanes 0-31 of y, and lanes 32-63 of x beside lanes 32-63 of y: (x, y) becomes what the low and the
// high half wave held of the first value (in lanes 0-31) and of the second (in lanes 32-63).
__device__ __forceinline__ void swap_halves(unsigned& x, unsigned& y)
{
    const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
    x = r[0];
    y = r[1];
}
__device__ __forceinline__ void swap_halves(float& x, float& y)
{
    unsigned a = __float_as_uint(x), b = __float_as_uint(y);
    swap_halves(a, b);
    x = __uint_as_float(a);
    y = __uint_as_float(b);
}

// ---------------------------------------------------------------------------------------------- the scan
// CLOSES: some of the tile's filters have weights that close windows. (Two bodies, so that the products of those take no registers in the other.)
// NT: sets of 32 filters that a wave takes (a workgroup of 16 waves: one, of 12: two, see takes_two).
template <int NT> constexpr int WAVES = NT == 2 ? 12 : NWAVE;
template <int PT, bool WANT_ARGMAX, int TB, int NT, bool CLOSES>
__device__ __forceinline__ void scanpool_digits_body(const digit_store& D, unsigned tile, unsigned split, const float* __restrict__ bias, unsigned f0, unsigned F,
                                                     const uint8_t* __restrict__ X, size_t N, size_t ndef, const uint32_t* __restrict__ R, unsigned P,
                                                     unsigned nsplit, float* __restrict__ pooled, uint32_t* __restrict__ argmax)
{
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int NI = product_count<TB>::N;
    const unsigned lane = threadIdx.x & 63u, wave = (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const unsigned col = lane & 31u, h = lane >> 5;
    unsigned* counter = reinterpret_cast<unsigned*>(smem);
    uint4* entries = reinterpret_cast<uint4*>(smem + 16) + (size_t)wave * ENTRIES;
    unsigned char* shut = smem + 16 + (size_t)WAVES<NT> * ENTRIES * 16;
    if (CLOSES) {
#pragma unroll
        for (int q = 0; q < NT; ++q) load_shut<TB>(D.shut + (size_t)(tile + q) * (TB * SLOT_BYTES), shut + q * SHUT_BYTES<TB>, WAVES<NT> * 64);
    }
    // this workgroup's regions
    const unsigned lo = (unsigned)((unsigned long long)P * split / nsplit), hi = (unsigned)((unsigned long long)P * (split + 1) / nsplit);
    if (threadIdx.x == 0) counter[0] = lo;
    const unsigned f = f0 + tile * FTILE + (NT == 2 ? lane : col);    // the filter whose results this lane writes (one set: lanes 0-31)
    // The sums come in units of 2^down, in which open windows and the bias stay below one half (`whole`), so that adding the bias and
    // rectifying is one instruction, which clamps to 0 .. 1. (16 of 61 vector instructions beside a tile's six products of 16 taps. The
    // whole call, us: max + average, 20 000 x 30-150 letters x 384 filters x 16 taps 231 -> 219; average, 30 000 x 101 x 256, 12 taps 208 -> 196, 24 taps 274 -> 262.)
    unsigned B[NT][NI][6];
    int s[NT][3];
    float bu[NT];
#pragma unroll
    for (int q = 0; q < NT; ++q) {
        const unsigned t = tile + q, g = f0 + t * FTILE + col;
        load_operands<TB>(D.digits + (size_t)t * (TB * NDIGIT * SLOT_BYTES), col, h, B[q]);
        const digit_facts& facts = D.facts[t * FTILE + col];
        const int down = 31 - facts.whole;
        bu[q] = g < F ? bias[g] * power_of_two(-down) : 0.0f;
        digit_scales(D.expo[t * FTILE + col] - down, facts.shut - (unsigned)down, h, s[q]);
    }
    const float bf = f < F ? bias[f] : 0.0f, unit = power_of_two(31 - D.facts[tile * FTILE + (NT == 2 ? lane : col)].whole);
    shut += (h * FTILE + col) * 24u;
    const unsigned rg = 4u * h;                                   // this half wave's rows lie 4 further down
    const unsigned at0 = first_operand<TB>(col, h), at1 = second_operand<TB>(col, h);
    __syncthreads();

    unsigned r = claim(counter, lane), rn = claim(counter, lane);                           // the region in work, the one after it
    unsigned a = 0u, b = 0u, an = 0u, bn = 0u;
    if (r < hi) { a = R[2 * (size_t)r]; b = R[2 * (size_t)r + 1]; }
    if (rn < hi) { an = R[2 * (size_t)rn]; bn = R[2 * (size_t)rn + 1]; }
    unsigned letters[3] = {0u, 0u, 0u};
    if (r < hi) load12(X, N, a, lane, letters);

    while (r < hi) {
        float mx[2] = {CLOSED, CLOSED}, sum[2] = {0.0f, 0.0f};
        unsigned xi[2] = {0u, 0u};
        unsigned c = a;
        bool last;
        do {
            const unsigned left = b > c ? b - c : 0u;             // rows of the region from this chunk on
            last = left <= CHUNK;
            stage(entries, lane, letters);
            // the next chunk's letters travel while this one is multiplied
            if (!last) load12(X, N, c + CHUNK, lane, letters);
            else if (rn < hi) load12(X, N, an, lane, letters);
            // ---- its tiles
            const unsigned nrow = last ? left : CHUNK;
            const unsigned defined = defined_rows(ndef, c);
            const uint4* src = entries;
            for (unsigned t0 = 0; t0 < nrow; t0 += ROWS, src += 34) {
                uint4 a0 = src[at0], a1 = TB >= 3 ? src[at1] : a0;
                if (t0 + ROWS > defined) close_undefined(a0, a1, t0 + col < defined);
                f32x16_t sums[NT];
#pragma unroll
                for (int q = 0; q < NT; ++q) {
#pragma unroll
                    for (int i = 0; i < 16; ++i) sums[q][i] = 0.0f;
                    if (CLOSES) sums[q] = closed_windows<TB, 2>(sums[q], a0, a1, shut + q * SHUT_BYTES<TB>, s[q][1]);
                }
                products<TB, NT, 0>(sums, a0, a1, B, s);
                if (left - t0 < (unsigned)ROWS) {
                    unsigned inside = left - t0;                  // (opaque: the comparisons stay in this branch)
                    asm volatile("" : "+v"(inside));
#pragma unroll
                    for (int i = 0; i < 16; ++i) {
                        const bool in = rg + ((i & 3) + 8 * (i >> 2)) < inside;
#pragma unroll
                        for (int q = 0; q < NT; ++q) sums[q][i] = in ? sums[q][i] : CLOSED;
                    }
                }
#pragma unroll
                for (int q = 0; q < NT; ++q) {
                    const f32x16_t& z = sums[q];
                    if (PT != DBK_PT_AVG) {
                        if (WANT_ARGMAX) {
                            float bm = z[0];
                            unsigned bi = 0u;
#pragma unroll
                            for (int i = 1; i < 16; ++i) {
                                const bool gt = z[i] > bm;
                                bm = gt ? z[i] : bm;
                                bi = gt ? (unsigned)i : bi;
                            }
                            if (bm > mx[q]) { mx[q] = bm; xi[q] = (c - a) + t0 + rg + (bi & 3u) + 8u * (bi >> 2); }
                        } else {
#pragma unroll
                            for (int i = 0; i < 16; i += 2) mx[q] = fmaxf(fmaxf(mx[q], z[i]), z[i + 1]);
                        }
                    }
                    if (PT != DBK_PT_MAX) {
                        float part = open_part(z[0], bu[q]);
#pragma unroll
                        for (int i = 1; i < 16; ++i) part += open_part(z[i], bu[q]);
                        sum[q] += part;                           // (a tile's sum first: sums of sums round less)
                    }
                }
            }
            c += CHUNK;
        } while (!last);
        // ---- the region's result: fold the two half waves (equal values keep the earlier row); two sets: the second's in lanes 32-63
        if (PT != DBK_PT_AVG) {
            if (NT == 2) swap_halves(mx[0], mx[1]); else mx[1] = __shfl_xor(mx[0], 32, 64);
            if (WANT_ARGMAX) {
                if (NT == 2) swap_halves(xi[0], xi[1]); else xi[1] = (unsigned)__shfl_xor((int)xi[0], 32, 64);
                if (mx[1] > mx[0] || (mx[1] == mx[0] && xi[1] < xi[0])) xi[0] = xi[1];
            }
            mx[0] = fmaxf(mx[0], mx[1]) * unit + bf;
            if (WANT_ARGMAX && !(mx[0] > 0.0f)) xi[0] = 0u;       // nothing open: the region's first row
            mx[0] = fmaxf(mx[0], 0.0f);
        }
        if (PT != DBK_PT_MAX) {
            if (NT == 2) swap_halves(sum[0], sum[1]); else sum[1] = __shfl_xor(sum[0], 32, 64);
            sum[0] = (sum[0] + sum[1]) / (float)(b - a) * unit;
        }
        if ((NT == 2 || h == 0u) && f < F) {
            const size_t j = (size_t)r * F + f;
            if (PT == DBK_PT_MAX) pooled[j] = mx[0];
            else if (PT == DBK_PT_AVG) pooled[j] = sum[0];
            else { pooled[2 * j] = mx[0]; pooled[2 * j + 1] = sum[0]; }
            if (WANT_ARGMAX) argmax[j] = (uint32_t)(((size_t)a + xi[0]) * F + f);
        }
        r = rn; a = an; b = bn;
        rn = claim(counter, lane);
        if (rn < hi) { an = R[2 * (size_t)rn]; bn = R[2 * (size_t)rn + 1]; }
    }
}

template <int PT, bool WANT_ARGMAX, int TB, int NT>
__global__ __launch_bounds__(WAVES<NT> * 64) __attribute__((amdgpu_waves_per_eu(WAVES<NT> / 4, WAVES<NT> / 4)))
void scanpool_digits_kernel(digit_store D, const float* __restrict__ bias, unsigned f0, unsigned F, const uint8_t* __restrict__ X, size_t N, size_t ndef,
                            const uint32_t* __restrict__ R, unsigned P, unsigned nsplit, float* __restrict__ pooled, uint32_t* __restrict__ argmax)
{
    const unsigned tile = NT * (blockIdx.x / nsplit), split = blockIdx.x % nsplit;
    if (left_out(D.flags, tile)) return;
    if (((D.flags[tile] | D.flags[tile + NT - 1]) & TILE_CLOSES) != 0u)
        scanpool_digits_body<PT, WANT_ARGMAX, TB, NT, true>(D, tile, split, bias, f0, F, X, N, ndef, R, P, nsplit, pooled, argmax);
    else
        scanpool_digits_body<PT, WANT_ARGMAX, TB, NT, false>(D, tile, split, bias, f0, F, X, N, ndef, R, P, nsplit, pooled, argmax);
}

// ---------------------------------------------------------------------------------------------- plain maxima
// Max pooling with filters of 17 to 32 taps: half the products. A region's maximum is one window, so the products only have
// to find its place; its value is then added up from the weights themselves, as whole numbers below 2^-29 of the most that an open
// window comes to, with one rounding in the end (weights that only close windows may wrap: no winning window holds them). The first NTOP digits of every weight give every
// window's sum to within what the digits left out can amount to. The value of the largest sum's window being known, it is
// the maximum unless the second largest sum plus the most that the left out digits can add to any window (`above`, per
// filter) reaches it. Where that is so (of normal weights over 500 random letters 0.1 % of the filters and regions), the region is
// scanned once more with all the digits, for the 32 filters concerned, to find the place. In sequences that repeat the windows
// tie in every filter: after two regions in a row that were unsure in both halves of its 64 filters a wave takes the next 15 to all the
// digits at once. A place that is sure is the one that those find (`above` has their rounding in it), so that a result does not depend
// on which regions a wave met before. Measured, 20 000 x 500 letters x 512 filters, ms, 24 / 32 taps: uniform letters 0.85 / 0.98, units of 7
// letters that repeat 1.30 / 2.4 (25 to 32 taps scan every region twice, as 24 did in 1.95; the table of 3-mer sums 1.35 / 2.7 whatever
// the letters).
//
// Sums of NTOP digits are whole numbers of 1/4 unit (a "mean of the four" counts quarters) below 2^18 units, which leaves
// float32 four bits below: a lane's 16 rows start from 15/64 .. 0 units instead of zero, so the maximum carries its row's
// number with it, and a tile only notes that it was the best so far. The second largest comes with the largest: v_max3 and
// v_med3 give the top two of three, 20 instructions for a tile's 16 rows and the two so far.
//
// A wave takes 64 filters at a time (the staging of the letters, the operand reads and the walk serve both halves), 12
// waves per workgroup: three per SIMD at up to 168 registers. At a region's end lanes 0-31 hold the
// first 32 filters and lanes 32-63 the others, and each adds up its own filter's window.
constexpr int MAX_WAVES = 12;
constexpr unsigned AT_ONCE = 15;              // regions that go to all the digits at once before the places are tried again
constexpr int PAIR = 2 * FTILE;               // filters per workgroup

template <int TB> struct place_count { static constexpr int N = TB == 3 ? 5 : 6; };

// which block and digit operand i of a tile holds; digit NTOP stands for an empty half
template <int TB> __device__ __forceinline__ void place_slot(int i, unsigned h, unsigned& block, unsigned& digit)
{
    if (TB == 3) {
        if (i < 3) { block = h; digit = 2 - i; }
        else { block = 2u; digit = i == 3 ? 1u + h : (h ? (unsigned)NTOP : 0u); }
    } else { block = (i & 1 ? 2u : 0u) + h; digit = 2 - i / 2; }
}

// In units of digit NTOP - 1: the digits' scales are the same for every filter. single: digits 0, 1, 2 by byte; pair: bytes
// for this half wave's digits (0, none) and (1, 2). The two halves' products take turns, so that none waits for the sum of the one
// before it, and each first one starts from the same registers: one half after the other, the second's start was copied for every tile.
// With that, and the comparisons of a region's last tile in a branch of their own instead of beside every tile's products, a tile takes 63
// vector instructions instead of 92: 100 000 x 500 letters x 1024 filters of 24 taps 8.26 -> 7.66 ms, 50 000 x 100-200 x 256 of 32 taps 0.52 -> 0.50.
template <int TB, int I>
__device__ __forceinline__ void place_sums(f32x16_t& z0, f32x16_t& z1, const uint4& a0, const uint4& a1, const unsigned (&B)[2][place_count<TB>::N][6], int single, int pair)
{
    if constexpr (I < place_count<TB>::N) {
        constexpr bool third = TB == 3 ? I >= 3 : (I & 1) != 0;   // operand of the third and fourth block
        constexpr int digit = TB == 3 ? (I < 3 ? 2 - I : 4 - I) : 2 - I / 2;
        const uint4& a = third ? a1 : a0;
        const int scale = TB == 3 && third ? pair : single;
        z0 = product<digit>(a, B[0][I], z0, scale);
        z1 = product<digit>(a, B[1][I], z1, scale);
        place_sums<TB, I + 1>(z0, z1, a0, a1, B, single, pair);
    }
}

// The maximum over a region from all the digits, and its row: this half wave's, without the bias, of the filters wanted (a bit each).
template <int TB, bool CLOSES>
__device__ __forceinline__ float2 region_maximum(const uint8_t* __restrict__ X, size_t N, size_t ndef, unsigned a, unsigned b, uint4* entries,
                                              const unsigned char* digits, const unsigned char* shut, unsigned lane, int expo, unsigned scale, unsigned wanted)
{
    asm volatile("" : "+v"(lane));                                // (opaque: nothing of this is held in registers across the regions)
    const unsigned col = lane & 31u, h = lane >> 5, at0 = first_operand<TB>(col, h), at1 = second_operand<TB>(col, h);
    int s[1][3];
    digit_scales(expo, scale, h, s[0]);
    shut += (h * FTILE + col) * 24u;
    unsigned B[1][product_count<TB>::N][6];
    load_operands<TB>(digits, col, h, B[0]);
    float mx = CLOSED;
    unsigned xi = 0u;
    for (unsigned c = a;; c += CHUNK) {
        const unsigned left = b > c ? b - c : 0u;
        unsigned letters[3];
        load12(X, N, c, lane, letters);
        stage(entries, lane, letters);
        const unsigned nrow = left < CHUNK ? left : CHUNK, defined = defined_rows(ndef, c);
        const uint4* src = entries;
        for (unsigned t0 = 0; t0 < nrow; t0 += ROWS, src += 34) {
            uint4 a0 = src[at0], a1 = TB >= 3 ? src[at1] : a0;
            if (t0 + ROWS > defined) close_undefined(a0, a1, t0 + col < defined);
            f32x16_t sums[1];
            f32x16_t& z = sums[0];
#pragma unroll
            for (int i = 0; i < 16; ++i) z[i] = 0.0f;
            if (CLOSES) z = closed_windows<TB, 2>(z, a0, a1, shut, s[0][1]);
            products<TB, 1, 0>(sums, a0, a1, B, s);
            if (left - t0 < (unsigned)ROWS) {
#pragma unroll
                for (int i = 0; i < 16; ++i) z[i] = 4u * h + ((i & 3) + 8 * (i >> 2)) < left - t0 ? z[i] : CLOSED;
            }
            float best = z[0];
#pragma unroll
            for (int i = 1; i < 15; i += 2) best = fmaxf(fmaxf(best, z[i]), z[i + 1]);
            best = fmaxf(best, z[15]);
            const bool further = best > mx && ((wanted >> col) & 1u) != 0u;
            if (__any(further)) {                                 // (where rows repeat, the first tiles alone)
                unsigned at = 15u;
#pragma unroll
                for (int i = 14; i >= 0; --i) at = z[i] == best ? (unsigned)i : at;
                if (further) { mx = best; xi = (c - a) + t0 + 4u * h + (at & 3u) + 8u * (at >> 2); }
            }
        }
        if (left <= CHUNK) break;
    }
    return make_float2(mx, __uint_as_float(xi));
}

// the two largest of a tile's 16 rows and of those so far; the tile of the largest
__device__ __forceinline__ void top_two(const f32x16_t& z, float& m1, float& m2, unsigned& t1, unsigned t)
{
    auto max3 = [](float x, float y, float w) { return fmaxf(fmaxf(x, y), w); };
    auto med3 = [](float x, float y, float w) { return __builtin_amdgcn_fmed3f(x, y, w); };
    float g[5], k[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        g[i] = max3(z[3 * i], z[3 * i + 1], z[3 * i + 2]);
        k[i] = med3(z[3 * i], z[3 * i + 1], z[3 * i + 2]);
    }
    const float u0 = max3(g[0], g[1], g[2]), v0 = med3(g[0], g[1], g[2]);
    const float u1 = max3(g[3], g[4], z[15]), v1 = med3(g[3], g[4], z[15]);
    const float top = max3(u0, u1, m1), v2 = med3(u0, u1, m1);
    m2 = max3(max3(max3(max3(m2, k[0], k[1]), k[2], k[3]), k[4], v0), v1, v2);
    t1 = top > m1 ? t : t1;
    m1 = top;
}

template <bool WANT_ARGMAX, int TB, bool CLOSES>
__device__ __forceinline__ void scanpool_digits_max_body(const digit_store& D, unsigned tile, unsigned split, bool two, const float* __restrict__ W,
                                                         const float* __restrict__ bias, unsigned f0, unsigned m, unsigned F, const uint8_t* __restrict__ X,
                                                         size_t N, size_t ndef, const uint32_t* __restrict__ R, unsigned P, unsigned nsplit,
                                                         float* __restrict__ pooled, uint32_t* __restrict__ argmax)
{
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr int NI = place_count<TB>::N;
    // (beside a fourth block of taps or the products of closing weights registers would spill: a repeating region costs both ways there)
    constexpr bool DIRECT = TB == 3 && !CLOSES;
    constexpr unsigned TAPS = 8u * TB, TILE_DIGITS = TB * NDIGIT * SLOT_BYTES;
    const unsigned lane = threadIdx.x & 63u, wave = (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const unsigned col = lane & 31u, h = lane >> 5;
    unsigned* counter = reinterpret_cast<unsigned*>(smem);
    uint4* entries = reinterpret_cast<uint4*>(smem + 16) + (size_t)wave * ENTRIES;
    int* table = reinterpret_cast<int*>(smem + 16 + MAX_WAVES * ENTRIES * 16);      // [8 TB taps][8 codes][64 filters]: the weights as whole numbers
    // all the digits, or (LDS does not hold both) the weights that close windows
    unsigned char* digits = reinterpret_cast<unsigned char*>(table + TAPS * 8 * PAIR);
    unsigned char* shut = digits;
    float4* about = reinterpret_cast<float4*>(digits + 2 * TILE_DIGITS);            // [64 filters]: bias, unit, above, exponents
    const unsigned lo = (unsigned)((unsigned long long)P * split / nsplit), hi = (unsigned)((unsigned long long)P * (split + 1) / nsplit);
    if (threadIdx.x == 0) counter[0] = lo;
    const unsigned fbase = f0 + tile * FTILE;
    if (CLOSES) {
        load_shut<TB>(D.shut + (size_t)tile * (TB * SLOT_BYTES), shut, MAX_WAVES * 64);
        if (two) load_shut<TB>(D.shut + (size_t)(tile + 1) * (TB * SLOT_BYTES), shut + SHUT_BYTES<TB>, MAX_WAVES * 64);
    } else {
        for (unsigned i = threadIdx.x; i < (two ? 2u : 1u) * TILE_DIGITS / 16; i += MAX_WAVES * 64)
            reinterpret_cast<uint4*>(digits)[i] = reinterpret_cast<const uint4*>(D.digits + (size_t)tile * TILE_DIGITS)[i];
    }
    for (unsigned i = threadIdx.x; i < TAPS * PAIR; i += MAX_WAVES * 64) {
        const unsigned tap = i / PAIR, fl = i % PAIR, f = fbase + fl;
        const bool in = tap < m && f < F && (two || fl < FTILE);
        const digit_facts k = D.facts[tile * FTILE + (in ? fl : 0u)];
        const float scale = __uint_as_float((unsigned)(127 + k.whole) << 23);
        float w[4];                                               // (what 32 bits do not hold is in no open window)
#pragma unroll
        for (int c = 0; c < 4; ++c) w[c] = in ? rintf(fmaxf(W[(size_t)(4 * tap + c) * F + f], k.lowest) * scale) : 0.0f;
        const double sum = ((double)w[0] + (double)w[1]) + ((double)w[2] + (double)w[3]);
        const int mean = (int)rint(fmax(0.25 * sum, -2147483647.0));
        int* row = table + (size_t)tap * 8 * PAIR + fl;
#pragma unroll
        for (int c = 0; c < 8; ++c) row[c * PAIR] = c < 4 ? (int)fmaxf(w[c & 3], -2147483520.0f) : (c == 6 ? 0 : mean);      // codes mod 8: 254 is 6
    }
    if (threadIdx.x < PAIR) {
        const unsigned f = fbase + threadIdx.x;
        const bool in = f < F && (two || threadIdx.x < FTILE);
        const digit_facts k = D.facts[tile * FTILE + (in ? threadIdx.x : 0u)];
        // (filters past the last: closed whatever their sums)
        about[threadIdx.x] = make_float4(in ? bias[f] : CLOSED, k.unit, k.above,
                                         __uint_as_float((unsigned)(k.whole + 128) << 24 | (unsigned)(D.expo[tile * FTILE + (in ? threadIdx.x : 0u)] + 128) << 16 | k.shut));
    }
    __syncthreads();
    unsigned B[2][NI][6];
    auto load_places = [&](unsigned ln) {
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                unsigned block, digit;
                place_slot<TB>(i, ln >> 5, block, digit);
                const bool none = digit == (unsigned)NTOP || (q == 1 && !two);
                const uint2* src = reinterpret_cast<const uint2*>(D.top + (none ? (size_t)0 : (size_t)(tile + q) * (TB * NTOP * SLOT_BYTES) +
                                                                            ((block * NTOP + digit) * FTILE + (ln & 31u)) * 24u));
#pragma unroll
                for (int k = 0; k < 3; ++k) { const uint2 v = src[k]; B[q][i][2 * k] = none ? 0u : v.x; B[q][i][2 * k + 1] = none ? 0u : v.y; }
            }
    };
    load_places(lane);
    // a unit is digit 2's step: digit p counts 2^(5 (2 - p)), stored in eighths
    const int single = 140 | 135 << 8 | 130 << 16, pair = 140 | (135 - 5 * (int)h) << 8;
    // (of weights that close windows: those of the first 32 filters, of the others)
    const int shut_scales = (int)(((__float_as_uint(about[col].w) >> 8) & 255u) | (__float_as_uint(about[FTILE + col].w) & 0xff00u));
    const unsigned char* shut_here = shut + (h * FTILE + col) * 24u;
    f32x16_t rows;                                                // what the rows start from, in 1/64 of a unit
#pragma unroll
    for (int i = 0; i < 16; ++i) rows[i] = (float)(15 - i) * (1.0f / 64.0f);
    // (opaque: as constants they would be copied from scalar registers for every tile)
    if constexpr (TB == 3 && !CLOSES) asm volatile("" : "+v"(rows));
    const unsigned at0 = first_operand<TB>(col, h), at1 = second_operand<TB>(col, h);

    unsigned r = claim(counter, lane), rn = claim(counter, lane); // the region in work, the one after it
    unsigned a = 0u, b = 0u, an = 0u, bn = 0u;
    if (r < hi) { a = R[2 * (size_t)r]; b = R[2 * (size_t)r + 1]; }
    if (rn < hi) { an = R[2 * (size_t)rn]; bn = R[2 * (size_t)rn + 1]; }
    a = (unsigned)__builtin_amdgcn_readfirstlane((int)a); b = (unsigned)__builtin_amdgcn_readfirstlane((int)b);
    unsigned letters[3] = {0u, 0u, 0u};
    if (r < hi) load12(X, N, a, lane, letters);

    // the value of a window (relative to the region), from the weights
    auto value_at = [&](unsigned mine, bool open, unsigned row, float exponents) -> float {
        const size_t at = (size_t)a + row;
        if (!open || at >= ndef) return 0.0f;
        unsigned v[2 * TB];
        if (at + TAPS <= N) __builtin_memcpy(v, X + at, TAPS);
        else load_tail<TAPS>(X, N, at, v);
        unsigned sum = 0u;                                        // (the sum fits, whatever its parts run through)
#pragma unroll
        for (int k = 0; k < 2 * TB; ++k) {
            if (odd_codes(v[k]) != 0u) v[k] = plain_codes(v[k]);
#pragma unroll
            for (int j = 0; j < 4; ++j) sum += (unsigned)(table + ((v[k] >> (8 * j)) & 7u) * PAIR + mine)[(4 * k + j) * 8 * PAIR];
        }
        return (float)(int)sum * __uint_as_float((unsigned)(127 + 128 - (int)(__float_as_uint(exponents) >> 24)) << 23);
    };
    // the place from all the digits, for the halves of `who`
    auto place_again = [&](unsigned mine, unsigned long long who, bool unsure, unsigned row) -> unsigned {
#pragma unroll 1
        for (unsigned q = 0; q < 2; ++q) {
            if ((unsigned)(who >> (32u * q)) == 0u) continue;
            const unsigned expo = __float_as_uint(about[32u * q + (mine & 31u)].w);
            const float2 all = region_maximum<TB, CLOSES>(X, N, ndef, a, b, entries, CLOSES ? D.digits + (size_t)(tile + q) * TILE_DIGITS : digits + q * TILE_DIGITS,
                                                          shut + q * SHUT_BYTES<TB>, mine, (int)((expo >> 16) & 255u) - 128, expo & 255u,
                                                          (unsigned)(who >> (32u * q)));
            const float oz = __shfl_xor(all.x, 32, 64);
            const unsigned xi = __float_as_uint(all.y), oi = (unsigned)__shfl_xor((int)xi, 32, 64);
            if (unsure && (mine >> 5) == q) row = oz > all.x || (oz == all.x && oi < xi) ? oi : xi;
        }
        return row;
    };
    auto keep = [&](unsigned mine, float value, unsigned row) {
        const unsigned f = fbase + mine;
        if (f < F && (two || mine < FTILE)) {
            const size_t j = (size_t)r * F + f;
            pooled[j] = value;
            if (WANT_ARGMAX) argmax[j] = (uint32_t)(((size_t)a + (value > 0.0f ? row : 0u)) * F + f);   // nothing open: the first row
        }
    };
    auto next_region = [&]() {
        r = rn;
        a = (unsigned)__builtin_amdgcn_readfirstlane((int)an); b = (unsigned)__builtin_amdgcn_readfirstlane((int)bn);
        rn = claim(counter, lane);
        if (rn < hi) { an = R[2 * (size_t)rn]; bn = R[2 * (size_t)rn + 1]; }
    };
    while (r < hi) {
        unsigned ties = 0u;                                           // regions in a row that were unsure in both halves
        while (r < hi && ties < 2u) {
            float m1[2] = {CLOSED, CLOSED}, m2[2] = {CLOSED, CLOSED}; // the two largest sums so far
            unsigned t1[2] = {0u, 0u}, t = 0u;                        // the tile of the largest, the tile in work
            unsigned c = a;
            bool last;
            do {
                const unsigned left = b > c ? b - c : 0u;             // rows of the region from this stretch on
                last = left <= CHUNK;
                stage(entries, lane, letters);
                // the next stretch's letters travel while this one is multiplied
                if (!last) load12(X, N, c + CHUNK, lane, letters);
                else if (rn < hi) load12(X, N, (unsigned)__builtin_amdgcn_readfirstlane((int)an), lane, letters);
                const unsigned nrow = last ? left : CHUNK;
                const unsigned defined = defined_rows(ndef, c);
                const uint4* src = entries;
                for (unsigned t0 = 0; t0 < nrow; t0 += ROWS, src += 34, ++t) {
                    uint4 a0 = src[at0], a1 = TB >= 3 ? src[at1] : a0;
                    if (t0 + ROWS > defined) close_undefined(a0, a1, t0 + col < defined);
                    const unsigned rest = left - t0;              // (rows of the region from this tile on)
                    f32x16_t z0, z1;                              // the first 32 filters' sums, the others'
                    if constexpr (CLOSES) {
                        float zero = 0.0f;                        // (opaque: the rows' numbers are formed anew, for their registers)
                        asm volatile("" : "+v"(zero));
#pragma unroll
                        for (int i = 0; i < 16; ++i) z0[i] = zero + (float)(15 - i) * (1.0f / 64.0f);
                        z1 = closed_windows<TB, 1>(z0, a0, a1, shut_here + SHUT_BYTES<TB>, shut_scales);
                        z0 = closed_windows<TB, 0>(z0, a0, a1, shut_here, shut_scales);
                    } else {
                        z0 = rows;
                        z1 = rows;
                    }
                    place_sums<TB, 0>(z0, z1, a0, a1, B, single, pair);
                    if (rest < (unsigned)ROWS) {
                        int inside = (int)rest - 4 * (int)h;      // (opaque: the comparisons stay in this branch)
                        asm volatile("" : "+v"(inside));
#pragma unroll
                        for (int i = 0; i < 16; ++i) {
                            const bool in = (i & 3) + 8 * (i >> 2) < inside;
                            z0[i] = in ? z0[i] : CLOSED;
                            z1[i] = in ? z1[i] : CLOSED;
                        }
                    }
                    top_two(z0, m1[0], m2[0], t1[0], t);
                    top_two(z1, m1[1], m2[1], t1[1], t);
                }
                c += CHUNK;
            } while (!last);
            // ---- each filter's two half waves side by side: the largest sum, its place, the second largest
            unsigned mine = lane;                                     // (opaque: addresses are formed from it here, not held in registers)
            asm volatile("" : "+v"(mine));
            swap_halves(m1[0], m1[1]);
            swap_halves(m2[0], m2[1]);
            swap_halves(t1[0], t1[1]);
            const bool upper = m1[1] > m1[0];
            const float best = fmaxf(m1[0], m1[1]), second = fmaxf(fminf(m1[0], m1[1]), fmaxf(m2[0], m2[1]));
            const unsigned i = 15u - ((unsigned)(int)(best * 64.0f) & 15u);
            unsigned row = (upper ? t1[1] : t1[0]) * ROWS + (upper ? 4u : 0u) + (i & 3u) + 8u * (i >> 2);
            const float4 filter = about[mine];
            // else every window's rectified value is zero (a region without rows has no best)
            const bool open = best > CLOSED && (best + filter.z) * filter.y + filter.x > 0.0f;
            // ---- its value from the weights
            float value = value_at(mine, open, row, filter.w);
            const bool unsure = open && filter.y > 0.0f && !((second + filter.z) * filter.y < value);     // (windows all alike: the first row)
            const unsigned long long who = __ballot(unsure);
            if (DIRECT) ties = (unsigned)who != 0u && (unsigned)(who >> 32) != 0u ? ties + 1u : 0u;
            if (who != 0ull) {
                // ---- too close to call: its place from all the digits, for the 32 filters concerned
                const unsigned found = place_again(mine, who, unsure, row);
                if (__any(found != row)) value = value_at(mine, open, found, about[mine].w);
                row = found;
                load_places(mine);                                    // (not held over the pass: its operands take their registers)
            }
            keep(mine, open ? fmaxf(value + filter.x, 0.0f) : 0.0f, row);
            next_region();
        }
        // ---- two regions in a row were unsure in both halves (sequences that repeat: their windows tie): the next ones go to all the
        // digits at once, before the places are tried again
        if (!DIRECT) break;
#pragma unroll 1
        for (unsigned k = 0; k < AT_ONCE && r < hi; ++k) {
            unsigned mine = lane;
            asm volatile("" : "+v"(mine));
            const bool open = b > a;
            const unsigned row = place_again(mine, open ? ~0ull : 0ull, open, 0u);
            const float4 filter = about[mine];
            keep(mine, open ? fmaxf(value_at(mine, open, row, filter.w) + filter.x, 0.0f) : 0.0f, row);
            next_region();
        }
        unsigned again = lane;
        asm volatile("" : "+v"(again));
        load_places(again);                                       // (not held meanwhile, on any path)
        if (r < hi) load12(X, N, a, again, letters);
    }
}

template <bool WANT_ARGMAX, int TB>
__global__ __launch_bounds__(MAX_WAVES * 64) __attribute__((amdgpu_waves_per_eu(MAX_WAVES / 4, MAX_WAVES / 4)))
void scanpool_digits_max_kernel(digit_store D, unsigned ntile, const float* __restrict__ W, const float* __restrict__ bias, unsigned f0, unsigned m, unsigned F,
                                const uint8_t* __restrict__ X, size_t N, size_t ndef, const uint32_t* __restrict__ R, unsigned P, unsigned nsplit,
                                float* __restrict__ pooled, uint32_t* __restrict__ argmax)
{
    const unsigned tile = 2u * (blockIdx.x / nsplit), split = blockIdx.x % nsplit;
    const bool two = tile + 1u < ntile;                           // (an odd last tile is scanned beside nothing)
    if (left_out(D.flags, tile)) return;
    if (((D.flags[tile] | (two ? D.flags[tile + 1] : 0u)) & TILE_CLOSES) != 0u)
        scanpool_digits_max_body<WANT_ARGMAX, TB, true>(D, tile, split, two, W, bias, f0, m, F, X, N, ndef, R, P, nsplit, pooled, argmax);
    else
        scanpool_digits_max_body<WANT_ARGMAX, TB, false>(D, tile, split, two, W, bias, f0, m, F, X, N, ndef, R, P, nsplit, pooled, argmax);
}

// workgroups per group of filters: one workgroup per CU in all, each with a region at least. (Fewer regions than waves lie side by side on all the
// CUs, with waves that have none, not in full workgroups on some: one set of filters, 600 regions of 500 rows x 64 filters of 8 taps 19.3 -> 16.5 us, max + average.)
inline unsigned splits(unsigned groups, size_t P)
{
    unsigned n = 256u / groups;
    if (n < 1) n = 1;
    return n < P ? n : (unsigned)P;
}

constexpr size_t max_smem(int tb)
{
    return 16 + (size_t)MAX_WAVES * ENTRIES * 16 + (size_t)tb * (8 * 8 * PAIR * sizeof(int) + 2 * NDIGIT * SLOT_BYTES) + PAIR * 16;
}
static_assert(max_smem(4) <= 160 * 1024 && SHUT_BYTES<4> <= 3 * NDIGIT * SLOT_BYTES, "LDS of a CU");

template <bool WANT_ARGMAX, int TB>
int launch_max(hipStream_t st, const digit_store& D, const float* W, const float* bias, unsigned f0, unsigned ntile, size_t m, size_t F, const uint8_t* X,
               size_t N, size_t ndef, const uint32_t* R, size_t P, float* pooled, uint32_t* argmax)
{
    auto kern = scanpool_digits_max_kernel<WANT_ARGMAX, TB>;
    DBK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)max_smem(TB)));
    const unsigned groups = (ntile + 1) / 2, nsplit = splits(groups, P);
    hipLaunchKernelGGL(kern, dim3(groups * nsplit), dim3(MAX_WAVES * 64), max_smem(TB), st, D, ntile, W, bias, f0, (unsigned)m, (unsigned)F, X, N, ndef, R,
                       (unsigned)P, nsplit, pooled, argmax);
    return 0;
}

template <int TB, int NT> constexpr size_t scan_smem() { return 16 + (size_t)WAVES<NT> * ENTRIES * 16 + NT * SHUT_BYTES<TB>; }

// Whether a wave takes two sets of 32 filters at a time: one staging of the letters, one read of a tile's operands and one walk serve both,
// and their products take turns instead of waiting for each other's sums. Up to 16 taps, whose digits leave the registers for it (24 taps, us, one /
// two: average, 30 000 x 101 x 256 251 / 254, max + average 271 / 303). An odd last set is scanned beside nothing, which many others pay for. Of the
// 3072 waves of two sets (4096 of one) the last round is to have most at work, or to be one of many: a wave has twice the products and no more
// than two others beside it. us, one / two, max + average, 500 rows x 128 filters: 16 taps, 600 regions (0.4 rounds of the waves of two sets) 22.3 / 25.4, 1200 (0.8) 27.8 / 28.4
// (maxima with their places, 12 taps, 27.8 / 29.8), 2000 (1.3)
// 34.7 / 40.6, 3000 (1.95) 44.3 / 44.4; 64 filters, 3000 (0.98) 31.0 / 29.5; 256 filters, 2000 (2.6) 55.5 / 53.1; 8 taps, 128 filters, 600 18.7 / 20.2, 2000 27.6 / 31.3,
// 3000 32.6 / 32.9 (average 32.9 / 30.6), 256 filters, 1200 (1.6) 29.8 / 32.1, 2000 41.0 / 38.3.
// Whole calls, us, one / two: max + average, 20 000 x 30-150 letters x 384 filters x 16 taps 205 / 193, 60 000 x 20-40 x 128 142 / 131; maximum,
// 60 000 x 101 x 256, 8 taps 225 / 195, 16 taps 328 / 304; average, 30 000 x 101 x 256 x 12 taps 186 / 174; 5000 x 101 x 64 x 16 taps 25.5 / 25.4.
template <int TB>
inline bool takes_two(unsigned ntile, size_t P)
{
    if (ntile % 2 != 0 && ntile <= 16) return false;
    const double rounds = (double)((ntile + 1) / 2) * (double)P / (256 * WAVES<2>);
    return rounds <= 1.0 ? rounds >= (TB == 1 ? 0.75 : 0.9) : rounds >= (TB == 1 ? 1.8 : 2.2);
}

template <int PT, bool WANT_ARGMAX, int TB, int NT>
int launch_sets(hipStream_t st, const digit_store& D, const float* bias, unsigned f0, unsigned ntile, size_t F, const uint8_t* X, size_t N, size_t ndef,
                const uint32_t* R, size_t P, float* pooled, uint32_t* argmax)
{
    auto kern = scanpool_digits_kernel<PT, WANT_ARGMAX, TB, NT>;
    constexpr size_t smem = scan_smem<TB, NT>();
    DBK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
    const unsigned groups = (ntile + NT - 1) / NT, nsplit = splits(groups, P);
    hipLaunchKernelGGL(kern, dim3(groups * nsplit), dim3(WAVES<NT> * 64), smem, st, D, bias, f0, (unsigned)F, X, N, ndef, R, (unsigned)P, nsplit, pooled, argmax);
    return 0;
}

template <int PT, bool WANT_ARGMAX, int TB>
int launch_pt(hipStream_t st, const digit_store& D, const float* bias, unsigned f0, unsigned ntile, size_t F, const uint8_t* X, size_t N, size_t ndef,
              const uint32_t* R, size_t P, float* pooled, uint32_t* argmax)
{
    if constexpr (TB <= 2) {
        if (takes_two<TB>(ntile, P)) return launch_sets<PT, WANT_ARGMAX, TB, 2>(st, D, bias, f0, ntile, F, X, N, ndef, R, P, pooled, argmax);
    }
    return launch_sets<PT, WANT_ARGMAX, TB, 1>(st, D, bias, f0, ntile, F, X, N, ndef, R, P, pooled, argmax);
}

// the filters f0 .. f0 + 32 * ntile - 1: their digits, then the scan (half: plain maxima with half the products)
template <int TB>
int launch(hipStream_t st, const digit_store& D, const float* W, const float* bias, unsigned f0, unsigned ntile, unsigned nflag, size_t m, size_t F,
           const uint8_t* X, size_t N, const uint32_t* R, size_t P, int ptype, bool half, float* pooled, uint32_t* argmax)
{
    constexpr bool ARG = TB < 4;                                   // (filters of more than 24 taps come without an argmax)
    const size_t ndef = N >= m ? N - m + 1 : 0;                    // rows the scan defines
    hipLaunchKernelGGL(weight_digits_kernel<TB>, dim3(nflag), dim3(256 * TB), 0, st, W, bias, (unsigned)m, (unsigned)F, f0, D);
    if constexpr (TB >= 3) {
        if (half)
            return ARG && argmax ? launch_max<ARG, TB>(st, D, W, bias, f0, ntile, m, F, X, N, ndef, R, P, pooled, argmax)
                                 : launch_max<false, TB>(st, D, W, bias, f0, ntile, m, F, X, N, ndef, R, P, pooled, argmax);
    }
    if (ptype == DBK_PT_AVG) return launch_pt<DBK_PT_AVG, false, TB>(st, D, bias, f0, ntile, F, X, N, ndef, R, P, pooled, argmax);
    if (ptype == DBK_PT_MAX)
        return ARG && argmax ? launch_pt<DBK_PT_MAX, ARG, TB>(st, D, bias, f0, ntile, F, X, N, ndef, R, P, pooled, argmax)
                             : launch_pt<DBK_PT_MAX, false, TB>(st, D, bias, f0, ntile, F, X, N, ndef, R, P, pooled, argmax);
    return ARG && argmax ? launch_pt<DBK_PT_ALL, ARG, TB>(st, D, bias, f0, ntile, F, X, N, ndef, R, P, pooled, argmax)
                         : launch_pt<DBK_PT_ALL, false, TB>(st, D, bias, f0, ntile, F, X, N, ndef, R, P, pooled, argmax);
}

// Whether plain maxima go through half the products: filters of more than 16 taps, more than 32 of them (a wave takes 64),
// regions of 80 rows on average and eight of them per wave. Measured, all the products / half of them, 24 taps: 100 000 x
// 500 letters x 1024 filters 10.4 / 8.1 ms (7.35 since the halves take turns), 65 536 x 101 x 256 0.515 / 0.461, 8192 x 101 x 256 0.080 / 0.078, 100 000 x 40 x
// 64 0.134 / 0.137, 2000 x 500 x 64 0.034 / 0.049; 16 taps, 65 536 x 101 x 256 0.361 / 0.368. A caller who asks for this
// path by name gets them whatever the number of regions; the regions' average length still decides, so a region's last bit may differ
// between calls of short and of long company.
bool half_the_products(size_t m, size_t F, size_t N, size_t P, int ptype, bool force)
{
    if (ptype != DBK_PT_MAX || m <= 16 || F <= FTILE || N < 80 * P) return false;
    return force || P * dbk::divup(F, PAIR) >= (size_t)256 * MAX_WAVES * 8;
}

// Whether a call of this size goes to the digit kernel when the choice is left to the library, in rows x 64-filter tiles
// (what the general path's time follows). The smallest call takes three launches (digits, scan, the look at the
// flags), 16-18 us. Measured break-even without argmax, 25 to 400 letters, 16 to 384 filters: up to 8 taps, where
// the general path has no matrix-core kernel, 0.15-0.25 M (at 0.5 M 17 us against 36, at 4 M 47 against 257); 9 to 32 taps
// 0.45-0.55 M (24 taps, 101 letters x 64 filters: 20 us against 19 at 0.5 M, 27 / 33 at 1 M, 72 / 129 at 4 M; 32 taps
// 26 / 26, 37 / 46, 107 / 171). With an argmax (a training step's forward pass) it lies at 0.9 M rows x tiles; such calls
// come here from the size on at which a group of models is better stepped alone than in the shared launches.
bool takes(size_t m, size_t F, size_t N, size_t P, bool argmax)
{
    if (m > (argmax ? 24u : 32u) || N == 0 || N > 0x7fffff00u || P > 0x7fff0000u) return false;
    if (argmax) return (double)N * dbk::divup(F, FTILE) >= (m > 12 ? 4.0e6 : 2.0e6);
    return (double)N * dbk::divup(F, 2 * FTILE) >= (m > 8 ? 0.6e6 : 0.25e6);
}

// A call's scratch: one flag per 32 filters (an even number of them: the launch behind looks at pairs), then the digits of
// up to PASS_TILES tiles; more filters than that are taken in several passes.
constexpr unsigned PASS_TILES = 1024;
inline size_t flag_bytes(size_t F) { return (2 * (size_t)dbk::divup(F, 2 * FTILE) * sizeof(unsigned) + 255) & ~(size_t)255; }
inline size_t scratch_bytes(size_t m, size_t F)
{
    const size_t nflag = 2 * (size_t)dbk::divup(F, 2 * FTILE), tiles = nflag < PASS_TILES ? nflag : PASS_TILES;
    return flag_bytes(F) + tiles * tile_bytes((unsigned)((m + 7) / 8));
}

// force: take this path whenever the shape allows, regardless of problem size.
// ws: device scratch of scratch_bytes(m, F) bytes the caller provides, or null to take the stream's grow-on-demand buffer.
int fprop_impl(hipStream_t st, const float* W, const float* bias, size_t m, size_t F, const uint8_t* X, size_t N,
               const uint32_t* R, size_t P, int ptype, float* pooled, uint32_t* argmax, bool force, unsigned char* ws = nullptr)
{
    if (ptype != DBK_PT_MAX && ptype != DBK_PT_AVG && ptype != DBK_PT_ALL) return -1;
    if (ptype == DBK_PT_AVG && argmax != nullptr) return -1;
    if (m > 32 || (force && m > 24) || N == 0 || N > 0x7fffff00u || P > 0x7fff0000u) return -1;
    if (!force && !takes(m, F, N, P, argmax != nullptr)) return -1;
    const unsigned tb = (unsigned)((m + 7) / 8), ntile = dbk::divup(F, FTILE), nflag = 2 * dbk::divup(F, 2 * FTILE);
    DBK_CHECK(nflag / 2 <= 65535u, "ValueError: too many filters (%zu) for one launch", F);
    if (!ws) {
        ws = (unsigned char*)dbk::workspace(scratch_bytes(m, F), st);
        // (a stream under capture whose scratch has not grown yet, or no memory: the general path needs none)
        if (!ws && !force) return -1;
        if (!ws) { dbk::set_error("MemoryError: could not allocate %zu bytes of scratch (%s)", scratch_bytes(m, F), dbk::workspace_error()); return 1; }
    }
    unsigned* flags = reinterpret_cast<unsigned*>(ws);
    const bool half = half_the_products(m, F, N, P, ptype, force);
    for (unsigned t0 = 0; t0 < ntile; t0 += PASS_TILES) {
        const unsigned nt = ntile - t0 < PASS_TILES ? ntile - t0 : PASS_TILES, nf = nflag - t0 < PASS_TILES ? nflag - t0 : PASS_TILES;
        const digit_store D = store_at(flags + t0, ws + flag_bytes(F), nf, tb);
        int rc;
        switch (tb) {
        case 1: rc = launch<1>(st, D, W, bias, t0 * FTILE, nt, nf, m, F, X, N, R, P, ptype, half, pooled, argmax); break;
        case 2: rc = launch<2>(st, D, W, bias, t0 * FTILE, nt, nf, m, F, X, N, R, P, ptype, half, pooled, argmax); break;
        case 3: rc = launch<3>(st, D, W, bias, t0 * FTILE, nt, nf, m, F, X, N, R, P, ptype, half, pooled, argmax); break;
        default: rc = launch<4>(st, D, W, bias, t0 * FTILE, nt, nf, m, F, X, N, R, P, ptype, half, pooled, argmax); break;
        }
        if (rc != 0) return rc;
    }
    // filters whose weights the digits do not express, by the tiles' flags, so that no host synchronisation is needed
    return dbk_scanpool_general::fprop_left(st, W, bias, m, F, X, N, R, P, ptype, pooled, argmax, flags);
}

int fprop(hipStream_t st, const float* W, const float* bias, size_t m, size_t F, const uint8_t* X, size_t N,
          const uint32_t* R, size_t P, int ptype, float* pooled, uint32_t* argmax)
{
    return fprop_impl(st, W, bias, m, F, X, N, R, P, ptype, pooled, argmax, false);
}

// ---- scratch that is part of the loaded code object, for callers that must not allocate ------------------
// Every device the library runs on holds its own copy of this array, at its own address, from the moment the code
// object is loaded there until the process ends. The array's name is a host-side handle, not a device address:
// host code asks the runtime for the address once per device and passes that pointer to the kernels.
// (24 taps: 1024 tiles' digits, 24.4 MB; flags of the 65 535 x 64 filters a launch may have, 0.5 MB)
constexpr size_t STATIC_SCRATCH_BYTES = size_t(24) << 20;
constexpr size_t STATIC_SEQUENCE_BYTES = (size_t(64) << 20) - 127; // sequence bytes a call may bring: the entry point's contract; the scratch does not depend on them
static_assert(131070 * sizeof(unsigned) + 256 + PASS_TILES * (FTILE * (sizeof(int) + sizeof(digit_facts)) + 3 * (NDIGIT + NTOP + 1) * SLOT_BYTES) <= STATIC_SCRATCH_BYTES, "the largest call must fit");
static __device__ __align__(256) unsigned char scratch[STATIC_SCRATCH_BYTES];
static unsigned char* g_static_scratch[64] = {nullptr};
static std::mutex g_static_scratch_mutex;

// Address of the current device's copy of `scratch` (looked up on the first call per device); null on failure.
static unsigned char* static_scratch()
{
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) { dbk::set_error("RuntimeError: no current device below 64"); return nullptr; }
    std::lock_guard<std::mutex> lock(g_static_scratch_mutex);
    if (!g_static_scratch[dev]) {
        unsigned char* p = nullptr;
        hipError_t e = hipGetSymbolAddress((void**)&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            dbk::set_error("RuntimeError: hipGetSymbolAddress(scratch) failed on device %d: %s", dev, hipGetErrorString(e));
            return nullptr;
        }
        g_static_scratch[dev] = p;
    }
    return g_static_scratch[dev];
}

}  // namespace dbk_scanpool_digits

extern "C" int dbk_scanpool_fprop_kmer_static(dbk_stream_t stream, const float* W, const float* bias, size_t m, size_t nfilter,
                                              const uint8_t* X, size_t N, const uint32_t* regions, size_t nregion, int ptype,
                                              float* pooled, uint32_t* argmax)
{
    using namespace dbk_scanpool_digits;
    DBK_CHECK(m >= 1, "ValueError: filter length must be >= 1");
    if (nfilter == 0 || nregion == 0) { dbk::clear_error(); return 0; }
    DBK_CHECK(W && bias && X && regions && pooled, "ValueError: null pointer argument");
    DBK_CHECK(!(argmax && ptype == DBK_PT_AVG), "ValueError: pooledmaps_argmax can only be used for max/all pooling.");
    DBK_CHECK(!argmax || (double)N * (double)nfilter <= 4294967296.0,
              "ValueError: %zu rows x %zu filters overflow the 32-bit argmax index; score in smaller batches or without argmax", N, nfilter);
    DBK_CHECK(N <= STATIC_SEQUENCE_BYTES,
              "ValueError: %zu sequence bytes; the entry point with the built-in buffer takes at most %zu per call; "
              "score in smaller batches or call dbk_scanpool_fprop_kmer", N, STATIC_SEQUENCE_BYTES);
    unsigned char* ws = static_scratch();
    if (!ws) return 2;
    // The flags and the digits are rewritten from the weights by the call's first launch, so nothing of an earlier call's
    // contents is read.
    int rc = fprop_impl(dbk::as_stream(stream), W, bias, m, nfilter, X, N, regions, nregion, ptype, pooled, argmax, true, ws);
    DBK_CHECK(rc >= 0, "NotImplementedError: the bulk path takes max / avg / all pooling and filter length <= 24");
    return rc;
}

extern "C" int dbk_scanpool_fprop_kmer(dbk_stream_t stream, const float* W, const float* bias, size_t m, size_t nfilter,
                                       const uint8_t* X, size_t N, const uint32_t* regions, size_t nregion, int ptype,
                                       float* pooled, uint32_t* argmax)
{
    DBK_CHECK(m >= 1, "ValueError: filter length must be >= 1");
    if (nfilter == 0 || nregion == 0) { dbk::clear_error(); return 0; }
    DBK_CHECK(W && bias && X && regions && pooled, "ValueError: null pointer argument");
    DBK_CHECK(!(argmax && ptype == DBK_PT_AVG), "ValueError: pooledmaps_argmax can only be used for max/all pooling.");
    DBK_CHECK(!argmax || (double)N * (double)nfilter <= 4294967296.0,
              "ValueError: %zu rows x %zu filters overflow the 32-bit argmax index; score in smaller batches or without argmax", N, nfilter);
    int rc = dbk_scanpool_digits::fprop_impl(dbk::as_stream(stream), W, bias, m, nfilter, X, N, regions, nregion, ptype, pooled, argmax, true);
    DBK_CHECK(rc >= 0, "NotImplementedError: the bulk path takes max / avg / all pooling and filter length <= 24");
    return rc;
}
