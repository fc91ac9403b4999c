// Device side of the prediction-time callers: packing of sequence text into the scan's input stream, the scores of every
// single-letter change of a batch (mutation maps), and the compaction of gradient maps.
//
// Reference: kangaroo/kangaroo/util.py:50-56,68-74 (letters), data.py:274-354 (packed stream, reverse-complement rows),
// predict.py:145-345 (predictions, mutation maps, window scans). There every change is one full pass of the net over the
// whole batch, the stream mutated on the host.
#include <type_traits>
#include "dbk_common.h"
#include "scan_common.h"

namespace {

using namespace dbk_scan;

constexpr double MAX_BOUND = 4294967295.0;                          // region bounds are 32-bit

__device__ __forceinline__ unsigned code_of_char(unsigned c)
{
    c |= 32u;                                                       // (letters only differ in this bit from their capitals)
    return c == 'a' ? 0u : c == 'c' ? 1u : c == 'g' ? 2u : (c == 't' || c == 'u') ? 3u : 255u;
}
__device__ __forceinline__ uint8_t strand_code(unsigned ch, bool rev)
{
    // 'A'..'z' is the only range where setting bit 5 maps a letter to a letter: '!'..'Z' minus 32 are no letters
    const unsigned c = ch >= 'A' ? code_of_char(ch) : 255u;
    return (uint8_t)(rev && c < 4u ? 3u - c : c);
}

// One wave per row (strand of a sequence): its leading pad, then its letters; the last row adds the closing pad.
// Row r of sequence s starts at padding * r + (strands * offsets[s] + (reverse row ? length : 0)).
__global__ __launch_bounds__(256) void k_pack_text(const uint8_t* __restrict__ text, const uint32_t* __restrict__ offsets, size_t nseq,
                                                   unsigned padding, unsigned strands, uint8_t* __restrict__ X, uint32_t* __restrict__ R)
{
    const unsigned lane = threadIdx.x & 63;
    const size_t nrow = nseq * strands, step = (size_t)gridDim.x * (blockDim.x >> 6);
    for (size_t r = (size_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); r < nrow; r += step) {
        const size_t s = strands == 2 ? r >> 1 : r;
        const bool rev = strands == 2 && (r & 1);
        const uint32_t o = offsets[s], len = offsets[s + 1] - o;
        const size_t a = (size_t)padding * r + (size_t)strands * o + (rev ? len : 0);
        for (uint32_t i = lane; i < padding; i += 64) X[a + i] = 255;
        uint8_t* dst = X + a + padding;
        for (uint32_t i = lane; i < len; i += 64) dst[i] = strand_code(text[o + (rev ? len - 1 - i : i)], rev);
        if (r + 1 == nrow)
            for (uint32_t i = lane; i < padding; i += 64) dst[len + i] = 255;
        if (lane == 0) { R[2 * r] = (uint32_t)a; R[2 * r + 1] = (uint32_t)(a + padding + len); }
    }
}

// Windows of `window` letters every `stride` letters of every sequence, N past its ends; the first window of a sequence
// starts window - 1 letters before it. first[s] .. first[s + 1] - 1 are sequence s's windows. One thread per byte of X.
__global__ __launch_bounds__(256) void k_pack_windows(const uint8_t* __restrict__ text, const uint32_t* __restrict__ offsets,
                                                      const uint32_t* __restrict__ first, unsigned nseq, unsigned window, unsigned stride,
                                                      unsigned padding, unsigned strands, size_t nbyte, uint8_t* __restrict__ X, uint32_t* __restrict__ R)
{
    const unsigned span = padding + window;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < nbyte; e += (size_t)gridDim.x * blockDim.x) {
        const size_t r = e / span;
        const unsigned o = (unsigned)(e - r * span);
        const size_t w = strands == 2 ? r >> 1 : r;
        if (o == 0 && w < first[nseq]) { R[2 * r] = (uint32_t)e; R[2 * r + 1] = (uint32_t)(e + span); }
        uint8_t v = 255;
        if (o >= padding && w < first[nseq]) {
            unsigned lo = 0, hi = nseq - 1;                         // the sequence that holds window w
            while (lo < hi) { const unsigned mid = (lo + hi + 1) >> 1; if (first[mid] <= w) lo = mid; else hi = mid - 1; }
            const bool rev = strands == 2 && (r & 1);
            const unsigned in = rev ? window - 1 - (o - padding) : o - padding;
            const long at = (long)((w - first[lo]) * stride) + in - (long)(window - 1);
            const uint32_t base = offsets[lo], len = offsets[lo + 1] - base;
            if (at >= 0 && at < (long)len) v = strand_code(text[base + at], rev);
        }
        X[e] = v;
    }
}

// ---------------------------------------------------------------------------------------------
// mutation maps
// ---------------------------------------------------------------------------------------------
// S[4 * p + c] = the net's output for the region around stream position p with the letter at p changed to c, for every
// letter p of every region (not its leading pad).
//
// A change at p moves the `m` rows whose windows hold p and nothing else, so a workgroup takes a few consecutive letters
// of one region: it scans the region once (16 lanes of filters x 16 lanes of rows, the letter table of 16 filters in
// LDS), keeps the maximum and the sum of the rows no change of its letters can reach and, one by one, the rows some change
// can; a wave then takes a letter at a time, its lanes being 4 quarters of the m rows x 16 filters: the rows are scanned anew without that
// letter, in two halves of its other taps, which leaves one addition for each of the four new ones, and pooled with what is kept (maps' error
// against float64 1.1e-6 to 7.1e-6, 1.3e-6 to 8.8e-6 with every tap in one chain). That adds a row's taps in another order than the forward pass does, and the
// rows of a mean in one that depends on where the workgroup's letters lie, so what a change is measured against is the score of the letter that is there
// from the same pass (k_mutation_map): letters of equal weight differ by nothing. An unknown letter and a change in two regions (below) have no such
// score: where filters have equal weights at a tap, their rows are scanned with each new letter in its place, in the order of the rows as they are (scan_changed).
// More than 16 filters take further passes; pooled values meet the dense head in LDS.
// What bounds it is instruction issue and LDS reads, one per (row, tap): m * m / 4 per letter and filter tile and lane (m * m with a lane per new
// letter, each of which scanned the rows by itself), where the reference's way (a pass of the
// whole net per change) scans length + m - 1 rows per change, and launches 15 kernels for it.
// Measured: 32 sequences of 60-101 letters, both strands, 16 filters of 24 taps: 25 us (a lane per new letter 47), the whole call
// 98 us from strings to host arrays (127) (74-84 ms when the batch was re-scored once per letter and base).
//
// The reference changes letter i of EVERY region in pass i; where a region is shorter than its neighbour's i that lands in
// the pad behind it, which is the next region's leading pad. Those entries are scored with both changes, the rows of either window anew.
constexpr unsigned MUT_F = 16, MUT_MAXK = 128, MUT_MAXH = 64;
constexpr unsigned MUT_NT = 256;                                    // threads per workgroup
constexpr unsigned MUT_TILE = 512;                                  // rows of the region scanned between two stagings of letters

struct mut_args {
    const float *W, *bias, *W1, *b1, *W2, *b2, *in_scale;
    const uint8_t* X;
    const uint32_t* R;
    size_t N, P;
    unsigned m, F, k, hidden, pos;                                  // pos: letters per workgroup
    int ptype, logistic, strands;
    float *S, *base;                                                // changed scores (4 per stream position), unchanged ones (per region)
};

// The letter table of filters c0 .. c0 + 15 (filters >= c1: zeros), [tap][letter][16], by all `nt` threads of the workgroup. Whether one of
// this thread's taps has the same weight, other than zero, for two letters (an unknown one counts their mean).
__device__ __forceinline__ bool letter_table16(float* __restrict__ lut, const float* __restrict__ W, unsigned m, size_t F, unsigned c0, unsigned c1,
                                               unsigned nt)
{
    bool ties = false;
    for (unsigned e = threadIdx.x; e < m * MUT_F; e += nt) {
        const unsigned j = e / MUT_F, c = c0 + e % MUT_F;
        float w[4];
#pragma unroll
        for (int l = 0; l < 4; ++l) w[l] = c < c1 ? W[(size_t)(4 * j + l) * F + c] : 0.0f;
        float z = w[0];
        z += w[1]; z += w[2]; z += w[3];
        float* t = lut + (size_t)j * NL * MUT_F + e % MUT_F;
        t[0] = w[0]; t[MUT_F] = w[1]; t[2 * MUT_F] = w[2]; t[3 * MUT_F] = w[3]; t[4 * MUT_F] = z * 0.25f; t[5 * MUT_F] = 0.0f;
        const float v[5] = {w[0], w[1], w[2], w[3], z * 0.25f};
#pragma unroll
        for (int a = 0; a < 4; ++a)
#pragma unroll
            for (int b = a + 1; b < 5; ++b) ties |= v[a] == v[b] && v[a] != 0.0f;
    }
    return ties;
}

// Rows p .. p + 3 of the staged letters (each already x 16) for this lane's filter, taps ascending. A letter is read once for the four rows it meets, a tap
// ahead of its use (one letter more than the rows need). us a launch, by the reads of its own tap as the compiler orders them / this: 4140 windows of 40 letters, 16 taps
// 18.3 / 17.1, 64 sequences of 101, 24 taps 6.8 / 6.6, of 300, 32 taps 11.6 / 10.3.
__device__ __forceinline__ void scan4(const float* __restrict__ lut_f, const uint8_t* __restrict__ let, unsigned p, unsigned m, float (&z)[4])
{
    z[0] = z[1] = z[2] = z[3] = 0.0f;
    unsigned l[4], ahead = let[p + 3];
#pragma unroll
    for (unsigned u = 0; u < 3; ++u) l[u + 1] = let[p + u];
#pragma unroll 4
    for (unsigned j = 0; j < m; ++j) {
        l[0] = l[1]; l[1] = l[2]; l[2] = l[3]; l[3] = ahead;
        ahead = let[p + 4 + j];
        const float* t = lut_f + j * NL * MUT_F;
#pragma unroll
        for (unsigned u = 0; u < 4; ++u) z[u] += t[l[u]];
    }
}

// Rows p .. p + NR - 1, in two halves of the taps, each ascending. FLY: taps whose reads are in flight.
template <unsigned NR, unsigned FLY>
__device__ __forceinline__ void scan_rows(const float* __restrict__ lut_f, const uint8_t* __restrict__ let, unsigned p, unsigned m, float (&z)[NR])
{
    float first[NR];
    unsigned l[NR];
#pragma unroll
    for (unsigned u = 0; u < NR; ++u) z[u] = 0.0f;
#pragma unroll
    for (unsigned u = 0; u + 1 < NR; ++u) l[u + 1] = let[p + u];
    auto taps = [&](unsigned from, unsigned to) __attribute__((always_inline)) {
#pragma unroll FLY
        for (unsigned j = from; j < to; ++j) {
#pragma unroll
            for (unsigned u = 0; u + 1 < NR; ++u) l[u] = l[u + 1];
            l[NR - 1] = let[p + NR - 1 + j];
            const float* t = lut_f + j * NL * MUT_F;
#pragma unroll
            for (unsigned u = 0; u < NR; ++u) z[u] += t[l[u]];
        }
    };
    const unsigned half = m / 2u;
    taps(0u, half);
#pragma unroll
    for (unsigned u = 0; u < NR; ++u) { first[u] = z[u]; z[u] = 0.0f; }
    taps(half, m);
#pragma unroll
    for (unsigned u = 0; u < NR; ++u) z[u] += first[u];
}

// Row p with each of the four letters at the indexes one and two (~0: none), its taps in the order of scan_rows.
__device__ __forceinline__ void scan_changed(const float* __restrict__ lut_f, const uint8_t* __restrict__ let, unsigned p, unsigned m, unsigned one, unsigned two,
                                             float (&z)[4])
{
    float first[4];
#pragma unroll
    for (unsigned c = 0; c < 4; ++c) z[c] = 0.0f;
#pragma unroll 1
    for (unsigned half = 0; half < 2u; ++half) {
#pragma unroll
        for (unsigned c = 0; c < 4; ++c) { first[c] = z[c]; z[c] = 0.0f; }
        const unsigned to = half ? m : m / 2u;
#pragma unroll 1
        for (unsigned j = half ? m / 2u : 0u; j < to; ++j) {
            const float* t = lut_f + j * NL * MUT_F;
            const bool changed = p + j == one || p + j == two;
            const unsigned l = let[p + j];
#pragma unroll
            for (unsigned c = 0; c < 4; ++c) z[c] += t[changed ? c * MUT_F : l];
        }
    }
#pragma unroll
    for (unsigned c = 0; c < 4; ++c) z[c] += first[c];
}

// LDS, in this order: letter table [m][NL][16], rows a change can reach [pos + m - 1][16] (rectified), two fold areas [2][NT / 16][16],
// pooled values [pos + 1][4][k], rows of the region's head, i.e. those whose windows hold letters of its leading pad, [m][16]; letters of a
// tile of rows and their windows, letters of the rows a change can reach, letters of the head rows, each wave's letters without the one it changes.
// (The scans of a quarter of the rows run up to 11 rows past the last one, and look up to 7 further.) The head's first weights [k][hidden] where they are few.
__host__ __device__ inline unsigned mut_tile_letters(unsigned m) { return (MUT_TILE + m + 7 + 3) & ~3u; }
__host__ __device__ inline unsigned mut_reach_letters(unsigned pos, unsigned m) { return (pos + 2 * m + 20 + 3) & ~3u; }
__host__ __device__ inline unsigned mut_head_weights(unsigned k, unsigned hidden) { const unsigned n = k * (hidden > 0 ? hidden : 1u); return n <= 2048u ? n : 0u; }
inline size_t mut_smem(unsigned pos, size_t m, size_t k, size_t hidden)
{
    return ((size_t)m * NL * MUT_F + (pos + m - 1) * MUT_F + 2 * MUT_NT / 16 * MUT_F + (pos + 1) * 4 * k + m * MUT_F + mut_head_weights((unsigned)k, (unsigned)hidden)) * sizeof(float) +
           mut_tile_letters((unsigned)m) + (1 + MUT_NT / 64) * mut_reach_letters(pos, (unsigned)m) + mut_reach_letters(0, (unsigned)m);
}
// what a call may ask for (65 536 bytes, while a workgroup had 256 threads and neither the head's weights nor the waves' letters in LDS)
inline bool mut_fits(size_t m, size_t k)
{
    return mut_smem(16, m, k, 4096) - MUT_NT / 64 * mut_reach_letters(16, (unsigned)m) - 2 * (MUT_NT - 256) * sizeof(float) <= 65536 + 36;
}

// Pass `pass` of the reference changes letter `pass` of every region: whether what it does to the region [pa, pb) before this one (none: !before)
// lands at stream position pad + pa + pass in the leading pad of this one, which begins at ra.
__device__ __forceinline__ bool spilled_pass(unsigned pass, unsigned pad, bool before, unsigned pa, unsigned pb, unsigned ra)
{
    return before && pb - pa > pass && pad + pa + pass >= pb && pad + pa + pass < ra + pad;
}

// v[c] of the four quarters of a wave put together: lanes 16 c .. 16 c + 15 get the one of v[c]
template <typename Op>
__device__ __forceinline__ float quarters(const float (&v)[4], Op op)
{
    float half[2];
#pragma unroll
    for (unsigned c = 0; c < 2; ++c) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v[c]), __float_as_uint(v[c + 2]), false, false);
        half[c] = op(__uint_as_float(r[0]), __uint_as_float(r[1]));
    }
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(half[0]), __float_as_uint(half[1]), false, false);
    return op(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// NR: rows that a lane scans at a time, of the quarter that it has. SPILLS: one strand only, where a change may lie in two regions (above).
// Few taps are all latency: a letter's rows take less than fetching them, so their kernels keep fewer reads in flight for the registers' sake and six
// or five waves per SIMD instead of four. (Up to 12 taps went through the kernel of four rows, of which one, two or three were any. us, with the letters
// per workgroup chosen below, and the kernel of a lane per new letter: 128 sequences of 60-101, one strand, 4 taps 33 -> 23 / 21, 8 taps 34 -> 27 / 27, 12 taps
// 39 -> 33 / 35; 64 on both strands 8 taps 28 -> 22 / 24, 12 taps 32 -> 25 / 30.) Eight rows at a time (25 to 64 taps) do not fit the registers of four waves:
// 26 spills of 108 bytes a lane. Four rows take none, and 79 against 87 us at 25 taps (128 sequences, both strands), but 91 against 88 at 32 and 238 against 227 at 64.
constexpr int mut_waves(unsigned nr) { return nr <= 2 ? 6 : nr == 3 ? 5 : 4; }
template <unsigned NR, bool SPILLS>
__global__ __launch_bounds__(MUT_NT, mut_waves(NR)) void k_mutation_scores(const mut_args a)
{
    constexpr unsigned FLY = NR <= 3 ? 2 : 4;
    extern __shared__ __align__(16) float msm[];
    const unsigned m = a.m, pad = m - 1;
    const size_t r = blockIdx.x;
    const unsigned tid = threadIdx.x, lane = tid & 63, wave = (unsigned)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    float* lut = msm;
    float* rows = lut + m * NL * MUT_F;
    float* fold = rows + (a.pos + m - 1) * MUT_F;
    float* pooled = fold + 2 * MUT_NT / 16 * MUT_F;
    float* head = pooled + (a.pos + 1) * 4 * a.k;
    float* head_w = head + m * MUT_F;
    const unsigned nhead_w = mut_head_weights(a.k, a.hidden);
    // (the weights are on their way before the region's bounds and letters)
    for (unsigned e = tid; e < nhead_w; e += MUT_NT) head_w[e] = a.W1[e];
    bool ties = letter_table16(lut, a.W, m, a.F, 0, a.F, MUT_NT);   // (of this thread's taps, then of the sixteen filters)
    const unsigned hl = tid & 15u;
    float hidden_b[MUT_MAXH / 16], hidden_w[MUT_MAXH / 16];         // this lane's hidden units'
#pragma unroll
    for (unsigned q = 0; q < MUT_MAXH / 16; ++q) {
        const bool one = hl + 16u * q < a.hidden;
        hidden_b[q] = one ? a.b1[hl + 16u * q] : 0.0f;
        hidden_w[q] = one ? a.W2[hl + 16u * q] : 0.0f;
    }
    const float last_b = a.hidden > 0 ? a.b2[0] : a.b1[0];
    const unsigned ra = a.R[2 * r], rb = a.R[2 * r + 1];
    const unsigned len = rb - ra > pad ? rb - ra - pad : 0u;
    const unsigned i0 = blockIdx.y * a.pos;
    if (i0 >= len && blockIdx.y != 0) return;
    const unsigned npos = i0 < len ? (len - i0 < a.pos ? len - i0 : a.pos) : 0u;
    uint8_t* tile = reinterpret_cast<uint8_t*>(head_w + nhead_w);
    uint8_t* let = tile + mut_tile_letters(m);
    uint8_t* hlet = let + mut_reach_letters(a.pos, m);
    uint8_t* mine = hlet + mut_reach_letters(0, m) + wave * mut_reach_letters(a.pos, m);
    const size_t n = a.N >= m ? a.N - m + 1 : 0;                   // rows the scan defines; later rows are relu(bias)
    // rows some change of these letters reaches: [s0, s1)
    const unsigned q0 = ra + pad + i0;                             // stream position of the first letter
    const unsigned s0 = q0 - pad, s1 = npos ? q0 + npos : s0;
    auto stage = [&](uint8_t* to, size_t from, unsigned count) {   // letters as offsets into a tap's part of the table
        for (unsigned e = tid; e < count; e += MUT_NT) to[e] = (uint8_t)((from + e < a.N ? letter_of(a.X[from + e]) : 5u) * MUT_F);
    };
    stage(let, s0, mut_reach_letters(a.pos, m));
    // the change of the region before this one that lands in this one's leading pad
    const bool shorter_before = SPILLS && r > 0;
    const unsigned pa = shorter_before ? a.R[2 * r - 2] : 0u, pb = shorter_before ? a.R[2 * r - 1] : 0u;
    auto spills = [&](unsigned pass) { return spilled_pass(pass, pad, shorter_before, pa, pb, ra); };
    bool spill_here = false;
    if (SPILLS)
        for (unsigned i = 0; i < npos; ++i) spill_here |= spills(i0 + i);
    // rows of the head that no change of these letters reaches: with a spill they are kept one by one as well
    const unsigned h1 = spill_here ? (s0 < ra + pad ? s0 : ra + pad) : ra;
    if (spill_here) stage(hlet, ra, mut_reach_letters(0, m));
    const unsigned f = tid & 15u, rl = tid >> 4;
    const unsigned kper = a.ptype == DBK_PT_ALL ? 2u : 1u;
    const float count = (float)(rb - ra);
    const float* lut_f = lut + f;

    for (unsigned f0 = 0; f0 < a.F; f0 += MUT_F) {
        const bool on = f0 + f < a.F;
        const float bf = on ? a.bias[f0 + f] : 0.0f;
        if (f0 > 0) {
            __syncthreads();                                        // the previous tile's table and rows are no longer read
            ties = letter_table16(lut, a.W, m, a.F, f0, a.F, MUT_NT);
        }
        // ---- the region as it is: rows out of reach folded, rows in reach kept
        float mx = 0.0f, sum = 0.0f;
        for (unsigned t0 = ra; t0 < rb; t0 += MUT_TILE) {
            __syncthreads();
            stage(tile, t0, mut_tile_letters(m));
            __syncthreads();
            const unsigned t1 = rb - t0 < MUT_TILE ? rb : t0 + MUT_TILE;
            for (unsigned p = t0 + 4 * rl; p < t1; p += MUT_NT / 4) {
                float z[4];
                scan_rows<4, FLY>(lut_f, tile, p - t0, m, z);
#pragma unroll
                for (unsigned u = 0; u < 4; ++u) {
                    if (p + u >= t1) break;
                    float v = (p + u < n ? z[u] : 0.0f) + bf;
                    v = v > 0.0f ? v : 0.0f;
                    if (p + u >= s0 && p + u < s1) rows[(p + u - s0) * MUT_F + f] = v;
                    else if (p + u < h1) head[(p + u - ra) * MUT_F + f] = v;
                    else { mx = v > mx ? v : mx; sum += v; }
                }
            }
        }
        fold[rl * MUT_F + f] = mx;
        fold[(MUT_NT / 16 + rl) * MUT_F + f] = sum;
        ties = __syncthreads_or(ties) != 0;
        mx = 0.0f; sum = 0.0f;
#pragma unroll
        for (unsigned t = 0; t < MUT_NT / 16; ++t) {
            const float v = fold[t * MUT_F + f];
            mx = v > mx ? v : mx;
            sum += fold[(MUT_NT / 16 + t) * MUT_F + f];
        }
        // ---- one letter per wave at a time (the item behind the last one is the region unchanged): lane = (quarter of the rows, filter)
        const unsigned g = lane >> 4;
        for (unsigned i = wave; i < npos + (i0 == 0 ? 1u : 0u); i += MUT_NT / 64) {
            float bm[4] = {mx, mx, mx, mx}, bs[4] = {0.0f, 0.0f, 0.0f, 0.0f};      // with each new letter, of this quarter
            float km = 0.0f, ks = g == 0u ? sum : 0.0f;                             // of rows that no new letter changes
            auto kept = [&](const float* values, unsigned lo, unsigned hi) __attribute__((always_inline)) {
                for (unsigned p = lo + g; p < hi; p += 4) { const float v = values[p * MUT_F + f]; km = v > km ? v : km; ks += v; }
            };
            // rows [lo, hi) among the kept ones are scanned anew: those of letter q0 + i's windows, and with a spill the head as well
            const bool both = SPILLS && i < npos && spills(i0 + i);
            const unsigned q2 = pad + pa + i0 + i, rest = s1 - s0;
            unsigned hp = 0;                                         // rows of the head to scan anew
            if (both) {
                hp = q2 + 1 - ra;                                    // rows ra .. q2 hold it
                if (hp > h1 - ra) hp = h1 - ra;
            }
            kept(head, hp, h1 - ra);
            unsigned lo = i < npos ? i : rest, hi = i < npos ? i + m : rest;
            if (both && q2 >= s0) lo = 0;
            kept(rows, 0u, lo);
            kept(rows, hi, rest);
            // the rows, then (spills) those of the head: row 0 at stream position `first`, the letters at indexes `at` and `at2` (~0: none) changed
            unsigned first = s0, at = i + pad, at2 = both ? q2 - s0 : ~0u;
            const uint8_t* letters = let;
            for (unsigned part = 0; part < (both ? 2u : 1u); ++part) {
                if (ties && (both || letters[at] >= 4u * MUT_F)) {
#pragma unroll 1
                    for (unsigned p = lo + g; p < hi; p += 4) {
                        float z[4];
                        scan_changed(lut_f, letters, p, m, at, at2, z);
#pragma unroll
                        for (unsigned c = 0; c < 4; ++c) {
                            float v = ((size_t)first + p < n ? z[c] : 0.0f) + bf;
                            v = v > 0.0f ? v : 0.0f;
                            bm[c] = v > bm[c] ? v : bm[c];
                            bs[c] += v;
                        }
                    }
                    lo = hi;                                         // (nothing left for the quarters)
                }
                const unsigned each = (hi - lo + 3u) / 4u, shown = hi > lo ? hi - lo + 3u + NR + m : 0u;
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                for (unsigned e = lane; e < shown; e += 64) mine[e] = lo + e == at || lo + e == at2 ? (uint8_t)(5u * MUT_F) : letters[lo + e];
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                const unsigned stop = n > first ? (n - first < hi ? (unsigned)(n - first) : hi) : 0u;      // rows that the scan defines
                for (unsigned u0 = 0; u0 < each; u0 += NR) {
                    const unsigned p0 = lo + g * each + u0;
                    float z[NR], w[NR][4];
                    // what the new letters put in the place of the old (no tap of this row's: nothing)
#pragma unroll
                    for (unsigned u = 0; u < NR; ++u) {
                        const bool here = at - (p0 + u) < m;        // (a row past the letter wraps round)
                        const float* t = lut_f + (here ? at - (p0 + u) : 0u) * NL * MUT_F;
#pragma unroll
                        for (unsigned c = 0; c < 4; ++c) w[u][c] = here ? t[c * MUT_F] : 0.0f;
                    }
                    if (SPILLS && both) {
#pragma unroll
                        for (unsigned u = 0; u < NR; ++u) {
                            const bool there = at2 - (p0 + u) < m;
                            const float* t = lut_f + (there ? at2 - (p0 + u) : 0u) * NL * MUT_F;
#pragma unroll
                            for (unsigned c = 0; c < 4; ++c) w[u][c] += there ? t[c * MUT_F] : 0.0f;
                        }
                    }
                    scan_rows<NR, FLY>(lut_f, mine, p0 - lo, m, z);
#pragma unroll
                    for (unsigned u = 0; u < NR; ++u) {
                        const bool counts = u0 + u < each && p0 + u < hi, in = p0 + u < stop;
#pragma unroll
                        for (unsigned c = 0; c < 4; ++c) {
                            float v = (in ? z[u] + w[u][c] : 0.0f) + bf;
                            v = counts && v > 0.0f ? v : 0.0f;
                            bm[c] = v > bm[c] ? v : bm[c];
                            bs[c] += v;
                        }
                    }
                }
                letters = hlet; first = ra; lo = 0u; hi = hp; at = q2 - ra; at2 = ~0u;
            }
            // ---- the quarters together, quarter g with new letter g
#pragma unroll
            for (unsigned c = 0; c < 4; ++c) { bm[c] = km > bm[c] ? km : bm[c]; bs[c] += ks; }
            const float best = quarters(bm, [](float x, float y) { return x > y ? x : y; }), total = quarters(bs, [](float x, float y) { return x + y; });
            if (on) {
                float* to = pooled + (i * 4 + g) * a.k + (f0 + f) * kper;
                if (a.ptype == DBK_PT_MAX) to[0] = best;
                else if (a.ptype == DBK_PT_AVG) to[0] = total / count;
                else { to[0] = best; to[1] = total / count; }
            }
        }
    }
    __syncthreads();
    // ---- the dense head: 16 lanes per (letter, change) item, hidden units dealt over them
    const float sc = a.in_scale ? a.in_scale[0] : 1.0f;
    const float* w1 = nhead_w ? head_w : a.W1;
    const unsigned nitem = (npos + (i0 == 0 ? 1u : 0u)) * 4;
    for (unsigned it = tid >> 4; it < nitem; it += MUT_NT / 16) {
        const float* x = pooled + it * a.k;
        float out = 0.0f;
        if (a.hidden > 0) {
#pragma unroll
            for (unsigned q = 0; q < MUT_MAXH / 16; ++q) {
                const unsigned h = hl + 16u * q;
                if (h >= a.hidden) break;
                float z = 0.0f;
#pragma unroll 8
                for (unsigned kk = 0; kk < a.k; ++kk) z = __builtin_fmaf(x[kk] * sc, w1[(size_t)kk * a.hidden + h], z);
                z += hidden_b[q];
                out += (z > 0.0f ? z : 0.0f) * hidden_w[q];
            }
        } else {
            for (unsigned kk = hl; kk < a.k; kk += 16) out += x[kk] * sc * w1[kk];
        }
#pragma unroll
        for (int d = 8; d >= 1; d >>= 1) out += __shfl_xor(out, d, 16);
        out += last_b;
        if (a.logistic) out = 1.0f / (1.0f + expf(-out));
        if (hl == 0) {
            const unsigned i = it >> 2, c = it & 3u;
            if (i < npos) a.S[4 * ((size_t)q0 + i) + c] = out;
            else if (c == 0) a.base[r] = out;
        }
    }
}

// ---------------------------------------------------------------------------------------------
// scores of few sequences
// ---------------------------------------------------------------------------------------------
// Scan, pooling and dense head of one (region, model) per workgroup of NT threads, for calls that are all latency: 16 lanes of
// filters x NT / 16 lanes of rows, four rows each at a time; lane h of the first wave holds hidden unit h's weights, on
// their way while the region is scanned. One launch and two round trips to memory (bounds, then letters and weights) where
// the scan kernel and the head cost a launch and three each. KM: pooled features per model, at most.
// Measured: 64 sequences x 101 nt, 16 filters of 24 taps, 16 -> 32 -> 1: 5.9 us, the whole call 10.0 with its host side (scan kernel
// 11.5 + head 4.1, the call 17.8).
struct small_args {
    const float *W, *bias, *W1, *b1, *W2, *b2, *in_scale;
    const uint8_t* X;
    const uint32_t* R;
    size_t N;
    unsigned m, nmodel, nfilter, k, hidden;
    int ptype, logistic;
    float* scores;
};

inline size_t small_smem(size_t m, unsigned nt) { return ((size_t)m * NL * MUT_F + nt / 64 * 2 * MUT_F + 2 * MUT_F) * sizeof(float) + mut_tile_letters((unsigned)m); }

template <int KM, int NT>
__global__ __launch_bounds__(NT) void k_predict_small(const small_args a)
{
    extern __shared__ __align__(16) float msm[];
    const unsigned m = a.m, tid = threadIdx.x, lane = tid & 63, wave = (unsigned)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const unsigned b = blockIdx.y, f = tid & 15u, rl = tid >> 4;
    const size_t r = blockIdx.x;
    float* lut = msm;
    float* part = lut + m * NL * MUT_F;                             // [waves][2][16]: maxima, sums
    float* x = part + NT / 64 * 2 * MUT_F;                          // pooled features
    uint8_t* tile = reinterpret_cast<uint8_t*>(x + 2 * MUT_F);
    const unsigned ra = a.R[2 * r], rb = a.R[2 * r + 1];
    const unsigned c0 = b * a.nfilter;
    const size_t F = (size_t)a.nmodel * a.nfilter;
    const float bf = f < a.nfilter ? a.bias[c0 + f] : 0.0f;
    letter_table16(lut, a.W, m, F, c0, c0 + a.nfilter, NT);
    float w[KM], b1v = 0.0f, w2v = 0.0f;
    if (wave == 0) {
        const unsigned h1 = a.hidden ? a.hidden : 1u;
        const bool in = lane < h1;
        // without a hidden layer lane l holds input l's weight
        if (a.hidden) {
#pragma unroll
            for (int kk = 0; kk < KM; ++kk) w[kk] = in && kk < (int)a.k ? a.W1[((size_t)b * a.k + kk) * h1 + lane] : 0.0f;
            w2v = in ? a.W2[(size_t)b * h1 + lane] : 0.0f;
        } else w[0] = lane < a.k ? a.W1[(size_t)b * a.k + lane] : 0.0f;
        b1v = in ? a.b1[(size_t)b * h1 + lane] : 0.0f;
    }
    const size_t n = a.N >= m ? a.N - m + 1 : 0;                   // rows the scan defines; later rows are relu(bias)
    float mx = 0.0f, sum = 0.0f;
    for (unsigned t0 = ra; t0 < rb; t0 += MUT_TILE) {
        if (t0 != ra) __syncthreads();
        const unsigned t1 = rb - t0 < MUT_TILE ? rb : t0 + MUT_TILE, count = t1 - t0 + m + 3;
        for (unsigned e = tid; e < count; e += NT) tile[e] = (uint8_t)((t0 + (size_t)e < a.N ? letter_of(a.X[t0 + (size_t)e]) : 5u) * MUT_F);
        __syncthreads();
        for (unsigned p = t0 + 4 * rl; p < t1; p += NT / 4) {
            float z[4];
            scan4(lut + f, tile, p - t0, m, z);
#pragma unroll
            for (unsigned u = 0; u < 4; ++u)
                if (p + u < t1) {
                    float v = (p + u < n ? z[u] : 0.0f) + bf;
                    v = v > 0.0f ? v : 0.0f;
                    mx = v > mx ? v : mx;
                    sum += v;
                }
        }
    }
#pragma unroll
    for (int d = 16; d <= 32; d <<= 1) {
        const float v = __shfl_xor(mx, d, 64);
        mx = v > mx ? v : mx;
        sum += __shfl_xor(sum, d, 64);
    }
    if (lane < MUT_F) { part[(2 * wave) * MUT_F + f] = mx; part[(2 * wave + 1) * MUT_F + f] = sum; }
    __syncthreads();
    if (wave != 0) return;
    if (lane < MUT_F) {
        for (unsigned v = 1; v < NT / 64; ++v) {
            const float o = part[(2 * v) * MUT_F + f];
            mx = o > mx ? o : mx;
            sum += part[(2 * v + 1) * MUT_F + f];
        }
        const float sc = a.in_scale ? a.in_scale[b] : 1.0f, avg = sum / (float)(rb - ra);
        if (a.ptype == DBK_PT_ALL) { x[2 * f] = mx * sc; x[2 * f + 1] = avg * sc; }
        else x[f] = (a.ptype == DBK_PT_MAX ? mx : avg) * sc;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    float out;
    if (a.hidden) {
        float z = 0.0f;
#pragma unroll
        for (int kk = 0; kk < KM; ++kk) z = __builtin_fmaf(kk < (int)a.k ? x[kk] : 0.0f, w[kk], z);
        z += b1v;
        out = (z > 0.0f ? z : 0.0f) * w2v;
    } else out = lane < a.k ? x[lane] * w[0] : 0.0f;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) out += __shfl_xor(out, d, 64);
    if (lane == 0) {
        out += a.hidden ? a.b2[b] : b1v;
        if (a.logistic) out = 1.0f / (1.0f + expf(-out));
        a.scores[r * a.nmodel + b] = out;
    }
}

// ---------------------------------------------------------------------------------------------
// gradient maps
// ---------------------------------------------------------------------------------------------
// One workgroup per sequence takes it from its letters to the map: both strands scanned (as k_predict_small does, keeping each
// filter's first largest row and, where a mean is pooled, a bit per row and filter that says the rectifier let it through) and
// put through the head; then the winning strand's score goes back through the head, the pooling and the filters. A letter's
// windows are rows of its own sequence, so nothing leaves the workgroup, no feature map is written, and the strand that lost is not
// taken back at all. Layer by layer the same took 23 launches over three maps of rows x filters.
// What bounds it is latency with the maximum, LDS reads with the mean (16 bytes per letter, base, tap and four filters). Measured: 1000 sequences of 101
// letters, both strands, 16 filters of 24 taps: 26 us a launch (layer by layer 170 us of kernels,
// 210 until the last of them ended), the call from strings to host arrays 0.90 -> 0.55 ms.
constexpr unsigned GRAD_MAXROWS = 2048;                             // rows of a region: their bits are 2 x 2 bytes of LDS each

struct grad_args {
    const float *W, *bias, *W1, *b1, *W2, *b2, *in_scale;
    const uint8_t* text;
    const uint32_t* offsets;
    unsigned m, F, k, hidden, rows_max;
    int ptype, logistic, strands;
    float *Z, *map;
    uint8_t* letters;
};

__host__ __device__ inline unsigned grad_letters(unsigned rows_max, unsigned m) { return (rows_max + m + 3 + 3 + 3) & ~3u; }
inline size_t grad_smem(size_t m, unsigned rows_max)
{
    return ((size_t)m * (NL + 4) * MUT_F + 3 * 16 * MUT_F + 2 * 2 * MUT_F + 2 * 64 + 2 * 2 * MUT_F + 2 * MUT_F + 4) * sizeof(float) +
           2 * ((rows_max + 1) & ~1u) * sizeof(uint16_t) + grad_letters(rows_max, (unsigned)m);
}

__global__ __launch_bounds__(256) void k_gradient_map(const grad_args a)
{
    extern __shared__ __align__(16) float msm[];
    const unsigned m = a.m, pad = m - 1, tid = threadIdx.x, lane = tid & 63;
    const unsigned f = tid & 15u, rl = tid >> 4;
    const size_t s = blockIdx.x;
    const unsigned base = a.offsets[s], len = a.offsets[s + 1] - base, rows = pad + len;
    float* lut = msm;                                               // [tap][letter][16]
    float* wt = lut + m * NL * MUT_F;                               // [tap][base][16], times the mean's gradient
    float* fold = wt + m * 4 * MUT_F;                               // largest value [16][16], sum [16][16], its row [16][16]
    unsigned* frow = reinterpret_cast<unsigned*>(fold + 2 * 16 * MUT_F);
    float* x = fold + 3 * 16 * MUT_F;                               // pooled features of either strand [2][32]
    float* hid = x + 2 * 2 * MUT_F;                                 // hidden units [2][64]
    unsigned* arg = reinterpret_cast<unsigned*>(hid + 2 * 64);      // row of the maximum [2][16]
    float* dmax = reinterpret_cast<float*>(arg + 2 * MUT_F);        // gradients of the pooled values [16], [16]
    float* davg = dmax + MUT_F;
    float* zs = davg + 3 * MUT_F;                                   // scores [2]
    uint16_t* bits = reinterpret_cast<uint16_t*>(zs + 4);           // [2][rows]
    const unsigned nbits = (a.rows_max + 1) & ~1u;
    uint8_t* tile = reinterpret_cast<uint8_t*>(bits + 2 * nbits);
    const bool mean = a.ptype != DBK_PT_MAX;
    const float bf = f < a.F ? a.bias[f] : 0.0f, sc = a.in_scale ? a.in_scale[0] : 1.0f;
    letter_table16(lut, a.W, m, a.F, 0, a.F, 256);
    for (int st = 0; st < a.strands; ++st) {
        __syncthreads();                                            // the other strand's letters are no longer read
        for (unsigned e = tid; e < rows + m + 3; e += 256) {
            const unsigned i = e - pad;                             // (wraps for the pad before the letters)
            tile[e] = (uint8_t)((i < len ? letter_of(strand_code(a.text[base + (st ? len - 1 - i : i)], st != 0)) : 4u) * MUT_F);
        }
        __syncthreads();
        float mx = -1.0f, sum = 0.0f;
        unsigned at = ~0u;
        for (unsigned p = 4 * rl; p < rows; p += 64) {
            float z[4];
            scan4(lut + f, tile, p, m, z);
#pragma unroll
            for (unsigned u = 0; u < 4; ++u) {
                float v = z[u] + bf;
                v = v > 0.0f && p + u < rows ? v : 0.0f;
                if (v > mx && p + u < rows) { mx = v; at = p + u; }
                sum += v;
                if (mean) {
                    const unsigned on = (unsigned)(__ballot(v > 0.0f) >> (lane & 48u));
                    if (f == 0 && p + u < rows) bits[st * nbits + p + u] = (uint16_t)on;
                }
            }
        }
        fold[rl * MUT_F + f] = mx;
        fold[(16 + rl) * MUT_F + f] = sum;
        frow[rl * MUT_F + f] = at;
        __syncthreads();
        if (tid < 64) {
            if (tid < a.F) {
                mx = -1.0f; sum = 0.0f; at = ~0u;
#pragma unroll
                for (unsigned t = 0; t < 16; ++t) {
                    const float v = fold[t * MUT_F + tid];
                    const unsigned r = frow[t * MUT_F + tid];
                    if (v > mx || (v == mx && r < at)) { mx = v; at = r; }       // the first of equal rows
                    sum += fold[(16 + t) * MUT_F + tid];
                }
                const float avg = sum / (float)rows;
                if (a.ptype == DBK_PT_ALL) { x[st * 2 * MUT_F + 2 * tid] = mx; x[st * 2 * MUT_F + 2 * tid + 1] = avg; }
                else x[st * 2 * MUT_F + tid] = a.ptype == DBK_PT_MAX ? mx : avg;
                arg[st * MUT_F + tid] = mx > 0.0f ? at : ~0u;        // (a maximum of nothing has no gradient)
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            const float* xs = x + st * 2 * MUT_F;
            float out = 0.0f;
            if (a.hidden > 0) {
                if (lane < a.hidden) {
                    float z = 0.0f;
#pragma unroll 8
                    for (unsigned kk = 0; kk < a.k; ++kk) z = __builtin_fmaf(xs[kk] * sc, a.W1[(size_t)kk * a.hidden + lane], z);
                    z += a.b1[lane];
                    z = z > 0.0f ? z : 0.0f;
                    hid[st * 64 + lane] = z;
                    out = z * a.W2[lane];
                }
            } else if (lane < a.k) out = xs[lane] * sc * a.W1[lane];
#pragma unroll
            for (int d = 32; d >= 1; d >>= 1) out += __shfl_xor(out, d, 64);
            out += a.hidden > 0 ? a.b2[0] : a.b1[0];
            if (a.logistic) out = 1.0f / (1.0f + expf(-out));
            if (lane == 0) zs[st] = out;
        }
    }
    __syncthreads();
    // ---- the strand that predicts more (the forward one wins ties), and its score's way back: eight lanes per pooled value
    const unsigned win = a.strands == 2 && zs[0] < zs[1] ? 1u : 0u;
    float dz = zs[win];
    if (a.strands == 2 && !(zs[0] >= zs[1]) && win == 0) dz = 0.0f;  // (scores that do not compare pick neither row of the pair)
    {
        const unsigned kk = tid >> 3, h8 = tid & 7u;
        float d = 0.0f;
        if (kk < a.k) {
            if (a.hidden > 0) {
                for (unsigned h = h8; h < a.hidden; h += 8)
                    d += (hid[win * 64 + h] > 0.0f ? dz * a.W2[h] : 0.0f) * a.W1[(size_t)kk * a.hidden + h];
            } else if (h8 == 0) d = dz * a.W1[kk];
        }
#pragma unroll
        for (int w = 4; w >= 1; w >>= 1) d += __shfl_xor(d, w, 8);
        if (h8 == 0) {
            d *= sc;
            if (a.ptype == DBK_PT_ALL) {
                if (kk & 1u) davg[kk >> 1] = kk < a.k ? d / (float)rows : 0.0f;
                else dmax[kk >> 1] = kk < a.k ? d : 0.0f;
            } else if (kk < MUT_F) {
                if (a.ptype == DBK_PT_MAX) dmax[kk] = kk < a.k ? d : 0.0f;
                else davg[kk] = kk < a.k ? d / (float)rows : 0.0f;
            }
        }
    }
    __syncthreads();
    if (mean) {
        for (unsigned e = tid; e < m * 4 * MUT_F; e += 256) {
            const unsigned j = e / (4 * MUT_F), c = e / MUT_F % 4;
            wt[e] = davg[e % MUT_F] * lut[(j * NL + c) * MUT_F + e % MUT_F];
        }
        __syncthreads();
    }
    for (unsigned e = tid; e < 4 * len; e += 256) {
        const unsigned q = pad + (e >> 2), c = e & 3u;               // the letter's place among the region's rows
        float g = 0.0f;
        if (mean) {
            const uint16_t* on = bits + win * nbits + q;
#pragma unroll 2
            for (unsigned j = 0; j < m; ++j) {
                const unsigned b = on[-(int)j];
                const float4* w = reinterpret_cast<const float4*>(wt + (j * 4 + c) * MUT_F);
#pragma unroll
                for (unsigned t = 0; t < 4; ++t) {
                    const float4 v = w[t];
                    g += b & (1u << (4 * t)) ? v.x : 0.0f;
                    g += b & (2u << (4 * t)) ? v.y : 0.0f;
                    g += b & (4u << (4 * t)) ? v.z : 0.0f;
                    g += b & (8u << (4 * t)) ? v.w : 0.0f;
                }
            }
        }
        if (a.ptype != DBK_PT_AVG)
            for (unsigned t = 0; t < a.F; ++t) {
                const unsigned j = q - arg[win * MUT_F + t];         // (wraps past m where the maximum is another window's)
                if (j < m) g += dmax[t] * lut[(j * NL + c) * MUT_F + t];
            }
        a.map[4 * (size_t)base + e] = g;
    }
    for (unsigned i = tid; i < len; i += 256) {
        const unsigned c = strand_code(a.text[base + (win ? len - 1 - i : i)], win != 0);
        a.letters[(size_t)base + i] = (uint8_t)(c == 0 ? 'A' : c == 1 ? 'C' : c == 2 ? 'G' : c == 3 ? 'T' : 'N');
    }
    if (tid == 0) a.Z[s] = a.strands == 2 && !(zs[0] >= zs[1]) && win == 0 ? __uint_as_float(0x7fc00000u) : zs[win];
}

// The map of a sequence: (changed score - score) where the larger of the two is positive, else 0; with both strands a score
// is the larger of the pair's, the reverse row changed at the mirrored letter to the complement. The score to take off is that of the letter that is
// there, its rows added in the order of the changed ones; where that is none of ACGT, or the pass changes the region twice, the score as
// k_mutation_scores formed it of the region as it is. One workgroup per sequence.
__global__ __launch_bounds__(256) void k_mutation_map(const uint32_t* __restrict__ R, unsigned pad, int strands, const uint8_t* __restrict__ X,
                                                      const float* __restrict__ S, const float* __restrict__ base, float* __restrict__ Z,
                                                      float* __restrict__ map)
{
    const size_t s = blockIdx.x, r = s * (unsigned)strands;
    const unsigned ra = R[2 * r], len = R[2 * r + 1] - ra - pad;
    const size_t out = ((size_t)ra - (size_t)pad * r) / (unsigned)strands;       // letters of the sequences before this one
    float z = base[r];
    if (strands == 2) z = base[r + 1] > z ? base[r + 1] : z;
    const unsigned mirror = strands == 2 ? R[2 * r + 3] - 1 : 0u;
    const bool before = strands == 1 && r > 0;
    const unsigned pa = before ? R[2 * r - 2] : 0u, pb = before ? R[2 * r - 1] : 0u;
    for (unsigned e = threadIdx.x; e < 4 * len; e += blockDim.x) {
        const unsigned i = e >> 2, c = e & 3u;
        const size_t at = (size_t)ra + pad + i;
        auto score = [&](unsigned letter) {
            float v = S[4 * at + letter];
            if (strands == 2) {
                const float w = S[4 * (size_t)(mirror - i) + 3 - letter];
                v = w > v ? w : v;
            }
            return v;
        };
        const unsigned own = X[at];
        const float v = score(c), from = own < 4u && !spilled_pass(i, pad, before, pa, pb, ra) ? score(own) : z;
        // (a product with 1 or 0, so that scores that are infinite or not a number show)
        const float d = v - from;
        map[4 * out + e] = (z > v ? z : v) > 0.0f ? d : v == v && z == z ? d * 0.0f : d;
    }
    if (threadIdx.x == 0) Z[s] = z;
}

// The rows of dX (4 values per stream position) that belong to the winning strand's letters, one sequence after another.
// Z: the rows' predictions; with both strands the forward row wins ties. One workgroup per sequence.
template <typename T, typename T4>
__global__ __launch_bounds__(256) void k_gather_maps(const uint32_t* __restrict__ R, unsigned pad, int strands, const T* __restrict__ Z,
                                                     const T4* __restrict__ dX, T4* __restrict__ map)
{
    const size_t s = blockIdx.x;
    size_t r = s * (unsigned)strands;
    const size_t out = ((size_t)R[2 * r] - (size_t)pad * r) / (unsigned)strands;
    if (strands == 2 && Z[r] < Z[r + 1]) r += 1;
    const unsigned ra = R[2 * r], len = R[2 * r + 1] - ra - pad;
    for (unsigned i = threadIdx.x; i < len; i += blockDim.x) map[out + i] = dX[(size_t)ra + pad + i];
}

}  // namespace

extern "C" {

int dbk_pack_text(dbk_stream_t stream, const uint8_t* text, const uint32_t* offsets, size_t nseq, size_t padding, int strands,
                  uint8_t* X, uint32_t* R)
{
    DBK_CHECK(strands == 1 || strands == 2, "ValueError: strands must be 1 or 2");
    if (nseq == 0) { dbk::clear_error(); return 0; }
    // (the letters, which only the device knows here, count too: the caller sizes X and sees to it)
    DBK_CHECK((double)nseq * strands * (double)padding <= MAX_BOUND, "ValueError: the stream of %zu sequences has more than 2^32 - 1 bytes", nseq);
    DBK_CHECK(offsets && X && R, "ValueError: null pointer argument");
    unsigned grid = dbk::divup(nseq * strands, 4);
    if (grid > 8192u) grid = 8192u;
    hipLaunchKernelGGL(k_pack_text, dim3(grid), dim3(256), 0, dbk::as_stream(stream), text, offsets, nseq, (unsigned)padding, (unsigned)strands, X, R);
    DBK_LAUNCH_OK();
}

int dbk_pack_windows(dbk_stream_t stream, const uint8_t* text, const uint32_t* offsets, const uint32_t* first, size_t nseq, size_t nwindow,
                     size_t window, size_t stride, size_t padding, int strands, uint8_t* X, uint32_t* R)
{
    DBK_CHECK(strands == 1 || strands == 2, "ValueError: strands must be 1 or 2");
    DBK_CHECK(window >= 1 && stride >= 1, "ValueError: window and stride must be >= 1");
    if (nseq == 0 || nwindow == 0) { dbk::clear_error(); return 0; }
    DBK_CHECK((double)nwindow * strands * ((double)padding + (double)window) <= MAX_BOUND, "ValueError: the stream of %zu windows has more than 2^32 - 1 bytes", nwindow);
    DBK_CHECK(offsets && first && X && R, "ValueError: null pointer argument");
    const size_t nbyte = nwindow * strands * (padding + window) + padding;
    hipLaunchKernelGGL(k_pack_windows, dim3(dbk::ew_grid(nbyte)), dim3(256), 0, dbk::as_stream(stream), text, offsets, first, (unsigned)nseq,
                       (unsigned)window, (unsigned)stride, (unsigned)padding, (unsigned)strands, nbyte, X, R);
    DBK_LAUNCH_OK();
}

int dbk_predict_small_takes(size_t m, size_t nmodel, size_t nfilter, size_t N, size_t nregion, int ptype, size_t hidden)
{
    // Every workgroup stages its model's weights: worth it while the call is a few waves of latency. One model's 16 filters leave the scan
    // kernel 48 of a tile's 64 lanes idle: up to 6e6 rows x taps (us a call, this kernel / scan kernel + head: 24 taps, 2000 x 101 nt 15 /
    // 18; 4 taps, 65 217 x 20 nt 94 / 240; 8 taps, 3358 x 60 nt 15 / 26). Where models share a tile, the workgroups that a GPU holds
    // at once, 2048, are the line besides: 16 models of 8 filters of 8 taps, 69 x 60 nt 6.6 / 10.4, 699 x 60 nt 41 / 17; of 4 taps, 4076 x
    // 20 nt 71 / 39. Of 3758 calls of 4 to 64 taps, 20 to 2000 nt, 1 to 64 models of 1 to 16 filters, 37 of those it takes are more than 5 %
    // slower than the scan kernel + head, by at most 9 us.
    return m >= 1 && m <= 64 && nfilter >= 1 && nfilter <= MUT_F && hidden <= 64 && N * nmodel * m <= 6000000 && nregion < ((size_t)1 << 31) && nmodel <= 65535 &&
           (nmodel == 1 || nregion * nmodel <= 2048) &&
           (ptype == DBK_PT_MAX || ptype == DBK_PT_AVG || ptype == DBK_PT_ALL);
}

int dbk_predict_small(dbk_stream_t stream, const float* W, const float* bias, size_t m, size_t nmodel, size_t nfilter, const uint8_t* X, size_t N,
                      const uint32_t* regions, size_t nregion, int ptype, size_t hidden, const float* W1, const float* b1, const float* W2,
                      const float* b2, const float* in_scale, int apply_logistic, float* scores)
{
    if (nregion == 0) { dbk::clear_error(); return 0; }
    DBK_CHECK(dbk_predict_small_takes(m, nmodel, nfilter, N, nregion, ptype, hidden), "NotImplementedError: dbk_predict_small takes up to 6e6 rows x models x taps, "
              "one model or up to 2048 regions x models, models of up to 16 filters of up to 64 taps and 64 hidden units");
    DBK_CHECK(W && bias && X && regions && W1 && b1 && scores, "ValueError: null pointer argument");
    DBK_CHECK(hidden == 0 || (W2 && b2), "ValueError: hidden layer requested but W2/b2 are null");
    small_args a;
    a.W = W; a.bias = bias; a.W1 = W1; a.b1 = b1; a.W2 = W2; a.b2 = b2; a.in_scale = in_scale; a.X = X; a.R = regions; a.N = N;
    a.m = (unsigned)m; a.nmodel = (unsigned)nmodel; a.nfilter = (unsigned)nfilter; a.k = (unsigned)(nfilter * (ptype == DBK_PT_ALL ? 2 : 1));
    a.hidden = (unsigned)hidden; a.ptype = ptype; a.logistic = apply_logistic; a.scores = scores;
    const bool wide = N > 64 * nregion;                             // 512 threads scan 128 rows at once
    auto kern = a.k <= 16 ? (wide ? k_predict_small<16, 512> : k_predict_small<16, 256>) : (wide ? k_predict_small<32, 512> : k_predict_small<32, 256>);
    const unsigned nt = wide ? 512u : 256u;
    hipLaunchKernelGGL(kern, dim3((unsigned)nregion, (unsigned)nmodel), dim3(nt), small_smem(m, nt), dbk::as_stream(stream), a);
    DBK_LAUNCH_OK();
}

int dbk_mutation_map_takes(size_t m, size_t nfilter, int ptype, size_t hidden)
{
    const size_t k = nfilter * (ptype == DBK_PT_ALL ? 2 : 1);
    return m >= 1 && m <= 64 && nfilter >= 1 && k <= MUT_MAXK && hidden <= MUT_MAXH &&
           (ptype == DBK_PT_MAX || ptype == DBK_PT_AVG || ptype == DBK_PT_ALL) && mut_fits(m, k);
}

int dbk_mutation_map(dbk_stream_t stream, const float* W, const float* bias, size_t m, size_t nfilter, const uint8_t* X, size_t N,
                     const uint32_t* regions, size_t nregion, size_t longest, int ptype, size_t hidden, const float* W1, const float* b1,
                     const float* W2, const float* b2, const float* in_scale, int apply_logistic, int strands, float* Z, float* map)
{
    DBK_CHECK(strands == 1 || (strands == 2 && nregion % 2 == 0), "ValueError: strands must be 1, or 2 with an even number of regions");
    DBK_CHECK(dbk_mutation_map_takes(m, nfilter, ptype, hidden), "NotImplementedError: the mutation map kernel does not take %zu filters of %zu taps with %zu hidden units and pooling %d",
              nfilter, m, hidden, ptype);
    if (nregion == 0) { dbk::clear_error(); return 0; }
    DBK_CHECK(W && bias && X && regions && W1 && b1 && Z && (longest == 0 || map), "ValueError: null pointer argument");
    DBK_CHECK(hidden == 0 || (W2 && b2), "ValueError: hidden layer requested but W2/b2 are null");
    // letters per workgroup: 16 where that still gives every CU six workgroups, 8 where it has two, else 4, as a workgroup's first scan of
    // its region costs less than an idle CU. Whole calls, us, 4 / 8 / 16: one sequence of 101 letters 72 / 77 / 88; 64 regions of 60-101, 24 taps
    // 111 / 104 / 114, 32 taps 145 / 144 / 163; 100 regions of 40-80, 8 taps 132 / 130 / 136; 256 regions of 101 227 / 209 / 200.
    // Up to 12 taps a letter costs little beside the first scan and the workgroups are to be on the GPU all at once: the next larger number where
    // they would not be (regions count as long as the longest). us, 4 / 8 / 16, 8 taps: 50 regions of 60-101 19 / 21 / 26, 64 on both strands 20 / 16 / 20, 128 of one strand
    // 30 / 27 / 28, 200 on both strands 37 / 31 / 28; 12 taps: 50 regions 20 / 23 / 30, 128 37 / 35 / 33.
    const size_t letters = longest > 0 ? longest : 1;
    const unsigned pos = m <= 12 ? (nregion * dbk::divup(letters, 8) > (m <= 8 ? 1920 : 1600) ? 16u : nregion * dbk::divup(letters, 4) > 1400 ? 8u : 4u)
                                 : (nregion * dbk::divup(letters, 16) >= 1536 ? 16u : nregion * dbk::divup(letters, 8) >= 512 ? 8u : 4u);
    const unsigned gy = dbk::divup(letters, pos);
    DBK_CHECK(nregion <= 0x7fffffffu && gy <= 65535u, "ValueError: too many regions (%zu) or letters per region (%zu) for one launch", nregion, longest);
    hipStream_t st = dbk::as_stream(stream);
    float* scratch = (float*)dbk::workspace((4 * N + nregion) * sizeof(float), st);
    DBK_CHECK(scratch != nullptr, "MemoryError: could not allocate %zu bytes of scratch (%s)", (4 * N + nregion) * sizeof(float), dbk::workspace_error());
    mut_args a;
    a.W = W; a.bias = bias; a.W1 = W1; a.b1 = b1; a.W2 = W2; a.b2 = b2; a.in_scale = in_scale;
    a.X = X; a.R = regions; a.N = N; a.P = nregion;
    a.m = (unsigned)m; a.F = (unsigned)nfilter; a.k = (unsigned)(nfilter * (ptype == DBK_PT_ALL ? 2 : 1)); a.hidden = (unsigned)hidden;
    a.ptype = ptype; a.logistic = apply_logistic; a.strands = strands;
    a.S = scratch; a.base = scratch + 4 * N;
    a.pos = pos;
    // (a lane takes a quarter of the m rows)
    auto pick = [&](auto spills) {
        constexpr bool S = decltype(spills)::value;
        return m <= 4 ? k_mutation_scores<1, S> : m <= 8 ? k_mutation_scores<2, S> : m <= 12 ? k_mutation_scores<3, S> : m <= 16 ? k_mutation_scores<4, S> : m <= 24 ? k_mutation_scores<6, S> : k_mutation_scores<8, S>;
    };
    auto kern = strands == 1 ? pick(std::true_type{}) : pick(std::false_type{});
    const size_t smem = mut_smem(pos, m, a.k, hidden);
    if (smem > 65536) DBK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
    hipLaunchKernelGGL(kern, dim3((unsigned)nregion, gy), dim3(MUT_NT), smem, st, a);
    hipLaunchKernelGGL(k_mutation_map, dim3((unsigned)(nregion / strands)), dim3(256), 0, st, regions, (unsigned)(m - 1), strands, X,
                       (const float*)a.S, (const float*)a.base, Z, map);
    DBK_LAUNCH_OK();
}

int dbk_gradient_map_takes(size_t m, size_t nfilter, size_t shortest, size_t longest, int ptype, size_t hidden)
{
    // One workgroup per sequence: a long one would keep it busy where the layer-by-layer kernels fill the chip. (An empty region
    // - no letters and filters of one tap - has no rows of its own: the layers say what it gives.)
    return m >= 1 && m <= 64 && nfilter >= 1 && nfilter <= MUT_F && hidden <= 64 && shortest + m > 1 && longest + m - 1 <= GRAD_MAXROWS &&
           (ptype == DBK_PT_MAX || ptype == DBK_PT_AVG || ptype == DBK_PT_ALL) && grad_smem(m, (unsigned)(longest + m - 1)) <= 65536;
}

int dbk_gradient_map(dbk_stream_t stream, const float* W, const float* bias, size_t m, size_t nfilter, const uint8_t* text, const uint32_t* offsets,
                     size_t nseq, size_t shortest, size_t longest, int ptype, size_t hidden, const float* W1, const float* b1, const float* W2,
                     const float* b2, const float* in_scale, int apply_logistic, int strands, float* Z, float* map, uint8_t* letters)
{
    DBK_CHECK(strands == 1 || strands == 2, "ValueError: strands must be 1 or 2");
    DBK_CHECK(dbk_gradient_map_takes(m, nfilter, shortest, longest, ptype, hidden), "NotImplementedError: the gradient map kernel does not take %zu filters of "
              "%zu taps with %zu hidden units, pooling %d and sequences of %zu to %zu letters", nfilter, m, hidden, ptype, shortest, longest);
    if (nseq == 0) { dbk::clear_error(); return 0; }
    DBK_CHECK(nseq <= 0x7fffffffu, "ValueError: too many sequences (%zu) for one launch", nseq);
    DBK_CHECK(W && bias && offsets && W1 && b1 && Z && (longest == 0 || (text && map && letters)), "ValueError: null pointer argument");
    DBK_CHECK(hidden == 0 || (W2 && b2), "ValueError: hidden layer requested but W2/b2 are null");
    grad_args a;
    a.W = W; a.bias = bias; a.W1 = W1; a.b1 = b1; a.W2 = W2; a.b2 = b2; a.in_scale = in_scale; a.text = text; a.offsets = offsets;
    a.m = (unsigned)m; a.F = (unsigned)nfilter; a.k = (unsigned)(nfilter * (ptype == DBK_PT_ALL ? 2 : 1)); a.hidden = (unsigned)hidden;
    a.rows_max = (unsigned)(longest + m - 1); a.ptype = ptype; a.logistic = apply_logistic; a.strands = strands;
    a.Z = Z; a.map = map; a.letters = letters;
    hipLaunchKernelGGL(k_gradient_map, dim3((unsigned)nseq), dim3(256), grad_smem(m, a.rows_max), dbk::as_stream(stream), a);
    DBK_LAUNCH_OK();
}

int dbk_gather_maps(dbk_stream_t stream, int dtype, const uint32_t* regions, size_t nregion, size_t padding, int strands, const void* Z,
                    const void* dX, void* map)
{
    DBK_DTYPE_OK(dtype);
    DBK_CHECK(strands == 1 || (strands == 2 && nregion % 2 == 0), "ValueError: strands must be 1, or 2 with an even number of regions");
    if (nregion == 0) { dbk::clear_error(); return 0; }
    DBK_CHECK(regions && Z && dX && map, "ValueError: null pointer argument");
    const dim3 grid((unsigned)(nregion / strands));
    if (dtype == DBK_F32)
        hipLaunchKernelGGL((k_gather_maps<float, float4>), grid, dim3(256), 0, dbk::as_stream(stream), regions, (unsigned)padding, strands,
                           (const float*)Z, (const float4*)dX, (float4*)map);
    else
        hipLaunchKernelGGL((k_gather_maps<double, double4>), grid, dim3(256), 0, dbk::as_stream(stream), regions, (unsigned)padding, strands,
                           (const double*)Z, (const double4*)dX, (double4*)map);
    DBK_LAUNCH_OK();
}

}  // extern "C"
