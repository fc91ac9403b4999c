// Fused motif scan + bias + ReLU + region pooling, forward and backward, general path.
//
// The (N, F) activation map is never written: a workgroup owns a tile of 64 filters (one lane per
// filter) and walks whole regions, each wave scanning 16 positions at a time in registers and
// folding them straight into the region's running max / argmax / sum. This path takes any filter
// length that fits in LDS, any region table and every letter code; the kernel of scanpool_digits.hip is the fast path
// for bulk scoring and leaves weights it cannot express to a launch of this file behind it.
//
// Backward: the max part is 1-sparse (one position per region and filter), the average part is
// dense and needs the forward recomputed for the ReLU mask. Both accumulate into per-wave private
// [tap][channel][filter] tables in LDS (a lane only ever touches its own filter column, so no
// atomics), the workgroup folds its waves in a fixed order into one slab in HBM, and a second
// kernel sums the slabs in a fixed tree: bit-reproducible gradients.
//
// Reference chain being fused: kangaroo/_ext/corr1ord.py:97-138, deepity/std/elemwise.py:71-82,162-180,
// kangaroo/_ext/poolrgn.py:56-82,153-180 with kernels corr1ord.cuh:139-157, poolrgn.cuh:44-160,
// poolrgn_bprop.cuh:45-127, corr1ord_bprop.cuh:91-137.
#include "dbk_common.h"
#include "scan_common.h"
#include <algorithm>

namespace dbk_scanpool_general {

using namespace dbk_scan;

constexpr unsigned XCH_SUBS = 4;          // sub-chunks of PSUB positions per wave and staging round

// A workgroup's place in its launch: (x, y) of a grid of gx by gy. The kernels of a training step take it as an
// argument instead of reading blockIdx / gridDim, so that one launch can hold the grids of several model groups.
struct wg_t { unsigned x, y, gx, gy; };
__device__ __forceinline__ wg_t this_wg() { return wg_t{blockIdx.x, blockIdx.y, gridDim.x, gridDim.y}; }

// Scans PSUB positions starting at chunk-relative p0 for this lane's filter.
__device__ __forceinline__ void scan16(const float* __restrict__ lut, const uint8_t* __restrict__ xl, unsigned m,
                                       unsigned p0, unsigned lane, float acc[PSUB])
{
#pragma unroll
    for (int p = 0; p < PSUB; ++p) acc[p] = 0.0f;
    for (unsigned j = 0; j < m; ++j) {
        const float* row = lut + (size_t)j * NL * FT + lane;
        const uint8_t* xs = xl + p0 + j;
#pragma unroll
        for (int p = 0; p < PSUB; ++p) acc[p] += row[(unsigned)xs[p] * FT];
    }
}

// MT > 0: filters of at most MT taps, letters held in scalar registers (scan16_window); MT == 0: any length.
template <int PT, bool WANT_ARGMAX, int MT>
__device__ __forceinline__ void scanpool_fprop_body(const wg_t wg, const float* __restrict__ W, const float* __restrict__ bias,
                                                    unsigned m, unsigned F, const uint8_t* __restrict__ X, size_t N,
                                                    const uint32_t* __restrict__ R, size_t P,
                                                    float* __restrict__ pooled, uint32_t* __restrict__ argmax,
                                                    unsigned long long* __restrict__ act)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const unsigned nw = blockDim.x >> 6;
    const unsigned chunk = nw * XCH_SUBS * PSUB;
    // up to 16 taps: the lane's filter weights live in register planes and the scan needs no table in LDS
    // (measured: 7.2 vs 9.1 us on a 128-sequence batch of width 16; with 24 taps the planes take 144 registers,
    // a CU holds two workgroups instead of three and the LDS table is the faster choice: 19.5 vs 21.7 us)
    constexpr bool PLANES = MT == 8 || MT == 16;
    constexpr int PMT = PLANES ? MT : 8;
    float* lut = reinterpret_cast<float*>(smem);
    float* red = lut + (PLANES ? 0 : (size_t)(MT ? MT : m) * NL * FT);   // [nw][3][FT]: max, index, sum
    uint8_t* xl = reinterpret_cast<uint8_t*>(red + (size_t)nw * 3 * FT);

    const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned f0 = wg.y * FT, f = f0 + lane;
    const size_t n = N + 1 >= (size_t)m + 1 ? N - m + 1 : 0;    // rows the scan defines; later rows are relu(bias)
    grad_planes<PMT> planes;
    if constexpr (PLANES) weight_planes_load<PMT>(planes, W, m, F, f);
    else build_letter_table(lut, W, m, F, f0, MT);
    const float bf = f < F ? bias[f] : 0.0f;

    for (size_t r = wg.x; r < P; r += wg.gx) {
        const size_t a = R[2 * r], b = R[2 * r + 1];
        float mx = -1.0f, sum = 0.0f;
        size_t xi = a;
        for (size_t c0 = a; c0 < b; c0 += chunk) {
            const unsigned rows = (unsigned)((b - c0) < chunk ? (b - c0) : chunk);
            __syncthreads();
            stage(xl, X, N, c0, MT ? window_span<MT ? MT : 1>(rows) : rows + m - 1);
            __syncthreads();
#pragma unroll 1
            for (unsigned s = 0; s < XCH_SUBS; ++s) {
                const unsigned p0 = (s * nw + wave) * PSUB;
                if (p0 >= rows) break;
                float acc[PSUB];
                if constexpr (PLANES) {
                    unsigned wq[window<PMT>::words];
                    load_window<PMT>(xl, p0, wq);
                    scan16_planes<PMT>(planes, wq, acc);
                } else if (MT) {
                    unsigned wq[window<MT ? MT : 1>::words];
                    load_window<MT ? MT : 1>(xl, p0, wq);
                    scan16_window<MT ? MT : 1>(lut, wq, lane, acc);
                } else {
                    scan16(lut, xl, m, p0, lane, acc);
                }
                if (act) {
                    // which rectifiers are open, for the backward pass: one 64-bit lane mask per (row, filter tile);
                    // lane p of the wave stores row p's
                    unsigned long long mine = 0;
#pragma unroll
                    for (int p = 0; p < PSUB; ++p) {
                        const size_t i = c0 + p0 + p;
                        const unsigned long long open = __ballot(((i < n ? acc[p] : 0.0f) + bf) > 0.0f);
                        if (lane == (unsigned)p) mine = open;
                    }
                    if (lane < (unsigned)PSUB && p0 + lane < rows) act[(c0 + p0 + lane) * wg.gy + wg.y] = mine;
                }
#pragma unroll
                for (int p = 0; p < PSUB; ++p) {
                    const size_t i = c0 + p0 + p;
                    if (p0 + p < rows) {
                        float z = (i < n ? acc[p] : 0.0f) + bf;
                        z = z > 0.0f ? z : 0.0f;
                        if (PT != DBK_PT_AVG) { if (z > mx) { mx = z; xi = i; } }
                        if (PT != DBK_PT_MAX) sum += z;
                    }
                }
            }
        }
        // fold the waves: larger value wins, equal values keep the earlier row
        red[(wave * 3 + 0) * FT + lane] = mx;
        red[(wave * 3 + 1) * FT + lane] = __uint_as_float((unsigned)(xi - a));
        red[(wave * 3 + 2) * FT + lane] = sum;
        __syncthreads();
        if (wave == 0 && f < F) {
            float bm = red[lane];
            unsigned bi = __float_as_uint(red[FT + lane]);
            float bs = red[2 * FT + lane];
            for (unsigned w = 1; w < nw; ++w) {
                float vm = red[(w * 3 + 0) * FT + lane];
                unsigned vi = __float_as_uint(red[(w * 3 + 1) * FT + lane]);
                if (vm > bm || (vm == bm && vi < bi)) { bm = vm; bi = vi; }
                bs += red[(w * 3 + 2) * FT + lane];
            }
            const size_t j = r * F + f;
            const float cnt = (float)(b - a);
            bm = bm > 0.0f ? bm : 0.0f;                          // only an empty region gets here with bm < 0
            if (PT == DBK_PT_MAX) pooled[j] = bm;
            else if (PT == DBK_PT_AVG) pooled[j] = bs / cnt;
            else { pooled[2 * j] = bm; pooled[2 * j + 1] = bs / cnt; }
            if (WANT_ARGMAX && PT != DBK_PT_AVG) argmax[j] = (uint32_t)((a + bi) * F + f);
        }
        __syncthreads();                                         // red[] is reused by the next region
    }
}

template <int PT, bool WANT_ARGMAX, int MT>
__global__ __launch_bounds__(256) void scanpool_fprop_kernel(const float* __restrict__ W, const float* __restrict__ bias,
                                                             unsigned m, unsigned F, const uint8_t* __restrict__ X, size_t N,
                                                             const uint32_t* __restrict__ R, size_t P,
                                                             float* __restrict__ pooled, uint32_t* __restrict__ argmax,
                                                             unsigned long long* __restrict__ act)
{
    scanpool_fprop_body<PT, WANT_ARGMAX, MT>(this_wg(), W, bias, m, F, X, N, R, P, pooled, argmax, act);
}

// The same forward pass with four filters per lane, for batches of many regions (filters of 17-24 taps).
//
// The kernel above spends one 4-byte LDS read per (position, tap, filter): a wave's read moves 256 bytes and the
// LDS delivers ~104 B/clk/CU of those, which is what bounds it once the GPU is full. Here a lane owns the four
// filters l, l+16, l+32, l+48 of the tile and the table row is laid out [16 lanes][4 filters], so the 16 lanes
// of a quarter wave read one aligned 256-byte line with ds_read_b128 (~216 B/clk/CU), and the four quarters of
// the wave work on four consecutive windows of 16 positions. A wave therefore takes 64 positions of ONE region
// at a time and the four waves of a workgroup walk four different regions: no workgroup barrier after the
// table is built. The letters of a quarter's window sit in ten vector registers (they differ between the
// quarters); one bit-field extract and one address add per letter serve up to 16 (position, tap) reads.
// Per position the taps are added in ascending order, as everywhere else: maxima and argmax are the bits of
// the kernel above; averages add the same rectified values in another order (quarter by quarter).
constexpr unsigned WIDE_SPAN = 4 * PSUB;                          // positions per wave and round

template <int PT, bool WANT_ARGMAX, int MT>
__device__ __forceinline__ void scanpool_fprop_wide_body(const wg_t wg, const float* __restrict__ W, const float* __restrict__ bias,
                                                         unsigned m, unsigned F, const uint8_t* __restrict__ X, size_t N,
                                                         const uint32_t* __restrict__ R, size_t P,
                                                         float* __restrict__ pooled, uint32_t* __restrict__ argmax,
                                                         unsigned long long* __restrict__ act)
{
    extern __shared__ __align__(16) unsigned char smem[];
    constexpr unsigned NWORD = wide_shape<MT>::words, XB = wide_shape<MT>::xbytes;
    const unsigned nw = blockDim.x >> 6;
    float* lut = reinterpret_cast<float*>(smem);                   // [MT*NL][16][4]
    // the wave's index, region bounds and loop control are wave-uniform: kept in scalar registers
    const unsigned lane = threadIdx.x & 63, wave = (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const unsigned qd = lane >> 4, l = lane & 15;
    uint8_t* xw = smem + (size_t)MT * NL * FT * sizeof(float) + (size_t)wave * XB;   // this wave's letters
    const unsigned f0 = wg.y * FT;
    const size_t n = N + 1 >= (size_t)m + 1 ? N - m + 1 : 0;    // rows the scan defines; later rows are relu(bias)
    build_letter_table<float, true>(lut, W, m, F, f0, MT);
    float bf[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) bf[c] = f0 + c * 16 + l < F ? bias[f0 + c * 16 + l] : 0.0f;
    __syncthreads();
    const float4* lut4 = reinterpret_cast<const float4*>(lut) + l;

    for (size_t r = (size_t)wg.x * nw + wave; r < P; r += (size_t)wg.gx * nw) {
        const size_t a = (unsigned)__builtin_amdgcn_readfirstlane((int)R[2 * r]), b = (unsigned)__builtin_amdgcn_readfirstlane((int)R[2 * r + 1]);
        float mx[4] = {-1.0f, -1.0f, -1.0f, -1.0f}, sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        unsigned xi[4] = {0u, 0u, 0u, 0u};                        // row of the maximum, relative to a
        for (size_t c0 = a; c0 < b; c0 += WIDE_SPAN) {
            const unsigned rows = (unsigned)((b - c0) < WIDE_SPAN ? (b - c0) : WIDE_SPAN);
            // ---- the round's letters, then this quarter's window: 16 positions x MT taps x 4 filters
            unsigned wq[NWORD];
            wide_stage<MT>(xw, X, N, c0, lane, wq);
            float4 acc[PSUB];
            scan16_wide<MT>(lut4, wq, acc);
            // ---- bias, rectifier, pooling; optionally the activity masks of the 64 rows
            const unsigned pq = PSUB * qd;                         // first position of this quarter's window
            unsigned long long mine = 0ull;
#pragma unroll
            for (int p = 0; p < PSUB; ++p) {
                const size_t i = c0 + pq + p;
                const bool defined = i < n;
                float z[4] = {acc[p].x, acc[p].y, acc[p].z, acc[p].w};
#pragma unroll
                for (int c = 0; c < 4; ++c) z[c] = (defined ? z[c] : 0.0f) + bf[c];
                if (act) {
                    // ballot c holds, for each quarter, 16 bits: filters 16c .. 16c+15 of that quarter's row p
                    unsigned lo = 0u, hi = 0u;
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const unsigned long long open = __ballot(z[c] > 0.0f);
                        const unsigned part = (unsigned)(open >> (16u * qd)) & 0xffffu;
                        if (c < 2) lo |= part << (16 * c);
                        else hi |= part << (16 * (c - 2));
                    }
                    if (l == (unsigned)p) mine = ((unsigned long long)hi << 32) | lo;
                }
                if (pq + p < rows) {
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const float zr = z[c] > 0.0f ? z[c] : 0.0f;
                        if (PT != DBK_PT_AVG) { if (zr > mx[c]) { mx[c] = zr; xi[c] = (unsigned)(i - a); } }
                        if (PT != DBK_PT_MAX) sum[c] += zr;
                    }
                }
            }
            if (act && pq + l < rows) act[(c0 + pq + l) * wg.gy + wg.y] = mine;
        }
        // ---- fold the four quarters: larger value wins, equal values keep the earlier row
#pragma unroll
        for (int c = 0; c < 4; ++c) {
#pragma unroll
            for (int d = 16; d <= 32; d <<= 1) {
                const float vm = __shfl_xor(mx[c], d, 64);
                const unsigned vi = (unsigned)__shfl_xor((int)xi[c], d, 64);
                const float vs = __shfl_xor(sum[c], d, 64);
                if (vm > mx[c] || (vm == mx[c] && vi < xi[c])) { mx[c] = vm; xi[c] = vi; }
                sum[c] += vs;
            }
        }
        if (qd == 0) {
            const float cnt = (float)(b - a);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const unsigned f = f0 + c * 16 + l;
                if (f >= F) continue;
                const size_t j = r * F + f;
                const float bm = mx[c] > 0.0f ? mx[c] : 0.0f;      // only an empty region gets here with a negative maximum
                if (PT == DBK_PT_MAX) pooled[j] = bm;
                else if (PT == DBK_PT_AVG) pooled[j] = sum[c] / cnt;
                else { pooled[2 * j] = bm; pooled[2 * j + 1] = sum[c] / cnt; }
                if (WANT_ARGMAX && PT != DBK_PT_AVG) argmax[j] = (uint32_t)((a + xi[c]) * F + f);
            }
        }
    }
}

template <int PT, bool WANT_ARGMAX, int MT>
__global__ __launch_bounds__(256) void scanpool_fprop_wide_kernel(const float* __restrict__ W, const float* __restrict__ bias,
                                                                  unsigned m, unsigned F, const uint8_t* __restrict__ X, size_t N,
                                                                  const uint32_t* __restrict__ R, size_t P,
                                                                  float* __restrict__ pooled, uint32_t* __restrict__ argmax,
                                                                  unsigned long long* __restrict__ act)
{
    scanpool_fprop_wide_body<PT, WANT_ARGMAX, MT>(this_wg(), W, bias, m, F, X, N, R, P, pooled, argmax, act);
}

}  // namespace dbk_scanpool_general

#include "scan_mfma.h"

namespace dbk_scanpool_general {

// What the bulk kernel (scanpool_digits.hip) leaves out: it writes a flag per 32 filters, and this launch, behind it on the
// stream, takes the 64-filter tiles of which one asks for it: finite weights on the matrix cores, in three bf16 pieces whatever
// their sizes; infinite and undefined ones, which a product would spread over windows that do not hold them, one by one from the
// letter table. The workgroups are dealt over the tiles that are left, not over all, so that a few of many have the whole GPU.
// Where nothing is left the launch costs 4-5 us. Measured, 20 000 x 500 letters x 512 filters, ms with nothing, one tile of eight and all
// tiles left: max pooling of 24 taps 0.98, 1.21, 2.36, of 8 taps 0.54, 0.66, 1.24, of 32 taps 1.11, 1.39, -; average of 24 taps 1.32, 1.53, 2.31.
// (One lookup per tap from the letter table, by a grid of all tiles of which most workgroups left at once: 24 taps 7.4 and 9.2, 8 taps 2.8 and 4.1.)
// (the form with its table in LDS: the register planes of 16 taps are pinned beyond the registers of three waves per SIMD)
constexpr int left_lookup_taps(int ks) { return ks == 8 ? 32 : 24; }
template <int PT, bool WANT_ARGMAX, int KS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 3))) void scanpool_fprop_left_kernel(const float* __restrict__ W, const float* __restrict__ bias,
                                                                  unsigned m, unsigned F, const uint8_t* __restrict__ X, size_t N,
                                                                  const uint32_t* __restrict__ R, size_t P,
                                                                  float* __restrict__ pooled, uint32_t* __restrict__ argmax,
                                                                  const unsigned* __restrict__ flags, unsigned ftiles)
{
    const unsigned lane = threadIdx.x & 63u;
    auto asked = [&](unsigned t0) -> unsigned long long {
        const unsigned t = t0 + lane;
        return __ballot(t < ftiles && ((flags[2 * t] | flags[2 * t + 1]) & (TILE_LEFT | TILE_NOT_FINITE)) != 0u);
    };
    unsigned left = 0u;
    for (unsigned t0 = 0; t0 < ftiles; t0 += 64u) left += (unsigned)__popcll(asked(t0));
    if (left == 0u) return;
    const unsigned gx = gridDim.x / left;                         // workgroups per tile (the grid has no fewer than tiles)
    if (blockIdx.x >= left * gx) return;
    unsigned t0 = 0u, nth = blockIdx.x % left;                     // the nth of the tiles that are left
    unsigned long long who = asked(0u);
    while ((unsigned)__popcll(who) <= nth) { nth -= (unsigned)__popcll(who); t0 += 64u; who = asked(t0); }
    for (; nth != 0u; --nth) who &= who - 1ull;
    const unsigned tile = t0 + (unsigned)__builtin_ctzll(who);
    const wg_t wg = {blockIdx.x / left, tile, gx, ftiles};
    if (((flags[2 * tile] | flags[2 * tile + 1]) & (TILE_INFINITE | TILE_NOT_FINITE)) != 0u)
        scanpool_fprop_body<PT, WANT_ARGMAX, left_lookup_taps(KS)>(wg, W, bias, m, F, X, N, R, P, pooled, argmax, nullptr);
    else
        scanpool_fprop_mfma_body<PT, WANT_ARGMAX, false, KS, true>(wg, W, bias, m, F, X, N, R, P, pooled, argmax, nullptr);
}

// ---------------------------------------------------------------------------------------------
// backward
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ void add_tap(float* cell, unsigned l, float g, float gq)
{
    if (l < 4u) {
        cell[l * FT] += g;
    } else if (l == 4u) {
        cell[0 * FT] += gq;
        cell[1 * FT] += gq;
        cell[2 * FT] += gq;
        cell[3 * FT] += gq;
    }
}

template <int PT>
__global__ __launch_bounds__(256) void scanpool_bprop_kernel(const float* __restrict__ W, const float* __restrict__ bias,
                                                             unsigned m, unsigned F, const uint8_t* __restrict__ X, size_t N,
                                                             const uint32_t* __restrict__ R, size_t P,
                                                             const float* __restrict__ pooled, const uint32_t* __restrict__ argmax,
                                                             const float* __restrict__ dpooled,
                                                             float* __restrict__ slabs, size_t stride)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const unsigned nw = blockDim.x >> 6;
    const unsigned chunk = nw * XCH_SUBS * PSUB;
    const unsigned tab = m * 4 * FT;
    float* lut = reinterpret_cast<float*>(smem);                   // only used when the average part is present
    float* acc_tab = lut + (PT == DBK_PT_MAX ? 0 : (size_t)m * NL * FT);
    float* dbacc = acc_tab + (size_t)nw * tab;                     // [nw][FT]
    uint8_t* xl = reinterpret_cast<uint8_t*>(dbacc + (size_t)nw * FT);

    const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned f0 = blockIdx.y * FT, f = f0 + lane;
    const size_t n = N + 1 >= (size_t)m + 1 ? N - m + 1 : 0;
    if (PT != DBK_PT_MAX) build_letter_table(lut, W, m, F, f0);
    for (unsigned e = threadIdx.x; e < nw * tab + nw * FT; e += blockDim.x) acc_tab[e] = 0.0f;
    const float bf = f < F ? bias[f] : 0.0f;
    float* mine = acc_tab + (size_t)wave * tab + lane;
    float db = 0.0f;
    __syncthreads();

    for (size_t r = blockIdx.x; r < P; r += gridDim.x) {
        const size_t a = R[2 * r], b = R[2 * r + 1];
        const size_t j0 = r * F + f;
        // ---- max part: one position per (region, filter); wave (r mod nw) does it
        if (PT != DBK_PT_AVG && (r % nw) == wave && f < F) {
            const float pv = PT == DBK_PT_MAX ? pooled[j0] : pooled[2 * j0];
            const float g = (pv > 0.0f) ? (PT == DBK_PT_MAX ? dpooled[j0] : dpooled[2 * j0]) : 0.0f;
            if (g != 0.0f) {
                const size_t i = argmax[j0] / F;
                db += g;
                if (i < n) {
                    const float gq = g * 0.25f;
                    for (unsigned j = 0; j < m; ++j) add_tap(mine + (size_t)j * 4 * FT, letter_of(X[i + j]), g, gq);
                }
            }
        }
        // ---- average part: recompute the map, mask by ReLU, spread davg/count
        if (PT != DBK_PT_MAX) {
            const float gavg = f < F ? (PT == DBK_PT_AVG ? dpooled[j0] : dpooled[2 * j0 + 1]) / (float)(b - a) : 0.0f;
            for (size_t c0 = a; c0 < b; c0 += chunk) {
                const unsigned rows = (unsigned)((b - c0) < chunk ? (b - c0) : chunk);
                __syncthreads();
                stage(xl, X, N, c0, rows + m - 1);
                __syncthreads();
    #pragma unroll 1
            for (unsigned s = 0; s < XCH_SUBS; ++s) {
                    const unsigned p0 = (s * nw + wave) * PSUB;
                    if (p0 >= rows) break;
                    float acc[PSUB];
                    scan16(lut, xl, m, p0, lane, acc);
#pragma unroll
                    for (int p = 0; p < PSUB; ++p) {
                        const size_t i = c0 + p0 + p;
                        if (p0 + p < rows) {
                            const float z = (i < n ? acc[p] : 0.0f) + bf;
                            const float g = z > 0.0f ? gavg : 0.0f;
                            db += g;
                            if (i < n) {
                                const float gq = g * 0.25f;
                                for (unsigned j = 0; j < m; ++j) add_tap(mine + (size_t)j * 4 * FT, xl[p0 + p + j], g, gq);
                            }
                        }
                    }
                }
            }
        }
    }
    dbacc[wave * FT + lane] = db;
    __syncthreads();
    float* outW = slabs + (size_t)blockIdx.x * stride;
    for (unsigned e = threadIdx.x; e < tab; e += blockDim.x) {
        float s = acc_tab[e];
        for (unsigned w = 1; w < nw; ++w) s += acc_tab[(size_t)w * tab + e];
        const unsigned row = e / FT, fl = e % FT;
        if (f0 + fl < F) outW[(size_t)row * F + f0 + fl] = s;
    }
    if (wave == 0 && f < F) {
        float s = dbacc[lane];
        for (unsigned w = 1; w < nw; ++w) s += dbacc[w * FT + lane];
        outW[(size_t)4 * m * F + f] = s;
    }
}

// For up to four positions i_u with gradients g_u: adds g_u at (tap j, letter of X[i_u+j]) for j < m into
// this lane's column of a [tap][channel][FT] table. Taps go eight at a time: the letters of all four
// positions are loaded first (32 independent global loads in flight), then each position's eight cells
// are read, updated and written (distinct taps are distinct cells), positions in ascending order.
// Adds g[u] at the MT-letter windows starting at pos[u], u = 0..3, into this lane's private column of the
// LDS slab, laid out [tap][A, C, G, T, mean-of-four][filter]: every letter, "mean of the four" included,
// touches exactly one cell, so a batch of eight taps is one LDS round trip (the mean row is spread over
// the four channels when the slab is written out).
constexpr int SPARSE_ROWS = 5;
template <int MT>
__device__ __forceinline__ void add_positions4(float* mine, const uint8_t* __restrict__ X, size_t N, const size_t (&pos)[4],
                                               const float (&g)[4], const bool (&on)[4], unsigned m)
{
    // The letters of all four windows first, so that their loads are in flight together: a window of MT
    // letters starting at any byte is MT/4 + 1 aligned 32-bit words shifted into place; a word is only
    // fetched if it starts before the end of the stream.
    static_assert(MT % 8 == 0, "windows are taken eight letters at a time");
    constexpr int NW = MT / 4 + 1;
    unsigned w[4][NW], sh[4];
    const uintptr_t xend = reinterpret_cast<uintptr_t>(X) + N;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const uintptr_t addr = reinterpret_cast<uintptr_t>(X) + pos[u];
        const uintptr_t base = addr & ~(uintptr_t)3;
        sh[u] = (unsigned)(addr & 3);
#pragma unroll
        for (int t = 0; t < NW; ++t)
            w[u][t] = (on[u] && base + 4 * t < xend) ? *reinterpret_cast<const unsigned*>(base + 4 * t) : 0xffffffffu;
    }
#pragma unroll
    for (unsigned j0 = 0; j0 < (unsigned)MT; j0 += 8) {
        if (j0 >= m) break;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const unsigned lo = __builtin_amdgcn_alignbyte(w[u][j0 / 4 + 1], w[u][j0 / 4], sh[u]);
            const unsigned hi = __builtin_amdgcn_alignbyte(w[u][j0 / 4 + 2], w[u][j0 / 4 + 1], sh[u]);     // j0/4 + 2 <= MT/4
            unsigned l[8];
#pragma unroll
            for (unsigned t = 0; t < 8; ++t) {
                const unsigned code = ((t < 4 ? lo : hi) >> ((t & 3) * 8)) & 0xffu;
                l[t] = (on[u] && j0 + t < m) ? letter_of(code) : 5u;
            }
            float v[8];
#pragma unroll
            for (unsigned t = 0; t < 8; ++t) v[t] = l[t] < 5u ? mine[((j0 + t) * SPARSE_ROWS + l[t]) * FT] : 0.0f;
#pragma unroll
            for (unsigned t = 0; t < 8; ++t)
                if (l[t] < 5u) mine[((j0 + t) * SPARSE_ROWS + l[t]) * FT] = v[t] + g[u];
        }
    }
}
// One wave; in a launch of wider workgroups only the first wave of a workgroup may enter.
// The end of a backward workgroup: its four waves hold their sums of the filter gradient in registers (lane = filter)
// and add them up in wave order into the workgroup's slab. Eight taps per round: every wave stores its 8 x 4 sums per
// lane side by side in LDS (128 KB would be needed for all 24 taps of four waves at once), then all 256 threads add
// the four copies of 8 elements each ((w0 + w1) + w2) + w3 and store them: two barriers per round and every LDS access of
// a round in flight together, where one wave after the other adding into one shared copy took four barriers and a
// dependent read-add-write per sum (measured on a calibration batch: 5.4 + 2.0 us of a 17.7 us workgroup; now 1.3).
constexpr int FOLD_TAPS = 8;
constexpr unsigned FOLD_ROUND = FOLD_TAPS * 4 * FT;              // floats of one wave's round
constexpr size_t FOLD_BYTES = (4 * (size_t)FOLD_ROUND + 4 * FT) * sizeof(float);   // four waves' rounds + their bias sums
template <int MT, typename V>
__device__ __forceinline__ void fold_waves_into_slab(unsigned char* smem_base, V value, float db, unsigned m, unsigned F, unsigned f0,
                                                     float* __restrict__ out)
{
    float* area = reinterpret_cast<float*>(smem_base);
    float* dbacc = area + 4 * FOLD_ROUND;
    const unsigned lane = threadIdx.x & 63, wave = (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), nw = blockDim.x >> 6;
#pragma unroll
    for (int t0 = 0; t0 < MT; t0 += FOLD_TAPS) {
        __syncthreads();                                           // whatever lay here, and the last round's sums, are no longer read
        if (t0 == 0) dbacc[wave * FT + lane] = db;
        float* mine = area + wave * FOLD_ROUND + lane;
#pragma unroll
        for (int j = 0; j < FOLD_TAPS; ++j)
#pragma unroll
            for (int c = 0; c < 4; ++c)
                if (t0 + j < MT) mine[(j * 4 + c) * FT] = value(t0 + j, c);
        __syncthreads();
#pragma unroll
        for (unsigned u = 0; u < FOLD_ROUND / 256; ++u) {
            const unsigned e = threadIdx.x + u * 256, row = (unsigned)t0 * 4 + e / FT, fl = e % FT;
            float v = area[e];
            for (unsigned w = 1; w < nw; ++w) v += area[w * FOLD_ROUND + e];
            if (row < 4 * m && f0 + fl < F) out[(size_t)row * F + f0 + fl] = v;
        }
    }
    if (wave == 0 && f0 + lane < F) {
        float t = dbacc[lane];
        for (unsigned w = 1; w < nw; ++w) t += dbacc[w * FT + lane];
        out[(size_t)4 * m * F + f0 + lane] = t;
    }
}

template <int PT, int MT>
__device__ __forceinline__ void scanpool_bprop_sparse_body(const wg_t wg, unsigned m, unsigned F, const uint8_t* __restrict__ X, size_t N,
                                                           size_t P, const float* __restrict__ pooled,
                                                           const uint32_t* __restrict__ argmax, const float* __restrict__ dpooled,
                                                           float* __restrict__ slabs, size_t stride)
{
    extern __shared__ __align__(16) unsigned char smem[];
    float* table = reinterpret_cast<float*>(smem);
    const unsigned lane = threadIdx.x;
    const unsigned f = wg.y * FT + lane;
    const size_t n = N + 1 >= (size_t)m + 1 ? N - m + 1 : 0;
    float* mine = table + lane;                                   // a lane only ever touches its own column: no barriers needed
    for (unsigned row = 0; row < SPARSE_ROWS * m; ++row) mine[row * FT] = 0.0f;
    float db = 0.0f;
    if (f < F) {
        const size_t gx = wg.gx;
        for (size_t r = wg.x; r < P; r += 4 * gx) {
            float g[4];
            size_t pos[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const size_t ru = r + u * gx;
                g[u] = 0.0f;
                pos[u] = 0;
                if (ru < P) {
                    const size_t j0 = ru * F + f;
                    const float pv = PT == DBK_PT_MAX ? pooled[j0] : pooled[2 * j0];
                    const float gd = PT == DBK_PT_MAX ? dpooled[j0] : dpooled[2 * j0];
                    pos[u] = argmax[j0] / F;
                    g[u] = pv > 0.0f ? gd : 0.0f;
                }
            }
            bool on[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (g[u] != 0.0f) db += g[u];
                on[u] = g[u] != 0.0f && pos[u] < n;
            }
            add_positions4<MT>(mine, X, N, pos, g, on, m);
        }
        float* out = slabs + (size_t)wg.x * stride;
        for (unsigned j = 0; j < m; ++j) {
            const float* tap = mine + (size_t)j * SPARSE_ROWS * FT;
            const float q = 0.25f * tap[4 * FT];
            float* o = out + (size_t)(4 * j) * F + f;
            o[0] = tap[0] + q;
            o[F] = tap[FT] + q;
            o[2 * (size_t)F] = tap[2 * FT] + q;
            o[3 * (size_t)F] = tap[3 * FT] + q;
        }
        out[(size_t)4 * m * F + f] = db;
    }
}

template <int PT, int MT>
__global__ __launch_bounds__(64) void scanpool_bprop_sparse_kernel(unsigned m, unsigned F, const uint8_t* __restrict__ X, size_t N,
                                                                   size_t P, const float* __restrict__ pooled,
                                                                   const uint32_t* __restrict__ argmax, const float* __restrict__ dpooled,
                                                                   float* __restrict__ slabs, size_t stride)
{
    scanpool_bprop_sparse_body<PT, MT>(this_wg(), m, F, X, N, P, pooled, argmax, dpooled, slabs, stride);
}

// Dense half of the backward pass (avg and max+avg pooling), filters of at most MT taps: every
// position of a region receives davg/count where the recomputed activation is positive. A lane keeps
// its filter's whole [tap][channel] gradient column in registers: the letter at a position is the
// same for all 64 lanes (lanes are filters), so it is read once into scalar registers, turned into
// four scalar weights (1 for the matching channel, 1/4 each for N, else 0) and applied as fused
// multiply-adds whose products are exact, i.e. one rounding per addition as in the reference's add.
template <int PT, int MT>
__global__ __launch_bounds__(256) void scanpool_bprop_dense_kernel(const float* __restrict__ W, const float* __restrict__ bias,
                                                                   unsigned m, unsigned F, const uint8_t* __restrict__ X, size_t N,
                                                                   const uint32_t* __restrict__ R, size_t P,
                                                                   const float* __restrict__ pooled, const uint32_t* __restrict__ argmax,
                                                                   const float* __restrict__ dpooled,
                                                                   float* __restrict__ slabs, size_t stride)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const unsigned nw = blockDim.x >> 6;
    const unsigned chunk = nw * XCH_SUBS * PSUB;
    float* lut = reinterpret_cast<float*>(smem);                   // [MT][NL][FT]; the memory is reused for the cross-wave fold at the end
    uint8_t* xl = reinterpret_cast<uint8_t*>(lut + (size_t)MT * NL * FT + (size_t)nw * FT);   // 4-byte aligned: everything before it is float

    const unsigned lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const unsigned f0 = blockIdx.y * FT, f = f0 + lane;
    const size_t n = N + 1 >= (size_t)m + 1 ? N - m + 1 : 0;
    build_letter_table(lut, W, m, F, f0, MT);
    const float bf = f < F ? bias[f] : 0.0f;
    float db = 0.0f;
    grad_planes<MT> planes;                                        // [letter][tap] accumulators in fixed registers
    planes.clear();

    for (size_t r = blockIdx.x; r < P; r += gridDim.x) {
        const size_t a = R[2 * r], b = R[2 * r + 1];
        const size_t j0 = r * F + f;
        const float gavg = f < F ? (PT == DBK_PT_AVG ? dpooled[j0] : dpooled[2 * j0 + 1]) / (float)(b - a) : 0.0f;
        // max+avg pooling: the maximum's gradient joins the average's at the winning row before the
        // rectifier, as it does in the unpooled gradient map of the layer-by-layer chain
        float gmax = 0.0f;
        size_t imax = ~(size_t)0;
        if (PT == DBK_PT_ALL && f < F && pooled[2 * j0] > 0.0f) { gmax = dpooled[2 * j0]; imax = argmax[j0] / F; }
        for (size_t c0 = a; c0 < b; c0 += chunk) {
            const unsigned rows = (unsigned)((b - c0) < chunk ? (b - c0) : chunk);
            __syncthreads();
            stage(xl, X, N, c0, window_span<MT>(rows));
            __syncthreads();
#pragma unroll 1
            for (unsigned s = 0; s < XCH_SUBS; ++s) {
                const unsigned p0 = (s * nw + wave) * PSUB;
                if (p0 >= rows) break;
                // letters of this sub-chunk's window, four per scalar register (letters past the region's
                // own window only ever meet zero table rows, g == 0 or taps >= m)
                unsigned wq[window<MT>::words];
                load_window<MT>(xl, p0, wq);
                float g[PSUB];
                scan16_window<MT>(lut, wq, lane, g);
#pragma unroll
                for (int p = 0; p < PSUB; ++p) {
                    const size_t i = c0 + p0 + p;
                    const float z = (i < n ? g[p] : 0.0f) + bf;
                    float gg = (p0 + p < rows && z > 0.0f) ? gavg : 0.0f;
                    if (PT == DBK_PT_ALL) gg += (p0 + p < rows && i == imax) ? gmax : 0.0f;
                    db += gg;
                    g[p] = i < n ? gg : 0.0f;                   // rows past the scan's end carry bias only
                }
                grad_planes_window<MT>(planes, wq, g);         // one add per (position, tap), the letter picks the plane
            }
        }
    }
    float aw[MT][4];
    grad_planes_read<MT>(planes, aw);
    // the waves' sums, added in wave order through the (now unused) letter table's memory, into the workgroup's slab
    fold_waves_into_slab<MT>(smem, [&](int j, int c) { return aw[j][c]; }, db, m, F, f0, slabs + (size_t)blockIdx.x * stride);
}

// Fixed-shape tree sum over slabs of nW + nB entries each: dW[e] += total (or = total with overwrite) for e < nW,
// dbias[e - nW] = total after that.
__global__ void reduce_slabs_kernel(float* __restrict__ dW, float* __restrict__ dbias, const float* __restrict__ slabs,
                                    size_t nW, size_t nB, unsigned nslab, bool overwrite)
{
    const size_t nelem = nW + nB;
    for (size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x; e < nelem; e += (size_t)gridDim.x * blockDim.x) {
        const float total = slab_sum(slabs, nelem, e, nslab);
        if (e < nW) dW[e] = overwrite ? total : dW[e] + total;
        else dbias[e - nW] = total;
    }
}

// The max-pooling gradient of short regions. It lands on one row per (region, filter): that row's letters are cut out of the
// region's letters held as one bit per (letter, position), from five ballots per chunk of 64 rows (wave-uniform, shifted in scalar
// registers), once per region. A wave walks whole regions; a lane keeps the 5 x MT sums of its filter in registers over all its
// regions (ascending), the waves fold them into the workgroup's slab as above. Deterministic.
template <int MT>
__device__ __forceinline__ void scanpool_bprop_bits_body(const wg_t wg, unsigned m, unsigned F, const uint8_t* __restrict__ X, size_t N,
                                                         const uint32_t* __restrict__ R, size_t P,
                                                         const float* __restrict__ pooled, const uint32_t* __restrict__ argmax,
                                                         const float* __restrict__ dpooled, float* __restrict__ slabs, size_t stride)
{
    extern __shared__ __align__(16) unsigned char smem[];
    const unsigned nw = blockDim.x >> 6;
    const unsigned lane = threadIdx.x & 63, wave = (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const unsigned f0 = wg.y * FT, f = f0 + lane;
    const size_t n = N + 1 >= (size_t)m + 1 ? N - m + 1 : 0;      // rows the scan defines; later rows carry bias only
    float acc[5][MT];
#pragma unroll
    for (int l = 0; l < 5; ++l)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[l][t] = 0.0f;
    float db = 0.0f;

    struct pooled_in { float pmax, dmax; unsigned arg; };
    auto load_pooled = [&](size_t r_) -> pooled_in {
        pooled_in q = { 0.0f, 0.0f, 0u };
        if (f < F && r_ < P) {
            const size_t j0 = r_ * F + f;
            q.pmax = pooled[j0]; q.dmax = dpooled[j0]; q.arg = argmax[j0];
        }
        return q;
    };
    auto bound = [&](size_t r_, unsigned which) -> size_t { return r_ < P ? (unsigned)__builtin_amdgcn_readfirstlane((int)R[2 * r_ + which]) : 0u; };
    struct raw { unsigned x0, x1; };                               // a chunk as loaded: two letters per lane
    auto load_chunk = [&](size_t c0) -> raw {
        raw w = { 254u, 254u };
        const size_t g0 = c0 + lane, g1 = g0 + 64;
        if (g0 < N) w.x0 = X[g0];
        if (lane < (unsigned)MT - 1 && g1 < N) w.x1 = X[g1];
        return w;
    };

    const size_t step = (size_t)wg.gx * nw;
    size_t r = (size_t)wg.x * nw + wave;
    size_t a = bound(r, 0), b = bound(r, 1), na = bound(r + step, 0), nb = bound(r + step, 1);
    size_t nna = bound(r + 2 * step, 0), nnb = bound(r + 2 * step, 1);
    pooled_in q = load_pooled(r), nq = load_pooled(r + step);
    size_t c0 = a;
    raw cur = r < P ? load_chunk(c0) : raw{ 254u, 254u };
    float gmax = 0.0f;
    size_t imax = ~(size_t)0;
    unsigned tm[5] = { 0u, 0u, 0u, 0u, 0u };                        // letters of the taps at the winning row: bit t of tm[l]
    while (r < P) {                                                // uniform over the wave
        // ---- the chunk after this one is requested before this one is worked on
        const bool last = c0 + 64 >= b;
        const size_t nc0 = last ? na : c0 + 64;
        const bool more = last ? r + step < P : true;
        raw nxt = { 254u, 254u };
        if (more) nxt = load_chunk(nc0);
        if (c0 == a) {
            gmax = 0.0f; imax = ~(size_t)0;
            if (q.pmax > 0.0f) { gmax = q.dmax; imax = q.arg / F; }
#pragma unroll
            for (int l = 0; l < 5; ++l) tm[l] = 0u;
        }
        // ---- one bit per (letter, position) of the chunk: positions c0 .. c0 + 63 and the MT - 1 behind them
        const unsigned v0 = letter_of(cur.x0), v1 = letter_of(cur.x1);
        unsigned long long L0[5], L1[5];
#pragma unroll
        for (int l = 0; l < 5; ++l) { L0[l] = __ballot(v0 == (unsigned)l); L1[l] = __ballot(v1 == (unsigned)l); }
        // ---- the winning row of this lane's filter, if it lies in the chunk: its taps' letters
        const bool here = imax >= c0 && imax - c0 < 64;
        const unsigned rel = here ? (unsigned)(imax - c0) : 0u;
        if (here) db += gmax;
        const bool counts = here && imax < n;
#pragma unroll
        for (int l = 0; l < 5; ++l) {
            const unsigned long long cut = rel == 0 ? L0[l] : (L0[l] >> rel) | (L1[l] << (64 - rel));
            tm[l] |= counts ? (unsigned)cut : 0u;                  // (MT <= 32 taps: the low word is all that is looked at)
        }
        // ---- on to the next chunk / region
        if (last) {
#pragma unroll
            for (int t = 0; t < MT; ++t) {
#pragma unroll
                for (int l = 0; l < 5; ++l) acc[l][t] = __builtin_fmaf(gmax, (float)((tm[l] >> t) & 1u), acc[l][t]);
            }
            r += step;
            a = na; b = nb; q = nq;
            na = nna; nb = nnb;
            nna = bound(r + 2 * step, 0); nnb = bound(r + 2 * step, 1);
            nq = load_pooled(r + step);
        }
        c0 = nc0;
        cur = nxt;
    }
    fold_waves_into_slab<MT>(smem, [&](int j, int c) { return acc[c][j] + 0.25f * acc[4][j]; }, db, m, F, f0, slabs + (size_t)wg.x * stride);
}

template <int MT>
__global__ __launch_bounds__(256) void scanpool_bprop_bits_kernel(unsigned m, unsigned F, const uint8_t* __restrict__ X, size_t N,
                                                                  const uint32_t* __restrict__ R, size_t P,
                                                                  const float* __restrict__ pooled, const uint32_t* __restrict__ argmax,
                                                                  const float* __restrict__ dpooled, float* __restrict__ slabs, size_t stride)
{
    scanpool_bprop_bits_body<MT>(this_wg(), m, F, X, N, R, P, pooled, argmax, dpooled, slabs, stride);
}

// The mask-driven backward of average (and max + average) pooling, counted on the matrix cores. At every row of a region
// whose rectifier is open the average-pooling gradient is the SAME number c = dpooled / rows, so the filter gradient needs
// no pass over the rows but counts:
//     dW[tap][letter][f] += c * #{rows of the region: open_f(row) and letter(row + tap) = letter}
// and the counts are a product of bits, letters (4m x rows) times open rows (rows x filters), which
// v_mfma_scale_f32_32x32x64_f8f6f4 forms 64 rows at a time and exactly: in its 4-bit format the bit pattern 0001 is 0.5, so
// a word of 32 bits is made an operand by three shifts and four masks (the order of the contraction index is free as long
// as both sides share it: dword d, nibble i is row 4 i + d). A letter is 0100 = 2, a "mean of the four" 0001 = 0.5 in all four
// of its rows: with the 0.5 of an open row the 1 and the quarter they count.
// The max-pooling gradient lands on one row per (region, filter): that is a column of bits too, with one set. A wave takes
// 16 filters; columns 0-15 of its products are their open rows, columns 16-31 their winning rows, and at the end of a region
// every column's counts are added to its sums with its own factor (a lane's, that is). The four waves of a workgroup share
// the regions and write the four quarters of its slab: no fold through LDS.
// The open rows come from the forward pass's activity masks, one 64-bit lane mask per row: a 16 x 16 bit transpose
// among the lanes (16 rows of this wave's 16 filters per row of lanes) makes them one word of 32 rows per column.
// Deterministic; c * count is rounded once where the kernels above add c count times, so the sums agree with theirs to
// rounding, not bit for bit. PT: DBK_PT_AVG or DBK_PT_ALL; DBK_PT_MAX (small batches of short regions, counts_takes_max) has the
// winning rows alone: a wave takes 32 filters, two waves a tile, and a workgroup two shares of the regions with a slab each.
// What bounds it: instruction issue, ~90 vector and as many scalar instructions per chunk and wave beside the m / 8 products (matrix
// cores busy a tenth of the time), with two to three waves per SIMD (sums, counts: 4 MT registers). Against one lane per filter that
// counts by population counts, 10 instructions per (tap, letter) and chunk (us, kernel and reduction of its slabs, before / after):
// 2048 regions of 90-200 rows x 128 filters, max + average, 32 taps 70 / 43, 24 taps 60 / 40, 8 taps 36 / 31; 20 000 x 101 x 256,
// 24 taps 356 / 227; 128 x 101 x 64, 24 taps 26 / 16; 50 x 3000 x 64 339 / 34. Requesting a chunk's inputs in the step before,
// with copies at its end, cost 15 to 25 % of that. Error of dW against float64 8.5e-8 (8.9e-8 before), of the bias 7.1e-8 (8.6e-8),
// a float64 sum per wave. Maxima alone: 8.1e-8 and 6.9e-8 (8.1e-8 and 7.9e-8 in the bit kernel).
typedef int i32x8_t __attribute__((ext_vector_type(8)));
// 32 bits as 32 values 0 or 0.5 of the 4-bit format
__device__ __forceinline__ i32x8_t bits_as_halves(unsigned w)
{
    const unsigned k = 0x11111111u;
    return i32x8_t{(int)(w & k), (int)((w >> 1) & k), (int)((w >> 2) & k), (int)((w >> 3) & k), 0, 0, 0, 0};
}
// ... as 0 or 2
__device__ __forceinline__ i32x8_t bits_as_twos(unsigned w)
{
    const unsigned k = 0x44444444u;
    return i32x8_t{(int)((w << 2) & k), (int)((w << 1) & k), (int)(w & k), (int)((w >> 1) & k), 0, 0, 0, 0};
}
__device__ __forceinline__ f32x16_t count_product(const i32x8_t& letters, const i32x8_t& rows, const f32x16_t& c)
{
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(letters, rows, c, 4, 4, 0, 127, 0, 127);      // (4-bit formats; block scales 1)
}
// Transposes a 16 x 16 bit matrix per row of 16 lanes: bit i of v is column i of this lane's row, afterwards row i of this lane's
// column. Four butterfly stages (block sizes 8 ... 1): a lane and its partner lane ^ d swap the off-diagonal d x d blocks they
// hold between them. The value is held twice, in both halves of the word, so that the shift of either side is a rotation.
struct transpose16 {
    unsigned keep[4], turn[4];
    __device__ __forceinline__ explicit transpose16(unsigned lane)
    {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const unsigned d = 8u >> k, clear = d == 8u ? 0x00ff00ffu : d == 4u ? 0x0f0f0f0fu : d == 2u ? 0x33333333u : 0x55555555u;
            keep[k] = lane & d ? ~clear : clear;
            turn[k] = lane & d ? d : 16u - d;
        }
    }
    __device__ __forceinline__ unsigned stage(unsigned v, unsigned partner, int k) const
    {
        const unsigned other = __builtin_amdgcn_alignbit(partner, partner, turn[k]);
        return other ^ ((v ^ other) & keep[k]);
    }
    __device__ __forceinline__ unsigned operator()(unsigned v) const
    {
        v |= v << 16;
        v = stage(v, (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x128, 0xf, 0xf, true), 0);       // lane ^ 8
        const int x7 = __builtin_amdgcn_mov_dpp((int)v, 0x141, 0xf, 0xf, true);                    // lane ^ 7
        v = stage(v, (unsigned)__builtin_amdgcn_mov_dpp(x7, 0x1b, 0xf, 0xf, true), 1);            // ^ 3: lane ^ 4
        v = stage(v, (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x4e, 0xf, 0xf, true), 2);        // lane ^ 2
        return stage(v, (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0xb1, 0xf, 0xf, true), 3);     // lane ^ 1
    }
};

template <int PT, int MT>
__device__ __forceinline__ void scanpool_bprop_counts_body(const wg_t wg, unsigned m, unsigned F, const uint8_t* __restrict__ X, size_t N,
                                                           const uint32_t* __restrict__ R, size_t P,
                                                           const float* __restrict__ pooled, const uint32_t* __restrict__ argmax,
                                                           const float* __restrict__ dpooled,
                                                           const unsigned long long* __restrict__ act,
                                                           float* __restrict__ slabs, size_t stride)
{
    constexpr bool DENSE = PT != DBK_PT_MAX, PEAK = PT != DBK_PT_AVG;
    constexpr int NB = MT / 8;                                     // blocks of eight taps: 32 rows (tap, letter) of the product
    constexpr unsigned NONE = ~0u;
    const unsigned lane = threadIdx.x & 63, wave = (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const unsigned col = lane & 31u, h = lane >> 5;
    const bool peak = !DENSE || (lane & 16u) != 0u;                // this lane's column: winning rows, or open rows
    const unsigned f = wg.y * FT + (DENSE ? 16u * wave + (lane & 15u) : 32u * (wave & 1u) + col);
    const unsigned share = DENSE ? wg.x : 2u * wg.x + (wave >> 1), shares = DENSE ? wg.gx : 2u * wg.gx;      // of the regions: a slab each
    const size_t n = N + 1 >= (size_t)m + 1 ? N - m + 1 : 0;      // rows the scan defines; later rows carry bias only
    const unsigned short* act16 = reinterpret_cast<const unsigned short*>(act) + 4 * (size_t)wg.y + wave;
    const transpose16 transpose(lane);
    // as a row of the letters' operand: letter col & 3 of tap col >> 2 of each block
    const unsigned not0 = col & 1u ? 0u : ~0u, not1 = col & 2u ? 0u : ~0u, tap = col >> 2;
    f32x16_t sums[NB], counts[NB];
#pragma unroll
    for (int t = 0; t < NB; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i) { sums[t][i] = 0.0f; counts[t][i] = 0.0f; }
    double db = 0.0;                                               // (the registers of two float32 chains, which round more)
    // A wave's regions are share, share + shares, ...: lane i holds the bounds of the i-th of 64 of them.
    const size_t step = shares;
    const unsigned nregion = N != 0 && share < P ? (unsigned)((P - share + step - 1) / step) : 0u;     // (without rows every region is empty)
    unsigned va = 0u, vb = 0u;
    auto load_bounds = [&](unsigned k) {
        const size_t e = share + ((size_t)k + lane) * step, r_ = e < P ? e : P - 1;
        va = R[2 * r_]; vb = R[2 * r_ + 1];
        __builtin_amdgcn_s_waitcnt(0x0f70);                        // vmcnt(0), here: else every step that may come this way waits for all that is under way
    };
    // What a chunk needs - its letters (two per lane) and masks, a region's first one its factors - is requested two chunks ahead, into
    // the registers that the chunk in work has just left (a copy on the way would wait for what is still under way), without
    // branches on the lane: past the end the last letter and row are read, and not used.
    struct chunk_in { unsigned x0, x1, mk, arg; float g, pmax; };
    struct place { unsigned k, a, b, c; };                         // a chunk: which of the wave's regions, its bounds, first row
    auto advance = [&](place& k) {
        if (k.b > k.c && k.b - k.c > 64u) { k.c += 64u; return; }
        ++k.k;
        if ((k.k & 63u) == 0u) load_bounds(k.k);
        k.a = k.c = (unsigned)__builtin_amdgcn_readlane((int)va, (int)(k.k & 63u));
        k.b = (unsigned)__builtin_amdgcn_readlane((int)vb, (int)(k.k & 63u));
    };
    // chunks up to here lie inside the text, and inside the rows that the scan defines
    const bool any_inside = N >= 128, any_defined = n >= 64;
    const unsigned inside = (unsigned)(N - 128 < 0xffffffffull ? N - 128 : 0xffffffffull), defined = (unsigned)(n - 64 < 0xffffffffull ? n - 64 : 0xffffffffull);
    const unsigned fe = f < F ? f : F - 1u, row_words = 4u * wg.gy;
    auto request_chunk = [&](const place& k, chunk_in& in) {
        size_t base = k.c;
        unsigned e0 = lane, e1 = lane + 64u, em = lane * row_words;
        if (!(any_inside && k.c <= inside)) {
            if (base >= N) base = N - 1;
            const unsigned more = N - 1 - base < 128 ? (unsigned)(N - 1 - base) : 128u;
            e0 = e0 < more ? e0 : more; e1 = e1 < more ? e1 : more; em = e0 * row_words;
        }
        in.x0 = (X + base)[e0];
        in.x1 = (X + base)[e1];
        if (DENSE) in.mk = (act16 + base * row_words)[em];
        if (k.c == k.a) {
            const size_t r_ = share + (size_t)k.k * step, j0 = (r_ < P ? r_ : P - 1) * F;
            if (PEAK && DENSE) { in.g = (dpooled + 2 * j0)[2u * fe + (peak ? 0u : 1u)]; in.pmax = (pooled + 2 * j0)[2u * fe]; in.arg = (argmax + j0)[fe]; }
            else if (PEAK) { in.g = (dpooled + j0)[fe]; in.pmax = (pooled + j0)[fe]; in.arg = (argmax + j0)[fe]; }
            else in.g = (dpooled + j0)[fe];
        }
    };
    chunk_in in0 = { 254u, 254u, 0u, 0u, 0.0f, 0.0f }, in1 = in0;
    place now = { 0u, 0u, 0u, 0u }, next = now;
    if (nregion != 0u) {
        load_bounds(0u);
        now.a = now.c = (unsigned)__builtin_amdgcn_readlane((int)va, 0);
        now.b = (unsigned)__builtin_amdgcn_readlane((int)vb, 0);
        request_chunk(now, in0);
        next = now;
        advance(next);
        request_chunk(next, in1);
    }
    float g = 0.0f;                                                // this column's factor
    unsigned top = NONE, open = 0u;                                // its winning row; how many of its bits were set (this half wave's)
    auto work = [&](chunk_in& in) {
        const unsigned c = now.c, left = now.b > c ? now.b - c : 0u;      // rows of the region from this chunk on
        const bool first = c == now.a, last = left <= 64u;
        // ---- the letters: one bit per (letter, position) of the chunk, positions c .. c + 63 and the MT - 1 behind them
        if (!(any_inside && c <= inside)) {
            if ((size_t)c + lane >= N) in.x0 = 254u;
            if ((size_t)c + 64 + lane >= N) in.x1 = 254u;
        }
        const unsigned long long V0 = __ballot(in.x0 < 4u), E0 = __ballot((in.x0 & 1u) != 0u), T0 = __ballot((in.x0 & 2u) != 0u);
        const unsigned V1 = (unsigned)__ballot(in.x1 < 4u), E1 = (unsigned)__ballot((in.x1 & 1u) != 0u), T1 = (unsigned)__ballot((in.x1 & 2u) != 0u);
        const unsigned long long Z0 = __ballot(in.x0 == 254u);
        const unsigned Z1 = (unsigned)__ballot(in.x1 == 254u);
        // ---- the columns: 32 rows' bits
        const unsigned v = DENSE ? transpose(lane < left ? in.mk : 0u) : 0u;
        if (first) {
            g = now.b > now.a && f < F ? in.g / (float)(now.b - now.a) : 0.0f;
            if (peak) {
                const bool any = PEAK && in.pmax > 0.0f && f < F;
                g = any ? in.g : 0.0f;
                top = any ? in.arg / F : NONE;
            }
        }
        // ---- what comes after the next chunk is on its way while this one is worked on
        place after = next;
        advance(after);
        request_chunk(after, in);
        if (now.k < nregion) {
            const auto halves = __builtin_amdgcn_permlane16_swap(v, v, false, false);
            unsigned bits = __builtin_amdgcn_perm(halves[1], halves[0], 0x05040100u);
            const unsigned rel = top - c - 32u * h;
            if (peak) bits = PEAK && top != NONE && rel < 32u ? 1u << (rel & 31u) : 0u;
            open += (unsigned)__popc(bits);
            if (!(any_defined && c <= defined)) {                      // rows that the scan does not define
                const size_t nrel = n > c ? n - c : 0;
                if (nrel < 64) bits &= (unsigned)(((1ull << nrel) - 1ull) >> (32u * h));
            }
            // ---- the counts
            const i32x8_t B = bits_as_halves(bits);
            auto letter = [&](unsigned v_, unsigned e, unsigned t) -> unsigned { return (e ^ not0) & (t ^ not1) & v_; };
            const unsigned w0 = letter((unsigned)V0, (unsigned)E0, (unsigned)T0), w1 = letter((unsigned)(V0 >> 32), (unsigned)(E0 >> 32), (unsigned)(T0 >> 32)), w2 = letter(V1, E1, T1);
            const unsigned wl = h ? w1 : w0, wh = h ? w2 : w1;         // from this half wave's first row on
            i32x8_t A[NB];
#pragma unroll
            for (int t = 0; t < NB; ++t) A[t] = bits_as_twos(__builtin_amdgcn_alignbit(wh, wl, 8u * t + tap));
            const unsigned long long M0 = ~(V0 | Z0);              // neither a letter nor nothing: the mean of the four
            const unsigned M1 = ~(V1 | Z1);
            if ((M0 | M1) != 0ull) {
                const unsigned ml = h ? (unsigned)(M0 >> 32) : (unsigned)M0, mh = h ? M1 : (unsigned)(M0 >> 32);
#pragma unroll
                for (int t = 0; t < NB; ++t) A[t] = A[t] | bits_as_halves(__builtin_amdgcn_alignbit(mh, ml, 8u * t + tap));
            }
            if (first) {
#pragma unroll
                for (int t = 0; t < NB; ++t) counts[t] = count_product(A[t], B, f32x16_t{});
            } else {
#pragma unroll
                for (int t = 0; t < NB; ++t) counts[t] = count_product(A[t], B, counts[t]);
            }
            // ---- a region's end
            if (last) {
                db = __builtin_fma((double)g, (double)open, db);
                open = 0u;
#pragma unroll
                for (int t = 0; t < NB; ++t)
#pragma unroll
                    for (int i = 0; i < 16; ++i) sums[t][i] = __builtin_fmaf(g, counts[t][i], sums[t][i]);
            }
        }
        now = next;
        next = after;
    };
    // (no way out between the two: the compiler's waits cover every path, and one that leaves a request out would make them longer)
    while (now.k < nregion) {                                      // uniform over the wave
        work(in0);
        work(in1);
    }
    // ---- this wave's quarter of the slab: a filter's two columns side by side, register i's sums in lanes 0-15 and 32-47, register
    // i + 1's in the others. Register i holds letter i & 3 of tap 2 (i >> 2) + h of its block.
    float bias_sum = (float)db;
    float* out = slabs + (size_t)share * stride;
    if (!DENSE) {                                                  // (a column per filter: this wave's half of its slab as it is)
#pragma unroll
        for (int t = 0; t < NB; ++t)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const unsigned j = 8u * t + 2u * (i >> 2) + h;
                if (j < m && f < F) out[(size_t)(4u * j + (i & 3)) * F + f] = sums[t][i];
            }
        const auto d32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(bias_sum), __float_as_uint(bias_sum), false, false);
        if (h == 0u && f < F) out[(size_t)4 * m * F + f] = __uint_as_float(d32[0]) + __uint_as_float(d32[1]);
        return;
    }
#pragma unroll
    for (int t = 0; t < NB; ++t)
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(sums[t][i]), __float_as_uint(sums[t][i + 1]), false, false);
            const unsigned j = 8u * t + 2u * (i >> 2) + h;
            if (j < m && f < F) out[(size_t)(4u * j + (i & 3) + (peak ? 1u : 0u)) * F + f] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
        }
    const auto d16 = __builtin_amdgcn_permlane16_swap(__float_as_uint(bias_sum), __float_as_uint(bias_sum), false, false);
    bias_sum = __uint_as_float(d16[0]) + __uint_as_float(d16[1]);
    const auto d32 = __builtin_amdgcn_permlane32_swap(__float_as_uint(bias_sum), __float_as_uint(bias_sum), false, false);
    if (lane < 16u && f < F) out[(size_t)4 * m * F + f] = __uint_as_float(d32[0]) + __uint_as_float(d32[1]);
}

template <int PT, int MT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(MT == 32 ? 2 : 3)))
void scanpool_bprop_counts_kernel(unsigned m, unsigned F, const uint8_t* __restrict__ X, size_t N, const uint32_t* __restrict__ R, size_t P,
                                  const float* __restrict__ pooled, const uint32_t* __restrict__ argmax, const float* __restrict__ dpooled,
                                  const unsigned long long* __restrict__ act, float* __restrict__ slabs, size_t stride)
{
    scanpool_bprop_counts_body<PT, MT>(this_wg(), m, F, X, N, R, P, pooled, argmax, dpooled, act, slabs, stride);
}

// Launch shapes, shared by the single-group launchers and the multi-group ones.
// forward: as many workgroups as are resident at once (three per CU; two with the register planes of 16 taps);
// each sets up its filter tile's weights once and then walks its share of the regions
inline unsigned fprop_grid_x(unsigned mt, unsigned ftiles, size_t P)
{
    unsigned gx = (mt == 16 ? 512u : 768u) / ftiles;
    if (gx < 1) gx = 1;
    if (gx > P) gx = (unsigned)P;
    return gx;
}
inline size_t fprop_smem(unsigned mt, size_t m)
{
    const unsigned nw = 4;
    const size_t taps = mt ? mt : m;
    const bool planes = mt == 8 || mt == 16;                     // weights in registers: no table in LDS
    return (planes ? 0 : taps * NL * FT * sizeof(float)) + nw * 3 * FT * sizeof(float) + ((nw * XCH_SUBS * PSUB + taps - 1 + 7) & ~(size_t)3);
}
// sparse half of the backward pass: ~2048 single-wave workgroups, at least four regions each (more regions per
// workgroup only lengthens its chain of dependent loads)
inline unsigned sparse_grid_x(unsigned ftiles, size_t P)
{
    unsigned gxs = 2048u / ftiles;
    if (gxs > (P + 3) / 4) gxs = (unsigned)((P + 3) / 4);
    if (gxs < 1) gxs = 1;
    return gxs;
}
// dense half: four-wave workgroups, as many as are resident at once (its register planes leave room for two per
// CU, three with 8 taps). A minibatch (a handful of regions per workgroup) takes one workgroup per CU instead:
// alone the kernel runs as fast (half as many partial sums to write and to reduce), and it leaves half of every
// CU's registers to whatever else is running, such as the other architectures of a calibration batch.
inline unsigned dense_grid_x(unsigned mt, unsigned ftiles, size_t P)
{
    unsigned gxd = (mt == 8 ? 768u : 512u) / ftiles;
    if (P < 8 * (size_t)gxd) gxd = 256u / ftiles;
    if (gxd < 1) gxd = 1;
    if (gxd > P) gxd = (unsigned)P;
    return gxd;
}
// The wide forward kernel (four filters per lane, a wave per region) pays off once there are enough (region, tile)
// items to keep every CU's LDS busy; a small batch is latency-bound and better off with four waves per region.
inline bool wide_takes(size_t m, unsigned ftiles, size_t P) { return m > 8 && m <= 24 && P * (size_t)ftiles >= 512; }
inline unsigned wide_tier(size_t m) { return m <= 16 ? 16u : 24u; }
// The matrix-core forward takes those batches (same break-even: it needs enough (region, tile) items to fill the GPU).
inline bool mfma_pays(size_t m, unsigned ftiles, size_t P) { return m > 8 && m <= 32 && P * (size_t)ftiles >= 512; }
inline unsigned wide_grid_x(unsigned ftiles, size_t P)
{
    unsigned gx = 768u / ftiles;                                  // three workgroups per CU are resident (150-160 registers)
    if (gx < 1) gx = 1;
    if (gx > (P + 3) / 4) gx = (unsigned)((P + 3) / 4);           // a workgroup walks four regions at a time
    return gx;
}
inline size_t wide_smem(unsigned mt) { return (size_t)mt * NL * FT * sizeof(float) + 4 * (mt == 16 ? wide_shape<16>::xbytes : wide_shape<24>::xbytes); }
// The bit kernel of max pooling: a wave per region, three workgroups per CU resident (its 5 x MT sums and the rest take ~150
// registers at 24 taps: three waves per SIMD; ~190 at 32: two);
// the smallest grid that gives every wave the same number of regions as the resident grid would.
inline unsigned bits_grid_x(unsigned mt, unsigned ftiles, size_t P)
{
    unsigned gx = (mt == 32 ? 512u : 768u) / ftiles;
    if (gx < 1) gx = 1;
    // at least two regions per wave: the fold of a workgroup's sums and its slab cost about as much as two regions
    // (measured on a calibration batch of 256 regions x 23 tiles: 26.7 us with two, 29.6 with three, 34.5 with five
    // regions per wave; the reduction of the slabs 7.9 / 7.1 / 6.5 us)
    if (gx > (P + 7) / 8) gx = (unsigned)((P + 7) / 8);
    const size_t per_wave = (P + (size_t)gx * 4 - 1) / ((size_t)gx * 4);
    return (unsigned)((P + 4 * per_wave - 1) / (4 * per_wave));
}
// The counting backward: as many workgroups as are resident at once (two per CU with 32 taps, else three, the third only
// where each of them gets many regions), every workgroup the same number of regions, at least eight chunks of 64 rows (the
// sums' way out and their reduction cost about as much). us with the third, without: 20 000 regions x 101 x 256 filters 240 / 277, 2048 x
// 145 x 128 42 / 41. us with eight regions, four: 128 x 101 x 64 17.8 / 14.6, 256 x 30 x 512 16.8 / 18.4; 50 x 3000 x 64 216 / 113, one 34.
inline unsigned counts_grid_x(unsigned mt, unsigned ftiles, size_t N, size_t P)
{
    size_t gx = (mt < 32 && P * ftiles >= 16 * 768 ? 768u : 512u) / ftiles;
    if (gx < 1) gx = 1;
    const size_t chunks = N / (64 * P) > 0 ? N / (64 * P) : 1, least = chunks < 8 ? (8 + chunks - 1) / chunks : 1;
    if (gx > (P + least - 1) / least) gx = (P + least - 1) / least;
    const size_t per_group = (P + gx - 1) / gx;
    return (unsigned)((P + per_group - 1) / per_group);
}
// Of max pooling it takes small batches of short regions (one chunk each, so that no chunk is walked for nothing); a workgroup has two
// shares of the regions there. us a call, bit kernel / this: 256 regions of 53 rows x 1440 filters of 24 taps 27 / 22, 171 x 512 17.2 / 15.7,
// 171 x 64 15.8 / 14.7, 512 x 16 of 8 taps 14.4 / 13.8, 768 of 61 x 256 of 32 taps 26.2 / 22.7, 768 of 37 x 512 of 8 taps 17.0 / 16.9; 128 of 119 rows x 64 16.0 / 16.4, 2048 of 77 rows x 256 of 8 taps 20.8 / 25.7, 20 000 of 60 x 64 50 / 57.
// Few taps leave the bit kernel little to do per region: it keeps the calls of many regions x filters (512 regions of 52 rows x 1024 filters
// of 8 taps 14.1 / 15.4, 768 x 1024 15.7 / 18.6, 768 x 256 12.2 / 12.9, 256 x 1024 13.1 / 11.8; 16 taps 768 x 1024 22.6 / 23.9, 500 x 1024 19.2 / 19.1).
inline bool counts_takes_max(unsigned mt, unsigned ftiles, size_t N, size_t P)
{
    return P <= (mt == 8 ? 512u : 768u) && N <= 64 * P && (mt > 16 || P * ftiles <= (mt == 8 ? 4096u : 8192u));
}
inline unsigned counts_max_grid_x(unsigned mt, unsigned ftiles, size_t N, size_t P) { return (counts_grid_x(mt, ftiles, N, P) + 1) / 2; }
// Max pooling goes through the bit kernel while the regions are short on average (it visits every 64-row chunk of a region to
// find each filter's winning row; the sparse kernel goes straight to that row).
inline bool bits_takes_max(size_t N, size_t P) { return N <= 128 * P; }
inline size_t bits_smem(unsigned) { return FOLD_BYTES; }
inline size_t sparse_smem(size_t m) { return m * SPARSE_ROWS * FT * sizeof(float); }
inline size_t dense_smem(unsigned mt)
{
    const size_t scan = ((size_t)mt * NL * FT + 4 * FT) * sizeof(float) + ((4 * XCH_SUBS * PSUB + mt - 1 + 7) & ~(size_t)3);
    return scan > FOLD_BYTES ? scan : FOLD_BYTES;                  // (the kernel's last act, the fold of its waves' sums, reuses the memory)
}

template <int PT, int MT>
int launch_fprop_mt(hipStream_t st, unsigned gx, unsigned ftiles, unsigned nw, size_t smem, const float* W, const float* bias, size_t m,
                     size_t F, const uint8_t* X, size_t N, const uint32_t* R, size_t P, float* pooled, uint32_t* argmax,
                     unsigned long long* act)
{
    if (argmax) {
        auto kern = scanpool_fprop_kernel<PT, true, MT>;
        DBK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        hipLaunchKernelGGL(kern, dim3(gx, ftiles), dim3(nw * 64), smem, st, W, bias, (unsigned)m, (unsigned)F, X, N, R, P, pooled, argmax, act);
    } else {
        auto kern = scanpool_fprop_kernel<PT, false, MT>;
        DBK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        hipLaunchKernelGGL(kern, dim3(gx, ftiles), dim3(nw * 64), smem, st, W, bias, (unsigned)m, (unsigned)F, X, N, R, P, pooled, argmax, act);
    }
    return 0;
}

template <int PT>
int launch_fprop_wide(hipStream_t st, unsigned ftiles, const float* W, const float* bias, size_t m, size_t F, const uint8_t* X, size_t N,
                      const uint32_t* R, size_t P, float* pooled, uint32_t* argmax, unsigned long long* act)
{
    const unsigned mt = wide_tier(m);
    const size_t smem = wide_smem(mt);
    DBK_CHECK(smem <= lds_limit(), "ValueError: the wide forward kernel needs %zu bytes of LDS (limit %zu)", smem, lds_limit());
    const unsigned gx = wide_grid_x(ftiles, P);
    auto kern = argmax ? (mt == 16 ? scanpool_fprop_wide_kernel<PT, true, 16> : scanpool_fprop_wide_kernel<PT, true, 24>)
                       : (mt == 16 ? scanpool_fprop_wide_kernel<PT, false, 16> : scanpool_fprop_wide_kernel<PT, false, 24>);
    DBK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
    hipLaunchKernelGGL(kern, dim3(gx, ftiles), dim3(256), smem, st, W, bias, (unsigned)m, (unsigned)F, X, N, R, P, pooled, argmax, act);
    DBK_LAUNCH_OK();
}

// The matrix-core forward: a workgroup holds a 64-filter tile (two waves per half) and walks two regions at a time.
inline unsigned mfma_grid_x(unsigned ftiles, size_t P)
{
    unsigned gx = 768u / ftiles;                                  // three workgroups per CU resident
    if (gx < 1) gx = 1;
    if (gx > (P + 1) / 2) gx = (unsigned)((P + 1) / 2);
    return gx;
}

template <int PT, int KS>
int launch_fprop_mfma_ks(hipStream_t st, unsigned ftiles, const float* W, const float* bias, size_t m, size_t F, const uint8_t* X, size_t N,
                         const uint32_t* R, size_t P, float* pooled, uint32_t* argmax, unsigned long long* act)
{
    const unsigned gx = mfma_grid_x(ftiles, P);
    auto kern = argmax ? (act ? scanpool_fprop_mfma_kernel<PT, true, true, KS> : scanpool_fprop_mfma_kernel<PT, true, false, KS>)
                       : (act ? scanpool_fprop_mfma_kernel<PT, false, true, KS> : scanpool_fprop_mfma_kernel<PT, false, false, KS>);
    hipLaunchKernelGGL(kern, dim3(gx, ftiles), dim3(256), MFMA_SMEM, st, W, bias, (unsigned)m, (unsigned)F, X, N, R, P, pooled, argmax, act);
    DBK_LAUNCH_OK();
}

template <int PT>
int launch_fprop_mfma(hipStream_t st, unsigned ftiles, const float* W, const float* bias, size_t m, size_t F, const uint8_t* X, size_t N,
                      const uint32_t* R, size_t P, float* pooled, uint32_t* argmax, unsigned long long* act)
{
    switch ((mfma_ksteps(m) + 1) / 2) {
    case 1:  return launch_fprop_mfma_ks<PT, 2>(st, ftiles, W, bias, m, F, X, N, R, P, pooled, argmax, act);
    case 2:  return launch_fprop_mfma_ks<PT, 4>(st, ftiles, W, bias, m, F, X, N, R, P, pooled, argmax, act);
    case 3:  return launch_fprop_mfma_ks<PT, 6>(st, ftiles, W, bias, m, F, X, N, R, P, pooled, argmax, act);
    default: return launch_fprop_mfma_ks<PT, 8>(st, ftiles, W, bias, m, F, X, N, R, P, pooled, argmax, act);
    }
}

template <int PT>
int launch_fprop_pt(hipStream_t st, const float* W, const float* bias, size_t m, size_t F, const uint8_t* X, size_t N,
                    const uint32_t* R, size_t P, float* pooled, uint32_t* argmax, unsigned long long* act)
{
    const unsigned nw = 4;
    const unsigned mt = m <= 8 ? 8 : (m <= 16 ? 16 : (m <= 24 ? 24 : (m <= 32 ? 32 : 0)));    // 0: any-length kernel
    const size_t smem = fprop_smem(mt, m);
    DBK_CHECK(smem <= lds_limit(), "ValueError: filter length %zu needs %zu bytes of LDS (limit %zu)", m, smem, lds_limit());
    unsigned ftiles = dbk::divup(F, FT);
    DBK_CHECK(ftiles <= 65535u, "ValueError: too many filters (%zu) for one launch", F);
    if (mfma_pays(m, ftiles, P)) return launch_fprop_mfma<PT>(st, ftiles, W, bias, m, F, X, N, R, P, pooled, argmax, act);
    const unsigned gx = fprop_grid_x(mt, ftiles, P);
    int rc = 0;
    switch (mt) {
    case 8:  rc = launch_fprop_mt<PT, 8>(st, gx, ftiles, nw, smem, W, bias, m, F, X, N, R, P, pooled, argmax, act); break;
    case 16: rc = launch_fprop_mt<PT, 16>(st, gx, ftiles, nw, smem, W, bias, m, F, X, N, R, P, pooled, argmax, act); break;
    case 24: rc = launch_fprop_mt<PT, 24>(st, gx, ftiles, nw, smem, W, bias, m, F, X, N, R, P, pooled, argmax, act); break;
    case 32: rc = launch_fprop_mt<PT, 32>(st, gx, ftiles, nw, smem, W, bias, m, F, X, N, R, P, pooled, argmax, act); break;
    default: rc = launch_fprop_mt<PT, 0>(st, gx, ftiles, nw, smem, W, bias, m, F, X, N, R, P, pooled, argmax, act); break;
    }
    if (rc) return rc;
    DBK_LAUNCH_OK();
}

template <int PT, int KS>
int launch_fprop_left_ks(hipStream_t st, const float* W, const float* bias, size_t m, size_t F, const uint8_t* X, size_t N, const uint32_t* R,
                         size_t P, float* pooled, uint32_t* argmax, const unsigned* flags)
{
    const unsigned ftiles = dbk::divup(F, FT);
    const size_t smem = std::max(MFMA_SMEM, fprop_smem(left_lookup_taps(KS), m)), items = ftiles * P;
    const unsigned grid = std::max(ftiles, items < 768 ? (unsigned)items : 768u);   // three workgroups per CU are resident
    constexpr bool ARG = PT != DBK_PT_AVG && KS < 8;               // (the bulk kernel takes more than 24 taps without an argmax only)
    auto kern = ARG && argmax ? scanpool_fprop_left_kernel<PT, ARG, KS> : scanpool_fprop_left_kernel<PT, false, KS>;
    DBK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
    hipLaunchKernelGGL(kern, dim3(grid), dim3(256), smem, st, W, bias, (unsigned)m, (unsigned)F, X, N, R, P, pooled, argmax, flags, ftiles);
    DBK_LAUNCH_OK();
}

template <int PT>
int launch_fprop_left(hipStream_t st, const float* W, const float* bias, size_t m, size_t F, const uint8_t* X, size_t N, const uint32_t* R,
                      size_t P, float* pooled, uint32_t* argmax, const unsigned* flags)
{
    switch ((mfma_ksteps(m) + 1) / 2) {
    case 1:  return launch_fprop_left_ks<PT, 2>(st, W, bias, m, F, X, N, R, P, pooled, argmax, flags);
    case 2:  return launch_fprop_left_ks<PT, 4>(st, W, bias, m, F, X, N, R, P, pooled, argmax, flags);
    case 3:  return launch_fprop_left_ks<PT, 6>(st, W, bias, m, F, X, N, R, P, pooled, argmax, flags);
    default: return launch_fprop_left_ks<PT, 8>(st, W, bias, m, F, X, N, R, P, pooled, argmax, flags);
    }
}

template <int PT, int MT>
int launch_counts(hipStream_t st, unsigned gx, unsigned ftiles, size_t m, size_t F, const uint8_t* X, size_t N, const uint32_t* R,
                  size_t P, const float* pooled, const uint32_t* argmax, const float* dpooled, const unsigned long long* act, float* slabs, size_t stride)
{
    auto kern = scanpool_bprop_counts_kernel<PT, MT>;
    hipLaunchKernelGGL(kern, dim3(gx, ftiles), dim3(256), 0, st, (unsigned)m, (unsigned)F, X, N, R, P, pooled, argmax, dpooled, act, slabs, stride);
    return 0;
}

template <int PT, int MT>
int launch_dense(hipStream_t st, unsigned gx, unsigned ftiles, size_t smem, const float* W, const float* bias, size_t m, size_t F,
                  const uint8_t* X, size_t N, const uint32_t* R, size_t P, const float* pooled, const uint32_t* argmax,
                  const float* dpooled, const unsigned long long* act, float* slabs, size_t stride)
{
    if (act) return launch_counts<PT, MT>(st, gx, ftiles, m, F, X, N, R, P, pooled, argmax, dpooled, act, slabs, stride);
    auto kern = scanpool_bprop_dense_kernel<PT, MT>;
    DBK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
    hipLaunchKernelGGL(kern, dim3(gx, ftiles), dim3(256), smem, st, W, bias, (unsigned)m, (unsigned)F, X, N, R, P, pooled, argmax, dpooled, slabs, stride);
    return 0;
}

template <int PT>
int launch_bprop_pt(hipStream_t st, const float* W, const float* bias, size_t m, size_t F, const uint8_t* X, size_t N,
                    const uint32_t* R, size_t P, const float* pooled, const uint32_t* argmax, const float* dpooled,
                    float* dW, float* dbias, bool overwrite, const unsigned long long* act)
{
    const unsigned ftiles = dbk::divup(F, FT);
    DBK_CHECK(ftiles <= 65535u, "ValueError: too many filters (%zu) for one launch", F);
    const size_t nW = 4 * m * F, stride = nW + F;
    const unsigned mt = m <= 8 ? 8 : (m <= 16 ? 16 : (m <= 24 ? 24 : (m <= 32 ? 32 : 0)));
    // Average pooling without the forward pass's activity masks: the matrix-core forward writes them again (into the
    // stream's second scratch buffer, with its pooled values beside them), and the counting kernel takes them from
    // there; less than half the time of recomputing the map through the letter table, whose registers moreover end at 24
    // taps: longer filters take this way at every size.
    const size_t mask_bytes = N * ftiles * sizeof(unsigned long long), pooled_bytes = P * F * 2 * sizeof(float);
    if (PT != DBK_PT_MAX && !act && !dbk::deferred() && (mfma_pays(m, ftiles, P) || mt == 32) && mask_bytes + pooled_bytes <= ((size_t)1 << 30)) {   // (at most 1 GiB of scratch for it)
        unsigned char* scratch = (unsigned char*)dbk::workspace(mask_bytes + pooled_bytes, st, 1);
        DBK_CHECK(scratch != nullptr, "MemoryError: could not allocate %zu bytes of scratch (%s)", mask_bytes + pooled_bytes, dbk::workspace_error());
        unsigned long long* masks = reinterpret_cast<unsigned long long*>(scratch);
        const int rc = launch_fprop_mfma<PT>(st, ftiles, W, bias, m, F, X, N, R, P, reinterpret_cast<float*>(scratch + mask_bytes), nullptr, masks);
        if (rc) return rc;
        act = masks;
    }
    if (mt == 0 || (mt == 32 && PT != DBK_PT_MAX && !act)) {
        // any filter length: one kernel does both halves through per-wave LDS tables
        unsigned nw = 4;
        const size_t lutb = PT == DBK_PT_MAX ? 0 : m * NL * FT * sizeof(float);
        auto need = [&](unsigned w) { return lutb + (size_t)w * (m * 4 * FT + FT) * sizeof(float) + w * XCH_SUBS * PSUB + m - 1; };
        while (nw > 1 && need(nw) > lds_limit()) nw >>= 1;
        const size_t smem = need(nw);
        DBK_CHECK(smem <= lds_limit(), "ValueError: filter length %zu needs %zu bytes of LDS (limit %zu)", m, smem, lds_limit());
        unsigned gx = 1024u / ftiles;
        if (gx < 1) gx = 1;
        if (gx > P) gx = (unsigned)P;
        float* slabs = (float*)dbk::workspace(stride * gx * sizeof(float), st);
        DBK_CHECK(slabs != nullptr, "MemoryError: could not allocate %zu bytes of scratch (%s)", stride * gx * sizeof(float), dbk::workspace_error());
        auto kern = scanpool_bprop_kernel<PT>;
        DBK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        hipLaunchKernelGGL(kern, dim3(gx, ftiles), dim3(nw * 64), smem, st, W, bias, (unsigned)m, (unsigned)F, X, N, R, P,
                           pooled, argmax, dpooled, slabs, stride);
        if (dbk::deferred_sums* later = dbk::deferred()) { later->slabs = slabs; later->slab_stride = stride; later->nslab = gx; }
        else hipLaunchKernelGGL(reduce_slabs_kernel, dim3(dbk::ew_grid(stride)), dim3(256), 0, st, dW, dbias, (const float*)slabs, nW, F, gx, overwrite);
        DBK_LAUNCH_OK();
    }
    // with max+avg pooling the dense half carries the maxima along
    const bool max_bits = PT == DBK_PT_MAX && bits_takes_max(N, P), max_counts = PT == DBK_PT_MAX && counts_takes_max(mt, ftiles, N, P);
    const unsigned gxs = PT == DBK_PT_MAX ? (max_counts ? 2 * counts_max_grid_x(mt, ftiles, N, P) : max_bits ? bits_grid_x(mt, ftiles, P) : sparse_grid_x(ftiles, P)) : 0u;
    const unsigned gxd = PT == DBK_PT_MAX ? 0u : act ? counts_grid_x(mt, ftiles, N, P) : dense_grid_x(mt, ftiles, P);
    const size_t smem_s = sparse_smem(m), smem_d = mt == 32 ? bits_smem(mt) : dense_smem(mt);
    DBK_CHECK(smem_s <= lds_limit() && smem_d <= lds_limit(), "ValueError: filter length %zu does not fit in LDS", m);
    float* slabs = (float*)dbk::workspace(stride * (gxs + gxd) * sizeof(float), st);
    DBK_CHECK(slabs != nullptr, "MemoryError: could not allocate %zu bytes of scratch (%s)", stride * (gxs + gxd) * sizeof(float), dbk::workspace_error());
    if (max_counts) {
        auto kern = mt == 8 ? scanpool_bprop_counts_kernel<DBK_PT_MAX, 8> : mt == 16 ? scanpool_bprop_counts_kernel<DBK_PT_MAX, 16>
                  : mt == 24 ? scanpool_bprop_counts_kernel<DBK_PT_MAX, 24> : scanpool_bprop_counts_kernel<DBK_PT_MAX, 32>;
        hipLaunchKernelGGL(kern, dim3(gxs / 2, ftiles), dim3(256), 0, st, (unsigned)m, (unsigned)F, X, N, R, P, pooled, argmax, dpooled,
                           (const unsigned long long*)nullptr, slabs, stride);
    } else if (gxs && max_bits) {
        auto kern = mt == 8 ? scanpool_bprop_bits_kernel<8> : mt == 16 ? scanpool_bprop_bits_kernel<16>
                  : mt == 24 ? scanpool_bprop_bits_kernel<24> : scanpool_bprop_bits_kernel<32>;
        const size_t smem_b = bits_smem(mt);
        DBK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem_b));
        hipLaunchKernelGGL(kern, dim3(gxs, ftiles), dim3(256), smem_b, st, (unsigned)m, (unsigned)F, X, N, R, P, pooled, argmax, dpooled,
                           slabs, stride);
    } else if (gxs) {
        constexpr int PS = PT == DBK_PT_AVG ? DBK_PT_MAX : PT;
        auto kern = mt == 8 ? scanpool_bprop_sparse_kernel<PS, 8> : mt == 16 ? scanpool_bprop_sparse_kernel<PS, 16>
                  : mt == 24 ? scanpool_bprop_sparse_kernel<PS, 24> : scanpool_bprop_sparse_kernel<PS, 32>;
        DBK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem_s));
        hipLaunchKernelGGL(kern, dim3(gxs, ftiles), dim3(64), smem_s, st, (unsigned)m, (unsigned)F, X, N, P, pooled, argmax, dpooled, slabs, stride);
    }
    if (gxd) {
        constexpr int PD = PT == DBK_PT_MAX ? DBK_PT_AVG : PT;
        float* sd = slabs + stride * gxs;
        int rc;
        if (mt == 8) rc = launch_dense<PD, 8>(st, gxd, ftiles, smem_d, W, bias, m, F, X, N, R, P, pooled, argmax, dpooled, act, sd, stride);
        else if (mt == 16) rc = launch_dense<PD, 16>(st, gxd, ftiles, smem_d, W, bias, m, F, X, N, R, P, pooled, argmax, dpooled, act, sd, stride);
        else if (mt == 24) rc = launch_dense<PD, 24>(st, gxd, ftiles, smem_d, W, bias, m, F, X, N, R, P, pooled, argmax, dpooled, act, sd, stride);
        else rc = launch_counts<PD, 32>(st, gxd, ftiles, m, F, X, N, R, P, pooled, argmax, dpooled, act, sd, stride);
        if (rc) return rc;
    }
    if (dbk::deferred_sums* later = dbk::deferred()) { later->slabs = slabs; later->slab_stride = stride; later->nslab = gxs + gxd; }
    else hipLaunchKernelGGL(reduce_slabs_kernel, dim3(dbk::ew_grid(stride)), dim3(256), 0, st, dW, dbias, (const float*)slabs, nW, F, gxs + gxd, overwrite);
    DBK_LAUNCH_OK();
}

int fprop_mfma(hipStream_t st, const float* W, const float* bias, size_t m, size_t F, const uint8_t* X, size_t N,
               const uint32_t* R, size_t P, int ptype, float* pooled, uint32_t* argmax, unsigned long long* act)
{
    const unsigned ftiles = dbk::divup(F, FT);
    DBK_CHECK(ftiles <= 65535u, "ValueError: too many filters (%zu) for one launch", F);
    switch (ptype) {
    case DBK_PT_MAX: return launch_fprop_mfma<DBK_PT_MAX>(st, ftiles, W, bias, m, F, X, N, R, P, pooled, argmax, act);
    case DBK_PT_AVG: return launch_fprop_mfma<DBK_PT_AVG>(st, ftiles, W, bias, m, F, X, N, R, P, pooled, nullptr, act);
    default:         return launch_fprop_mfma<DBK_PT_ALL>(st, ftiles, W, bias, m, F, X, N, R, P, pooled, argmax, act);
    }
}

int fprop_wide(hipStream_t st, const float* W, const float* bias, size_t m, size_t F, const uint8_t* X, size_t N,
               const uint32_t* R, size_t P, int ptype, float* pooled, uint32_t* argmax, unsigned long long* act)
{
    const unsigned ftiles = dbk::divup(F, FT);
    DBK_CHECK(ftiles <= 65535u, "ValueError: too many filters (%zu) for one launch", F);
    switch (ptype) {
    case DBK_PT_MAX: return launch_fprop_wide<DBK_PT_MAX>(st, ftiles, W, bias, m, F, X, N, R, P, pooled, argmax, act);
    case DBK_PT_AVG: return launch_fprop_wide<DBK_PT_AVG>(st, ftiles, W, bias, m, F, X, N, R, P, pooled, nullptr, act);
    default:         return launch_fprop_wide<DBK_PT_ALL>(st, ftiles, W, bias, m, F, X, N, R, P, pooled, argmax, act);
    }
}

int fprop(hipStream_t st, const float* W, const float* bias, size_t m, size_t F, const uint8_t* X, size_t N,
          const uint32_t* R, size_t P, int ptype, float* pooled, uint32_t* argmax, unsigned long long* act)
{
    switch (ptype) {
    case DBK_PT_MAX: return launch_fprop_pt<DBK_PT_MAX>(st, W, bias, m, F, X, N, R, P, pooled, argmax, act);
    case DBK_PT_AVG: return launch_fprop_pt<DBK_PT_AVG>(st, W, bias, m, F, X, N, R, P, pooled, nullptr, act);
    default:         return launch_fprop_pt<DBK_PT_ALL>(st, W, bias, m, F, X, N, R, P, pooled, argmax, act);
    }
}

// The tiles that the bulk kernel left out (flags: one per 32 filters), for filters of up to 32 taps.
int fprop_left(hipStream_t st, const float* W, const float* bias, size_t m, size_t F, const uint8_t* X, size_t N,
               const uint32_t* R, size_t P, int ptype, float* pooled, uint32_t* argmax, const unsigned* flags)
{
    switch (ptype) {
    case DBK_PT_MAX: return launch_fprop_left<DBK_PT_MAX>(st, W, bias, m, F, X, N, R, P, pooled, argmax, flags);
    case DBK_PT_AVG: return launch_fprop_left<DBK_PT_AVG>(st, W, bias, m, F, X, N, R, P, pooled, nullptr, flags);
    default:         return launch_fprop_left<DBK_PT_ALL>(st, W, bias, m, F, X, N, R, P, pooled, argmax, flags);
    }
}

// ---------------------------------------------------------------------------------------------
// several model groups in one launch
// ---------------------------------------------------------------------------------------------
// Workgroups first[g] .. first[g+1]-1 of the launch are group g's grid of gx[g] by ftiles[g], x fastest. The
// argument block travels by value in the kernel-argument segment.
struct multi_args {
    unsigned n, m;
    size_t N, P;
    const uint32_t* R;
    unsigned first[dbk::MULTI_MAX + 1], gx[dbk::MULTI_MAX], ftiles[dbk::MULTI_MAX];
    unsigned wide[dbk::MULTI_MAX];                                 // the group goes through the many-regions kernel body (forward: the matrix-core scan; backward: a wave per region)
    dbk::scan_group g[dbk::MULTI_MAX];
};

__device__ __forceinline__ unsigned multi_locate(const multi_args& a, wg_t& wg)
{
    unsigned g = 0;
    while (g + 1 < a.n && blockIdx.x >= a.first[g + 1]) ++g;
    const unsigned local = blockIdx.x - a.first[g];
    wg = wg_t{local % a.gx[g], local / a.gx[g], a.gx[g], a.ftiles[g]};
    return g;
}

template <int MT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(MT == 24 ? 3 : 1))) void scanpool_fprop_multi_kernel(const multi_args a)
{
    wg_t wg;
    const unsigned gi = multi_locate(a, wg);
    const dbk::scan_group& j = a.g[gi];
    if constexpr (MT == 16 || MT == 24 || MT == 32) {
        if (a.wide[gi]) {
            if (j.ptype == DBK_PT_MAX)
                scanpool_fprop_mfma_body<DBK_PT_MAX, true, false, MT / 4>(wg, j.W, j.bias, a.m, j.F, j.X, a.N, a.R, a.P, j.pooled, j.argmax, nullptr);
            else if (j.ptype == DBK_PT_ALL)
                scanpool_fprop_mfma_body<DBK_PT_ALL, true, true, MT / 4>(wg, j.W, j.bias, a.m, j.F, j.X, a.N, a.R, a.P, j.pooled, j.argmax, j.act);
            else
                scanpool_fprop_mfma_body<DBK_PT_AVG, false, true, MT / 4>(wg, j.W, j.bias, a.m, j.F, j.X, a.N, a.R, a.P, j.pooled, nullptr, j.act);
            return;
        }
    }
    if (j.ptype == DBK_PT_MAX)
        scanpool_fprop_body<DBK_PT_MAX, true, MT>(wg, j.W, j.bias, a.m, j.F, j.X, a.N, a.R, a.P, j.pooled, j.argmax, nullptr);
    else if (j.ptype == DBK_PT_ALL)
        scanpool_fprop_body<DBK_PT_ALL, true, MT>(wg, j.W, j.bias, a.m, j.F, j.X, a.N, a.R, a.P, j.pooled, j.argmax, j.act);
    else
        scanpool_fprop_body<DBK_PT_AVG, false, MT>(wg, j.W, j.bias, a.m, j.F, j.X, a.N, a.R, a.P, j.pooled, nullptr, j.act);
}

// The counting kernel; for max pooling the bit kernel, over long regions the one-wave sparse kernel in the first wave of the
// workgroup (the other waves leave at once).
template <int MT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(MT == 32 ? 2 : 3))) void scanpool_bprop_multi_kernel(const multi_args a)
{
    wg_t wg;
    const unsigned gi = multi_locate(a, wg);
    const dbk::scan_group& j = a.g[gi];
    if (j.ptype == DBK_PT_MAX) {
        if (a.wide[gi] == 2u)
            scanpool_bprop_counts_body<DBK_PT_MAX, MT>(wg, a.m, j.F, j.X, a.N, a.R, a.P, j.pooled, j.argmax, j.dpooled, nullptr, j.slabs, j.slab_stride);
        else if (a.wide[gi])
            scanpool_bprop_bits_body<MT>(wg, a.m, j.F, j.X, a.N, a.R, a.P, j.pooled, j.argmax, j.dpooled, j.slabs, j.slab_stride);
        else if (threadIdx.x < 64)
            scanpool_bprop_sparse_body<DBK_PT_MAX, MT>(wg, a.m, j.F, j.X, a.N, a.P, j.pooled, j.argmax, j.dpooled, j.slabs, j.slab_stride);
    } else if (j.ptype == DBK_PT_ALL) {
        scanpool_bprop_counts_body<DBK_PT_ALL, MT>(wg, a.m, j.F, j.X, a.N, a.R, a.P, j.pooled, j.argmax, j.dpooled, j.act, j.slabs, j.slab_stride);
    } else {
        scanpool_bprop_counts_body<DBK_PT_AVG, MT>(wg, a.m, j.F, j.X, a.N, a.R, a.P, j.pooled, j.argmax, j.dpooled, j.act, j.slabs, j.slab_stride);
    }
}

inline unsigned multi_tier(size_t m) { return m <= 8 ? 8u : (m <= 16 ? 16u : (m <= 24 ? 24u : (m <= 32 ? 32u : 0u))); }

template <typename K>
int launch_multi(K kern, hipStream_t st, size_t smem, const multi_args& a)
{
    DBK_HIP(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
    hipLaunchKernelGGL(kern, dim3(a.first[a.n]), dim3(256), smem, st, a);
    DBK_LAUNCH_OK();
}

}  // namespace dbk_scanpool_general

namespace dbk_scanpool_digits {
bool takes(size_t m, size_t F, size_t N, size_t P, bool argmax);
}

namespace dbk {

using namespace dbk_scanpool_general;

bool scan_multi_takes(size_t m, size_t N, size_t P, unsigned n, const scan_group* g)
{
    if (n < 1 || n > MULTI_MAX || multi_tier(m) == 0 || P == 0 || N == 0) return false;
    for (unsigned i = 0; i < n; ++i) {
        if (g[i].F == 0 || dbk::divup(g[i].F, FT) > 65535u) return false;
        if (g[i].ptype != DBK_PT_MAX && g[i].ptype != DBK_PT_AVG && g[i].ptype != DBK_PT_ALL) return false;
        if (g[i].ptype != DBK_PT_MAX && !g[i].act) return false;      // the dense backward kernel here is the mask-driven one
        if (g[i].ptype != DBK_PT_AVG && !g[i].argmax) return false;
        // a max-pooling group on a batch large enough for the bulk kernel goes there when stepped alone (other sums, other bits)
        if (g[i].ptype == DBK_PT_MAX && dbk_scanpool_digits::takes(m, g[i].F, N, P, true)) return false;
    }
    return fprop_smem(multi_tier(m), m) <= lds_limit() && wide_smem(24) <= lds_limit() && sparse_smem(m) <= lds_limit() && bits_smem(multi_tier(m)) <= lds_limit();
}

int scan_fprop_multi(hipStream_t st, size_t m, size_t N, const uint32_t* R, size_t P, unsigned n, const scan_group* g)
{
    const unsigned mt = multi_tier(m);
    multi_args a;
    a.n = n; a.m = (unsigned)m; a.N = N; a.P = P; a.R = R;
    a.first[0] = 0;
    bool any_wide = false;
    unsigned tiles = 0;
    for (unsigned i = 0; i < n; ++i) tiles += dbk::divup(g[i].F, FT);
    for (unsigned i = 0; i < n; ++i) {
        a.g[i] = g[i];
        a.ftiles[i] = dbk::divup(g[i].F, FT);
        a.wide[i] = mfma_pays(m, a.ftiles[i], P);                 // the kernel body the group's own launch would choose
        // the groups share the GPU: the grids are sized so that all of them are resident together, and a workgroup
        // amortises its filter tile's table over more regions (a region's results do not depend on the grid)
        a.gx[i] = a.wide[i] ? mfma_grid_x(tiles, P) : fprop_grid_x(mt, tiles, P);
        a.first[i + 1] = a.first[i] + a.gx[i] * a.ftiles[i];
        if (a.wide[i]) any_wide = true;
    }
    size_t smem = fprop_smem(mt, m);
    if (any_wide && MFMA_SMEM > smem) smem = MFMA_SMEM;
    if (mt == 8) return launch_multi(scanpool_fprop_multi_kernel<8>, st, smem, a);
    if (mt == 16) return launch_multi(scanpool_fprop_multi_kernel<16>, st, smem, a);
    if (mt == 24) return launch_multi(scanpool_fprop_multi_kernel<24>, st, smem, a);
    return launch_multi(scanpool_fprop_multi_kernel<32>, st, smem, a);
}

int scan_bprop_multi(hipStream_t st, size_t m, size_t N, const uint32_t* R, size_t P, unsigned n, scan_group* g)
{
    const unsigned mt = multi_tier(m);
    multi_args a;
    a.n = n; a.m = (unsigned)m; a.N = N; a.P = P; a.R = R;
    a.first[0] = 0;
    size_t total = 0;
    for (unsigned i = 0; i < n; ++i) {
        a.ftiles[i] = dbk::divup(g[i].F, FT);
        // as the group's own launch would choose: the counting kernel, for max pooling the bit kernel or, over long regions, the sparse one
        a.wide[i] = g[i].ptype != DBK_PT_MAX ? 1u : counts_takes_max(mt, a.ftiles[i], N, P) ? 2u : bits_takes_max(N, P) ? 1u : 0u;
        a.gx[i] = g[i].ptype != DBK_PT_MAX ? counts_grid_x(mt, a.ftiles[i], N, P) : a.wide[i] == 2u ? counts_max_grid_x(mt, a.ftiles[i], N, P)
                : a.wide[i] ? bits_grid_x(mt, a.ftiles[i], P) : sparse_grid_x(a.ftiles[i], P);
        a.first[i + 1] = a.first[i] + a.gx[i] * a.ftiles[i];
        g[i].slab_stride = 4 * m * (size_t)g[i].F + g[i].F;
        g[i].nslab = a.wide[i] == 2u ? 2 * a.gx[i] : a.gx[i];
        total += g[i].slab_stride * g[i].nslab;
    }
    float* slabs = (float*)dbk::workspace(total * sizeof(float), st);
    DBK_CHECK(slabs != nullptr, "MemoryError: could not allocate %zu bytes of scratch (%s)", total * sizeof(float), dbk::workspace_error());
    for (unsigned i = 0; i < n; ++i) {
        g[i].slabs = slabs;
        slabs += g[i].slab_stride * g[i].nslab;
        a.g[i] = g[i];
    }
    const size_t ss = sparse_smem(m), sd = bits_smem(mt);
    const size_t smem = ss > sd ? ss : sd;
    if (mt == 8) return launch_multi(scanpool_bprop_multi_kernel<8>, st, smem, a);
    if (mt == 16) return launch_multi(scanpool_bprop_multi_kernel<16>, st, smem, a);
    if (mt == 24) return launch_multi(scanpool_bprop_multi_kernel<24>, st, smem, a);
    return launch_multi(scanpool_bprop_multi_kernel<32>, st, smem, a);
}

}  // namespace dbk

namespace dbk_scanpool_digits {
// Bulk path (6-bit digits on the matrix cores); returns -1 when the shape is outside what it handles.
int fprop(hipStream_t st, const float* W, const float* bias, size_t m, size_t F, const uint8_t* X, size_t N,
          const uint32_t* R, size_t P, int ptype, float* pooled, uint32_t* argmax);
}

extern "C" {

int dbk_scanpool_fprop_general(dbk_stream_t stream, const float* W, const float* bias, size_t m, size_t nfilter,
                               const uint8_t* X, size_t N, const uint32_t* regions, size_t nregion, int ptype,
                               float* pooled, uint32_t* argmax, uint64_t* act)
{
    // sum pooling has no fused kernel: the operator chain computes it (no activity masks are written)
    if (ptype == DBK_PT_SUM) return dbk_scanpool_fprop_unfused(stream, W, bias, m, nfilter, X, N, regions, nregion, 2, ptype, pooled, argmax);
    DBK_CHECK(ptype == DBK_PT_MAX || ptype == DBK_PT_AVG || ptype == DBK_PT_ALL, "ValueError: unknown pooling type %d", ptype);
    DBK_CHECK(m >= 1, "ValueError: filter length must be >= 1");
    DBK_CHECK(!(argmax && ptype == DBK_PT_AVG), "ValueError: pooledmaps_argmax can only be used for max/all pooling.");
    // argmax entries are flat 32-bit indices row*nfilter + f into the (virtual) map, as in the reference (uindex_t)
    DBK_CHECK(!argmax || (double)N * (double)nfilter <= 4294967296.0,
              "ValueError: %zu rows x %zu filters overflow the 32-bit argmax index; score in smaller batches or without argmax", N, nfilter);
    if (nfilter == 0 || nregion == 0) { dbk::clear_error(); return 0; }
    DBK_CHECK(W && bias && X && regions && pooled, "ValueError: null pointer argument");
    return dbk_scanpool_general::fprop(dbk::as_stream(stream), W, bias, m, nfilter, X, N, regions, nregion, ptype, pooled, argmax,
                                       reinterpret_cast<unsigned long long*>(act));
}

int dbk_scanpool_fprop_wide(dbk_stream_t stream, const float* W, const float* bias, size_t m, size_t nfilter,
                            const uint8_t* X, size_t N, const uint32_t* regions, size_t nregion, int ptype,
                            float* pooled, uint32_t* argmax, uint64_t* act)
{
    DBK_CHECK(ptype == DBK_PT_MAX || ptype == DBK_PT_AVG || ptype == DBK_PT_ALL, "ValueError: fused pooling type must be max, avg or all (got %d)", ptype);
    DBK_CHECK(m > 8 && m <= 24, "NotImplementedError: the wide forward kernel takes filters of 9 to 24 taps (got %zu)", m);
    DBK_CHECK(!(argmax && ptype == DBK_PT_AVG), "ValueError: pooledmaps_argmax can only be used for max/all pooling.");
    DBK_CHECK(!argmax || (double)N * (double)nfilter <= 4294967296.0,
              "ValueError: %zu rows x %zu filters overflow the 32-bit argmax index; score in smaller batches or without argmax", N, nfilter);
    if (nfilter == 0 || nregion == 0) { dbk::clear_error(); return 0; }
    DBK_CHECK(W && bias && X && regions && pooled, "ValueError: null pointer argument");
    return dbk_scanpool_general::fprop_wide(dbk::as_stream(stream), W, bias, m, nfilter, X, N, regions, nregion, ptype, pooled, argmax,
                                            reinterpret_cast<unsigned long long*>(act));
}

int dbk_scanpool_fprop_mfma(dbk_stream_t stream, const float* W, const float* bias, size_t m, size_t nfilter,
                            const uint8_t* X, size_t N, const uint32_t* regions, size_t nregion, int ptype,
                            float* pooled, uint32_t* argmax, uint64_t* act)
{
    DBK_CHECK(ptype == DBK_PT_MAX || ptype == DBK_PT_AVG || ptype == DBK_PT_ALL, "ValueError: fused pooling type must be max, avg or all (got %d)", ptype);
    DBK_CHECK(dbk_scanpool_general::mfma_takes(m), "NotImplementedError: the matrix-core forward kernel takes filters of 1 to 32 taps (got %zu)", m);
    DBK_CHECK(!(argmax && ptype == DBK_PT_AVG), "ValueError: pooledmaps_argmax can only be used for max/all pooling.");
    DBK_CHECK(!argmax || (double)N * (double)nfilter <= 4294967296.0,
              "ValueError: %zu rows x %zu filters overflow the 32-bit argmax index; score in smaller batches or without argmax", N, nfilter);
    if (nfilter == 0 || nregion == 0) { dbk::clear_error(); return 0; }
    DBK_CHECK(W && bias && X && regions && pooled, "ValueError: null pointer argument");
    return dbk_scanpool_general::fprop_mfma(dbk::as_stream(stream), W, bias, m, nfilter, X, N, regions, nregion, ptype, pooled, argmax,
                                            reinterpret_cast<unsigned long long*>(act));
}

int dbk_scanpool_fprop(dbk_stream_t stream, const float* W, const float* bias, size_t m, size_t nfilter,
                       const uint8_t* X, size_t N, const uint32_t* regions, size_t nregion, int ptype,
                       float* pooled, uint32_t* argmax, uint64_t* act)
{
    // sum pooling has no fused kernel: the operator chain computes it (no activity masks are written)
    if (ptype == DBK_PT_SUM) return dbk_scanpool_fprop_unfused(stream, W, bias, m, nfilter, X, N, regions, nregion, 2, ptype, pooled, argmax);
    DBK_CHECK(ptype == DBK_PT_MAX || ptype == DBK_PT_AVG || ptype == DBK_PT_ALL, "ValueError: unknown pooling type %d", ptype);
    DBK_CHECK(m >= 1, "ValueError: filter length must be >= 1");
    DBK_CHECK(!(argmax && ptype == DBK_PT_AVG), "ValueError: pooledmaps_argmax can only be used for max/all pooling.");
    // argmax entries are flat 32-bit indices row*nfilter + f into the (virtual) map, as in the reference (uindex_t)
    DBK_CHECK(!argmax || (double)N * (double)nfilter <= 4294967296.0,
              "ValueError: %zu rows x %zu filters overflow the 32-bit argmax index; score in smaller batches or without argmax", N, nfilter);
    if (nfilter == 0 || nregion == 0) { dbk::clear_error(); return 0; }
    DBK_CHECK(W && bias && X && regions && pooled, "ValueError: null pointer argument");
    // the activity masks are written by the general path only (the bulk kernel is for scoring, where no backward pass follows)
    if (!act) {
        int rc = dbk_scanpool_digits::fprop(dbk::as_stream(stream), W, bias, m, nfilter, X, N, regions, nregion, ptype, pooled, argmax);
        if (rc >= 0) return rc;
    }
    return dbk_scanpool_general::fprop(dbk::as_stream(stream), W, bias, m, nfilter, X, N, regions, nregion, ptype, pooled, argmax,
                                       reinterpret_cast<unsigned long long*>(act));
}

int dbk_scanpool_bprop(dbk_stream_t stream, const float* W, const float* bias, size_t m, size_t nfilter,
                       const uint8_t* X, size_t N, const uint32_t* regions, size_t nregion, int ptype,
                       const float* pooled, const uint32_t* argmax, const float* dpooled, float* dW, float* dbias, int overwrite,
                       const uint64_t* act)
{
    using namespace dbk_scanpool_general;
    if (ptype == DBK_PT_SUM && !dbk::deferred())
        return dbk_scanpool_bprop_unfused(stream, W, bias, m, nfilter, X, N, regions, nregion, 2, ptype, argmax, dpooled, dW, dbias, overwrite);
    DBK_CHECK(ptype == DBK_PT_MAX || ptype == DBK_PT_AVG || ptype == DBK_PT_ALL, "ValueError: fused pooling type must be max, avg or all (got %d)", ptype);
    DBK_CHECK(m >= 1, "ValueError: filter length must be >= 1");
    if (nfilter == 0) { dbk::clear_error(); return 0; }
    DBK_CHECK(W && bias && dW && dbias, "ValueError: null pointer argument");
    if (nregion == 0 && dbk::deferred()) {
        dbk::deferred()->slabs = nullptr;                          // zero slabs: the gradient is zero
        dbk::deferred()->slab_stride = 4 * m * nfilter + nfilter;
        dbk::deferred()->nslab = 0;
        dbk::clear_error();
        return 0;
    }
    if (nregion == 0) {
        // no regions: the bias gradient is written as zero by the slab reduction over zero slabs
        // (a kernel rather than a memset, so that the call can sit in a captured graph)
        hipLaunchKernelGGL(reduce_slabs_kernel, dim3(dbk::ew_grid(nfilter)), dim3(256), 0, dbk::as_stream(stream), dW, dbias,
                           (const float*)nullptr, (size_t)(overwrite ? 4 * m * nfilter : 0), nfilter, 0u, overwrite != 0);
        DBK_LAUNCH_OK();
    }
    DBK_CHECK(ptype == DBK_PT_AVG || argmax != nullptr, "ValueError: pooledmaps_argmax must be specified for max pooling.");
    DBK_CHECK(X && regions && pooled && dpooled, "ValueError: null pointer argument");
    hipStream_t st = dbk::as_stream(stream);
    const unsigned long long* am = reinterpret_cast<const unsigned long long*>(act);
    switch (ptype) {
    case DBK_PT_MAX: return launch_bprop_pt<DBK_PT_MAX>(st, W, bias, m, nfilter, X, N, regions, nregion, pooled, argmax, dpooled, dW, dbias, overwrite != 0, am);
    case DBK_PT_AVG: return launch_bprop_pt<DBK_PT_AVG>(st, W, bias, m, nfilter, X, N, regions, nregion, pooled, argmax, dpooled, dW, dbias, overwrite != 0, am);
    default:         return launch_bprop_pt<DBK_PT_ALL>(st, W, bias, m, nfilter, X, N, regions, nregion, pooled, argmax, dpooled, dW, dbias, overwrite != 0, am);
    }
}

}  // extern "C"
