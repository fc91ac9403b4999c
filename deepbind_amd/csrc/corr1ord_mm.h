// The two gradients of the drop-in scan as products on the 16 x 16 x 4 matrix instructions of their own float type
// (v_mfma_f64_16x16x4_f64, v_mfma_f32_16x16x4_f32): exact products, accumulation in the type itself, one fixed order.
// reference: corr1ord_bprop.cuh:57-139 (filters), corr1ord_bprop.cu:167-224 (inputs)
#pragma once
#include "scan_common.h"
#include "mfma_common.h"

namespace dbk_corr_mm {

using namespace dbk_scan;

// D (16 x 16) += A (16 x 4) . B (4 x 16). Lane l supplies row / column l & 15 and contraction value l >> 4; it receives column
// l & 15, rows row(0 .. 3, l >> 4).
template <typename T> struct mm16;
template <> struct mm16<double> {
    typedef double acc_t __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ acc_t mul(double a, double b, acc_t c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }
    static __device__ __forceinline__ unsigned row(unsigned i, unsigned g) { return 4u * i + g; }
    static __device__ __forceinline__ double share(unsigned letter, unsigned c)      // of a letter in channel c: 1, the mean's quarter, or nothing
    {
        return __hiloint2double(letter == c ? 0x3ff00000 : (letter == 4u ? 0x3fd00000 : 0), 0);
    }
};
template <> struct mm16<float> {
    typedef float acc_t __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ acc_t mul(float a, float b, acc_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
    static __device__ __forceinline__ unsigned row(unsigned i, unsigned g) { return 4u * g + i; }
    static __device__ __forceinline__ float share(unsigned letter, unsigned c)
    {
        return __uint_as_float(letter == c ? 0x3f800000u : (letter == 4u ? 0x3e800000u : 0u));
    }
};

// ---------------------------------------------------------------------------------------------
// filter gradient: dW (4m x F) = H^T (4m x n) . dZ (n x F), H the one-hot windows
// ---------------------------------------------------------------------------------------------
// A wave owns 16 filters and all taps (a tile of 16 rows of dW is 4 taps x 4 letters; TT tiles, in registers) and walks its rows
// four at a time. Of the one-hot operand nothing is stored: row i, contraction value k of tile t at row p is the letter at
// p + k + 4 t + (i >> 2) held against i & 3, so tile t at one step is tile 0 at t steps on: ONE new operand per step (a byte of
// LDS and three instructions) serves TT products. The rows of dZ are requested eight steps ahead. The four waves of a
// workgroup are folded in wave order, the workgroups' results by the reduction every filter gradient ends with.
// Bound by the matrix pipe: N F m / 4 / 16 products of 64 (float64) or 32 (float32) clocks. Measured, us
// a call with the reduction: float64, 123 000 rows x 64 filters of 24 taps 55 (the kernel with per-wave tables in LDS, one read-modify-
// write per row and tap: 876); float32, 250 000 x 16 filters of 24 taps 45 (one register add per row and tap: 68), 60 000 x 16 of 32 taps 21
// (tables in LDS: 497).
// A product with a zero of the one-hot operand is no zero where dZ is infinite or not a number: a wave that has met such a value adds
// its rows again one by one, each to the rows of dW its letters name and to no other.
constexpr unsigned CW_CHUNK = 256;                                  // rows whose letters a wave stages at a time
template <int TT> struct cw_lds { static constexpr unsigned letters = CW_CHUNK + 4 * TT + 4; };

template <typename T, int TT>
__global__ __launch_bounds__(256) void corr1ord_bprop_W_mm_kernel(T* __restrict__ partial, unsigned m, unsigned F, const uint8_t* __restrict__ X,
                                                                  size_t n, const T* __restrict__ dZ, unsigned rows_per_wave)
{
    typedef typename mm16<T>::acc_t acc_t;
    extern __shared__ __align__(16) unsigned char smem[];           // letters of the four waves, then (at the end) their tiles
    const unsigned lane = threadIdx.x & 63, wave = (unsigned)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const unsigned col = lane & 15u, k = lane >> 4, shift = k + (col >> 2), c = col & 3u;
    const unsigned f = blockIdx.x * 16u + col;
    const size_t N = n + m - 1;
    uint8_t* xl = smem + wave * cw_lds<TT>::letters;
    const size_t r0 = ((size_t)blockIdx.y * 4 + wave) * rows_per_wave;
    const size_t r1 = r0 + rows_per_wave < n ? r0 + rows_per_wave : n;
    acc_t acc[TT];
#pragma unroll
    for (int t = 0; t < TT; ++t) acc[t] = (acc_t)(T)0;
    const T* src = dZ + (f < F ? f : F - 1);
    bool odd = false;
    auto fetch = [&](size_t p, T (&b)[8]) {                         // rows p + k, p + 4 + k, ..: eight steps
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const size_t row = p + 4u * u + k;
            const T v = src[(row < n ? row : n - 1) * F];
            b[u] = row < r1 && f < F ? v : (T)0;
            odd |= !__builtin_isfinite(b[u]);
        }
    };
    T b[8], bn[8];
    if (r0 < r1) fetch(r0, b);
    for (size_t c0 = r0; c0 < r1; c0 += CW_CHUNK) {
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (unsigned e = 0; e < 2; ++e) {
            const unsigned at = 4u * lane + 256u * e;
            if (at < cw_lds<TT>::letters) {
                const unsigned v = dbk_mfma::load_letters4(X, N, c0 + at);
                unsigned l = 0;
#pragma unroll
                for (int t = 0; t < 4; ++t) l |= letter_of((v >> (8 * t)) & 0xffu) << (8 * t);
                *reinterpret_cast<unsigned*>(xl + at) = l;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        T a[8 + TT - 1];
#pragma unroll
        for (int t = 0; t < TT - 1; ++t) a[t] = mm16<T>::share(xl[4 * t + shift], c);
        for (unsigned s = 0; s < CW_CHUNK / 32; ++s) {
            if (c0 + 32u * s >= r1) break;
            fetch(c0 + 32u * (s + 1), bn);
#pragma unroll
            for (int u = 0; u < 8; ++u) a[TT - 1 + u] = mm16<T>::share(xl[32u * s + 4 * (TT - 1 + u) + shift], c);
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int t = 0; t < TT; ++t) acc[t] = mm16<T>::mul(a[u + t], b[u], acc[t]);
#pragma unroll
            for (int t = 0; t < TT - 1; ++t) a[t] = a[8 + t];
#pragma unroll
            for (int u = 0; u < 8; ++u) b[u] = bn[u];
        }
    }
    __syncthreads();                                                // (the letters are no longer read)
    T* tiles = reinterpret_cast<T*>(smem);                          // [wave][TT][16][16]
    if (__ballot(odd) == 0) {
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
            for (unsigned i = 0; i < 4; ++i) tiles[((wave * TT + t) * 16 + mm16<T>::row(i, k)) * 16 + col] = acc[t][i];
    } else {
        T* mine = tiles + wave * TT * 256u + col;                   // row 4 j + l of dW, this lane's filter; taps k, k + 4, .. are this lane's
        for (unsigned j = k; j < 4u * TT; j += 4)
            for (unsigned l = 0; l < 4; ++l) mine[(4 * j + l) * 16] = (T)0;
        for (size_t p = r0; p < r1 && f < F; ++p) {
            const T v = dZ[p * F + f];
            for (unsigned j = k; j < m; j += 4) {
                const unsigned letter = letter_of(X[p + j]);
                for (unsigned l = 0; l < 4; ++l)
                    if (letter == l || letter == 4u) mine[(4 * j + l) * 16] += letter == 4u ? v * (T)0.25 : v;
            }
        }
    }
    __syncthreads();
    T* out = partial + (size_t)blockIdx.y * 4 * m * F;
    for (unsigned e = threadIdx.x; e < TT * 256u; e += 256u) {
        const unsigned row = e >> 4, fl = blockIdx.x * 16u + (e & 15u);
        const T v = ((tiles[e] + tiles[TT * 256 + e]) + tiles[2 * TT * 256 + e]) + tiles[3 * TT * 256 + e];
        if (row < 4 * m && fl < F) out[(size_t)row * F + fl] = v;
    }
}

// ---------------------------------------------------------------------------------------------
// input gradient: dX[q, c] += sum over taps j and filters f of dZ[q - j, f] W[4j + c, f]
// ---------------------------------------------------------------------------------------------
// Four output rows side by side fill the instruction's 16 columns: with q = 4 r + s,
//     dX[4 r + s, c] = sum over d, f of dZ[4 r + d, f] . V_d[f, (s, c)],   V_d[f, (s, c)] = W[4 (s - d) + c, f] where 0 <= s - d < m, else 0,
// d from -(m - 1) to 3: m + 3 steps where m would do, and no sum over taps of an intermediate (rows x 4m) product. A
// workgroup takes 256 rows of dX (64 per wave) and passes over the filters 16 at a time: those columns of the rows of dZ and of
// W lie in LDS at a stride of 17, so that the 16 lanes that read rows four apart, or 16 rows of W, meet no bank twice. Per
// product one element of either operand per lane; one fixed order (filter tiles, d, filters, ascending), so that a row's bits do
// not depend on its place in the batch.
// The next 16 filters' columns are requested while these are multiplied and wait in registers (sized for up to MT taps): with the loads
// behind the barrier a call of few waves spent most of its time on their latency (us a call, before / now: 123 000 rows x 64 filters
// of 24 taps float64 70 / 48, float32 34 / 27; 20 000 x 256 95 / 48, 64 / 29; 250 000 x 64 of 8 taps 95 / 52, 42 / 28).
// Bound by the matrix pipe at F (m + 3) / 4 products of 64 (float64) or 32 (float32) clocks per 64 rows, the LDS reads of its operands beside
// it. Against the kernels before: float64, 123 000 x 64 444 us (one wave per row); float32, 250 000 x 16 filters 15 against 70
// (one wave per 96 rows and 64 filters, multiply-adds with the weights in registers), 123 000 x 64 55.
constexpr unsigned CX_ST = 17;
// NB blocks of 64 rows per workgroup: 4, a wave each; or 1, whose steps d the four waves share out (wave w takes d = w, w + 4, ..,
// and the four sums are added in wave order), for calls whose rows would otherwise leave CUs idle.
template <typename T> inline size_t cx_smem(size_t m, unsigned nb) { return ((64 * nb + m - 1) + (m + 6) * 4) * CX_ST * sizeof(T); }

template <typename T, unsigned NB, unsigned MT>
__global__ __launch_bounds__(256) void corr1ord_bprop_X_mm_kernel(T* __restrict__ dX, size_t n, const T* __restrict__ W, unsigned m, unsigned F,
                                                                  const T* __restrict__ dZ)
{
    static_assert(NB == 1 || NB == 4, "one block of rows per workgroup, or one per wave");
    typedef typename mm16<T>::acc_t acc_t;
    extern __shared__ __align__(16) unsigned char smem[];
    T* zs = reinterpret_cast<T*>(smem);                             // rows q0 - (m - 1) .. q0 + 64 NB - 1 of dZ, 16 filters
    T* ws = zs + (64 * NB + m - 1) * CX_ST;                         // rows of W for taps -3 .. m + 2 (zero outside 0 .. m - 1)
    const unsigned tid = threadIdx.x, lane = tid & 63, wave = (unsigned)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const unsigned col = lane & 15u, k = lane >> 4;
    const unsigned w0 = NB == 4 ? 64u * wave : 0u, d0 = NB == 4 ? 0u : wave;
    constexpr unsigned DSTEP = NB == 4 ? 1u : 4u;
    const size_t q0 = (size_t)blockIdx.x * (64 * NB);
    bool odd = false;
    acc_t acc = (acc_t)(T)0;
    const T* za = zs + (w0 + 4u * col) * CX_ST + k;                 // A: row 4 r + d of the wave's rows, r = col; d counted from -(m - 1)
    const T* wb = ws + ((m - 1 + 3) * 4u + col) * CX_ST + k;        // B: (s, c) = col at d = -(m - 1): tap s + m - 1
    constexpr unsigned ZE = ((64 * NB + MT - 1) * 16 + 255) / 256, WE = ((MT + 6) * 64 + 255) / 256;
    const unsigned nz = (64 * NB + m - 1) * 16, nw = (m + 6) * 64, er = tid >> 4, ef = tid & 15u;
    T zr[ZE], wr[WE];
    auto fetch = [&](unsigned f0) {                                 // the next 16 filters' columns: always an element of the matrix, kept or not below
        const unsigned fl = f0 + ef < F ? f0 + ef : F - 1;
#pragma unroll
        for (unsigned i = 0; i < ZE; ++i) {
            size_t row = q0 + er + 16 * i;                          // + (m - 1): offset by the rows before the workgroup's
            row = row < m - 1 ? 0 : row - (m - 1);
            zr[i] = dZ[(row < n ? row : n - 1) * F + fl];
        }
#pragma unroll
        for (unsigned i = 0; i < WE; ++i) {
            const unsigned r = er + 16 * i;
            wr[i] = W[(size_t)(r < 12 ? 0 : r - 12 < 4 * m ? r - 12 : 4 * m - 1) * F + fl];
        }
    };
    fetch(0);
    for (unsigned f0 = 0; f0 < F; f0 += 16) {
        __syncthreads();
#pragma unroll
        for (unsigned i = 0; i < ZE; ++i)
            if (tid + 256 * i < nz) {
                const size_t row = q0 + er + 16 * i;
                const T v = row >= m - 1 && row - (m - 1) < n && f0 + ef < F ? zr[i] : (T)0;
                zs[(er + 16 * i) * CX_ST + ef] = v;
                odd |= !__builtin_isfinite(v);
            }
#pragma unroll
        for (unsigned i = 0; i < WE; ++i)
            if (tid + 256 * i < nw) {
                const unsigned r = er + 16 * i;
                const T v = r >= 12 && r - 12 < 4 * m && f0 + ef < F ? wr[i] : (T)0;
                ws[r * CX_ST + ef] = v;
                odd |= !__builtin_isfinite(v);
            }
        __syncthreads();
        if (f0 + 16 < F) fetch(f0 + 16);
#pragma unroll 4
        for (unsigned d = d0; d < m + 3; d += DSTEP) {
#pragma unroll
            for (unsigned s = 0; s < 4; ++s) acc = mm16<T>::mul(za[d * CX_ST + 4 * s], wb[-(int)(d * 4 * CX_ST) + (int)(4 * s)], acc);
        }
    }
    // (a zero beside an infinite value or one that is not a number is no zero of the sum: such rows are added without it)
    if (__syncthreads_or(odd)) {
        for (unsigned e = tid; e < 64 * NB * 4; e += 256) {
            const size_t q = q0 + (e >> 2);
            if (q >= n) break;
            const T* w = W + (size_t)(e & 3u) * F;
            T sum = (T)0;
            for (unsigned j = 0; j < m && j <= q; ++j)
                for (unsigned f = 0; f < F; ++f) sum += dZ[(q - j) * F + f] * w[(size_t)4 * j * F + f];
            dX[q * 4 + (e & 3u)] += sum;
        }
        return;
    }
    if (NB == 1) {
        acc_t* parts = reinterpret_cast<acc_t*>(smem);              // [wave][lane]: less than the staged rows
        parts[tid] = acc;
        __syncthreads();
        if (wave != 0) return;
        acc = ((parts[lane] + parts[64 + lane]) + parts[128 + lane]) + parts[192 + lane];
    }
#pragma unroll
    for (unsigned i = 0; i < 4; ++i) {
        const size_t q = q0 + w0 + 4u * mm16<T>::row(i, k) + (col >> 2);
        if (q < n) dX[q * 4 + (col & 3u)] += acc[i];
    }
}

}  // namespace dbk_corr_mm
