// Region pooling over the rows of an (N, F) feature map and its gradient.
//
// One thread per (region, column): the 64 lanes of a wave take 64 consecutive columns, so every
// row visit is one coalesced 256-byte read (or read-modify-write) of HBM. Rows are visited in
// ascending order, which fixes both the argmax tie rule (first strict maximum) and the order of
// the running sum.
//
// Reference semantics: kangaroo_smat/poolrgn.cuh:44-160 (forward), poolrgn_bprop.cuh:45-127 (gradient).
#include "dbk_common.h"

namespace {

struct region_t { size_t a, b, step, count; };

__device__ __forceinline__ region_t load_region(const uint32_t* __restrict__ R, size_t r, bool per_step)
{
    const uint32_t* p = R + r * (per_step ? 3 : 2);
    region_t g;
    g.a = p[0];
    g.b = p[1];
    g.step = per_step ? p[2] : 1;
    if (g.step == 0) g.step = 1;
    g.count = (g.b - g.a + g.step - 1) / g.step;
    return g;
}

template <typename T, int PT>
__global__ __launch_bounds__(256) void poolrgn_kernel(const T* __restrict__ U, size_t F, const uint32_t* __restrict__ R,
                                                      size_t P, bool per_step, T* __restrict__ pooled,
                                                      uint32_t* __restrict__ argmax)
{
    const size_t f = (size_t)blockIdx.y * 64 + (threadIdx.x & 63);
    const size_t r = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (f >= F || r >= P) return;
    const region_t g = load_region(R, r, per_step);
    size_t xi = g.a * F + f;
    T x = U[xi];
    T y = x;
    auto take = [&](size_t i, T v) {
        if (PT == DBK_PT_MAX || PT == DBK_PT_ALL) {
            if (v > x) { x = v; xi = i * F + f; }
        }
        if (PT != DBK_PT_MAX) y += v;
    };
    // eight rows per round: the loads of a round are in flight together, the rows are still taken in ascending order
    size_t i = g.a + g.step;
    for (; i + 7 * g.step < g.b; i += 8 * g.step) {
        T v[8];
#pragma unroll
        for (int t = 0; t < 8; ++t) v[t] = U[(i + t * g.step) * F + f];
#pragma unroll
        for (int t = 0; t < 8; ++t) take(i + t * g.step, v[t]);
    }
    for (; i < g.b; i += g.step) take(i, U[i * F + f]);
    const size_t j = r * F + f;
    if (PT == DBK_PT_MAX) {
        pooled[j] = x;
    } else if (PT == DBK_PT_SUM) {
        pooled[j] = y;
    } else if (PT == DBK_PT_AVG) {
        pooled[j] = y / (T)g.count;
    } else {
        pooled[2 * j] = x;
        pooled[2 * j + 1] = y / (T)g.count;
    }
    if ((PT == DBK_PT_MAX || PT == DBK_PT_ALL) && argmax) argmax[j] = (uint32_t)xi;
}

// ---- sixteen bytes per lane -----------------------------------------------------------------------------------
// When a row is a whole number of 16-byte packs (four floats, two doubles) a lane takes one pack of one region: V
// neighbouring columns, each pooled exactly as poolrgn_kernel pools it. Thread t owns pack t % (F / V) of region
// t / (F / V), so the lanes of a wave read consecutive packs - whole rows when the map has 256 columns, 16 short
// regions side by side when it has 16 (where the one-column kernel leaves 48 of its 64 lanes idle) - and the map streams
// at 6 TB/s instead of 5.
template <typename T> struct pack_t {
    static constexpr int V = 16 / sizeof(T);
    typedef T type __attribute__((ext_vector_type(16 / sizeof(T))));
    typedef uint32_t index_type __attribute__((ext_vector_type(16 / sizeof(T))));
};

template <typename T, int PT>
__global__ __launch_bounds__(256) void poolrgn_pack_kernel(const T* __restrict__ U, unsigned F, const uint32_t* __restrict__ R,
                                                           unsigned P, bool per_step, T* __restrict__ pooled,
                                                           uint32_t* __restrict__ argmax)
{
    using V4 = typename pack_t<T>::type;
    using I4 = typename pack_t<T>::index_type;
    constexpr int V = pack_t<T>::V;
    const unsigned Fp = F / V;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)P * Fp) return;
    const unsigned r = (unsigned)(t / Fp), f = (unsigned)(t - (size_t)r * Fp) * V;      // region; first of this lane's columns
    const region_t g = load_region(R, r, per_step);
    const V4* Up = reinterpret_cast<const V4*>(U + f);               // row i of the lane's pack: Up[i * Fp]
    V4 x = Up[g.a * Fp], y = x;
    I4 xr;                                                           // row of each column's maximum
#pragma unroll
    for (int k = 0; k < V; ++k) xr[k] = (uint32_t)g.a;
    auto take = [&](size_t i, const V4& v) {
#pragma unroll
        for (int k = 0; k < V; ++k) {
            if (PT == DBK_PT_MAX || PT == DBK_PT_ALL) {
                const bool gt = v[k] > x[k];
                x[k] = gt ? v[k] : x[k];
                xr[k] = gt ? (uint32_t)i : xr[k];
            }
            if (PT != DBK_PT_MAX) y[k] += v[k];
        }
    };
    // ROUND rows per round: the loads of a round are in flight together, the rows are still taken in ascending order
    constexpr int ROUND = 8;
    size_t i = g.a + g.step;
    for (; i + (ROUND - 1) * g.step < g.b; i += ROUND * g.step) {
        V4 v[ROUND];
#pragma unroll
        for (int q = 0; q < ROUND; ++q) v[q] = Up[(i + q * g.step) * Fp];
#pragma unroll
        for (int q = 0; q < ROUND; ++q) take(i + q * g.step, v[q]);
    }
    for (; i < g.b; i += g.step) take(i, Up[i * Fp]);
    I4 xi;
#pragma unroll
    for (int k = 0; k < V; ++k) xi[k] = (uint32_t)((size_t)xr[k] * F + f + k);
    const size_t j = (size_t)r * F + f;
    if (PT == DBK_PT_MAX) {
        *reinterpret_cast<V4*>(pooled + j) = x;
    } else if (PT == DBK_PT_SUM) {
        *reinterpret_cast<V4*>(pooled + j) = y;
    } else if (PT == DBK_PT_AVG) {
        V4 o;
#pragma unroll
        for (int k = 0; k < V; ++k) o[k] = y[k] / (T)g.count;
        *reinterpret_cast<V4*>(pooled + j) = o;
    } else {
        V4 o[2];
#pragma unroll
        for (int k = 0; k < V; ++k) {
            o[(2 * k) / V][(2 * k) % V] = x[k];
            o[(2 * k + 1) / V][(2 * k + 1) % V] = y[k] / (T)g.count;
        }
        reinterpret_cast<V4*>(pooled + 2 * j)[0] = o[0];
        reinterpret_cast<V4*>(pooled + 2 * j)[1] = o[1];
    }
    if ((PT == DBK_PT_MAX || PT == DBK_PT_ALL) && argmax) *reinterpret_cast<I4*>(argmax + j) = xi;
}

// Maximum pooling of few (region, pack) items: SPLIT lanes share an item, each taking a run of the region's rows; the runs'
// maxima meet by lane exchanges, the earlier run winning ties, so the result is the first strict maximum as above (a region's
// first row counts whatever it holds, later rows only where they exceed: a NaN behaves as in the one-lane kernel). With a lane per
// item 2000 regions x 16 columns keep 125 waves busy with 124 dependent rows each: 34 us for 16 MB, under 9 this way; 1000
// regions x 64 doubles 35 us, 14.
template <typename T, int SPLIT>
__global__ __launch_bounds__(256) void poolrgn_max_split_kernel(const T* __restrict__ U, unsigned F, const uint32_t* __restrict__ R, unsigned P, bool per_step,
                                                                T* __restrict__ pooled, uint32_t* __restrict__ argmax)
{
    using V4 = typename pack_t<T>::type;
    using I4 = typename pack_t<T>::index_type;
    constexpr int V = pack_t<T>::V;
    constexpr unsigned ITEMS = 64 / SPLIT;                           // items of a wave: neighbouring packs, so that a run reads ITEMS x 16 bytes at once
    const unsigned Fp = F / V, lane = threadIdx.x & 63, run = lane / ITEMS;
    const size_t wave = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    size_t t = wave * ITEMS + lane % ITEMS;
    const bool live = t < (size_t)P * Fp;
    if (!live) t = (size_t)P * Fp - 1;
    const unsigned r = (unsigned)(t / Fp), f = (unsigned)(t - (size_t)r * Fp) * V;
    const region_t g = load_region(R, r, per_step);
    const V4* Up = reinterpret_cast<const V4*>(U + f);
    V4 x;
    I4 xr;
#pragma unroll
    for (int k = 0; k < V; ++k) { x[k] = (T)-INFINITY; xr[k] = (uint32_t)g.a; }
    size_t per = (g.count + SPLIT - 1) / SPLIT;
    if (per < 1) per = 1;
    size_t n0 = run * per, n1 = n0 + per < g.count ? n0 + per : g.count;    // rows of the region, counted from its first
    if (run == 0) { x = Up[g.a * Fp]; n0 = 1; }                      // (also where the region is empty, as the one-lane kernel does)
    auto take = [&](size_t i, const V4& v) {
#pragma unroll
        for (int k = 0; k < V; ++k) {
            const bool gt = v[k] > x[k];
            x[k] = gt ? v[k] : x[k];
            xr[k] = gt ? (uint32_t)i : xr[k];
        }
    };
    size_t q = n0;
    for (; q + 7 < n1; q += 8) {
        V4 v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = Up[(g.a + (q + u) * g.step) * Fp];
#pragma unroll
        for (int u = 0; u < 8; ++u) take(g.a + (q + u) * g.step, v[u]);
    }
    for (; q < n1; ++q) take(g.a + q * g.step, Up[(g.a + q * g.step) * Fp]);
#pragma unroll
    for (unsigned d = ITEMS; d < 64; d <<= 1) {
#pragma unroll
        for (int k = 0; k < V; ++k) {
            const T ox = __shfl_down(x[k], d, 64);
            const uint32_t orow = (uint32_t)__shfl_down((int)xr[k], d, 64);
            const bool gt = ox > x[k];
            x[k] = gt ? ox : x[k];
            xr[k] = gt ? orow : xr[k];
        }
    }
    if (run != 0 || !live) return;
    const size_t j = (size_t)r * F + f;
    *reinterpret_cast<V4*>(pooled + j) = x;
    if (argmax) {
        I4 xi;
#pragma unroll
        for (int k = 0; k < V; ++k) xi[k] = (uint32_t)((size_t)xr[k] * F + f + k);
        *reinterpret_cast<I4*>(argmax + j) = xi;
    }
}

// LDS the packed forward asks for without using it: 40 KB leave four workgroups per CU instead of eight, and with fewer
// regions being read at the same time the map streams ~6 % faster (5.3 -> 5.6 TB/s at 8192 regions x 124 rows x 256).
constexpr size_t PACK_LDS_CAP = 40 * 1024;
template <typename T>
bool pack_shape(const void* U, size_t F, size_t P, const void* pooled, const void* index)
{
    constexpr size_t V = 16 / sizeof(T);
    return F % V == 0 && (double)P * (double)(F / V) < 2147483648.0 * 256.0 && F < 0x80000000u && P < 0x80000000u &&
           ((reinterpret_cast<uintptr_t>(U) | reinterpret_cast<uintptr_t>(pooled)) & 15u) == 0 &&
           (reinterpret_cast<uintptr_t>(index) & (4 * V - 1)) == 0;
}

// flag[0] = 1 when regions are sorted, unit-step and non-overlapping (each map element then has a
// single writer in the gradient kernel), else 0.
__device__ __forceinline__ bool disjoint_at(const uint32_t* __restrict__ R, size_t P, bool per_step, size_t r)
{
    const unsigned rc = per_step ? 3 : 2;
    const unsigned a = R[r * rc], b = R[r * rc + 1], step = per_step ? R[r * rc + 2] : 1u, next = r + 1 < P ? R[(r + 1) * rc] : b;
    return b >= a && step == 1u && next >= b;
}

__global__ void regions_disjoint_kernel(const uint32_t* __restrict__ R, size_t P, bool per_step, unsigned* flag)
{
    bool bad = false;
    for (size_t r = threadIdx.x; r < P; r += blockDim.x) bad |= !disjoint_at(R, P, per_step, r);
    bad = __syncthreads_or(bad) != 0;
    if (threadIdx.x == 0) flag[0] = bad ? 0u : 1u;
}

// Few regions: every workgroup looks through the whole table itself, and one launch takes the place of three (the look, the kernel for disjoint
// regions, the one for others, one of which has nothing to do). Up to 1024 regions that is no slower whatever the columns; up to 2048 while all
// workgroups together read no more than 4.6 M entries of the table (the kernel of single columns, which maxima take, has one per 4 regions and 64 columns).
// us, three launches / one, regions of 60 rows: maxima, float32, 1000 regions x 64 columns 6.3 / 4.1, x 1024 31.9 / 30.7, x 4096 182 / 177; 1500 x 512 (4.5 M) 25.7 / 25.4, x 1024 (9 M)
// 49.9 / 52.9; 2048 x 256 19.4 / 18.6, x 512 (8 M) 33.3 / 34.7, x 1024 73.5 / 82.1, float64 76.9 / 90.1; average, rows of 12, 2048 x 512 (2 M) 21.9 / 22.1, x 1024 (4 M)
// 37.9 / 38.2, x 4096 165 / 170, float64 x 1024 67.5 / 71.4. All threads of the workgroup come here.
constexpr size_t CHECK_ALWAYS = 1024, CHECK_REGIONS = 2048, CHECK_ENTRIES = 4600000;
__device__ __forceinline__ bool all_disjoint(const uint32_t* __restrict__ R, unsigned P, bool per_step)
{
    bool bad = false;
    for (unsigned r = threadIdx.x; r < P; r += 256u) bad |= !disjoint_at(R, P, per_step, r);
    return __syncthreads_or(bad) == 0;
}

template <bool ATOMIC, typename T>
__device__ __forceinline__ void accumulate(T* p, T v)
{
    if (ATOMIC) atomicAdd(p, v);
    else *p += v;
}

// One (region, column). ATOMIC=false: regions are disjoint (plain read-modify-write, reproducible); true: they may overlap (same accumulation
// races as any scatter-add).
template <typename T, int PT, bool ATOMIC>
__device__ __forceinline__ void poolrgn_bprop_element(size_t r, size_t f, T* __restrict__ dU, size_t F, const uint32_t* __restrict__ R, bool per_step,
                                                      const T* __restrict__ dP, const uint32_t* __restrict__ argmax)
{
    const region_t g = load_region(R, r, per_step);
    const size_t j = r * F + f;
    // The argmax index is caller data. One that lies in this thread's own column and region (what the forward
    // pass produces) has this thread as its only writer when regions are disjoint: a plain add. Any other index
    // may point anywhere in the map and is added atomically.
    auto scatter = [&](T v) {
        const size_t ai = argmax[j], row = ai / F;
        if (!ATOMIC && ai - row * F == f && row >= g.a && row < g.b) dU[ai] += v;
        else atomicAdd(&dU[ai], v);
    };
    if (PT == DBK_PT_MAX) {
        scatter(dP[j]);
        return;
    }
    T dy;
    if (PT == DBK_PT_ALL) dy = dP[2 * j + 1] / (T)g.count;
    else if (PT == DBK_PT_AVG) dy = dP[j] / (T)g.count;
    else dy = dP[j];
    size_t i = g.a;
    if (!ATOMIC) {
        // eight rows per round: read, add, write, with the eight reads in flight together
        for (; i + 7 * g.step < g.b; i += 8 * g.step) {
            T v[8];
#pragma unroll
            for (int t = 0; t < 8; ++t) v[t] = dU[(i + t * g.step) * F + f];
#pragma unroll
            for (int t = 0; t < 8; ++t) dU[(i + t * g.step) * F + f] = v[t] + dy;
        }
    }
    for (; i < g.b; i += g.step) accumulate<ATOMIC>(&dU[i * F + f], dy);
    if (PT == DBK_PT_ALL) scatter(dP[2 * j]);
}

template <typename T, int PT, bool ATOMIC>
__global__ __launch_bounds__(256) void poolrgn_bprop_kernel(T* __restrict__ dU, size_t F, const uint32_t* __restrict__ R, size_t P, bool per_step,
                                                            const T* __restrict__ dP, const uint32_t* __restrict__ argmax,
                                                            const unsigned* __restrict__ flag)
{
    if ((flag[0] != 0) == ATOMIC) return;
    const size_t f = (size_t)blockIdx.y * 64 + (threadIdx.x & 63), r = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (f < F && r < P) poolrgn_bprop_element<T, PT, ATOMIC>(r, f, dU, F, R, per_step, dP, argmax);
}

template <typename T, int PT>
__global__ __launch_bounds__(256) void poolrgn_bprop_check_kernel(T* __restrict__ dU, size_t F, const uint32_t* __restrict__ R, unsigned P, bool per_step,
                                                                  const T* __restrict__ dP, const uint32_t* __restrict__ argmax)
{
    const bool disjoint = all_disjoint(R, P, per_step);
    const size_t f = (size_t)blockIdx.y * 64 + (threadIdx.x & 63), r = (size_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (f >= F || r >= P) return;
    if (disjoint) poolrgn_bprop_element<T, PT, false>(r, f, dU, F, R, per_step, dP, argmax);
    else poolrgn_bprop_element<T, PT, true>(r, f, dU, F, R, per_step, dP, argmax);
}

// The gradient of average / sum / max+average pooling with sixteen bytes per lane (regions disjoint, rows whole packs):
// thread t adds to pack t % (F / V) of every row of region t / (F / V), as poolrgn_pack_kernel reads them; every column
// receives what poolrgn_bprop_kernel<.., false> gives it, in the same order (the share of the average first, then the
// maximum's).
// PASS (max+average): the maximum's share goes in as its row passes, with the same additions, instead of in four reads and writes of single
// elements behind the loop, each of a whole line that has left the caches by then: 8192 regions x 124 rows x 256 float32 545 -> 434 us,
// 20 000 x 60 x 64 163 -> 131. A map that stays in the caches is faster without (1000 x 123 x 64: 21 us against 24).
// CHECK: the workgroup looks through the table of regions itself (flag is not read).
template <typename T, int PT, bool PASS, bool CHECK = false>
__global__ __launch_bounds__(256) void poolrgn_bprop_pack_kernel(T* __restrict__ dU, unsigned F, const uint32_t* __restrict__ R, unsigned P,
                                                                 bool per_step, const T* __restrict__ dP,
                                                                 const uint32_t* __restrict__ argmax, const unsigned* __restrict__ flag)
{
    using V4 = typename pack_t<T>::type;
    constexpr int V = pack_t<T>::V;
    bool disjoint = true;
    if (CHECK) disjoint = all_disjoint(R, P, per_step);
    else if (flag[0] == 0) return;                                   // overlapping regions: the atomic kernel runs instead
    const unsigned Fp = F / V;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (size_t)P * Fp) return;
    const unsigned r = (unsigned)(t / Fp), f = (unsigned)(t - (size_t)r * Fp) * V;
    if (CHECK && !disjoint) {
#pragma unroll 1
        for (int k = 0; k < V; ++k) poolrgn_bprop_element<T, PT, true>(r, f + k, dU, F, R, per_step, dP, argmax);
        return;
    }
    const region_t g = load_region(R, r, per_step);
    const size_t j = (size_t)r * F + f;
    V4 dy;
    if (PT == DBK_PT_ALL) {
        const V4 a = reinterpret_cast<const V4*>(dP + 2 * j)[0], b = reinterpret_cast<const V4*>(dP + 2 * j)[1];
#pragma unroll
        for (int k = 0; k < V; ++k) dy[k] = ((2 * k + 1) / V ? b : a)[(2 * k + 1) % V] / (T)g.count;
    } else {
        dy = *reinterpret_cast<const V4*>(dP + j);
        if (PT == DBK_PT_AVG) {
#pragma unroll
            for (int k = 0; k < V; ++k) dy[k] = dy[k] / (T)g.count;
        }
    }
    V4 peak = dy;
    size_t top[V];                                                   // rows of the maxima, none where the index is another lane's
#pragma unroll
    for (int k = 0; k < V; ++k) top[k] = ~(size_t)0;
    if (PASS) {
#pragma unroll
        for (int k = 0; k < V; ++k) {
            const size_t ai = argmax[j + k], row = ai / F;
            peak[k] = dP[2 * (j + k)];
            const bool own = ai - row * F == f + k && row >= g.a && row < g.b && (!per_step || (row - g.a) % g.step == 0);
            top[k] = own ? row : ~(size_t)0;
        }
    }
    auto share = [&](V4 x, size_t i) {
        x = x + dy;
        if (PASS) {
#pragma unroll
            for (int k = 0; k < V; ++k) x[k] = i == top[k] ? x[k] + peak[k] : x[k];
        }
        return x;
    };
    V4* Dp = reinterpret_cast<V4*>(dU + f);                          // row i of the lane's pack: Dp[i * Fp]
    size_t i = g.a;
    for (; i + 7 * g.step < g.b; i += 8 * g.step) {
        V4 v[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) v[q] = Dp[(i + q * g.step) * Fp];
#pragma unroll
        for (int q = 0; q < 8; ++q) Dp[(i + q * g.step) * Fp] = share(v[q], i + q * g.step);
    }
    for (; i < g.b; i += g.step) Dp[i * Fp] = share(Dp[i * Fp], i);
    if (PT == DBK_PT_ALL) {
        // a plain add where the index lies in this lane's own column and region, else atomic
#pragma unroll
        for (int k = 0; k < V; ++k) {
            if (PASS && top[k] != ~(size_t)0) continue;
            const size_t ai = argmax[j + k], row = ai / F;
            const T v = dP[2 * (j + k)];
            if (ai - row * F == f + k && row >= g.a && row < g.b) dU[ai] += v;
            else atomicAdd(&dU[ai], v);
        }
    }
}

template <typename T>
int launch_fwd(hipStream_t st, const T* U, size_t F, const uint32_t* R, size_t P, bool per_step, T* pooled,
               uint32_t* argmax, int ptype)
{
    if (pack_shape<T>(U, F, P, pooled, argmax)) {
        const dim3 grid(dbk::divup(P * (F / (16 / sizeof(T))), 256)), block(256);
        const unsigned F32 = (unsigned)F, P32 = (unsigned)P;
        const size_t items = P * (F / (16 / sizeof(T)));
        // Too few items to fill the GPU with a lane each. The regions' lengths are only known on the device: the lines lie where regions of a
        // few rows are no slower either. us, lane per item / this, for regions of 12 and of 124 rows: 16 000 items, 16 lanes each, 4.0 / 4.0
        // and 34 / 10 (at 32 000 items 3.9 / 5.1 and 33 / 18); 32 000, eight lanes, 4.0 / 3.9 and 35 / 13.6; 64 000, four, 3.9 / 3.8 and
        // 35 / 20 (at 130 000 5.4 / 6.5 for 12 rows).
        if (ptype == DBK_PT_MAX && items <= 98304) {
            if (items <= 16384)
                hipLaunchKernelGGL((poolrgn_max_split_kernel<T, 16>), dim3(dbk::divup(items, 16)), block, 0, st, U, F32, R, P32, per_step, pooled, argmax);
            else if (items <= 32768)
                hipLaunchKernelGGL((poolrgn_max_split_kernel<T, 8>), dim3(dbk::divup(items, 32)), block, 0, st, U, F32, R, P32, per_step, pooled, argmax);
            else
                hipLaunchKernelGGL((poolrgn_max_split_kernel<T, 4>), dim3(dbk::divup(items, 64)), block, 0, st, U, F32, R, P32, per_step, pooled, argmax);
            DBK_LAUNCH_OK();
        }
        switch (ptype) {
        case DBK_PT_MAX: hipLaunchKernelGGL((poolrgn_pack_kernel<T, DBK_PT_MAX>), grid, block, PACK_LDS_CAP, st, U, F32, R, P32, per_step, pooled, argmax); break;
        case DBK_PT_AVG: hipLaunchKernelGGL((poolrgn_pack_kernel<T, DBK_PT_AVG>), grid, block, PACK_LDS_CAP, st, U, F32, R, P32, per_step, pooled, argmax); break;
        case DBK_PT_SUM: hipLaunchKernelGGL((poolrgn_pack_kernel<T, DBK_PT_SUM>), grid, block, PACK_LDS_CAP, st, U, F32, R, P32, per_step, pooled, argmax); break;
        default:         hipLaunchKernelGGL((poolrgn_pack_kernel<T, DBK_PT_ALL>), grid, block, PACK_LDS_CAP, st, U, F32, R, P32, per_step, pooled, argmax); break;
        }
        DBK_LAUNCH_OK();
    }
    dim3 grid(dbk::divup(P, 4), dbk::divup(F, 64)), block(256);
    DBK_CHECK(grid.y <= 65535u, "ValueError: too many feature maps (%zu) for one launch", F);
    switch (ptype) {
    case DBK_PT_MAX: hipLaunchKernelGGL((poolrgn_kernel<T, DBK_PT_MAX>), grid, block, 0, st, U, F, R, P, per_step, pooled, argmax); break;
    case DBK_PT_AVG: hipLaunchKernelGGL((poolrgn_kernel<T, DBK_PT_AVG>), grid, block, 0, st, U, F, R, P, per_step, pooled, argmax); break;
    case DBK_PT_SUM: hipLaunchKernelGGL((poolrgn_kernel<T, DBK_PT_SUM>), grid, block, 0, st, U, F, R, P, per_step, pooled, argmax); break;
    default:         hipLaunchKernelGGL((poolrgn_kernel<T, DBK_PT_ALL>), grid, block, 0, st, U, F, R, P, per_step, pooled, argmax); break;
    }
    DBK_LAUNCH_OK();
}

template <typename T, int PT>
void launch_bwd_pt(hipStream_t st, T* dU, size_t F, const uint32_t* R, size_t P, bool per_step, const T* dP,
                   const uint32_t* argmax, const unsigned* flag)
{
    dim3 grid(dbk::divup(P, 4), dbk::divup(F, 64)), block(256);
    if (PT != DBK_PT_MAX && pack_shape<T>(dU, F, P, dP, nullptr)) {
        // (the map's rows are only known on the device: 262 144 packs of regions of ~60 rows and more leave the caches)
        const size_t packs = P * (F / (16 / sizeof(T)));
        const dim3 wgs(dbk::divup(packs, 256));
        if (!flag) {
            auto kern = PT == DBK_PT_ALL && packs >= 262144 ? poolrgn_bprop_pack_kernel<T, PT, PT == DBK_PT_ALL, true> : poolrgn_bprop_pack_kernel<T, PT, false, true>;
            hipLaunchKernelGGL(kern, wgs, block, PACK_LDS_CAP, st, dU, (unsigned)F, R, (unsigned)P, per_step, dP, argmax, flag);
            return;
        }
        auto kern = PT == DBK_PT_ALL && packs >= 262144 ? poolrgn_bprop_pack_kernel<T, PT, PT == DBK_PT_ALL> : poolrgn_bprop_pack_kernel<T, PT, false>;
        hipLaunchKernelGGL(kern, wgs, block, PACK_LDS_CAP, st, dU, (unsigned)F, R, (unsigned)P, per_step, dP, argmax, flag);
    } else if (!flag) {
        hipLaunchKernelGGL((poolrgn_bprop_check_kernel<T, PT>), grid, block, 0, st, dU, F, R, (unsigned)P, per_step, dP, argmax);
        return;
    } else
        hipLaunchKernelGGL((poolrgn_bprop_kernel<T, PT, false>), grid, block, 0, st, dU, F, R, P, per_step, dP, argmax, flag);
    hipLaunchKernelGGL((poolrgn_bprop_kernel<T, PT, true>), grid, block, 0, st, dU, F, R, P, per_step, dP, argmax, flag);
}

template <typename T>
int launch_bwd(hipStream_t st, T* dU, size_t F, const uint32_t* R, size_t P, bool per_step, const T* dP,
               const uint32_t* argmax, int ptype)
{
    DBK_CHECK(dbk::divup(F, 64) <= 65535u, "ValueError: too many feature maps (%zu) for one launch", F);
    const bool packs = ptype != DBK_PT_MAX && pack_shape<T>(dU, F, P, dP, nullptr);
    const size_t wgs = packs ? dbk::divup(P * (F / (16 / sizeof(T))), 256) : (size_t)dbk::divup(P, 4) * dbk::divup(F, 64);
    unsigned* flag = nullptr;
    if (P > CHECK_REGIONS || (P > CHECK_ALWAYS && wgs * P > CHECK_ENTRIES)) {
        flag = (unsigned*)dbk::workspace(256, st);
        // (without the word - a stream under capture that has no scratch yet - few enough regions are looked at by every workgroup all the same)
        DBK_CHECK(flag != nullptr || P <= CHECK_REGIONS, "MemoryError: could not allocate scratch (%s)", dbk::workspace_error());
        if (flag) hipLaunchKernelGGL(regions_disjoint_kernel, dim3(1), dim3(1024), 0, st, R, P, per_step, flag);
    }
    switch (ptype) {
    case DBK_PT_MAX: launch_bwd_pt<T, DBK_PT_MAX>(st, dU, F, R, P, per_step, dP, argmax, flag); break;
    case DBK_PT_AVG: launch_bwd_pt<T, DBK_PT_AVG>(st, dU, F, R, P, per_step, dP, argmax, flag); break;
    case DBK_PT_SUM: launch_bwd_pt<T, DBK_PT_SUM>(st, dU, F, R, P, per_step, dP, argmax, flag); break;
    default:         launch_bwd_pt<T, DBK_PT_ALL>(st, dU, F, R, P, per_step, dP, argmax, flag); break;
    }
    DBK_LAUNCH_OK();
}

}  // namespace

extern "C" {

int dbk_poolrgn(dbk_stream_t stream, int dtype, const void* unpooledmaps, size_t nfeaturemap,
                const uint32_t* regions, size_t nregion, int per_region_step,
                void* pooledmaps, uint32_t* pooledmaps_argmax, int ptype)
{
    DBK_DTYPE_OK(dtype);
    DBK_CHECK(ptype >= DBK_PT_MAX && ptype <= DBK_PT_ALL, "ValueError: unknown pooling type %d", ptype);
    DBK_CHECK(!pooledmaps_argmax || ptype == DBK_PT_MAX || ptype == DBK_PT_ALL,
              "ValueError: pooledmaps_argmax can only be used for max/all pooling.");
    if (nfeaturemap == 0 || nregion == 0) { dbk::clear_error(); return 0; }
    DBK_CHECK(unpooledmaps && regions && pooledmaps, "ValueError: null pointer argument");
    if (dtype == DBK_F32)
        return launch_fwd<float>(dbk::as_stream(stream), (const float*)unpooledmaps, nfeaturemap, regions, nregion,
                                 per_region_step != 0, (float*)pooledmaps, pooledmaps_argmax, ptype);
    return launch_fwd<double>(dbk::as_stream(stream), (const double*)unpooledmaps, nfeaturemap, regions, nregion,
                              per_region_step != 0, (double*)pooledmaps, pooledmaps_argmax, ptype);
}

int dbk_poolrgn_bprop(dbk_stream_t stream, int dtype, void* unpooledmaps, size_t nfeaturemap,
                      const uint32_t* regions, size_t nregion, int per_region_step,
                      const void* pooledmaps, const uint32_t* pooledmaps_argmax, int ptype)
{
    DBK_DTYPE_OK(dtype);
    DBK_CHECK(ptype >= DBK_PT_MAX && ptype <= DBK_PT_ALL, "ValueError: unknown pooling type %d", ptype);
    if (ptype == DBK_PT_MAX || ptype == DBK_PT_ALL)
        DBK_CHECK(pooledmaps_argmax != nullptr, "ValueError: pooledmaps_argmax must be specified for max pooling.");
    else
        DBK_CHECK(pooledmaps_argmax == nullptr, "ValueError: pooledmaps_argmax can only be specified for max pooling.");
    if (nfeaturemap == 0 || nregion == 0) { dbk::clear_error(); return 0; }
    DBK_CHECK(unpooledmaps && regions && pooledmaps, "ValueError: null pointer argument");
    if (dtype == DBK_F32)
        return launch_bwd<float>(dbk::as_stream(stream), (float*)unpooledmaps, nfeaturemap, regions, nregion,
                                 per_region_step != 0, (const float*)pooledmaps, pooledmaps_argmax, ptype);
    return launch_bwd<double>(dbk::as_stream(stream), (double*)unpooledmaps, nfeaturemap, regions, nregion,
                              per_region_step != 0, (const double*)pooledmaps, pooledmaps_argmax, ptype);
}

}  // extern "C"
