// Auxiliary kernels: buffer fills, HU -> density calibration, the
// statistical-uncertainty reduction, Dij compaction into CSR, and the Dij
// forward (D w) / adjoint (D^T g) sparse products.
#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>

#include "mqi_aux.h"
#include "mqi_device.hpp"
#include "mqi_kernels.h"

#define MQI_TABLE_QUALIFIER static __constant__
#include "mqi_tables.inc"

namespace mqi_aux
{

// ------------------------------------------------------------------ fills
// Grid-stride fills; used instead of hipMemsetAsync so a captured graph
// re-clears its buffers on every replay.
__global__ void k_fill_u64(unsigned long long* p, unsigned long long v, uint64_t n) {
    for (uint64_t i = (uint64_t) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t) gridDim.x * blockDim.x)
        p[i] = v;
}
__global__ void k_fill_u32(uint32_t* p, uint32_t v, uint64_t n) {
    for (uint64_t i = (uint64_t) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t) gridDim.x * blockDim.x)
        p[i] = v;
}

static int
grid_for(uint64_t n) {
    uint64_t b = (n + 255) / 256;
    if (b > 65536) b = 65536;
    if (b < 1) b = 1;
    return (int) b;
}

__global__ void k_queue_init(unsigned long long* q, uint64_t total) {
    const int i = threadIdx.x;
    if (i < MQI_QUEUES) q[i * MQI_QUEUE_STRIDE] = mqi_range_begin(total, i);
}

int
queue_init(unsigned long long* q, uint64_t total, hipStream_t s) {
    hipLaunchKernelGGL(k_queue_init, dim3(1), dim3(64), 0, s, q, total);
    return (int) hipGetLastError();
}

int
fill_u64(void* p, unsigned long long v, uint64_t n, hipStream_t s) {
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_fill_u64, dim3(grid_for(n)), dim3(256), 0, s, (unsigned long long*) p, v, n);
    return (int) hipGetLastError();
}
int
fill_u32(void* p, uint32_t v, uint64_t n, hipStream_t s) {
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_fill_u32, dim3(grid_for(n)), dim3(256), 0, s, (uint32_t*) p, v, n);
    return (int) hipGetLastError();
}

// ------------------------------------------------------------------ calibration
// rho = hu_to_density(HU) * scale (mqi_tps_env.hpp:766-769)
__global__ void k_hu_to_density(const int16_t* hu, float* rho, uint64_t n, float scale) {
    __shared__ float corr[3996];
    for (int i = threadIdx.x; i < 3996; i += blockDim.x) corr[i] = kDensityCorrection[i];
    __syncthreads();
    for (uint64_t i = (uint64_t) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t) gridDim.x * blockDim.x)
        rho[i] = mqi_dev::hu_to_density(hu[i], corr) * scale;
}

int
hu_to_density(const int16_t* hu, float* rho, uint64_t n, float scale, hipStream_t s) {
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_hu_to_density, dim3(grid_for(n)), dim3(256), 0, s, hu, rho, n, scale);
    return (int) hipGetLastError();
}

// ------------------------------------------------------------------ math probe
// The portable functions evaluated on the device (verification of the exact build).
__global__ void k_math_probe(int fn, const double* x, const double* y, double* out, int64_t n) {
    int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double r;
    switch (fn) {
    case 0: r = mqi_pm::pm_log(x[i]); break;
    case 1: r = mqi_pm::pm_exp(x[i]); break;
    case 2: r = mqi_pm::pm_pow(x[i], y[i]); break;
    case 3: r = mqi_pm::pm_sin(x[i]); break;
    case 4: r = mqi_pm::pm_cos(x[i]); break;
    case 5: r = mqi_pm::pm_acos(x[i]); break;
    case 6: r = mqi_pm::pm_sqrt(x[i]); break;
    case 7: r = (double) ((float) x[i] / (float) y[i]); break;   // IEEE float division
    case 8: r = x[i] / y[i]; break;                              // IEEE double division
    default: r = (double) __builtin_sqrtf((float) x[i]); break;
    }
    out[i] = r;
}

int
math_probe(int fn, const double* x, const double* y, double* out, int64_t n, hipStream_t s) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_math_probe, dim3((unsigned) ((n + 255) / 256)), dim3(256), 0, s, fn, x, y, out, n);
    return (int) hipGetLastError();
}

// ------------------------------------------------------------------ atomic probe
// n_updates FP64 atomic adds of 1.0 to slots picked by a 64-bit hash of the
// update index over n_slots: the scoring pattern of the transport (random
// voxels, device-scope adds whose results are not read) without the rest of
// the step, to measure the part's throughput for such atomics.
MQI_DI uint32_t fmix32(uint32_t h) {   // the murmur3 32-bit finaliser
    h ^= h >> 16;
    h *= 0x85EBCA6Bu;
    h ^= h >> 13;
    h *= 0xC2B2AE35u;
    h ^= h >> 16;
    return h;
}

// slot = a hash of i scaled to [0, n_slots) by a high multiply (n_slots <=
// 2^32): a few integer operations per update, so the probe measures the
// atomic stream, not a 64-bit modulo.  window > 0: the wave's 64 updates
// (i with the same i / 64) share one window [base, base + window).
__global__ void k_atomic_probe(double* a, uint64_t n_slots, uint64_t n_updates, uint64_t window) {
    for (uint64_t i = (uint64_t) blockIdx.x * blockDim.x + threadIdx.x; i < n_updates;
         i += (uint64_t) gridDim.x * blockDim.x) {
        uint64_t slot;
        if (window == 0) {
            slot = ((uint64_t) fmix32((uint32_t) i) * n_slots) >> 32;
        } else {
            const uint64_t base = ((uint64_t) fmix32((uint32_t) (i >> 6) ^ 0x9E3779B9u) * (n_slots - window)) >> 32;
            slot                = base + (fmix32((uint32_t) i) & (uint32_t) (window - 1));
        }
        atomicAdd(a + slot, 1.0);
    }
}

int
atomic_probe(double* a, uint64_t n_slots, uint64_t n_updates, uint64_t window, hipStream_t s) {
    if (n_slots == 0 || n_updates == 0) return 0;
    if (n_slots > (1ull << 32)) return (int) hipErrorInvalidValue;
    if (window != 0 && (window >= n_slots || (window & (window - 1)) != 0)) return (int) hipErrorInvalidValue;
    hipLaunchKernelGGL(k_atomic_probe, dim3(65536), dim3(256), 0, s, a, n_slots, n_updates, window);
    return (int) hipGetLastError();
}

// ------------------------------------------------------------------ statistics
// calculate_standard_deviation (mqi_variables.hpp:21-48) fused with the
// reduction of calculate_stat (mqi_tps_env.hpp:1396-1425):
//   mean_i = S1_i / N, sd_i = sqrtf((S2_i/N - mean_i^2) / (N - 1)),
//   stat = mean over {i : mean_i > thr * max mean} of sd_i / mean_i.
// Pass 1: max of the float means.  Pass 2: sum and count above threshold.
__global__ void k_stat_max(const double* s1, uint64_t n, double N, float* out_max) {
    float m = 0.0f;
    for (uint64_t i = (uint64_t) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t) gridDim.x * blockDim.x) {
        float mu = (float) (s1[i] / N);
        m        = mu > m ? mu : m;
    }
    typedef hipcub::BlockReduce<float, 256> BR;
    __shared__ typename BR::TempStorage tmp;
    float bm = BR(tmp).Reduce(m, hipcub::Max());
    if (threadIdx.x == 0) atomicMax((int*) out_max, __float_as_int(bm));   // non-negative floats order as ints
}

__global__ void k_stat_sum(const double* s1, const double* s2, uint64_t n, double N, const float* max_mu, float thr,
                           double* out_sum, unsigned long long* out_cnt) {
    // dose_mean[i] > dose_max * stat_threshold with dose_max a double
    // (mqi_tps_env.hpp:1409-1425)
    const double lim = (double) *max_mu * (double) thr;
    double      acc = 0.0;
    unsigned long long cnt = 0;
    for (uint64_t i = (uint64_t) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t) gridDim.x * blockDim.x) {
        if (s1[i] == 0.0 && s2[i] == 0.0) continue;   // untouched slot (key1 == empty_pair)
        float mu = (float) (s1[i] / N);
        float sd = sqrtf((float) (((s2[i] / N) - ((s1[i] / N) * (s1[i] / N))) / (N - 1)));
        if ((double) mu > (double) lim) {
            acc += (double) (sd / mu);
            cnt += 1;
        }
    }
    typedef hipcub::BlockReduce<double, 256>             BRd;
    typedef hipcub::BlockReduce<unsigned long long, 256> BRu;
    __shared__ typename BRd::TempStorage t1;
    __shared__ typename BRu::TempStorage t2;
    double                               bs = BRd(t1).Sum(acc);
    __syncthreads();
    unsigned long long bc = BRu(t2).Sum(cnt);
    if (threadIdx.x == 0) {
        atomicAdd(out_sum, bs);
        atomicAdd(out_cnt, bc);
    }
}

int
stat_reduce(const double* s1, const double* s2, uint64_t n, double N, float thr, float* d_max, double* d_sum,
            unsigned long long* d_cnt, hipStream_t s) {
    fill_u32(d_max, 0u, 1, s);
    fill_u64(d_sum, 0ull, 1, s);
    fill_u64(d_cnt, 0ull, 1, s);
    int g = grid_for(n);
    if (g > 2048) g = 2048;
    hipLaunchKernelGGL(k_stat_max, dim3(g), dim3(256), 0, s, s1, n, N, d_max);
    hipLaunchKernelGGL(k_stat_sum, dim3(g), dim3(256), 0, s, s1, s2, n, N, d_max, thr, d_sum, d_cnt);
    return (int) hipGetLastError();
}

// rescale of scorers by N_target / N_tracked (calculate_average, mqi_variables.hpp:51-66)
// dose[i] += w * (stat[i] - snap[i]) outside voxel 0 of every scenario block
__global__ void k_dose_from_stat(double* dose, const double* stat, const double* snap, uint64_t n, uint64_t nvox,
                                 double w) {
    for (uint64_t i = (uint64_t) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t) gridDim.x * blockDim.x)
        if (i % nvox != 0) dose[i] += w * (stat[i] - snap[i]);
}

int
dose_from_stat(double* dose, const double* stat, const double* snap, uint64_t n, uint64_t nvox, double w,
               hipStream_t s) {
    if (n == 0 || nvox == 0) return 0;
    hipLaunchKernelGGL(k_dose_from_stat, dim3(grid_for(n)), dim3(256), 0, s, dose, stat, snap, n, nvox, w);
    return (int) hipGetLastError();
}

__global__ void k_scale(double* p, uint64_t n, double w) {
    for (uint64_t i = (uint64_t) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t) gridDim.x * blockDim.x)
        p[i] *= w;
}
int
scale(double* p, uint64_t n, double w, hipStream_t s) {
    if (n == 0) return 0;
    hipLaunchKernelGGL(k_scale, dim3(grid_for(n)), dim3(256), 0, s, p, n, w);
    return (int) hipGetLastError();
}

// ------------------------------------------------------------------ Dij compaction
// The hash table of an item (spot of a scenario), slots [off[item],
// off[item + 1]) of keys/vals, is scanned by `chunks` workgroups: the item's
// maximum, the entries >= rel_thr * max per chunk, and these entries (voxel,
// spot and value) from each chunk's place in the row-major list, in no order
// within a row (prepare_products sorts).  The scans are bound by the 8 bytes
// per slot they read: a slot's value is 0 until a key owns it, so the values
// alone tell the entries, and a key is read for an entry only.  One workgroup
// per item and a block-wide scan per 256 slots before: 3.8 ms for 400 tables
// of 290 k slots (1.39 GB), 0.65 ms now (0.16 + 0.16 at 5.8 TB/s, 0.33).
MQI_DI uint64_t chunk_begin(uint64_t cap, uint32_t chunk, uint32_t chunks) {
    return cap / chunks * chunk + min((uint64_t) chunk, cap % chunks);
}
#define MQI_SCAN 4   // slots a lane has in flight

// item_max (zeroed): values are positive, so their bits order as they do
__global__ void __launch_bounds__(256)
k_dij_max(const double* __restrict__ vals, const uint64_t* __restrict__ off, uint32_t chunks,
          unsigned long long* __restrict__ item_max) {
    const uint32_t item = blockIdx.x / chunks, chunk = blockIdx.x % chunks;
    const uint64_t o = off[item], cap = off[item + 1] - o;
    const uint64_t e = o + chunk_begin(cap, chunk + 1, chunks);
    double         m = 0.0;
    for (uint64_t i = o + chunk_begin(cap, chunk, chunks) + threadIdx.x; i < e; i += 256 * MQI_SCAN) {
        double v[MQI_SCAN];
#pragma unroll
        for (int j = 0; j < MQI_SCAN; ++j) v[j] = i + 256 * j < e ? vals[i + 256 * j] : 0.0;
#pragma unroll
        for (int j = 0; j < MQI_SCAN; ++j)
            if (v[j] > m) m = v[j];
    }
    typedef hipcub::BlockReduce<double, 256> BR;
    __shared__ typename BR::TempStorage tmp;
    const double                        bm = BR(tmp).Reduce(m, hipcub::Max());
    if (threadIdx.x == 0) atomicMax(item_max + item, (unsigned long long) __double_as_longlong(bm));
}

// counts[item * chunks + chunk]
__global__ void __launch_bounds__(256)
k_dij_count(const double* __restrict__ vals, const uint64_t* __restrict__ off, uint32_t chunks,
            const double* __restrict__ item_max, double rel_thr, uint32_t* __restrict__ counts) {
    const uint32_t item = blockIdx.x / chunks, chunk = blockIdx.x % chunks;
    const uint64_t o = off[item], cap = off[item + 1] - o;
    const uint64_t e   = o + chunk_begin(cap, chunk + 1, chunks);
    const double   lim = item_max[item] * rel_thr;
    uint32_t       n   = 0;
    for (uint64_t i = o + chunk_begin(cap, chunk, chunks) + threadIdx.x; i < e; i += 256 * MQI_SCAN) {
        double v[MQI_SCAN];
#pragma unroll
        for (int j = 0; j < MQI_SCAN; ++j) v[j] = i + 256 * j < e ? vals[i + 256 * j] : 0.0;
#pragma unroll
        for (int j = 0; j < MQI_SCAN; ++j) n += v[j] > 0.0 && v[j] >= lim ? 1u : 0u;
    }
    typedef hipcub::BlockReduce<uint32_t, 256> BR;
    __shared__ typename BR::TempStorage tmp;
    const uint32_t                      bn = BR(tmp).Sum(n);
    if (threadIdx.x == 0) counts[blockIdx.x] = bn;
}

// items [item0, item0 + gridDim.x / chunks); start[item * chunks + chunk]:
// the chunk's first place.  A wave takes places for its entries of a load at
// once, from the workgroup's counter.
__global__ void __launch_bounds__(256)
k_dij_write(const uint32_t* __restrict__ keys, const double* __restrict__ vals, const uint64_t* __restrict__ off,
            uint32_t item0, uint32_t chunks, const double* __restrict__ item_max, double rel_thr,
            const uint32_t* __restrict__ start, uint32_t* __restrict__ vox, uint64_t* __restrict__ packed) {
    const uint32_t spot = blockIdx.x / chunks, chunk = blockIdx.x % chunks, item = item0 + spot;
    const uint64_t o = off[item], cap = off[item + 1] - o;
    const uint64_t b = o + chunk_begin(cap, chunk, chunks), e = o + chunk_begin(cap, chunk + 1, chunks);
    const double   lim = item_max[item] * rel_thr;
    __shared__ uint32_t next;
    if (threadIdx.x == 0) next = start[(uint64_t) item * chunks + chunk];
    __syncthreads();
    for (uint64_t i = b + threadIdx.x; i - threadIdx.x < e; i += 256 * MQI_SCAN) {
        double v[MQI_SCAN];
#pragma unroll
        for (int j = 0; j < MQI_SCAN; ++j) v[j] = i + 256 * j < e ? vals[i + 256 * j] : 0.0;
#pragma unroll
        for (int j = 0; j < MQI_SCAN; ++j) {
            const bool               keep = v[j] > 0.0 && v[j] >= lim;
            const unsigned long long m    = __ballot(keep);
            if (!m) continue;
            uint32_t at = 0;
            if ((threadIdx.x & 63) == 0) at = atomicAdd(&next, (uint32_t) __popcll(m));
            at = __builtin_amdgcn_readfirstlane(at);
            if (keep) {
                at += __builtin_amdgcn_mbcnt_hi((uint32_t) (m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t) m, 0u));
                vox[at]    = keys[i + 256 * j];
                packed[at] = ((uint64_t) spot << 32) | (uint64_t) __float_as_uint((float) v[j]);
            }
        }
    }
}

// every entry of every table added to its scenario's Dose
__global__ void __launch_bounds__(256)
k_dij_dose(const uint32_t* __restrict__ keys, const double* __restrict__ vals, const uint64_t* __restrict__ off,
           uint32_t chunks, uint32_t n_spots, uint64_t stride, double* __restrict__ dose) {
    const uint32_t item = blockIdx.x / chunks, chunk = blockIdx.x % chunks;
    const uint64_t o = off[item], cap = off[item + 1] - o;
    const uint64_t e   = o + chunk_begin(cap, chunk + 1, chunks);
    double*        out = dose + stride * (item / n_spots);
    for (uint64_t i = o + chunk_begin(cap, chunk, chunks) + threadIdx.x; i < e; i += 256 * MQI_SCAN) {
        double v[MQI_SCAN];
#pragma unroll
        for (int j = 0; j < MQI_SCAN; ++j) v[j] = i + 256 * j < e ? vals[i + 256 * j] : 0.0;
#pragma unroll
        for (int j = 0; j < MQI_SCAN; ++j)
            if (v[j] != 0.0) atomicAdd(out + keys[i + 256 * j], v[j]);
    }
}
int
dose_from_dij(const uint32_t* keys, const double* vals, const uint64_t* off, uint32_t n_items, uint32_t chunks,
              uint32_t n_spots, uint64_t stride, double* dose, hipStream_t s) {
    if (n_items == 0) return 0;
    hipLaunchKernelGGL(k_dij_dose, dim3(n_items * chunks), dim3(256), 0, s, keys, vals, off, chunks, n_spots, stride,
                       dose);
    return (int) hipGetLastError();
}

int
dij_count(const double* vals, const uint64_t* off, uint32_t n_items, uint32_t chunks, double rel_thr,
          double* item_max, uint32_t* counts, hipStream_t s) {
    if (n_items == 0) return 0;
    const int e = fill_u64(item_max, 0ull, n_items, s);
    if (e) return e;
    hipLaunchKernelGGL(k_dij_max, dim3(n_items * chunks), dim3(256), 0, s, vals, off, chunks,
                       (unsigned long long*) item_max);
    hipLaunchKernelGGL(k_dij_count, dim3(n_items * chunks), dim3(256), 0, s, vals, off, chunks, item_max, rel_thr,
                       counts);
    return (int) hipGetLastError();
}

int
dij_write(const uint32_t* keys, const double* vals, const uint64_t* off, uint32_t item0, uint32_t n_spots,
          uint32_t chunks, const double* item_max, double rel_thr, const uint32_t* start, uint32_t* vox,
          uint64_t* packed, hipStream_t s) {
    if (n_spots == 0) return 0;
    hipLaunchKernelGGL(k_dij_write, dim3(n_spots * chunks), dim3(256), 0, s, keys, vals, off, item0, chunks, item_max,
                       rel_thr, start, vox, packed);
    return (int) hipGetLastError();
}

// ------------------------------------------------------------------ both orders of a matrix
// A matrix arrives as (voxel; spot, value) with the spots ascending and, from
// the Dij tables, no order within a spot.  A stable radix sort on the voxel
// gives the voxel-major copy with each voxel's spots ascending whatever the
// scheduling was; its voxels, their ranks and row pointers are read off the
// sorted keys tile by tile, and a second stable sort on the spot, carrying
// (rank, value), gives the rows in voxel order.  The products' tables of a
// field's matrix (400 spots, 9 M nonzeros, 8.4 M voxels) take 2.8 ms, against
// 27 ms with a segmented sort of the rows and the voxels counted, ranked and
// marked on the host; nine scenarios of 60 spots on 3.1 M voxels 9 ms
// against 60.
int
sort_pairs(uint32_t* keys, uint32_t* keys_tmp, uint64_t* vals, uint64_t* vals_tmp, int64_t n, int bits, void* scratch,
           size_t* scratch_bytes, int* in_tmp, hipStream_t s) {
    hipcub::DoubleBuffer<uint32_t> k(keys, keys_tmp);
    hipcub::DoubleBuffer<uint64_t> v(vals, vals_tmp);
    const hipError_t e = hipcub::DeviceRadixSort::SortPairs(scratch, *scratch_bytes, k, v, (size_t) n, 0, bits, s);
    if (scratch && in_tmp) *in_tmp = k.Current() != keys ? 1 : 0;
    return (int) e;
}

__global__ void k_pack_rows(const int64_t* __restrict__ indptr, const float* __restrict__ val, int64_t n_rows,
                            uint64_t* __restrict__ packed) {
    const int     lane  = threadIdx.x & 63;
    const int64_t wave  = ((int64_t) blockIdx.x * blockDim.x + threadIdx.x) >> 6;
    const int64_t waves = ((int64_t) gridDim.x * blockDim.x) >> 6;
    for (int64_t r = wave; r < n_rows; r += waves)
        for (int64_t k = indptr[r] + lane; k < indptr[r + 1]; k += 64)
            packed[k] = ((uint64_t) (uint32_t) r << 32) | (uint64_t) __float_as_uint(val[k]);
}
int
pack_rows(const int64_t* indptr, const float* val, int64_t n_rows, uint64_t* packed, hipStream_t s) {
    if (n_rows <= 0) return 0;
    hipLaunchKernelGGL(k_pack_rows, dim3(4096), dim3(256), 0, s, indptr, val, n_rows, packed);
    return (int) hipGetLastError();
}

// voxels beginning in each tile of the sorted keys
__global__ void __launch_bounds__(256)
k_tile_heads(const uint32_t* __restrict__ key, int64_t n, uint32_t* __restrict__ heads) {
    __shared__ uint32_t total;
    if (threadIdx.x == 0) total = 0;
    __syncthreads();
    uint32_t c = 0;
#pragma unroll 4
    for (int j = 0; j < MQI_TILE / 256; ++j) {
        const int64_t            i = (int64_t) blockIdx.x * MQI_TILE + 256 * j + threadIdx.x;
        const bool               h = i < n && (i == 0 || key[i] != key[i - 1]);
        const unsigned long long m = __ballot(h);
        c += (uint32_t) __popcll(m);
    }
    if ((threadIdx.x & 63) == 0) atomicAdd(&total, c);
    __syncthreads();
    if (threadIdx.x == 0) heads[blockIdx.x] = total;
}
// x[0 .. n) to its exclusive prefix sums, the total to x[n]; one workgroup
__global__ void __launch_bounds__(1024) k_scan_u32(uint32_t* __restrict__ x, int64_t n) {
    typedef hipcub::BlockScan<uint32_t, 1024> BS;
    __shared__ typename BS::TempStorage tmp;
    uint32_t                            base = 0;
    for (int64_t i0 = 0; i0 < n; i0 += 1024) {
        const int64_t i = i0 + threadIdx.x;
        uint32_t      at, tot;
        BS(tmp).ExclusiveSum(i < n ? x[i] : 0u, at, tot);
        if (i < n) x[i] = base + at;
        base += tot;
        __syncthreads();
    }
    if (threadIdx.x == 0) x[n] = base;
}
int
tile_heads(const uint32_t* key, int64_t n, uint32_t* heads, hipStream_t s) {
    if (n <= 0) return 0;
    const int64_t tiles = (n + MQI_TILE - 1) / MQI_TILE;
    hipLaunchKernelGGL(k_tile_heads, dim3((unsigned) tiles), dim3(256), 0, s, key, n, heads);
    hipLaunchKernelGGL(k_scan_u32, dim3(1), dim3(1024), 0, s, heads, tiles);
    return (int) hipGetLastError();
}

// The voxel-major copy from the sorted (voxel; spot, value): the voxels'
// list, row pointers (64-bit, and 32-bit for the host's plan) and bits, the
// spots (T: 16-bit columns for at most 65536 spots) and values, and for the
// sort back (spot; rank, value).
template<typename T>
__global__ void __launch_bounds__(256)
k_voxel_rows(const uint32_t* __restrict__ key, const uint64_t* __restrict__ packed, int64_t n,
             const uint32_t* __restrict__ heads, int32_t* __restrict__ nzvox, int64_t* __restrict__ tptr,
             uint32_t* __restrict__ tptr32, uint32_t* __restrict__ bits, T* __restrict__ tcol,
             float* __restrict__ tval, uint32_t* __restrict__ spot, uint64_t* __restrict__ ranked) {
    __shared__ uint32_t wave_heads[MQI_TILE / 64];
    const int           lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int64_t       i0 = (int64_t) blockIdx.x * MQI_TILE;
    // each wave of the tile's 64 runs of 64 keys: its voxels
#pragma unroll 4
    for (int j = w; j < MQI_TILE / 64; j += 4) {
        const int64_t            i = i0 + 64 * j + lane;
        const bool               h = i < n && (i == 0 || key[i] != key[i - 1]);
        const unsigned long long m = __ballot(h);
        if (lane == 0) wave_heads[j] = (uint32_t) __popcll(m);
    }
    __syncthreads();
    if (w == 0) {
        const uint32_t x = wave_heads[lane];
        uint32_t       p = x;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t y = __shfl_up(p, d);
            if (lane >= d) p += y;
        }
        wave_heads[lane] = heads[blockIdx.x] + p - x;
    }
    __syncthreads();
#pragma unroll 4
    for (int j = w; j < MQI_TILE / 64; j += 4) {
        const int64_t            i  = i0 + 64 * j + lane;
        const bool               in = i < n;
        const uint32_t           v  = in ? key[i] : 0u;
        const bool               h  = in && (i == 0 || v != key[i - 1]);
        const unsigned long long m  = __ballot(h);
        // the row of entry i: the voxels that begin up to and with it, less 1
        const uint32_t row = wave_heads[j] - 1u + (h ? 1u : 0u) +
                             __builtin_amdgcn_mbcnt_hi((uint32_t) (m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t) m, 0u));
        if (!in) continue;
        if (h) {
            nzvox[row]  = (int32_t) v;
            tptr[row]   = i;
            tptr32[row] = (uint32_t) i;
            atomicOr(bits + (v >> 5), 1u << (v & 31));
        }
        const uint64_t p = packed[i];
        tcol[i]          = (T) (uint32_t) (p >> 32);
        tval[i]          = __uint_as_float((uint32_t) p);
        spot[i]          = (uint32_t) (p >> 32);
        ranked[i]        = ((uint64_t) row << 32) | (uint64_t) (uint32_t) p;
        if (i == n - 1) {
            tptr[row + 1]   = n;
            tptr32[row + 1] = (uint32_t) n;
            for (int k = 0; k < MQI_SEG_PAD; ++k) {
                tcol[n + k] = (T) 0;
                tval[n + k] = 0.0f;
            }
        }
    }
}
int
voxel_rows(const uint32_t* key, const uint64_t* packed, int64_t n, const uint32_t* heads, int32_t* nzvox,
           int64_t* tptr, uint32_t* tptr32, uint32_t* bits, int64_t cols, uint16_t* tcol16, int32_t* tcol,
           float* tval, uint32_t* spot, uint64_t* ranked, hipStream_t s) {
    if (n <= 0) return 0;
    const int e = fill_u32(bits, 0u, (uint64_t) (cols + 31) / 32, s);
    if (e) return e;
    const dim3 g((unsigned) ((n + MQI_TILE - 1) / MQI_TILE));
    if (tcol16)
        hipLaunchKernelGGL(k_voxel_rows<uint16_t>, g, dim3(256), 0, s, key, packed, n, heads, nzvox, tptr, tptr32,
                           bits, tcol16, tval, spot, ranked);
    else
        hipLaunchKernelGGL(k_voxel_rows<int32_t>, g, dim3(256), 0, s, key, packed, n, heads, nzvox, tptr, tptr32,
                           bits, tcol, tval, spot, ranked);
    return (int) hipGetLastError();
}

// the rows from (rank, value) in spot-major order: columns, compacted
// columns and values
__global__ void k_spot_rows(const uint64_t* __restrict__ ranked, const int32_t* __restrict__ nzvox, int64_t n,
                            int32_t* __restrict__ col, int32_t* __restrict__ ccol, float* __restrict__ val) {
    for (int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t) gridDim.x * blockDim.x) {
        const uint64_t p = ranked[i];
        const int32_t  r = (int32_t) (p >> 32);
        ccol[i]          = r;
        col[i]           = nzvox[r];
        val[i]           = __uint_as_float((uint32_t) p);
    }
}
int
spot_rows(const uint64_t* ranked, const int32_t* nzvox, int64_t n, int32_t* col, int32_t* ccol, float* val,
          hipStream_t s) {
    if (n <= 0) return 0;
    hipLaunchKernelGGL(k_spot_rows, dim3(grid_for((uint64_t) n)), dim3(256), 0, s, ranked, nzvox, n, col, ccol, val);
    return (int) hipGetLastError();
}

// ------------------------------------------------------------------ sparse products
// y = alpha * A x (+ y) for a CSR matrix A (float values, int32 columns) with
// FP64 accumulation, in the CSR-Adaptive form (J. L. Greathouse and M. Daga,
// "Efficient sparse matrix-vector multiplication on GPUs using the CSR storage
// format", SC'14): the nonzeros are tiled into segments at build time.
//   partial segment  a piece (<= MQI_SEG_LONG entries) of one long row; the
//                    wave streams it with 16-byte loads and leaves its sum in
//                    part[s]; a second pass adds the pieces of each split row
//                    in order.
//   packed segment   whole rows, <= MQI_SEG_SHORT entries and <= MQI_SEG_ROWS
//                    rows: the wave forms the products into LDS with
//                    coalesced loads, then each row is summed by L lanes
//                    (the largest power of two with L * rows <= 64; strided
//                    parts, then shuffles within the group).
// Every sum runs in a fixed order, so results do not depend on scheduling.
// seg_info[s] = first row | (partial << 31); seg_k[s] = first nonzero;
// entry n_seg of both is the sentinel (rows, nnz).
typedef float    f32x4 __attribute__((ext_vector_type(4)));
typedef int32_t  i32x4 __attribute__((ext_vector_type(4)));
typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// four columns in one load: int32 columns, or 16-bit ones (D w over at most
// 65536 spots)
template<typename TC> struct col4;
template<> struct col4<int32_t> { typedef i32x4 type; };
template<> struct col4<uint16_t> { typedef u16x4 type; };

// a packed segment is loaded as at most 4 x 64 vectors of four entries, which
// may begin up to three entries before it
static_assert(MQI_SEG_SHORT + 3 <= MQI_SEG_BUF && MQI_SEG_BUF == 1024, "segments are loaded as at most 256 vectors");

// a wave's LDS accesses are performed in order: only the compiler must keep it
MQI_DI void lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// One wave's walk over segments, with MQI_SEG_SHORT doubles of LDS of its own.
// OBJ: instead of y, the quadratic objective of y (quad_obj): per row
// c_r (y_r - p_r)^2 summed over each packed segment into o.part[s] (0 for a
// long-row segment, whose rows k_quad_split finishes), and
// o.g[r] = two_inv_n c_r (y_r - p_r) when o.g is set
template<typename TY, typename TC, bool OBJ>
MQI_DI void csr_walk(const int64_t* __restrict__ indptr, const TC* __restrict__ col, const float* __restrict__ val,
                     const float* __restrict__ x, const int64_t* __restrict__ seg_k,
                     const uint32_t* __restrict__ seg_info, int64_t first, int64_t stride, int64_t n_seg,
                     double* __restrict__ part, TY* __restrict__ y, double alpha, const double* __restrict__ up,
                     int accumulate, const quad_obj& o, const int32_t* __restrict__ rowmap, double* buf) {
    const int lane = threadIdx.x & 63;
    // plain grid-stride walk: a remap giving each XCD a contiguous run of
    // segments measured ~7 % slower on the 5000-spot Dij
    for (int64_t s = first; s < n_seg; s += stride) {
        const uint32_t info = seg_info[s];
        const int64_t  kb = seg_k[s], ke = seg_k[s + 1];
        if (info >> 31) {
            double  acc = 0.0;
            int64_t ka  = (kb + 3) & ~(int64_t) 3;
            if (ka > ke) ka = ke;
            if (lane < ka - kb) acc += (double) val[kb + lane] * (double) x[col[kb + lane]];
            const int64_t n4 = (ke - ka) >> 2;
            typedef typename col4<TC>::type c4t;
            const f32x4*  v4 = reinterpret_cast<const f32x4*>(val + ka);
            const c4t*    c4 = reinterpret_cast<const c4t*>(col + ka);
            int64_t       i  = lane;
            for (; i + 192 < n4; i += 256) {
                f32x4 v[4];
                c4t   c[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    v[u] = __builtin_nontemporal_load(v4 + i + 64 * u);
                    c[u] = __builtin_nontemporal_load(c4 + i + 64 * u);
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    acc += (double) v[u].x * (double) x[c[u].x];
                    acc += (double) v[u].y * (double) x[c[u].y];
                    acc += (double) v[u].z * (double) x[c[u].z];
                    acc += (double) v[u].w * (double) x[c[u].w];
                }
            }
            for (; i < n4; i += 64) {
                const f32x4 v = __builtin_nontemporal_load(v4 + i);
                const c4t   c = __builtin_nontemporal_load(c4 + i);
                acc += (double) v.x * (double) x[c.x];
                acc += (double) v.y * (double) x[c.y];
                acc += (double) v.z * (double) x[c.z];
                acc += (double) v.w * (double) x[c.w];
            }
            const int64_t kt = ka + (n4 << 2);
            if (lane < ke - kt) acc += (double) val[kt + lane] * (double) x[col[kt + lane]];
            for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
            if (lane == 0) {
                part[s] = acc;
                if (OBJ) o.part[s] = 0.0;
            }
        } else {
            const int64_t r0 = info, r1 = seg_info[s + 1] & 0x7fffffffu;
            // products into LDS: the segment's aligned body as 16-byte loads
            // (four consecutive entries per lane, the whole segment in flight
            // at once: at most 1024 entries, 256 vectors), head and tail of
            // up to three entries one per lane
            typedef typename col4<TC>::type c4t;
            int64_t ka = (kb + 3) & ~(int64_t) 3;
            if (ka > ke) ka = ke;
            const int64_t n4 = (ke - ka) >> 2;
            const int64_t kt = ka + (n4 << 2);
            const f32x4*  v4 = reinterpret_cast<const f32x4*>(val + ka);
            const c4t*    c4 = reinterpret_cast<const c4t*>(col + ka);
            f32x4         v[4];
            c4t           c[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int64_t i = lane + 64 * u;
                if (i < n4) {
                    v[u] = __builtin_nontemporal_load(v4 + i);
                    c[u] = __builtin_nontemporal_load(c4 + i);
                }
            }
            if (lane < ka - kb) buf[lane] = (double) val[kb + lane] * (double) x[col[kb + lane]];
            if (lane < ke - kt) buf[kt - kb + lane] = (double) val[kt + lane] * (double) x[col[kt + lane]];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int64_t i = lane + 64 * u;
                if (i < n4) {
                    double* b = buf + (ka - kb) + 4 * i;
                    b[0]      = (double) v[u].x * (double) x[c[u].x];
                    b[1]      = (double) v[u].y * (double) x[c[u].y];
                    b[2]      = (double) v[u].z * (double) x[c[u].z];
                    b[3]      = (double) v[u].w * (double) x[c[u].w];
                }
            }
            lds_fence();
            // L lanes per row (a power of two, L * rows <= 64): each sums a
            // strided part, then the group adds its parts with shuffles
            const int64_t nr = r1 - r0;
            int           L  = 1;
            while (L < 64 && 2 * L * nr <= 64) L *= 2;
            const int sub = lane & (L - 1);
            double    obj = 0.0;   // this lane's rows' objective terms, in row order
            for (int64_t rb = r0; rb < r1; rb += 64 / L) {
                const int64_t r   = rb + lane / L;
                double        acc = 0.0;
                // the row's prescription and weight are loaded with its
                // pointers, not after its sum (one round trip per row)
                // row r of the matrix is element v of y (rowmap: the voxel of
                // each row of a matrix with its empty rows left out)
                const int64_t v  = (rowmap && r < r1) ? (int64_t) rowmap[r] : r;
                double        pr = 0.0, cw = 1.0;
                if (OBJ && r < r1 && sub == 0) {
                    pr = o.p[v];
                    if (o.c) cw = (double) o.c[v];
                }
                if (r < r1) {
                    const int64_t e = indptr[r + 1] - kb;
                    for (int64_t k = indptr[r] - kb + sub; k < e; k += L) acc += buf[k];
                }
                for (int off = L >> 1; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
                if (r < r1 && sub == 0) {
                    const double out = up ? alpha * acc * *up : alpha * acc;
                    if (OBJ) {
                        const double res = out - pr;
                        obj += cw * res * res;
                        if (o.g) o.g[v] = (float) (o.two_inv_n * cw * res);
                    } else {
                        y[v] = accumulate ? (TY) ((double) y[v] + out) : (TY) out;
                    }
                }
            }
            if (OBJ) {
                for (int off = 32; off > 0; off >>= 1) obj += __shfl_xor(obj, off);
                if (lane == 0) o.part[s] = obj;
            }
            lds_fence();
        }
    }
}

// y = 0 at the elements no row reaches (bit clear in nonempty): part b of n
template<typename TY>
MQI_DI void zero_empty(const uint32_t* __restrict__ nonempty, int64_t n_y, TY* __restrict__ y, int b, int n) {
    // eight elements per lane and pass, their mask words loaded together
    const int64_t zs = (int64_t) n * 64;
    for (int64_t v0 = (int64_t) b * 64 + (threadIdx.x & 63); v0 < n_y; v0 += 8 * zs) {
        uint32_t bits[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) bits[j] = (v0 + j * zs < n_y) ? nonempty[(v0 + j * zs) >> 5] : 0xffffffffu;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int64_t v = v0 + j * zs;
            if (v < n_y && !((bits[j] >> (v & 31)) & 1u)) y[v] = (TY) 0;
        }
    }
}

// x behind the waves' buffers, and the wave's index in the grid (a scalar)
MQI_DI const float* stage_x(const float* __restrict__ x, int n_x, double* lds) {
    float* xs = (float*) (lds + (blockDim.x >> 6) * MQI_SEG_BUF);
    for (int i = threadIdx.x; i < n_x; i += blockDim.x) xs[i] = x[i];
    __syncthreads();
    return xs;
}
MQI_DI int64_t wave_index() {
    return (int64_t) blockIdx.x * (blockDim.x >> 6) + __builtin_amdgcn_readfirstlane((int) (threadIdx.x >> 6));
}

// up (device): y = alpha * A x * *up, rounded as the two products
template<typename TY, typename TC>
__global__ void __launch_bounds__(64) k_csr_adaptive(const int64_t* __restrict__ indptr,
                                                     const TC* __restrict__ col,
                                                     const float* __restrict__ val, const float* __restrict__ x,
                                                     const int64_t* __restrict__ seg_k,
                                                     const uint32_t* __restrict__ seg_info, int64_t n_seg,
                                                     double* __restrict__ part, TY* __restrict__ y, double alpha,
                                                     const double* __restrict__ up, int accumulate,
                                                     const int32_t* __restrict__ rowmap,
                                                     const uint32_t* __restrict__ nonempty, int64_t n_y,
                                                     int zero_blocks) {
    __shared__ double buf[MQI_SEG_BUF];
    // the first zero_blocks workgroups write y = 0 at the elements no row
    // reaches, alongside the segments' workgroups
    if ((int) blockIdx.x < zero_blocks) {
        zero_empty(nonempty, n_y, y, blockIdx.x, zero_blocks);
        return;
    }
    csr_walk<TY, TC, false>(indptr, col, val, x, seg_k, seg_info, (int64_t) blockIdx.x - zero_blocks,
                            (int64_t) gridDim.x - zero_blocks, n_seg, part, y, alpha, up, accumulate, quad_obj{},
                            rowmap, buf);
}

// ------------------------------------------------------------------ D w, large matrices
// The same with x in LDS and the next segment under way, for 16-bit columns.
// k_csr_adaptive's waves load, gather, sum and write one segment after
// another, and their gathers of x (64 lanes, as many lines of the vector
// cache) take about a clock a lane: 6 bytes an entry at 2.2 to 2.8 TB/s.  Here
// workgroups of 8 to 16 waves share a copy of x and stay; a wave loads its
// next segment's entries, row pointers and voxels once this segment's products
// are in LDS, before it sums them.  D w of 1000 spots on 8.4 M voxels (42 M
// entries) 116 -> 91 us, 8000 spots (219 M) 465 -> 356, 24576 spots (672 M)
// 1755 -> 1431; their objective with weights and gradient 156 -> 127, 514 ->
// 377 and 1816 -> 1414.  (The loads alone stream 6.8 TB/s, with sums of rows
// of 27 entries and the gathers 5.2; what is left between is the row data, the
// scattered writes and the last, partly filled round of segments.)
//
// A segment's entries are read as the whole 16-byte vectors that cover it: at
// most 256, as a packed segment has at most MQI_SEG_SHORT entries; what is
// read around it belongs to its neighbours or to the arrays' padding.
struct seg_rows {   // a packed segment, as a wave holds it
    int64_t kb, r0;
    int     n4, nr, L;          // vectors, rows, lanes per row
    int     ea, eb;             // the lane's first row: its entries in the buffer
    int32_t va;                 // and its element of y
};
struct seg_data {
    f32x4 v[4];
    u16x4 c[4];
};
MQI_DI void seg_load(const int64_t* __restrict__ indptr, const uint16_t* __restrict__ col,
                     const float* __restrict__ val, int64_t kb, int64_t ke, int64_t r0, int64_t r1,
                     const int32_t* __restrict__ rowmap, seg_rows& q, seg_data& d) {
    const int lane = threadIdx.x & 63;
    q.kb           = kb & ~(int64_t) 3;
    q.r0           = r0;
    q.n4           = (int) ((ke + 3 - q.kb) >> 2);
    q.nr           = (int) (r1 - r0);
    q.L            = 1;
    while (q.L < 64 && 2 * q.L * q.nr <= 64) q.L *= 2;
    const f32x4* v4 = reinterpret_cast<const f32x4*>(val + q.kb);
    const u16x4* c4 = reinterpret_cast<const u16x4*>(col + q.kb);
#pragma unroll
    for (int u = 0; u < 4; ++u)
        if (lane + 64 * u < q.n4) {
            d.v[u] = __builtin_nontemporal_load(v4 + lane + 64 * u);
            d.c[u] = __builtin_nontemporal_load(c4 + lane + 64 * u);
        }
    const int ra = lane / q.L;
    if (ra < q.nr) {
        q.ea = (int) (indptr[r0 + ra] - q.kb);
        q.eb = (int) (indptr[r0 + ra + 1] - q.kb);
        q.va = rowmap ? rowmap[r0 + ra] : (int32_t) (r0 + ra);
    }
}

// wave `wave` of `waves`' segments of a matrix: as csr_walk
template<typename TY, bool OBJ>
MQI_DI void csr_stream(const int64_t* __restrict__ indptr, const uint16_t* __restrict__ col,
                       const float* __restrict__ val, const float* xs, const int64_t* __restrict__ seg_k,
                       const uint32_t* __restrict__ seg_info, int64_t wave, int64_t waves, int64_t n_seg,
                       double* __restrict__ part, TY* __restrict__ y, double alpha, int accumulate, const quad_obj& o,
                       const int32_t* __restrict__ rowmap, double* buf) {
    const int lane = threadIdx.x & 63;
    seg_rows  q;
    seg_data  d;
    bool      loaded = false;
    for (int64_t s = wave; s < n_seg; s += waves) {
        const uint32_t info = seg_info[s];
        if (info >> 31) {   // a piece of a long row
            csr_walk<TY, uint16_t, OBJ>(indptr, col, val, xs, seg_k, seg_info, s, 1, s + 1, part, y, alpha, nullptr,
                                        accumulate, o, rowmap, buf);
            continue;
        }
        if (!loaded)
            seg_load(indptr, col, val, seg_k[s], seg_k[s + 1], info, seg_info[s + 1] & 0x7fffffffu, rowmap, q, d);
        const seg_rows h  = q;
        const int      ra = lane / h.L, sub = lane & (h.L - 1);
        double         pa = 0.0, ca = 1.0;
        if (OBJ && ra < h.nr && sub == 0) {
            pa = o.p[h.va];
            if (o.c) ca = (double) o.c[h.va];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (lane + 64 * u < h.n4) {
                double* b = buf + 4 * (lane + 64 * u);
                b[0]      = (double) d.v[u].x * (double) xs[d.c[u].x];
                b[1]      = (double) d.v[u].y * (double) xs[d.c[u].y];
                b[2]      = (double) d.v[u].z * (double) xs[d.c[u].z];
                b[3]      = (double) d.v[u].w * (double) xs[d.c[u].w];
            }
        const int64_t  nx = s + waves;
        const uint32_t ni = nx < n_seg ? seg_info[nx] : 1u << 31;
        loaded            = !(ni >> 31);
        if (loaded)
            seg_load(indptr, col, val, seg_k[nx], seg_k[nx + 1], ni, seg_info[nx + 1] & 0x7fffffffu, rowmap, q, d);
        lds_fence();
        double obj = 0.0;   // this lane's rows' objective terms, in row order
        for (int rb = 0; rb < h.nr; rb += 64 / h.L) {
            const int r   = rb + ra;
            double    acc = 0.0, pr = pa, cw = ca;
            int       i = h.ea, e = h.eb;
            int32_t   v = h.va;
            if (rb > 0 && r < h.nr) {
                i = (int) (indptr[h.r0 + r] - h.kb);
                e = (int) (indptr[h.r0 + r + 1] - h.kb);
                v = rowmap ? rowmap[h.r0 + r] : (int32_t) (h.r0 + r);
                if (OBJ && sub == 0) {
                    pr = o.p[v];
                    if (o.c) cw = (double) o.c[v];
                }
            }
            if (r < h.nr) {
                // in order, four LDS reads in flight
                i += sub;
                for (; i + 3 * h.L < e; i += 4 * h.L) {
                    const double a0 = buf[i], a1 = buf[i + h.L], a2 = buf[i + 2 * h.L], a3 = buf[i + 3 * h.L];
                    acc += a0;
                    acc += a1;
                    acc += a2;
                    acc += a3;
                }
                for (; i < e; i += h.L) acc += buf[i];
            }
            for (int off = h.L >> 1; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
            if (r < h.nr && sub == 0) {
                const double out = alpha * acc;
                if (OBJ) {
                    const double res = out - pr;
                    obj += cw * res * res;
                    if (o.g) o.g[v] = (float) (o.two_inv_n * cw * res);
                } else {
                    y[v] = accumulate ? (TY) ((double) y[v] + out) : (TY) out;
                }
            }
        }
        if (OBJ) {
            for (int off = 32; off > 0; off >>= 1) obj += __shfl_xor(obj, off);
            if (lane == 0) o.part[s] = obj;
        }
        lds_fence();
    }
}

template<typename TY>
__global__ void __launch_bounds__(1024)
k_csr_lds(const int64_t* __restrict__ indptr, const uint16_t* __restrict__ col, const float* __restrict__ val,
          const float* __restrict__ x, int n_x, const int64_t* __restrict__ seg_k,
          const uint32_t* __restrict__ seg_info, int64_t n_seg, double* __restrict__ part, TY* __restrict__ y,
          double alpha, int accumulate, const int32_t* __restrict__ rowmap, const uint32_t* __restrict__ nonempty,
          int64_t n_y, int zero) {
    extern __shared__ double lds[];
    const float*  xs    = stage_x(x, n_x, lds);
    const int64_t waves = (int64_t) gridDim.x * (blockDim.x >> 6), wave = wave_index();
    if (zero) zero_empty(nonempty, n_y, y, (int) wave, (int) waves);
    csr_stream<TY, false>(indptr, col, val, xs, seg_k, seg_info, wave, waves, n_seg, part, y, alpha, accumulate,
                              quad_obj{}, rowmap, lds + (threadIdx.x >> 6) * MQI_SEG_BUF);
}

// rows split over partial segments [split_seg[2i], split_seg[2i+1]): their
// pieces' sum in order
MQI_DI double split_row(const int32_t* __restrict__ split_seg, int64_t i, const double* __restrict__ part) {
    double acc = 0.0;
    for (int32_t s = split_seg[2 * i]; s < split_seg[2 * i + 1]; ++s) acc += part[s];
    return acc;
}
MQI_DI int64_t split_element(const uint32_t* __restrict__ seg_info, const int32_t* __restrict__ split_seg, int64_t i,
                             const int32_t* __restrict__ rowmap) {
    const int64_t r = seg_info[split_seg[2 * i]] & 0x7fffffffu;
    return rowmap ? (int64_t) rowmap[r] : r;
}

// y[r] = alpha * sum of the pieces (+ y[r])
template<typename TY>
__global__ void k_csr_split_rows(const uint32_t* __restrict__ seg_info, const int32_t* __restrict__ split_seg,
                                 int64_t n_split, const double* __restrict__ part, TY* __restrict__ y, double alpha,
                                 const double* __restrict__ up, int accumulate, const int32_t* __restrict__ rowmap) {
    const int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n_split) return;
    const int64_t r   = split_element(seg_info, split_seg, i, rowmap);
    const double  acc = split_row(split_seg, i, part);
    const double  out = up ? alpha * acc * *up : alpha * acc;
    y[r]              = accumulate ? (TY) ((double) y[r] + out) : (TY) out;
}

int
csr_split_rows(const uint32_t* seg_info, const int32_t* split_seg, int64_t n_split, double* part, void* y,
               int y_is_double, double alpha, const double* up, int accumulate, const int32_t* rowmap, hipStream_t s) {
    if (n_split > 0) {
        const int b = (int) ((n_split + 255) / 256);
        if (y_is_double)
            hipLaunchKernelGGL(k_csr_split_rows<double>, dim3(b), dim3(256), 0, s, seg_info, split_seg, n_split, part,
                               (double*) y, alpha, up, accumulate, rowmap);
        else
            hipLaunchKernelGGL(k_csr_split_rows<float>, dim3(b), dim3(256), 0, s, seg_info, split_seg, n_split, part,
                               (float*) y, alpha, up, accumulate, rowmap);
    }
    return (int) hipGetLastError();
}

// Workgroups with x in LDS: waves a group, groups and LDS bytes; false where
// the segments are too few to stay for, or too few waves would share a CU with
// x (the kernels' registers allow 16).
struct lds_shape {
    int    waves, blocks;
    size_t bytes;
};
bool
lds_launch(int64_t n_x, int64_t n_seg, lds_shape& L) {
    const int64_t w = std::min<int64_t>(16, (MQI_LDS - 4 * n_x) / (8 * MQI_SEG_BUF));
    if (n_x <= 0 || w < MQI_LDS_WAVES || n_seg < MQI_LDS_SEGS) return false;
    L.waves  = (int) w;
    L.bytes  = (size_t) (8 * MQI_SEG_BUF * w + 4 * n_x);
    L.blocks = MQI_CUS;
    return true;
}

template<typename TC>
int
csr_adaptive_t(const int64_t* indptr, const TC* col, const float* val, const float* x, const int64_t* seg_k,
               const uint32_t* seg_info, int64_t n_seg, const int32_t* split_seg, int64_t n_split, double* part,
               void* y, int y_is_double, double alpha, const double* up, int accumulate, const int32_t* rowmap,
               const uint32_t* nonempty, int64_t n_y, hipStream_t s) {
    if (rowmap && !accumulate && (!nonempty || n_y <= 0)) return (int) hipErrorInvalidValue;
    if (n_seg <= 0) return 0;
    const int blocks = (int) (n_seg < 262144 ? n_seg : 262144);
    const int zb     = (rowmap && !accumulate) ? MQI_ZERO_BLOCKS : 0;
    if (y_is_double)
        hipLaunchKernelGGL((k_csr_adaptive<double, TC>), dim3(blocks + zb), dim3(64), 0, s, indptr, col, val, x, seg_k,
                           seg_info, n_seg, part, (double*) y, alpha, up, accumulate, rowmap, nonempty, n_y, zb);
    else
        hipLaunchKernelGGL((k_csr_adaptive<float, TC>), dim3(blocks + zb), dim3(64), 0, s, indptr, col, val, x, seg_k,
                           seg_info, n_seg, part, (float*) y, alpha, up, accumulate, rowmap, nonempty, n_y, zb);
    return csr_split_rows(seg_info, split_seg, n_split, part, y, y_is_double, alpha, up, accumulate, rowmap, s);
}

int
csr_adaptive(const int64_t* indptr, const int32_t* col, const float* val, const float* x, const int64_t* seg_k,
             const uint32_t* seg_info, int64_t n_seg, const int32_t* split_seg, int64_t n_split, double* part,
             void* y, int y_is_double, double alpha, const double* up, int accumulate, const int32_t* rowmap,
             const uint32_t* nonempty, int64_t n_y, hipStream_t s) {
    return csr_adaptive_t(indptr, col, val, x, seg_k, seg_info, n_seg, split_seg, n_split, part, y, y_is_double,
                          alpha, up, accumulate, rowmap, nonempty, n_y, s);
}
int
csr_adaptive16(const int64_t* indptr, const uint16_t* col, const float* val, const float* x, int64_t n_x,
               const int64_t* seg_k, const uint32_t* seg_info, int64_t n_seg, const int32_t* split_seg,
               int64_t n_split, double* part, void* y, int y_is_double, double alpha, int accumulate,
               const int32_t* rowmap, const uint32_t* nonempty, int64_t n_y, hipStream_t s) {
    lds_shape L;
    if (!lds_launch(n_x, n_seg, L))
        return csr_adaptive_t(indptr, col, val, x, seg_k, seg_info, n_seg, split_seg, n_split, part, y, y_is_double,
                              alpha, nullptr, accumulate, rowmap, nonempty, n_y, s);
    const int zero = rowmap && !accumulate;
    if (zero && (!nonempty || n_y <= 0)) return (int) hipErrorInvalidValue;
    if (y_is_double)
        hipLaunchKernelGGL(k_csr_lds<double>, dim3(L.blocks), dim3(64 * L.waves), L.bytes, s, indptr, col, val, x,
                           (int) n_x, seg_k, seg_info, n_seg, part, (double*) y, alpha, accumulate, rowmap, nonempty,
                           n_y, zero);
    else
        hipLaunchKernelGGL(k_csr_lds<float>, dim3(L.blocks), dim3(64 * L.waves), L.bytes, s, indptr, col, val, x,
                           (int) n_x, seg_k, seg_info, n_seg, part, (float*) y, alpha, accumulate, rowmap, nonempty,
                           n_y, zero);
    return csr_split_rows(seg_info, split_seg, n_split, part, y, y_is_double, alpha, nullptr, accumulate, rowmap, s);
}

// ------------------------------------------------------------------ quadratic objective
// f_i = inv_n * (sum of c (d_i - p)^2) of up to MQI_QUAD_MATS matrices over one
// x, p and c.  One launch forms the terms: per matrix, `empty` workgroups take
// the elements no row reaches (d = 0) and the others its segments, side by
// side; a second launch sums each matrix' terms.  Four launches per matrix
// before (elements without a row, segments, chunk sums, sum): each drained
// the device and cost 4 us and its share of the host's time.
struct quad_set {
    int      n;
    quad_mat m[MQI_QUAD_MATS];
    uint32_t unit0[MQI_QUAD_MATS + 1];   // first unit of each matrix
};

// the objective's terms of the elements of y no row reaches (bit v of
// nonempty clear): c p^2 per element, summed per workgroup into part[b], and
// g = -two_inv_n c p there
MQI_DI void quad_empty(const uint32_t* __restrict__ nonempty, int64_t n, const quad_obj& o, uint32_t b,
                       uint32_t blocks, double* __restrict__ part) {
    // eight elements per lane and pass, their loads issued together (one load
    // in flight per lane left the pass latency-bound); the lane's sum runs
    // over its elements in index order
    constexpr int U      = 8;
    const int64_t stride = (int64_t) blocks * 64;
    double        acc    = 0.0;
    for (int64_t v0 = (int64_t) b * 64 + (threadIdx.x & 63); v0 < n; v0 += U * stride) {
        uint32_t bits[U];
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const int64_t v = v0 + j * stride;
            bits[j]         = v < n ? nonempty[v >> 5] : 0xffffffffu;
        }
        double p[U], cw[U];
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const int64_t v     = v0 + j * stride;
            const bool    empty = v < n && !((bits[j] >> (v & 31)) & 1u);
            p[j]                = empty ? o.p[v] : 0.0;
            cw[j]               = (empty && o.c) ? (double) o.c[v] : 1.0;
        }
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const int64_t v = v0 + j * stride;
            if (v >= n || ((bits[j] >> (v & 31)) & 1u)) continue;
            acc += cw[j] * p[j] * p[j];
            if (o.g) o.g[v] = (float) (-o.two_inv_n * cw[j] * p[j]);
        }
    }
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    if ((threadIdx.x & 63) == 0) part[b] = acc;
}

// unit `u` of the set: a part of a matrix' elements without a row, or a segment
template<typename TC>
MQI_DI void quad_unit(const quad_set& S, const float* __restrict__ x, quad_obj& o, int64_t n_y, uint32_t u,
                      double* buf) {
    int i = 0;
    while (i + 1 < S.n && u >= S.unit0[i + 1]) ++i;
    const quad_mat& m = S.m[i];
    const uint32_t  b = u - S.unit0[i];
    o.part            = m.terms;
    if (b < m.empty)
        quad_empty(m.nonempty, n_y, o, b, m.empty, m.terms + m.n_seg + m.n_split);
    else
        csr_walk<double, TC, true>(m.indptr, (const TC*) m.col, m.val, x, m.seg_k, m.seg_info, b - m.empty, 1,
                                   b - m.empty + 1, m.part, nullptr, m.alpha, nullptr, 0, o, m.rowmap, buf);
}
template<typename TC>
__global__ void __launch_bounds__(64)
k_quad(quad_set S, const float* __restrict__ x, quad_obj o, int64_t n_y) {
    __shared__ double buf[MQI_SEG_BUF];
    for (uint32_t u = blockIdx.x; u < S.unit0[S.n]; u += gridDim.x) quad_unit<TC>(S, x, o, n_y, u, buf);
}
// with x in LDS (k_csr_lds); block0: the first workgroup of each matrix
struct quad_blocks {
    uint32_t b[MQI_QUAD_MATS + 1];
};
__global__ void __launch_bounds__(1024)
k_quad_lds(quad_set S, quad_blocks block0, const float* __restrict__ x, int n_x, quad_obj o, int64_t n_y) {
    extern __shared__ double lds[];
    const float* xs = stage_x(x, n_x, lds);
    int          i  = 0;
    while (i + 1 < S.n && blockIdx.x >= block0.b[i + 1]) ++i;
    const quad_mat& m     = S.m[i];
    const int64_t   waves = (int64_t) (block0.b[i + 1] - block0.b[i]) * (blockDim.x >> 6);
    const int64_t   wave  = wave_index() - (int64_t) block0.b[i] * (blockDim.x >> 6);
    o.part                = m.terms;
    for (int64_t b = wave; b < m.empty; b += waves)
        quad_empty(m.nonempty, n_y, o, (uint32_t) b, m.empty, m.terms + m.n_seg + m.n_split);
    csr_stream<double, true>(m.indptr, (const uint16_t*) m.col, m.val, xs, m.seg_k, m.seg_info, wave, waves, m.n_seg,
                             m.part, nullptr, m.alpha, 0, o, m.rowmap, lds + (threadIdx.x >> 6) * MQI_SEG_BUF);
}

// the split rows' terms, after the packed segments' ones (blockIdx.y: matrix)
__global__ void k_quad_split(quad_set S, quad_obj o) {
    const quad_mat& m = S.m[blockIdx.y];
    const int64_t   i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= m.n_split) return;
    const int64_t r   = split_element(m.seg_info, m.split_seg, i, m.rowmap);
    const double  res = m.alpha * split_row(m.split_seg, i, m.part) - o.p[r];
    const double  cw  = o.c ? (double) o.c[r] : 1.0;
    m.terms[m.n_seg + i] = cw * res * res;
    if (o.g) o.g[r] = (float) (o.two_inv_n * cw * res);
}

MQI_DI int64_t quad_terms(const quad_mat& m) { return m.n_seg + m.n_split + m.empty; }

// this thread's elements of a[0 .. n) in index order, four loads in flight
MQI_DI double strided_sum(const double* __restrict__ a, int64_t n, int t) {
    double  acc = 0.0;
    int64_t i   = threadIdx.x;
    for (; i + 3 * t < n; i += 4 * t) {
        const double a0 = a[i], a1 = a[i + t], a2 = a[i + 2 * t], a3 = a[i + 3 * t];
        acc += a0;
        acc += a1;
        acc += a2;
        acc += a3;
    }
    for (; i < n; i += t) acc += a[i];
    return acc;
}

// Fixed-order sums.  A matrix of more than MQI_QUAD_ONE terms has them summed
// in MQI_QUAD_SUM_BLOCKS chunks by as many workgroups first (one workgroup
// over the 3.8e5 terms of a 3e8-nonzero matrix took 0.35 ms); one workgroup
// then sums the chunk sums, or the terms.
__global__ void __launch_bounds__(256) k_quad_chunks(quad_set S) {
    const quad_mat& m = S.m[blockIdx.y];
    const int64_t   n = quad_terms(m);
    if (n <= MQI_QUAD_ONE) return;
    const int64_t ch = (n + gridDim.x - 1) / gridDim.x, b0 = (int64_t) blockIdx.x * ch;
    const int64_t len = b0 + ch < n ? ch : n - b0;
    const double  acc = strided_sum(m.terms + b0, len, 256);
    typedef hipcub::BlockReduce<double, 256> BR;
    __shared__ typename BR::TempStorage tmp;
    const double t = BR(tmp).Sum(acc);
    if (threadIdx.x == 0) m.terms[n + blockIdx.x] = t;
}
__global__ void __launch_bounds__(1024) k_quad_sum(quad_set S, double inv_n, double* __restrict__ f) {
    const quad_mat& m   = S.m[blockIdx.x];
    const int64_t   n   = quad_terms(m);
    const double    acc = n > MQI_QUAD_ONE ? strided_sum(m.terms + n, MQI_QUAD_SUM_BLOCKS, 1024)
                                           : strided_sum(m.terms, n, 1024);
    typedef hipcub::BlockReduce<double, 1024> BR;
    __shared__ typename BR::TempStorage tmp;
    const double t = BR(tmp).Sum(acc);
    if (threadIdx.x == 0) f[blockIdx.x] = inv_n * t;
}

int
csr_quadratic(const quad_mat* mats, int n, int cols16, const float* x, int64_t n_x, const double* p, const float* c,
              float* g, int64_t n_y, double* f, hipStream_t s) {
    if (n < 1 || n > MQI_QUAD_MATS || !p || !f || n_y <= 0 || (g && n != 1)) return (int) hipErrorInvalidValue;
    quad_set S{};
    S.n            = n;
    int64_t units = 0, segs = 0, split = 0, terms = 0;
    for (int i = 0; i < n; ++i) {
        quad_mat& m = S.m[i];
        m           = mats[i];
        if (m.n_seg <= 0 || !m.terms || (m.rowmap && !m.nonempty)) return (int) hipErrorInvalidValue;
        m.empty     = m.rowmap ? (uint32_t) std::min<int64_t>(MQI_QUAD_EMPTY_BLOCKS, (n_y + 511) / 512) : 0;
        S.unit0[i]  = (uint32_t) units;
        units += m.empty + m.n_seg;
        segs += m.n_seg;
        split = std::max(split, m.n_split);
        terms = std::max(terms, m.n_seg + m.n_split + (int64_t) m.empty);
    }
    if (units > (int64_t) UINT32_MAX) return (int) hipErrorInvalidValue;
    S.unit0[n] = (uint32_t) units;
    quad_obj o{};
    o.p         = p;
    o.c         = c;
    o.g         = g;
    o.two_inv_n = 2.0 / (double) n_y;
    lds_shape  L;
    const dim3 blocks((unsigned) std::min<int64_t>(units, 262144));
    if (cols16 && lds_launch(n_x, segs, L)) {
        // workgroups by the matrices' work, at least one each
        quad_blocks bl{};
        for (int i = 0; i < n; ++i)
            bl.b[i + 1] = bl.b[i] + (uint32_t) std::max<int64_t>(
                                        1, (int64_t) L.blocks * (S.unit0[i + 1] - S.unit0[i]) / units);
        hipLaunchKernelGGL(k_quad_lds, dim3(bl.b[n]), dim3(64 * L.waves), L.bytes, s, S, bl, x, (int) n_x, o, n_y);
    } else if (cols16)
        hipLaunchKernelGGL(k_quad<uint16_t>, blocks, dim3(64), 0, s, S, x, o, n_y);
    else
        hipLaunchKernelGGL(k_quad<int32_t>, blocks, dim3(64), 0, s, S, x, o, n_y);
    if (split > 0)
        hipLaunchKernelGGL(k_quad_split, dim3((unsigned) ((split + 255) / 256), (unsigned) n), dim3(256), 0, s, S, o);
    if (terms > MQI_QUAD_ONE)
        hipLaunchKernelGGL(k_quad_chunks, dim3(MQI_QUAD_SUM_BLOCKS, (unsigned) n), dim3(256), 0, s, S);
    hipLaunchKernelGGL(k_quad_sum, dim3((unsigned) n), dim3(1024), 0, s, S, 1.0 / (double) n_y, f);
    return (int) hipGetLastError();
}

// ------------------------------------------------------------------ D^T g over column deltas
// Index compression of the CSR stream (delta coding of the column indices,
// after K. Kourtis, G. Goumas and N. Koziris, "Optimizing sparse
// matrix-vector multiplication using index and value compression", CF'08):
// a nonzero keeps its value and the difference of its column to the
// previous nonzero of its row.  The nonzeros are cut into pieces of <=
// MQI_PIECE entries of one row, also where a row skips more than 65535
// columns; a piece keeps the column its first delta adds to (pbase).  For
// the product the pieces are restaged: padded with zero values and zero
// deltas to whole batches of 256 nonzeros, each batch lane-major (the
// 16-byte value load of lane l holds the batch's nonzeros l, l + 64,
// l + 128 and l + 192, its 4-byte delta load their deltas), so that each of
// the four gathers of a batch reads the columns of 64 consecutive nonzeros:
// few distinct cache lines per gather instruction instead of every fourth
// column of 256.  A delta takes one byte; the 1.2 % of deltas of 255 and
// more (the steps between the rows and slices of a spot's footprint on the
// 5000-spot Dij) are escapes, kept in order in the piece's escape list:
// 5.02 bytes per nonzero instead of 8.
// One wave per piece rebuilds the columns with wave prefix sums of the
// deltas and forms the FP64 sum of the piece into part[piece]; a second pass
// adds each row's pieces in a fixed order, so results do not depend on
// scheduling or on the order the pieces run in.  (Offsets from each batch's
// first column instead of deltas need no prefix sums, but the sparse halo of
// a spot spans more than 65535 columns in 256 nonzeros so often that the
// cuts it needs made the pieces tiny: 13x slower on the 5000-spot Dij.)

// dcol[k] = col[k] - col[k - 1] where that is in [1, 65535], else 0; the
// positions with a larger step are listed in gaps[] (count in *n_gaps, at
// most cap written).  Row starts are cleared afterwards (k_row_starts).
__global__ void k_deltas(const int32_t* __restrict__ col, int64_t nnz, uint16_t* __restrict__ dcol,
                         unsigned long long* __restrict__ n_gaps, int64_t* __restrict__ gaps, int64_t cap) {
    for (int64_t k = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; k < nnz; k += (int64_t) gridDim.x * blockDim.x) {
        const int64_t d = k > 0 ? (int64_t) col[k] - (int64_t) col[k - 1] : 0;
        const bool    ok = d >= 1 && d <= 65535;
        dcol[k]          = ok ? (uint16_t) d : (uint16_t) 0;
        if (!ok && d > 65535) {
            const unsigned long long at = atomicAdd(n_gaps, 1ull);
            if ((int64_t) at < cap) gaps[at] = k;
        }
    }
}

__global__ void k_row_starts(const int64_t* __restrict__ indptr, int64_t rows, uint16_t* __restrict__ dcol) {
    const int64_t r = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (r < rows && indptr[r + 1] > indptr[r]) dcol[indptr[r]] = 0;
}

// pbase[p] = col[pk[p]] - dcol[pk[p]]: the column the piece's first delta
// adds to (0 for the empty piece of an empty row)
__global__ void k_piece_base(const int32_t* __restrict__ col, const uint16_t* __restrict__ dcol,
                             const int64_t* __restrict__ pk, int64_t n_p, int32_t* __restrict__ pbase) {
    const int64_t p = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (p < n_p) pbase[p] = pk[p] < pk[p + 1] ? col[pk[p]] - (int32_t) dcol[pk[p]] : 0;
}

// deltas of 255 and more are escapes: the byte holds 255 and the piece's
// escape list (in nonzero order) the delta
#define MQI_ESC 255

// ecount[p]: the escapes of piece p; one workgroup of 256 per piece
__global__ void k_piece_escapes(const uint16_t* __restrict__ dcol, const int64_t* __restrict__ pk, int64_t n_p,
                                uint32_t* __restrict__ ecount) {
    typedef hipcub::BlockReduce<uint32_t, 256> BR;
    __shared__ typename BR::TempStorage tmp;
    for (int64_t p = blockIdx.x; p < n_p; p += gridDim.x) {
        const int64_t kb = pk[p], len = pk[p + 1] - kb;
        uint32_t      n  = 0;
        for (int64_t i = threadIdx.x; i < len; i += 256) n += dcol[kb + i] >= MQI_ESC ? 1u : 0u;
        const uint32_t t = BR(tmp).Sum(n);
        if (threadIdx.x == 0) ecount[p] = t;
        __syncthreads();
    }
}

// pb[p]: the piece's first staged slot (a multiple of 256); pb[n_p]: total.
// Nonzero i of a piece goes to batch i / 256, lane i % 64, byte (i / 64) % 4
// of the lane's word; its escape (if any) to esc[ebase[p] + the escapes
// before it in the piece].  One workgroup of 256 per piece.
__global__ void k_stage_pieces(const float* __restrict__ val, const uint16_t* __restrict__ dcol,
                               const int64_t* __restrict__ pk, const int64_t* __restrict__ pb,
                               const uint32_t* __restrict__ ebase, int64_t n_p, float* __restrict__ sval,
                               uint8_t* __restrict__ sd8, uint16_t* __restrict__ esc) {
    typedef hipcub::BlockScan<uint32_t, 256> BS;
    __shared__ typename BS::TempStorage tmp;
    for (int64_t p = blockIdx.x; p < n_p; p += gridDim.x) {
        const int64_t kb = pk[p], len = pk[p + 1] - kb, base = pb[p], padded = pb[p + 1] - base;
        uint32_t      e  = ebase[p];
        for (int64_t i0 = 0; i0 < padded; i0 += 256) {   // padded is a multiple of 256
            const int64_t  i   = i0 + threadIdx.x;
            const int64_t  j   = i & 255;
            const int64_t  dst = base + i0 + ((j & 63) << 2) + (j >> 6);
            const uint16_t d   = i < len ? dcol[kb + i] : (uint16_t) 0;
            const uint32_t f   = d >= MQI_ESC ? 1u : 0u;
            uint32_t       off, tot;
            BS(tmp).ExclusiveSum(f, off, tot);
            sval[dst] = i < len ? val[kb + i] : 0.0f;
            sd8[dst]  = (uint8_t) (f ? MQI_ESC : d);
            if (f) esc[e + off] = d;
            e += tot;
            __syncthreads();
        }
    }
}

// inclusive prefix sum over the wave: DPP row shifts within the four rows
// of 16 lanes, then the row broadcasts of lanes 15 and 31
MQI_DI uint32_t wave_scan_dpp(uint32_t x) {
    x += (uint32_t) __builtin_amdgcn_update_dpp(0, (int) x, 0x111, 0xf, 0xf, false);   // row_shr:1
    x += (uint32_t) __builtin_amdgcn_update_dpp(0, (int) x, 0x112, 0xf, 0xf, false);   // row_shr:2
    x += (uint32_t) __builtin_amdgcn_update_dpp(0, (int) x, 0x114, 0xf, 0xf, false);   // row_shr:4
    x += (uint32_t) __builtin_amdgcn_update_dpp(0, (int) x, 0x118, 0xf, 0xf, false);   // row_shr:8
    x += (uint32_t) __builtin_amdgcn_update_dpp(0, (int) x, 0x142, 0xa, 0xf, false);   // row_bcast:15
    x += (uint32_t) __builtin_amdgcn_update_dpp(0, (int) x, 0x143, 0xc, 0xf, false);   // row_bcast:31
    return x;
}

// One wave per piece, MQI_PIECE_BATCHES batches (2048 nonzeros) in flight;
// the pieces run in the order of their headers (first columns ascending:
// pieces that run at the same time gather from the same stretch of x).
// The wave keeps the next 64 escapes of its piece in a register (one per
// lane) and hands them to the lanes whose byte is an escape.
__global__ void __launch_bounds__(64 * MQI_PIECE_WAVES)
    k_pieces_staged(const float* __restrict__ sval, const uint8_t* __restrict__ sd8, const uint16_t* __restrict__ esc,
                    const float* __restrict__ x, const piece_hdr* __restrict__ hdr, int64_t n_p,
                    double* __restrict__ part) {
    constexpr int U    = MQI_PIECE_BATCHES;
    const int     lane = threadIdx.x & 63;
    const int64_t w    = (int64_t) blockIdx.x * MQI_PIECE_WAVES + (threadIdx.x >> 6);
    const int64_t nw   = (int64_t) gridDim.x * MQI_PIECE_WAVES;
    for (int64_t i = w; i < n_p; i += nw) {
        // the whole header in two 16-byte loads
        const u32x4     h  = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(hdr + i));
        const u32x4     h2 = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(hdr + i) + 1);
        const int64_t   p  = (int32_t) h.w;
        const int64_t   b0 = h.x, nb = h.y;
        const f32x4*    v4 = reinterpret_cast<const f32x4*>(sval) + b0 * 64;
        const uint32_t* d4 = reinterpret_cast<const uint32_t*>(sd8) + b0 * 64;
        uint32_t        run = h.z;
        // escapes: esc[e_ptr + lane] in e_reg, e_off of them used
        uint32_t        e_ptr = h2.x, e_off = 0;
        uint32_t        e_reg = esc[e_ptr + lane];   // the list is padded by 64
        double          acc   = 0.0;
        for (int64_t b = 0; b < nb; b += U) {
            f32x4    v[U];
            uint32_t d[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (b + u < nb) {
                    v[u] = __builtin_nontemporal_load(v4 + (b + u) * 64 + lane);
                    d[u] = __builtin_nontemporal_load(d4 + (b + u) * 64 + lane);
                } else {
                    v[u] = f32x4{ 0.0f, 0.0f, 0.0f, 0.0f };
                    d[u] = 0u;
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                // quarter q of the batch (nonzeros 64 q .. 64 q + 63, one per
                // lane): byte q of the lane's word, its columns a prefix sum
                // over the wave
                uint32_t c[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    uint32_t                 dq = (d[u] >> (8 * q)) & 0xffu;
                    const unsigned long long m  = __ballot(dq == MQI_ESC);
                    if (m) {
                        const uint32_t n = (uint32_t) __popcll(m);
                        if (e_off + n > 64) {
                            e_ptr += e_off;
                            e_off = 0;
                            e_reg = esc[e_ptr + lane];
                        }
                        const uint32_t k  = e_off + (uint32_t) __builtin_amdgcn_mbcnt_hi(
                                                       (uint32_t) (m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t) m, 0u));
                        const uint32_t ev = (uint32_t) __shfl((int) e_reg, (int) (k & 63u));
                        if (dq == MQI_ESC) dq = ev;
                        e_off += n;
                    }
                    c[q] = dq;
                }
                const uint32_t s0 = wave_scan_dpp(c[0]);
                const uint32_t t0 = (uint32_t) __builtin_amdgcn_readlane((int) s0, 63);
                const uint32_t s1 = wave_scan_dpp(c[1]);
                const uint32_t t1 = (uint32_t) __builtin_amdgcn_readlane((int) s1, 63);
                const uint32_t s2 = wave_scan_dpp(c[2]);
                const uint32_t t2 = (uint32_t) __builtin_amdgcn_readlane((int) s2, 63);
                const uint32_t s3 = wave_scan_dpp(c[3]);
                const uint32_t t3 = (uint32_t) __builtin_amdgcn_readlane((int) s3, 63);
                acc += (double) v[u].x * (double) x[run + s0];
                acc += (double) v[u].y * (double) x[run + t0 + s1];
                acc += (double) v[u].z * (double) x[run + t0 + t1 + s2];
                acc += (double) v[u].w * (double) x[run + t0 + t1 + t2 + s3];
                run += t0 + t1 + t2 + t3;
            }
        }
        for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
        if (lane == 0) part[p] = acc;
    }
}

// y[r] = alpha * (the pieces row_piece[r] .. row_piece[r + 1] - 1) (* *up)
// (+ y[r]):
// one wave per row, lane l takes pieces q0 + l + 64 k, the wave adds them in
// a fixed tree order
template<typename TY>
__global__ void k_piece_rows(const int32_t* __restrict__ row_piece, int64_t rows, const double* __restrict__ part,
                             TY* __restrict__ y, double alpha, const double* __restrict__ up, int accumulate) {
    const int64_t r    = (int64_t) blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int     lane = threadIdx.x & 63;
    if (r >= rows) return;
    const int32_t q0 = row_piece[r], q1 = row_piece[r + 1];
    double        acc = 0.0;
    for (int32_t q = q0 + lane; q < q1; q += 64) acc += part[q];
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    if (lane == 0) {
        const double out = up ? alpha * acc * *up : alpha * acc;
        y[r]             = accumulate ? (TY) ((double) y[r] + out) : (TY) out;
    }
}

int
deltas16(const int64_t* indptr, const int32_t* col, int64_t rows, int64_t nnz, uint16_t* dcol,
         unsigned long long* n_gaps, int64_t* gaps, int64_t cap, hipStream_t s) {
    if (nnz <= 0) return 0;
    int e = fill_u64(n_gaps, 0ull, 1, s);
    if (e) return e;
    hipLaunchKernelGGL(k_deltas, dim3(grid_for((uint64_t) nnz)), dim3(256), 0, s, col, nnz, dcol, n_gaps, gaps, cap);
    if (rows > 0)
        hipLaunchKernelGGL(k_row_starts, dim3((unsigned) ((rows + 255) / 256)), dim3(256), 0, s, indptr, rows, dcol);
    return (int) hipGetLastError();
}

int
piece_base(const int32_t* col, const uint16_t* dcol, const int64_t* pk, int64_t n_p, int32_t* pbase, hipStream_t s) {
    if (n_p <= 0) return 0;
    hipLaunchKernelGGL(k_piece_base, dim3((unsigned) ((n_p + 255) / 256)), dim3(256), 0, s, col, dcol, pk, n_p, pbase);
    return (int) hipGetLastError();
}

int
piece_escapes(const uint16_t* dcol, const int64_t* pk, int64_t n_p, uint32_t* ecount, hipStream_t s) {
    if (n_p <= 0) return 0;
    hipLaunchKernelGGL(k_piece_escapes, dim3((unsigned) (n_p < 65536 ? n_p : 65536)), dim3(256), 0, s, dcol, pk, n_p,
                       ecount);
    return (int) hipGetLastError();
}

int
stage_pieces(const float* val, const uint16_t* dcol, const int64_t* pk, const int64_t* pb, const uint32_t* ebase,
             int64_t n_p, float* sval, uint8_t* sd8, uint16_t* esc, hipStream_t s) {
    if (n_p <= 0) return 0;
    hipLaunchKernelGGL(k_stage_pieces, dim3((unsigned) (n_p < 65536 ? n_p : 65536)), dim3(256), 0, s, val, dcol, pk, pb,
                       ebase, n_p, sval, sd8, esc);
    return (int) hipGetLastError();
}

int
pieces_staged(const float* sval, const uint8_t* sd8, const uint16_t* esc, const float* x, const piece_hdr* hdr,
              int64_t n_p, const int32_t* row_piece, int64_t rows, double* part, void* y, int y_is_double,
              double alpha, const double* up, int accumulate, hipStream_t s) {
    if (n_p > 0) {
        const int64_t b = (n_p + MQI_PIECE_WAVES - 1) / MQI_PIECE_WAVES;
        hipLaunchKernelGGL(k_pieces_staged, dim3((unsigned) (b < 65536 ? b : 65536)), dim3(64 * MQI_PIECE_WAVES), 0,
                           s, sval, sd8, esc, x, hdr, n_p, part);
    }
    if (rows > 0) {
        const unsigned b = (unsigned) ((rows + 3) / 4);
        if (y_is_double)
            hipLaunchKernelGGL(k_piece_rows<double>, dim3(b), dim3(256), 0, s, row_piece, rows, part, (double*) y,
                               alpha, up, accumulate);
        else
            hipLaunchKernelGGL(k_piece_rows<float>, dim3(b), dim3(256), 0, s, row_piece, rows, part, (float*) y,
                               alpha, up, accumulate);
    }
    return (int) hipGetLastError();
}

// Compacted x for D^T g: xc[i] = x[nzvox[i]] (nzvox: the voxels that appear
// in some row, ascending), rounded to float here if x is double: a conversion
// of the whole vector first reads and writes every voxel (20 us for 8.4 M).
// four entries per thread: 16-byte index loads and stores
template<typename TX>
__global__ void k_gather_x(const TX* __restrict__ x, const int32_t* __restrict__ nzvox, int64_t n,
                           float* __restrict__ xc) {
    const int64_t n4 = n >> 2;
    for (int64_t i = (int64_t) blockIdx.x * blockDim.x + threadIdx.x; i < n4; i += (int64_t) gridDim.x * blockDim.x) {
        const i32x4 v = __builtin_nontemporal_load(reinterpret_cast<const i32x4*>(nzvox) + i);
        f32x4       o;
        o.x = (float) x[v.x];
        o.y = (float) x[v.y];
        o.z = (float) x[v.z];
        o.w = (float) x[v.w];
        __builtin_nontemporal_store(o, reinterpret_cast<f32x4*>(xc) + i);
    }
    const int64_t t = (n4 << 2) + (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    if (blockIdx.x == 0 && t < n) xc[t] = (float) x[nzvox[t]];
}

int
gather_x(const void* x, int x_double, const int32_t* nzvox, int64_t n, float* xc, hipStream_t s) {
    if (n <= 0) return 0;
    const dim3 g(grid_for((uint64_t) (n + 3) / 4));
    if (x_double)
        hipLaunchKernelGGL(k_gather_x<double>, g, dim3(256), 0, s, (const double*) x, nzvox, n, xc);
    else
        hipLaunchKernelGGL(k_gather_x<float>, g, dim3(256), 0, s, (const float*) x, nzvox, n, xc);
    return (int) hipGetLastError();
}

}   // namespace mqi_aux

namespace mqi_aux
{
// out[s][i] += pair[stride i + s] for s < ns over n elements (stride 2 or 4);
// the pair array is cleared where it held a sum
struct fold_outs {
    double* o[4];
};
__global__ void k_pair_fold(fold_outs out, int ns, int stride, double* __restrict__ pair, uint64_t n) {
    for (uint64_t i = (uint64_t) blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t) gridDim.x * blockDim.x) {
        double* e = pair + (uint64_t) stride * i;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            if (s >= ns) break;
            const double x = e[s];
            if (x != 0.0) {
                out.o[s][i] += x;
                e[s] = 0.0;
            }
        }
    }
}
int
pair_fold(double* const* out, int ns, int stride, double* pair, uint64_t n, hipStream_t s) {
    if (n == 0) return 0;
    if (ns < 1 || ns > 4 || ns > stride) return (int) hipErrorInvalidValue;
    fold_outs o{};
    for (int k = 0; k < ns; ++k) o.o[k] = out[k];
    hipLaunchKernelGGL(k_pair_fold, dim3(grid_for(n)), dim3(256), 0, s, o, ns, stride, pair, n);
    return (int) hipGetLastError();
}
}   // namespace mqi_aux
