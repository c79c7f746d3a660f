// Device execution of an application's generalized-reduction functor table
// with keyed reduction objects.
//
// The reference runs map over 5,000-unit tasks, inserting (key, value) pairs
// into an LDS hash per thread group; when an insert finds the object full the
// map returns false, the group merges its LDS object into the device object
// and runs the unit again (kmeans/regular/gpu_kernel.cu:39-183, ros.cu:15-170,
// rog.cu:17-310), with per-bucket spin locks throughout.  Here:
//
//  * ro_map: each wavefront takes a contiguous run of units and owns an LDS
//    hash table (SO, api/regular/objects.h) whose inserts the lanes make
//    together, each key's values folded in lane order -- no locks, a fixed
//    fold order;
//  * a refused insert (table full) makes the wavefront merge its LDS table
//    into its own table in device memory, clear it, and run the refused
//    units' maps again; a map that returns false is run again the same way
//    (the reference's contract).  A map whose refused insert followed an
//    accepted one cannot be run again without inserting twice: that is an
//    error, as is a unit whose values do not fit an empty LDS table.  A
//    wavefront that was never refused writes its LDS records out as they are;
//  * ro_claim: every record of every wavefront looks its key up in the final
//    buckets, claiming an empty one by compare-and-swap.  A bucket holds the
//    place of the record that claimed it, written by the kernel before, so
//    a key is compared at once and no thread waits for another.  The record's
//    place goes into the bucket's row of the matrix, one column a wavefront;
//  * ro_fold: one workgroup per claimed bucket folds its row in column order,
//    a run of columns a thread, then the threads' values in a tree, and
//    writes the final record.
//
// What bounds it: latencies, of the LDS rounds in ro_map and of the dependent
// record reads in ro_fold; the bytes are few.  One fold workgroup walking
// every wavefront's buckets and inserts one lane at a time took, for 1 M
// points of kmeans' map1 (40 keys), 9.7 + 3.6 ms, and for 500,000 values in
// 5,003 keys 32 + 54 ms; these kernels take 0.12 + 0.04 + 0.02 ms (map, claim,
// fold) and 0.04 + 0.06 + 0.10 ms.
//
// Every key's value is therefore the same fold over the units every run.
// The library (pat_regular_*) sizes the tables and reads the final one.
//
//     #define GPU_KERNEL
//     #include "regular.h"
//     #include "gpu/regular_table.hpp"
//     PAT_GR_TABLE(FFGPU::map_function_table, FFGPU::reduce_function_table)
#ifndef PAT_GPU_REGULAR_TABLE_HPP_
#define PAT_GPU_REGULAR_TABLE_HPP_

#include <hip/hip_runtime.h>

#include <cstdint>
#include <utility>

#include "pattern.h"
#include "regular/objects.h"

namespace pat_gpu {

// LDS of a wavefront's table, one wavefront per workgroup: 512 buckets and 8
// KiB of records, so that the keys of a few hundred units fit without a merge
// and fifteen wavefronts still fit a CU.
constexpr int kRoLdsBuckets = 512;
constexpr int kRoLdsPool = 2048;
constexpr uint32_t kRoPending = 0xffffffffu;
constexpr int kRoFoldThreads = 256;
constexpr int kRoFoldWords = 16;  // a value up to this many words is folded in LDS, a larger one in place

enum RoError { kRoWaveFull = 1, kRoUnitTooLarge = 2, kRoPartialRefusal = 4, kRoFinalFull = 8 };
enum RoStatus { kRoError = 0, kRoMerges = 1, kRoReruns = 2, kRoSlots = 3, kRoWords = 4 };

__device__ __forceinline__ ro_word *ro_wave_buckets(const pat_gr_object &a, int64_t w)
{
    return (ro_word *)a.wave_tables + (size_t)w * ((size_t)a.table_buckets + (size_t)a.table_pool_words);
}
__device__ __forceinline__ ro_word *ro_wave_pool(const pat_gr_object &a, int64_t w)
{
    return ro_wave_buckets(a, w) + a.table_buckets;
}

// One record of the wavefront's LDS table into its table in device memory.
// The lanes insert distinct keys together: a bucket another lane is filling
// (kRoPending) never holds this key.
template <typename R>
__device__ bool ro_insert_wave(const pat_gr_object &a, ro_word *bk, ro_word *pool, ro_word *top, const ro_word *rec,
                               R reduce)
{
    const int ks = (int)(rec[0] >> 16), vs = (int)(rec[0] & 0xffffu);
    const ro_word *key = rec + 1;
    const ro_word *val = rec + 1 + RoTable::key_words(ks);
    const uint32_t h = ro_hash((const unsigned char *)key, ks);
    for (int p = 0; p < a.table_buckets; p++) {
        const int b = (int)((h + (uint32_t)p) & (uint32_t)(a.table_buckets - 1));
        uint32_t st = __hip_atomic_load((uint32_t *)&bk[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (st == 0u) {
            st = atomicCAS((uint32_t *)&bk[b], 0u, kRoPending);
            if (st == 0u) {
                const int need = 1 + RoTable::key_words(ks) + ((vs + 3) >> 2);
                const uint32_t at = atomicAdd((uint32_t *)top, (uint32_t)need);
                if ((int64_t)at + need > a.table_pool_words) return false;  // the bucket stays claimed: the result is void
                ro_word *r = pool + at;
                for (int i = 0; i < need; i++) r[i] = rec[i];
                __threadfence_block();  // the record before its place: other lanes may read it as soon as they see that
                atomicExch((uint32_t *)&bk[b], at + 1u);
                return true;
            }
        }
        if (st == kRoPending) continue;
        __threadfence_block();  // the place before the record
        ro_word *r = pool + (st - 1u);
        if (r[0] == rec[0] && ro_equal(r + 1, key, ks)) {
            reduce((void *)(r + 1 + RoTable::key_words(ks)), (unsigned short)vs, (void *)val, (unsigned short)vs);
            return true;
        }
    }
    return false;
}

template <class Tab, int MI, int RI>
__global__ __launch_bounds__(64) void ro_map(pat_gr_object a)
{
    extern __shared__ ro_word ro_lds[];  // the table, then the pool counter of the table in device memory
    const int lane = (int)threadIdx.x;
    const int64_t w = (int64_t)blockIdx.x;
    // this wavefront's share of the final buckets, cleared for ro_claim
    for (int64_t b = w * 64 + lane; b < a.table_buckets; b += (int64_t)a.waves * 64) a.final_buckets[b] = 0ull;
    SO so;
    so.t = RoTable::at(ro_lds, a.lds_buckets, a.lds_pool_words);
    ro_word *wtop = ro_lds + RoTable::words(a.lds_buckets, a.lds_pool_words);
    so.t.clear(lane, 64);
    ro_wave_sync();
    ro_word *wbk = ro_wave_buckets(a, w), *wpool = ro_wave_pool(a, w);
    const auto reduce = Tab::template reduce<RI>();
    int err = 0, flushes = 0, reruns = 0;
    bool spilled = false;
    // moves the LDS table into the wavefront's table in device memory
    auto spill = [&]() {
        if (!spilled) {
            for (int b = lane; b < a.table_buckets; b += 64)
                __hip_atomic_store((uint32_t *)&wbk[b], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (lane == 0) *wtop = 0u;
            spilled = true;
        }
        __threadfence_block();
        ro_wave_sync();
        for (int b0 = 0; b0 < so.t.nb; b0 += 64) {
            const uint32_t st = b0 + lane < so.t.nb ? so.t.bk[b0 + lane] : 0u;
            if (st != 0u && !ro_insert_wave(a, wbk, wpool, wtop, so.t.pool + (st - 1u), reduce))
                err |= kRoWaveFull;
            // the next records may fold into the ones just written
            __threadfence_block();
            ro_wave_sync();
        }
    };
    const int64_t per = (a.num_units + a.waves - 1) / a.waves;
    const int64_t u0 = w * per, u1 = u0 + per < a.num_units ? u0 + per : a.num_units;
    for (int64_t base = u0; base < u1; base += 64) {
        const int64_t u = base + lane;
        bool pending = u < u1;
        // every round after a merge, the lowest pending lane inserts into an
        // empty table, so each round finishes at least one unit unless that
        // unit cannot fit an empty table: 65 rounds suffice
        for (int round = 0; round < 66 && __ballot(pending); round++) {
            so.full = false;
            so.accepted = 0;
            bool ok = true;
            if (pending) {
                const unsigned long long idx =
                    a.offsets ? (unsigned long long)a.offsets[u] : (unsigned long long)(u * a.unit_bytes);
                ok = Tab::template map<MI, RI>(&so, const_cast<void *>(a.data), idx, const_cast<void *>(a.param));
            }
            if (pending && so.full && so.accepted > 0) {
                err |= kRoPartialRefusal;  // part of the unit went in: it cannot run again
                pending = false;
            }
            const bool again = pending && (!ok || so.full);
            if (__ballot(again)) {
                spill();
                so.t.clear(lane, 64);
                ro_wave_sync();
                flushes++;
                reruns += __popcll(__ballot(again));
            }
            pending = again;
        }
        if (__ballot(pending)) err |= kRoUnitTooLarge;
    }
    ro_wave_sync();
    int count = a.table_buckets;  // a spilled table's buckets, or the records' places one after another
    if (spilled) {
        spill();
    } else {
        const int top = (int)*so.t.top;
        count = 0;
        for (int b0 = 0; b0 < so.t.nb; b0 += 64) {
            const uint32_t st = b0 + lane < so.t.nb ? so.t.bk[b0 + lane] : 0u;
            const bool have = st != 0u;
            const unsigned long long m = __ballot(have);
            const int at = count + __popcll(m & ((1ull << lane) - 1ull));
            if (have && at < a.table_buckets) wbk[at] = st;
            count += __popcll(m);
        }
        if (count > a.table_buckets || top > a.table_pool_words) {
            err |= kRoWaveFull;
            count = 0;
        } else {
            for (int i = lane; i < top; i += 64) wpool[i] = so.t.pool[i];
        }
    }
    int werr = 0;
    for (int bit = 1; bit <= kRoFinalFull; bit <<= 1)
        if (__ballot((err & bit) != 0)) werr |= bit;
    if (lane == 0) {
        // a table that overflowed holds claimed buckets without a record
        a.wave_counts[w] = werr & kRoWaveFull ? 0 : count;
        if (werr) atomicOr(&a.status[kRoError], werr);
        atomicAdd(&a.status[kRoMerges], flushes + 1);
        if (reruns) atomicAdd(&a.status[kRoReruns], reruns);
    }
}

// One workgroup per wavefront of ro_map: its records into the final buckets.
static __global__ __launch_bounds__(256) void ro_claim(pat_gr_object a)
{
    const int64_t w = (int64_t)blockIdx.x;
    const ro_word *base = (const ro_word *)a.wave_tables;
    const ro_word *wbk = ro_wave_buckets(a, w), *wpool = ro_wave_pool(a, w);
    const int count = a.wave_counts[w];
    for (int i = (int)threadIdx.x; i < count; i += (int)blockDim.x) {
        const uint32_t st = wbk[i];
        if (st == 0u) continue;
        const ro_word *r = wpool + (st - 1u);
        const int ks = (int)(r[0] >> 16);
        const uint32_t h = ro_hash((const unsigned char *)(r + 1), ks);
        const unsigned long long me = (unsigned long long)(r - base) + 1ull;
        bool placed = false;
        for (int p = 0; p < a.table_buckets && !placed; p++) {
            const int b = (int)((h + (uint32_t)p) & (uint32_t)(a.table_buckets - 1));
            unsigned long long o =
                __hip_atomic_load(&a.final_buckets[b], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (o == 0ull) {
                o = atomicCAS(&a.final_buckets[b], 0ull, me);
                if (o == 0ull) {
                    a.slots[atomicAdd(&a.status[kRoSlots], 1)] = b;  // at most one per bucket
                    o = me;
                }
            }
            const ro_word *q = base + (o - 1ull);
            placed = o == me || (q[0] == r[0] && ro_equal(q + 1, r + 1, ks));
            if (placed) a.matrix[(size_t)b * (size_t)a.waves + (size_t)w] = st;
        }
        if (!placed) atomicOr(&a.status[kRoError], (int)kRoFinalFull);
    }
}

// One workgroup per claimed bucket: its row of the matrix, folded in column
// order, into the final record; the row is cleared again for the next run.
template <class Tab, int RI>
__global__ __launch_bounds__(kRoFoldThreads) void ro_fold(pat_gr_object a)
{
    __shared__ ro_word vals[kRoFoldThreads][kRoFoldWords + 1];  // odd stride: no bank conflicts
    __shared__ ro_word *at[kRoFoldThreads];                     // each thread's value, or none
    const auto reduce = Tab::template reduce<RI>();
    const int t = (int)threadIdx.x;
    const int slots = a.status[kRoSlots];
    const int per = (a.waves + kRoFoldThreads - 1) / kRoFoldThreads;
    for (int s = (int)blockIdx.x; s < slots; s += (int)gridDim.x) {
        const int b = a.slots[s];
        const ro_word *first = (const ro_word *)a.wave_tables + (a.final_buckets[b] - 1ull);
        const uint32_t hdr = first[0];
        const int ks = (int)(hdr >> 16), vs = (int)(hdr & 0xffffu), kw = RoTable::key_words(ks);
        const bool in_lds = vs <= 4 * kRoFoldWords;
        uint32_t *row = a.matrix + (size_t)b * (size_t)a.waves;
        ro_word *acc = nullptr;
        for (int w = t * per; w < (t + 1) * per && w < a.waves; w++) {
            const uint32_t st = row[w];
            if (st == 0u) continue;
            row[w] = 0u;
            ro_word *v = ro_wave_pool(a, w) + st + kw;  // st - 1, header, key
            if (acc) {
                if (in_lds)
                    reduce((void *)vals[t], (unsigned short)vs, (void *)v, (unsigned short)vs);
                else
                    reduce((void *)acc, (unsigned short)vs, (void *)v, (unsigned short)vs);
            } else if (in_lds) {
                for (int i = 0; i < (vs + 3) / 4; i++) vals[t][i] = v[i];
                acc = vals[t];
            } else {
                acc = v;
            }
        }
        at[t] = acc;
        __syncthreads();
        for (int d = 1; d < kRoFoldThreads; d <<= 1) {
            if ((t & (2 * d - 1)) == 0 && at[t + d]) {
                if (!at[t]) {
                    if (in_lds) {
                        for (int i = 0; i < (vs + 3) / 4; i++) vals[t][i] = vals[t + d][i];
                        at[t] = vals[t];
                    } else {
                        at[t] = at[t + d];
                    }
                } else if (in_lds) {
                    reduce((void *)vals[t], (unsigned short)vs, (void *)vals[t + d], (unsigned short)vs);
                } else {
                    reduce((void *)at[t], (unsigned short)vs, (void *)at[t + d], (unsigned short)vs);
                }
            }
            __syncthreads();
        }
        if (t == 0) {
            const int need = 1 + kw + ((vs + 3) >> 2);
            const int64_t to = (int64_t)(uint32_t)atomicAdd(&a.status[kRoWords], need);
            if (to + need > a.table_pool_words) {
                atomicOr(&a.status[kRoError], (int)kRoFinalFull);
            } else {
                ro_word *r = (ro_word *)a.final_pool + to;
                r[0] = hdr;
                for (int i = 0; i < kw; i++) r[1 + i] = first[1 + i];
                for (int i = 0; i < (vs + 3) / 4; i++) r[1 + kw + i] = at[0][i];
            }
        }
        __syncthreads();
    }
}

template <class Tab, int MI, int RI>
int ro_launch(const pat_gr_object &a, hipStream_t st)
{
    if constexpr (!Tab::template valid<MI, RI>()) {
        return PAT_ERR_UNSUPPORTED;
    } else {
        const size_t lds = sizeof(uint32_t) * ((size_t)RoTable::words(a.lds_buckets, a.lds_pool_words) + 1);
        hipLaunchKernelGGL((ro_map<Tab, MI, RI>), dim3((unsigned)a.waves), dim3(64), lds, st, a);
        if (hipGetLastError() != hipSuccess) return PAT_ERR_HIP;
        hipLaunchKernelGGL(ro_claim, dim3((unsigned)a.waves), dim3(256), 0, st, a);
        if (hipGetLastError() != hipSuccess) return PAT_ERR_HIP;
        // enough workgroups to fill the chip with the buckets there may be
        const unsigned grid = (unsigned)(a.table_buckets < 4096 ? a.table_buckets : 4096);
        hipLaunchKernelGGL((ro_fold<Tab, RI>), dim3(grid), dim3(kRoFoldThreads), 0, st, a);
        return hipGetLastError() == hipSuccess ? PAT_OK : PAT_ERR_HIP;
    }
}

template <class Tab, int MI, std::size_t... RI>
int ro_dispatch_reduce(int ri, const pat_gr_object &a, hipStream_t st, std::index_sequence<RI...>)
{
    int rc = PAT_ERR_UNSUPPORTED;
    ((ri == (int)RI ? (void)(rc = ro_launch<Tab, MI, (int)RI>(a, st)) : (void)0), ...);
    return rc;
}

template <class Tab, std::size_t... MI>
int ro_dispatch(int mi, int ri, const pat_gr_object &a, hipStream_t st, std::index_sequence<MI...>)
{
    int rc = PAT_ERR_UNSUPPORTED;
    ((mi == (int)MI ? (void)(rc = ro_dispatch_reduce<Tab, (int)MI>(
                                 ri, a, st, std::make_index_sequence<(std::size_t)Tab::rcount>{}))
                    : (void)0),
     ...);
    return rc;
}

// pat_gr_table::map_reduce for the tables of Tab.
template <class Tab>
int ro_entry(int map_idx, int reduce_idx, const pat_gr_object *obj, void *stream)
{
    if (!obj || obj->layout != 0 || obj->waves <= 0 || !obj->wave_tables || !obj->wave_counts || !obj->matrix || !obj->final_buckets ||
        !obj->slots || !obj->final_pool || !obj->status || obj->lds_buckets <= 0 || obj->lds_buckets > kRoLdsBuckets ||
        (obj->lds_buckets & (obj->lds_buckets - 1)) || obj->lds_pool_words <= 0 ||
        obj->lds_pool_words > kRoLdsPool || obj->table_buckets <= 0 ||
        (obj->table_buckets & (obj->table_buckets - 1)))
        return PAT_ERR_INVALID;
    return ro_dispatch<Tab>(map_idx, reduce_idx, *obj, (hipStream_t)stream,
                            std::make_index_sequence<(std::size_t)Tab::mcount>{});
}

}  // namespace pat_gpu

// Defines pat_app_gr_table() for the application's map and reduce tables
// (__device__ constexpr arrays of map_fp / reduce_fp).
#define PAT_GR_TABLE(MAP_TABLE, REDUCE_TABLE)                                                                     \
    namespace {                                                                                                   \
    struct PatGrTab {                                                                                             \
        static constexpr int mcount = (int)(sizeof(MAP_TABLE) / sizeof(MAP_TABLE[0]));                            \
        static constexpr int rcount = (int)(sizeof(REDUCE_TABLE) / sizeof(REDUCE_TABLE[0]));                      \
        template <int MI, int RI>                                                                                 \
        static constexpr bool valid()                                                                             \
        {                                                                                                         \
            return MAP_TABLE[MI] != nullptr && REDUCE_TABLE[RI] != nullptr;                                       \
        }                                                                                                         \
        template <int RI>                                                                                         \
        __device__ static constexpr auto reduce()                                                                 \
        {                                                                                                         \
            return REDUCE_TABLE[RI];                                                                              \
        }                                                                                                         \
        template <int MI, int RI>                                                                                 \
        __device__ static bool map(SO *o, void *data, unsigned long long index, void *param)                      \
        {                                                                                                         \
            return MAP_TABLE[MI](o, data, index, param, 1, REDUCE_TABLE[RI]);                                     \
        }                                                                                                         \
    };                                                                                                            \
    }                                                                                                             \
    extern "C" const pat_gr_table *pat_app_gr_table(void)                                                         \
    {                                                                                                             \
        static const pat_gr_table t = {PatGrTab::mcount, PatGrTab::rcount, pat_gpu::kRoLdsBuckets,                \
                                       pat_gpu::kRoLdsPool, &pat_gpu::ro_entry<PatGrTab>};                        \
        return &t;                                                                                                \
    }

#endif
