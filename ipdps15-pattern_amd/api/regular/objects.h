// The reduction objects a generalized-reduction functor inserts into, with
// the insert(key, key_size, value, value_size, reduce_ptr) call of the
// reference (kmeans/regular/ros.h:33 on the GPU, roc.h:39 on the CPU): the
// first value for a key is copied, later ones are folded into it by the
// reduce functor; insert returns false when the object has no room.
//
// CO (host): a map from key bytes to value bytes, never full.
// SO (device, api/gpu/regular_table.hpp): a wavefront's own open-addressing
// hash table in LDS.  The lanes that call insert together look their keys up
// and add the new ones side by side; the values of one key are then folded
// in lane order, so the table needs no locks and every value is folded in a
// fixed order.  When it is full, insert returns false; the engine then moves
// the table into the wavefront's table in device memory, clears it and runs
// the unit's map again (the reference's merge-and-retry,
// kmeans/regular/gpu_kernel.cu:143-150).
//
// Also: ANY_KEY() (kmeans/regular/kernel_tools.h:15 -- 0 on the host, the
// thread index mod 41 on the device, spreading one logical key over 41
// buckets as the reference does) and copy_val.
#ifndef REGULAR_OBJECTS_H_
#define REGULAR_OBJECTS_H_

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

#include "data_type.h"

class CO {
  public:
    typedef void (*reduce_fn)(void *, unsigned short, void *, unsigned short);
    CO() = default;
    // kept for drivers that size a dense object: the bound is not needed
    CO(int max_keys, int value_size) { (void)max_keys, (void)value_size; }
    bool insert(void *key, unsigned short ksize, void *value, unsigned short vsize, reduce_fn reduce)
    {
        std::string k((const char *)key, ksize);
        auto it = vals_.find(k);
        if (it == vals_.end()) {
            Val v(vsize);
            memcpy(v.p, value, vsize);
            vals_.emplace(std::move(k), std::move(v));
        } else {
            reduce(it->second.p, (unsigned short)it->second.n, value, vsize);
        }
        return true;
    }
    // key bytes -> value bytes
    std::map<std::string, std::string> entries() const
    {
        std::map<std::string, std::string> r;
        for (const auto &e : vals_) r.emplace(e.first, std::string((const char *)e.second.p, e.second.n));
        return r;
    }
    // by an unsigned int key
    bool used(unsigned int k) const { return vals_.count(ukey(k)) != 0; }
    const void *value(unsigned int k) const { return vals_.at(ukey(k)).p; }

  private:
    // a value's bytes in malloc'd storage, which the functors read and write
    // as their own types
    struct Val {
        void *p = nullptr;
        size_t n = 0;
        explicit Val(size_t bytes) : p(std::malloc(bytes ? bytes : 1)), n(bytes) {}
        Val(Val &&o) noexcept : p(o.p), n(o.n) { o.p = nullptr; }
        Val(const Val &) = delete;
        Val &operator=(const Val &) = delete;
        ~Val() { std::free(p); }
    };
    static std::string ukey(unsigned int k) { return std::string((const char *)&k, sizeof(k)); }
    std::map<std::string, Val> vals_;
};

#ifdef __HIPCC__
#include <hip/hip_runtime.h>

namespace pat_gpu {

// Words of the tables: keys and values of any type are stored into and read
// out of them, so every access goes through a type that may alias the
// functors' own (float, double, struct) accesses to the same bytes.
typedef uint32_t __attribute__((__may_alias__)) ro_word;

// FNV-1a over the key bytes.
__device__ __forceinline__ uint32_t ro_hash(const unsigned char *k, int n)
{
    uint32_t h = 2166136261u;
    for (int i = 0; i < n; i++) h = (h ^ k[i]) * 16777619u;
    return h;
}

__device__ __forceinline__ void ro_copy(void *dst, const void *src, int n)
{
    if ((((uintptr_t)dst | (uintptr_t)src | (uintptr_t)n) & 3) == 0) {
        for (int i = 0; i < n / 4; i++) ((ro_word *)dst)[i] = ((const ro_word *)src)[i];
    } else {
        for (int i = 0; i < n; i++) ((unsigned char *)dst)[i] = ((const unsigned char *)src)[i];
    }
}

__device__ __forceinline__ bool ro_equal(const void *a, const void *b, int n)
{
    for (int i = 0; i < n; i++)
        if (((const unsigned char *)a)[i] != ((const unsigned char *)b)[i]) return false;
    return true;
}

// Orders a wavefront's LDS accesses for the compiler (the hardware keeps one
// wavefront's LDS operations in order).
__device__ __forceinline__ void ro_wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Bucket state of an LDS table besides 0 (empty) and 1 + a record's word
// offset in the pool.
constexpr uint32_t kRoClaim = 0x40000000u;  // | (63 - lane): being taken, within one insert only

// A wavefront's LDS hash table: nb buckets (a power of two), then the pool's
// fill counter, then pw pool words.  Record: a header word (key_size << 16 |
// value_size), the key and the value, each padded to whole words.
struct RoTable {
    ro_word *bk, *top, *pool;
    int nb, pw;

    __device__ static RoTable at(ro_word *base, int nb, int pw)
    {
        return RoTable{base, base + nb, base + nb + 1, nb, pw};
    }
    __host__ __device__ static int words(int nb, int pw) { return nb + 1 + pw; }
    __device__ void clear(int lane, int nlanes)
    {
        for (int b = lane; b < nb; b += nlanes) bk[b] = 0u;
        if (lane == 0) *top = 0u;
    }
    __device__ static int key_words(int ks) { return (ks + 3) >> 2; }

    // The record (1 + word offset) of each calling lane's key, added where it
    // is new (fresh: its value is still to be written), 0 where no bucket or
    // no pool room is left.  Keys of up to eight bytes.  The lanes probe
    // together; where several want one empty bucket the lowest takes it, and
    // new records take pool room in lane order, so that the same lanes are
    // refused every run.  A refused key leaves its bucket empty to the others
    // that wanted it.  Lanes with one key probe in step, so they get one
    // record in one round.
    __device__ uint32_t place(const void *key, int ks, int vs, bool &fresh)
    {
        const int lane = (int)__lane_id();
        uint32_t k0 = 0u, k1 = 0u;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (i < ks) k0 |= (uint32_t)((const unsigned char *)key)[i] << (8 * i);
            if (i + 4 < ks) k1 |= (uint32_t)((const unsigned char *)key)[i + 4] << (8 * i);
        }
        const uint32_t hdr = ((uint32_t)ks << 16) | (uint32_t)vs;
        const int need = 1 + key_words(ks) + ((vs + 3) >> 2);
        const uint32_t h = ro_hash((const unsigned char *)key, ks);
        uint32_t rec = 0u;
        bool open = true;
        fresh = false;
        int p = 0;  // buckets seen: all of them, and the lane is refused
        // (every round an open lane goes on by a bucket, or one is closed)
        for (int round = 0; __ballot(open) && round < nb + 64; round++) {
            const int b = (int)((h + (uint32_t)p) & (uint32_t)(nb - 1));
            bool want = false;
            if (open) {
                const uint32_t st = bk[b];
                want = st == 0u;
                if (!want) {
                    const ro_word *r = pool + (st - 1u);
                    if (r[0] == hdr && (ks < 1 || r[1] == k0) && (ks < 5 || r[2] == k1)) {
                        rec = st;
                        open = false;
                    } else {
                        open = ++p < nb;
                    }
                }
            }
            if (!__ballot(want)) continue;
            ro_wave_sync();
            if (want) atomicMax((uint32_t *)&bk[b], kRoClaim | (uint32_t)(63 - lane));
            ro_wave_sync();
            const int w = want ? 63 - (int)(bk[b] & 63u) : lane;
            const bool won = want && w == lane;
            // pool room for the winners, in lane order
            const unsigned long long wins = __ballot(won);
            const int used = (int)*top;
            int off = -1, end = used;
            const int first = __shfl(need, __ffsll((long long)wins) - 1);
            if (!__ballot(won && need != first)) {
                const int room = (pw - used) / first;
                const int rank = __popcll(wins & ((1ull << lane) - 1ull));
                if (won && rank < room) off = used + rank * first;
                const int taken = __popcll(wins);
                end = used + (taken < room ? taken : room) * first;
            } else {
                for (unsigned long long m = wins; m; m &= m - 1) {
                    const int l = __ffsll((long long)m) - 1;
                    const int n = __shfl(need, l);
                    if (end + n <= pw) {
                        if (lane == l) off = end;
                        end += n;
                    }
                }
            }
            ro_wave_sync();
            if (won) {
                *top = (uint32_t)end;
                if (off >= 0) {
                    ro_word *r = pool + off;
                    r[0] = hdr;
                    if (ks > 0) r[1] = k0;
                    if (ks > 4) r[2] = k1;
                    rec = (uint32_t)off + 1u;
                    fresh = true;
                }
                bk[b] = rec;
                open = false;
            }
            ro_wave_sync();
            const uint32_t wh = (uint32_t)__shfl((int)hdr, w), w0 = (uint32_t)__shfl((int)k0, w),
                           w1 = (uint32_t)__shfl((int)k1, w), wr = (uint32_t)__shfl((int)rec, w);
            if (want && !won) {
                if (wh == hdr && w0 == k0 && w1 == k1) {  // the winner's key: its record or its refusal
                    rec = wr;
                    fresh = wr != 0u;
                    open = false;
                } else if (wr != 0u) {
                    open = ++p < nb;
                }
            }
        }
        return rec;
    }

    // place() for keys of any size, one lane's turn: finds or adds.
    __device__ uint32_t place_one(const void *key, int ks, int vs, bool &fresh)
    {
        const uint32_t h = ro_hash((const unsigned char *)key, ks);
        const uint32_t hdr = ((uint32_t)ks << 16) | (uint32_t)vs;
        fresh = false;
        for (int p = 0; p < nb; p++) {
            const int b = (int)((h + (uint32_t)p) & (uint32_t)(nb - 1));
            const uint32_t st = bk[b];
            if (st == 0u) {
                const int need = 1 + key_words(ks) + ((vs + 3) >> 2);
                const uint32_t rec = *top;
                if ((int)rec + need > pw) return 0u;
                *top = rec + (uint32_t)need;
                ro_word *r = pool + rec;
                r[0] = hdr;
                for (int w = 0; w < key_words(ks); w++) r[1 + w] = 0u;
                ro_copy(r + 1, key, ks);
                bk[b] = rec + 1u;
                fresh = true;
                return rec + 1u;
            }
            ro_word *r = pool + (st - 1u);
            if (r[0] == hdr && ro_equal(r + 1, key, ks)) return st;
        }
        return 0u;
    }
};

}  // namespace pat_gpu

// A wavefront's LDS reduction object.  Per lane, over one map call: full = an
// insert was refused, accepted = inserts taken.
class SO {
  public:
    pat_gpu::RoTable t;
    bool full = false;
    int accepted = 0;

    // Lanes that call together are placed together (place; in turn for keys
    // beyond eight bytes).  The lanes of one record are then found by the
    // bits of its offset, and fold in lane order, the records side by side:
    // as many rounds as the most lanes that share a key, where one turn per
    // lane took 64.
    template <typename R>
    __device__ bool insert(void *key, unsigned short ksize, void *value, unsigned short vsize, R reduce_ptr)
    {
        const int lane = (int)__lane_id();
        uint32_t rec = 0u;
        bool fresh = false;
        if (!__ballot(ksize > 8)) {
            rec = t.place(key, ksize, vsize, fresh);
        } else {
            // a key placed earlier in this call is fresh for the later lanes
            // too; which of them copies is settled below by lane order
            const uint32_t before = *t.top;
            pat_gpu::ro_wave_sync();
            for (unsigned long long turn = __ballot(1); turn; turn &= turn - 1) {
                if (lane == __ffsll((long long)turn) - 1) rec = t.place_one(key, ksize, vsize, fresh);
                pat_gpu::ro_wave_sync();
            }
            fresh = rec > before;
        }
        const bool ok = rec != 0u;
        unsigned long long same = __ballot(ok);
        for (int bit = 0; (1 << bit) <= t.pw; bit++) {
            const bool one = (rec >> bit) & 1u;
            const unsigned long long m = __ballot(ok && one);
            same &= one ? m : ~m;
        }
        const int rank = __popcll(same & ((1ull << lane) - 1ull));
        pat_gpu::ro_wave_sync();
        for (int r = 0; __ballot(ok && rank >= r); r++) {
            if (ok && rank == r) {
                void *v = (void *)(t.pool + rec + pat_gpu::RoTable::key_words(ksize));  // rec - 1, header, key
                if (r == 0 && fresh)
                    pat_gpu::ro_copy(v, value, vsize);
                else
                    reduce_ptr(v, vsize, value, vsize);
            }
            pat_gpu::ro_wave_sync();
        }
        if (ok)
            accepted++;
        else
            full = true;
        return ok;
    }
};

__device__ __forceinline__ unsigned int ANY_KEY() { return threadIdx.x % 41; }
__device__ __forceinline__ void copy_val(void *dst, const void *src, unsigned size) { pat_gpu::ro_copy(dst, src, (int)size); }
#else
inline unsigned int ANY_KEY() { return 0; }
inline void copy_val(void *dst, const void *src, unsigned size) { memcpy(dst, src, size); }
#endif

#endif
