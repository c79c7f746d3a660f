// Generalized-reduction engine for gfx950: kmeans assignment + centroid
// accumulation (the reference's map1/reduce1 functors, kmeans/regular.h:
// 75-136, run by the regular compute_gpu kernel, kmeans/regular/
// gpu_kernel.cu:39-183, into an LDS hash reduction object, ros.cu:15-170).
//
// Reduction object.  map1 emits {x_0..x_{D-1}, 1, min_dist} under key =
// nearest centre and reduce1 adds values per key.  The reference adds FP32
// values in lock-acquisition order, which is not reproducible.  Here each
// coordinate (and min_dist) is rounded once to an integer multiple of 2^-s
// (s chosen so every rounded value fits in 31 bits and the largest possible
// sum in 62) and summed as int64:
// integer addition is associative, so every summation order -- LDS atomics
// within a workgroup, global atomics across workgroups, or the CPU oracle's
// loop -- gives identical bits, and so identical centroids every iteration.
// The dense per-workgroup object (K x D sums, K counts, K distance sums)
// lives in LDS and is flushed once per workgroup with global atomics.
//
// Assignment, plain path: the functor's arithmetic exactly -- for each centre
// in order, dist = sum_d (c_d - x_d)^2 in FP32 in dimension order, sqrt,
// strict < against min_dist starting at 65536*65 (lowest index wins ties).
// Compiled with -ffp-contract=off so no multiply-add is fused.
//
// Assignment, MFMA path: a wavefront takes 32 points and computes
// ||c||^2 - 2 x.c (up to a scale) for every centre with 32x32x16 MFMAs (FP32
// accumulation, the norm split into three terms on an extra K step).
// With NT = 3 terms, x and c are each split into FP16 high and low parts and
// the product is xl.ch + xh.cl + xh.ch (the dropped terms are O(2^-22)
// relative); with NT = 1 x and -2c are rounded to BF16 once (O(2^-8)).  A
// per-point bound E on the error of that value (operand rounding, the norm
// split, FP32 accumulation) plus the FP32 rounding of the reference's own
// difference form gives a margin:
// every centre whose approximate value is within the margin of the smallest
// is rescored with the plain path's exact FP32 arithmetic, and the exact
// results decide (same tie rule).  A centre outside the margin provably has a
// larger reference distance than the best one, so the assignment equals the
// plain path's bit for bit.  Shapes whose object is beyond LDS take the same
// steps against rows in global memory (km_wide).
#include <algorithm>
#include <cmath>
#include <iterator>
#include <vector>

#include "pat_common.hpp"
#include "pat_device.hpp"
#include "kmeans_dev.hpp"

namespace {

using pat::kWave;

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;
typedef __attribute__((__vector_size__(2 * sizeof(float)))) float f32x2;
typedef __attribute__((__vector_size__(4 * sizeof(unsigned)))) unsigned u32x4;

// (lo, hi) rounded to BF16 (nearest even, as a scalar conversion rounds)
// in one packed conversion: lo in bits 0-15, hi in bits 16-31.
__device__ __forceinline__ unsigned bf16_pair(float lo, float hi)
{
    return __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2){lo, hi}, bf16x2));
}
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16;

constexpr float kInitMin = 65536 * 65;  // map1's initial min_dist (kmeans/regular.h:86)

// Position of element e of centre row k in the MFMA operand array,
// stored in fragment order: for 32-row block b and K-step s, lane
// l = (k % 32) + 32 * ((e % 16) / 8) holds elements 8*(l/32) .. +8 of row
// b*32 + l%32 at 16-byte slot (b*NS + s)*64 + l, so a wavefront's operand
// read is 1 KB of consecutive LDS bytes (no bank conflicts).
__host__ __device__ __forceinline__ int64_t frag_index(int k, int e, int ns)
{
    const int b = k / 32, col = k % 32, s = e / 16, h = (e % 16) / 8, j = e % 8;
    return ((((int64_t)b * ns + s) * 2 + h) * 32 + col) * 8 + j;
}

// rint(v * 2^s) as a 64-bit two's-complement integer, with scale = 2^s an
// FP32 power of two chosen so that |v| 2^s <= 2^30 for every value summed:
// v * scale is exact, rounding it to an integer is exact in FP32, and the
// integer converts exactly to int32.  The same integer as
// rint((double)v * 2^s) in FP64.
__device__ __forceinline__ unsigned long long to_fixed(float v, float scale)
{
    return (unsigned long long)(long long)(int)__builtin_rintf(v * scale);
}

// ------------------------------------------------------------ shared parts

struct KmArgs {
    const float *x;         // N x D points
    const float *c;         // K x D centres (FP32)
    int64_t N;
    int D, K;
    float scale, dscale;    // fixed-point scales 2^s, 2^ds (FP32 powers of two)
    int32_t *assign;        // N
    float *mindist;         // N (may be null)
    unsigned long long *gsum;   // K x D
    unsigned long long *gcnt;   // K
    unsigned long long *gdsum;  // K
    int use_lds_acc;        // 1: LDS reduction object, 0: global atomics directly
    int defer_acc;          // 1: assignments only; the bucketed reduction (km_bucket_*) sums afterwards
    int rs;                 // row stride (8-byte words) of the coordinate sums: D in global memory,
                            // odd in LDS so that rows of different keys start in different banks
};

// Adds the wavefront's points [base, base+np) with keys key_of(j) into the
// reduction object.  Lanes cover (point, dimension) pairs so consecutive
// lanes touch consecutive 8-byte words.
template <typename KeyFn, typename DistFn>
__device__ __forceinline__ void accumulate_points(const KmArgs &a, int64_t base, int np, KeyFn key_of, DistFn dist_of,
                                                  unsigned long long *acc, unsigned long long *cnt,
                                                  unsigned long long *dsum)
{
    // Trip counts are uniform over the wavefront so that every lane is active
    // at each cross-lane read of the keys.
    const int lane = threadIdx.x % kWave;
    const int D = a.D;
    const int total = np * D;
    // lane covers flat index t = j*D + d, advanced by kWave per trip without
    // a division inside the loop
    const int step_j = kWave / D, step_d = kWave % D;
    int j = lane / D, d = lane % D;
    for (int t0 = 0; t0 < total; t0 += kWave) {
        const bool in = t0 + lane < total;
        const int k = key_of(in ? j : np - 1);
        if (in) {
            const float v = a.x[(base + j) * D + d];
            atomicAdd(&acc[(int64_t)k * a.rs + d], to_fixed(v, a.scale));
        }
        j += step_j;
        d += step_d;
        if (d >= D) {
            d -= D;
            j++;
        }
    }
    const int jj = lane < np ? lane : np - 1;
    const int k = key_of(jj);
    const float dist = dist_of(jj);
    if (lane < np) {
        atomicAdd(&cnt[k], 1ULL);
        atomicAdd(&dsum[k], to_fixed(dist, a.dscale));
    }
}

__device__ void flush_lds_object(const KmArgs &a, unsigned long long *acc, unsigned long long *cnt,
                                 unsigned long long *dsum)
{
    const int KD = a.K * a.D;
    for (int i = threadIdx.x; i < KD; i += blockDim.x) {
        const int k = i / a.D, d = i - k * a.D;
        const unsigned long long v = acc[(int64_t)k * a.rs + d];
        if (v) atomicAdd(&a.gsum[i], v);
    }
    for (int i = threadIdx.x; i < a.K; i += blockDim.x) {
        if (cnt[i]) atomicAdd(&a.gcnt[i], cnt[i]);
        if (dsum[i]) atomicAdd(&a.gdsum[i], dsum[i]);
    }
}

__device__ void zero_lds_object(const KmArgs &a, unsigned long long *acc, unsigned long long *cnt,
                                unsigned long long *dsum)
{
    for (int i = threadIdx.x; i < a.K * a.rs; i += blockDim.x) acc[i] = 0;
    for (int i = threadIdx.x; i < a.K; i += blockDim.x) {
        cnt[i] = 0;
        dsum[i] = 0;
    }
}

// Row stride of the LDS reduction object: D rounded up to odd, so that the
// rows of different keys start in different banks (with an even stride every
// row would start in the same bank, and the wavefront's atomics on one
// dimension of 32 points would serialise).
__host__ __device__ __forceinline__ int object_stride(int D) { return D | 1; }

// Words of the LDS reduction object, rounded up to a 16-byte boundary.
__host__ __device__ __forceinline__ int64_t object_words(int K, int D)
{
    return ((int64_t)K * object_stride(D) + 2 * K + 1) & ~1LL;
}

// LDS layout of the reduction object (when it fits).
__device__ __forceinline__ void lds_object(const KmArgs &a, unsigned long long *base, unsigned long long *&acc,
                                           unsigned long long *&cnt, unsigned long long *&dsum)
{
    if (a.use_lds_acc) {
        acc = base;
        cnt = base + (int64_t)a.K * a.rs;
        dsum = cnt + a.K;
    } else {
        acc = a.gsum;
        cnt = a.gcnt;
        dsum = a.gdsum;
    }
}

// ------------------------------------------------------------ plain path

// One thread per point; centres read from LDS when they fit (cs != null).
// BS threads per workgroup: the LDS object allows one workgroup per CU, so
// BS sets the waves per SIMD that hide LDS latency (4 at 1024 threads).
template <int DMAX, int BS>
__global__ __launch_bounds__(BS) void km_plain(KmArgs a, int centres_in_lds)
{
    extern __shared__ unsigned long long smem[];
    unsigned long long *acc, *cnt, *dsum;
    lds_object(a, smem, acc, cnt, dsum);
    // centres in LDS: rows of D4 = D rounded up to 4 floats, zero-padded
    float *cs = (float *)(smem + (a.use_lds_acc ? object_words(a.K, a.D) : 0));
    const int D = a.D, K = a.K, D4 = (D + 3) & ~3;
    if (a.use_lds_acc) zero_lds_object(a, acc, cnt, dsum);
    if (centres_in_lds)
        for (int i = threadIdx.x; i < K * D4; i += blockDim.x) {
            const int k = i / D4, d = i - k * D4;
            cs[i] = d < D ? a.c[(int64_t)k * D + d] : 0.0f;
        }
    __syncthreads();

    const int lane = threadIdx.x % kWave;
    const int64_t nwaves = (int64_t)gridDim.x * (blockDim.x / kWave);
    const int64_t w0 = (int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
    for (int64_t base = w0 * kWave; base < a.N; base += nwaves * kWave) {
        const int64_t p = base + lane;
        const bool live = p < a.N;
        float x[DMAX];
#pragma unroll
        for (int d = 0; d < DMAX; d++) x[d] = (live && d < D) ? a.x[p * D + d] : 0.0f;
        unsigned int key = 0;
        float min_dist = kInitMin;
        // dist = sum over d < D of (c_d - x_d)^2 in dimension order.  From
        // the LDS rows: groups of four dimensions (one 16-byte read, the same
        // address in every lane); past D both the row and x hold zeros, and
        // adding (0 - 0)^2 = +0 to the non-negative sum changes no bit.
        // From global memory: one guarded dimension at a time.
        auto dist_of = [&](int k) {
            float dist = 0;
            if (centres_in_lds) {
                const float *ci = cs + k * D4;
#pragma unroll
                for (int g = 0; g < DMAX / 4; g++) {
                    if (4 * g < D) {
                        const float4 c4 = *(const float4 *)(ci + 4 * g);
                        float t = c4.x - x[4 * g];
                        dist = dist + t * t;
                        t = c4.y - x[4 * g + 1];
                        dist = dist + t * t;
                        t = c4.z - x[4 * g + 2];
                        dist = dist + t * t;
                        t = c4.w - x[4 * g + 3];
                        dist = dist + t * t;
                    }
                }
            } else {
                const float *ci = a.c + (int64_t)k * D;
#pragma unroll
                for (int d = 0; d < DMAX; d++) {
                    if (d < D) {
                        const float t = ci[d] - x[d];
                        dist = dist + t * t;
                    }
                }
            }
            return sqrtf(dist);
        };
        int i = 0;
        for (; i + 4 <= K; i += 4) {
            // four independent chains for ILP; compared in index order
            float dv[4];
#pragma unroll
            for (int q = 0; q < 4; q++) dv[q] = dist_of(i + q);
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (dv[q] < min_dist) {
                    min_dist = dv[q];
                    key = i + q;
                }
        }
        for (; i < K; i++) {
            const float dist = dist_of(i);
            if (dist < min_dist) {
                min_dist = dist;
                key = i;
            }
        }
        if (live) {
            a.assign[p] = (int32_t)key;
            if (a.mindist) a.mindist[p] = min_dist;
        }
        const int np = (int)min<int64_t>(kWave, a.N - base);
        if (!a.defer_acc) {
            auto key_of = [&](int j) { return (int)__shfl((int)key, j, kWave); };
            auto dist_at = [&](int j) { return __shfl(min_dist, j, kWave); };
            // the LDS object addressed from the shared array itself, so that
            // its adds compile to LDS atomics
            if (a.use_lds_acc)
                accumulate_points(a, base, np, key_of, dist_at, smem, smem + K * a.rs, smem + K * a.rs + K);
            else
                accumulate_points(a, base, np, key_of, dist_at, a.gsum, a.gcnt, a.gdsum);
        }
    }
    if (a.use_lds_acc) {
        __syncthreads();
        flush_lds_object(a, acc, cnt, dsum);
    }
}

// ------------------------------------------------------------ MFMA path

typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8;
typedef __attribute__((__vector_size__(2 * sizeof(_Float16)))) _Float16 f16x2;

// Fragments of a centre's row (16 elements each): three terms take high and low
// parts, one term one; and the norm.
constexpr int mfma_fragments(int ks, int nt) { return (nt == 3 ? 2 : 1) * ks + 1; }

constexpr float kWideOne = 32768.0f;  // the norm parts' factor 2^15
constexpr float kWideFar = 60000.0f;  // first norm part of a row that never wins: above any value (2^28)

// Per-point bound inputs of the one-term form: u = 2^-8 (BF16 unit roundoff),
// g = FP32 accumulation over the MFMA's terms with a factor 2 of slack for any
// intermediate rounding mode.
struct MfmaBound {
    float c_dot;   // multiplies ||x|| * max||c||
    float c_norm;  // multiplies max||c||^2
    float c_ref;   // relative error of the reference's FP32 difference form
};

// Those of the FP16 parts (km_wide has the proof).
struct WideBound {
    float sx;                        // 2^a
    float c_dot, c_sum, c_cc, c_abs;  // error: c_dot X C + c_sum (X + C) + c_cc C^2 + c_abs
    float c_ref, ref_abs;            // the reference's FP32 difference form: relative, and for underflow
    float far;                       // half squared distances from here on may reach map1's initial minimum
};

// Four floats at any float's address (a 16-byte global load needs no more).
typedef float float4u __attribute__((ext_vector_type(4), aligned(4)));

// x[d .. d+3] of a row of D, zeros past its end.
__device__ __forceinline__ float4u ragged_4(const float *__restrict__ x, int d, int D)
{
    float4u q = {0.f, 0.f, 0.f, 0.f};
    if (d + 4 <= D) {
        q = *(const float4u *)(x + d);
    } else {
        if (d < D) q.x = x[d];
        if (d + 1 < D) q.y = x[d + 1];
        if (d + 2 < D) q.z = x[d + 2];
    }
    return q;
}

// Exact plain-path distance (sqrt of the FP32 difference form, dimensions in
// order) of point row xp to centre row ck, both read from memory (the point
// row was just loaded by the wavefront, so it is in cache).
__device__ __forceinline__ float exact_dist(const float *__restrict__ xp, const float *__restrict__ ck, int D)
{
    float dist = 0;
    int d = 0;
#pragma unroll 4
    for (; d + 4 <= D; d += 4) {
        const float4u cv = *(const float4u *)(ck + d), xv = *(const float4u *)(xp + d);
        float t = cv.x - xv.x;
        dist = dist + t * t;
        t = cv.y - xv.y;
        dist = dist + t * t;
        t = cv.z - xv.z;
        dist = dist + t * t;
        t = cv.w - xv.w;
        dist = dist + t * t;
    }
    for (; d < D; d++) {
        const float t = ck[d] - xp[d];
        dist = dist + t * t;
    }
    return sqrtf(dist);
}

// The same distance with the point row held by the wavefront's two halves
// (lane l and l+32 hold the point's dimensions 16s + 8*half + e in xo):
// v_permlane32_swap gives both lanes dimensions 16s + e in its first result
// and 16s + 8 + e in its second, so the row is read in order from registers
// instead of memory.  Called by every lane (the swap is cross-lane); the
// row is only formed where D == 16*KS.
template <int KS>
__device__ __forceinline__ void point_row(const float (&xo)[8 * KS], float (&row)[16 * KS])
{
#pragma unroll
    for (int s = 0; s < KS; s++)
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const unsigned v = __float_as_uint(xo[8 * s + e]);
            const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
            row[16 * s + e] = __uint_as_float(r[0]);
            row[16 * s + 8 + e] = __uint_as_float(r[1]);
        }
}

template <int KS>
__device__ __forceinline__ float exact_dist_row(const float (&row)[16 * KS], const float *__restrict__ ck)
{
    float dist = 0;
#pragma unroll
    for (int d = 0; d < 16 * KS; d += 4) {
        const float4 cv = *(const float4 *)(ck + d);
        float t = cv.x - row[d];
        dist = dist + t * t;
        t = cv.y - row[d + 1];
        dist = dist + t * t;
        t = cv.z - row[d + 2];
        dist = dist + t * t;
        t = cv.w - row[d + 3];
        dist = dist + t * t;
    }
    return sqrtf(dist);
}

// Approximate value v with its position idx (0..127) in the low 7 bits of
// the significand: a key that orders like v (up to 127 ulps) and carries its
// index through a plain float minimum.  |key - v| <= 2^-16 |v| + 2^-126.
// keep: ~127 held in a vector register (key_mask), so that with idx in a
// scalar register the packing is one v_and_or_b32 (an instruction reads at
// most one scalar operand, and the mask as a literal would be a second).
__device__ __forceinline__ float pack_key(float v, int idx, int keep)
{
    return __int_as_float((__float_as_int(v) & keep) | idx);
}

// ~127 in a vector register, opaque to constant folding.
__device__ __forceinline__ int key_mask()
{
    int m;
    asm volatile("v_mov_b32 %0, 0xffffff80" : "=v"(m));
    return m;
}

// base | i for a wavefront-uniform base, in one scalar register (a scalar
// ALU operation, opaque to the compiler, which would otherwise fold the OR
// into the packing as a second vector instruction).  It sets SCC.
__device__ __forceinline__ int scalar_or(int base, int i)
{
    int r;
    asm("s_or_b32 %0, %1, %2" : "=s"(r) : "s"(base), "s"(i) : "scc");
    return r;
}

// Stand-in for a value past the last centre row: finite (so its key is not
// a NaN) and above any threshold.
constexpr float kFar = 3.0e38f;

// KS: K-steps of 16 dimensions holding the data (D <= 16*KS); NT: terms
// (1 or 3), each KS steps; one more K-step holds the norm terms.  KB:
// 32-centre blocks per chunk.  cb: NT = 1: K_pad x 16 (KS + 1) BF16 rows
// [-2c | n1 n2 n3 0...]; padded rows have n1 = 1e30 (far, but finite so that
// their keys are numbers).  NT = 3: K_pad x 16 (2 KS + 1) FP16 rows (km_wide
// has their form, the value they give and its bound).  Data zero-padded to
// 16*KS, fragment order (frag_index).  cnorm: ||c_k|| (K entries).
//
// Per 32-point tile a wavefront (lanes l and l+32 hold halves of point l):
// computes the approximate values of every centre with MFMAs, packs the
// smaller of every two (one term: every value) with their index (pack_key) and
// keeps the three smallest keys of each half (the two smallest values per chunk
// when the index bits cannot tell the chunks apart).  The threshold is the
// minimum plus the error bound plus the packing error; when only the smallest
// key is under it (the usual case) its centres are rescored, of two one by each
// half, when a half's third key lies above it the kept keys under it are, and
// otherwise
// every centre under it is (the values recomputed chunk by chunk).  The exact
// FP32 results decide with map1's rule, and the point is added to the LDS
// reduction object from the registers holding its half rows.
//
// Bound by instruction issue, vector and matrix together: 2^24 x 32, K 256,
// 20 passes: 1.41 ms each (1.54 with BF16 parts and a key for every value; the
// wider bound of those left 2.3% of the points several candidates, one in every
// second tile; 0.3% now).  One block of centres per chunk at every KS: its two accumulators
// and the registers around them fit without spills (1 M x 8, K 16: 41 us with
// one, 54 with four; 1 M x 16, K 128: 55 and 64), and the matrix cores work on
// the next block during a scan.
// TAIL = false: D == 16*KS and the rows are 16-byte aligned, so every
// K-step is full and the loads need no per-element guard.
// GC: the form for K x D too large for LDS.  The workgroup's wavefronts
// step through the centre chunks together: before each chunk the
// workgroup copies its KB blocks of rows from global memory into one
// LDS chunk buffer (between two barriers) and every wavefront computes its
// own tile against it, so each copy of the rows serves 8 tiles.  Tiles are
// taken block-uniformly (a wavefront past the last tile computes with every
// lane dead) and the recompute path is a workgroup vote, so every wavefront
// reaches every barrier.
// BS: threads per workgroup (the LDS-resident centre rows and reduction
// object are shared by all its wavefronts, so larger workgroups raise the
// occupancy the LDS allows when the registers permit).
template <int KS, int KB, int NT, bool TAIL, bool GC, int BS = 512>
__global__ __launch_bounds__(BS) void km_mfma(KmArgs a, const void *__restrict__ cb, const float *__restrict__ cnorm,
                                               int K_pad, MfmaBound bd, WideBound wb,
                                               unsigned long long *__restrict__ rescored)
{
    constexpr bool F16 = NT == 3;
    constexpr int NS = NT * KS + 1;               // MFMAs per block of 32 centres
    constexpr int NF = mfma_fragments(KS, NT);    // fragments per block in cb (1 KiB each)
    static_assert(KB * 16 <= 128, "pack_key indexes at most 128 values per chunk");
    extern __shared__ unsigned long long smem[];
    unsigned long long *acc_o, *cnt_o, *dsum_o;
    lds_object(a, smem, acc_o, cnt_o, dsum_o);
    u32x4 *cbs = (u32x4 *)(smem + (a.use_lds_acc ? object_words(a.K, a.D) : 0));
    __shared__ float red[16];
    if (a.use_lds_acc) zero_lds_object(a, acc_o, cnt_o, dsum_o);
    // stage the centre rows in LDS (16-byte copies); the GC form stages one
    // chunk at a time (stage_chunk)
    if (!GC) {
        const int n16 = K_pad * NF * 2;
        const u32x4 *src = (const u32x4 *)cb;
        for (int i = threadIdx.x; i < n16; i += blockDim.x) cbs[i] = src[i];
    }
    // max ||c|| over the centres (for the bound)
    float cm = 0.0f;
    for (int i = threadIdx.x; i < a.K; i += blockDim.x) cm = fmaxf(cm, cnorm[i]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) cm = fmaxf(cm, __shfl_xor(cm, o, kWave));
    if (threadIdx.x % kWave == 0) red[threadIdx.x / kWave] = cm;
    __syncthreads();
    float cmax = 0.0f;
    for (int w = 0; w < (int)(blockDim.x / kWave); w++) cmax = fmaxf(cmax, red[w]);
    const float cc_max = cmax * cmax, C = cmax * wb.sx;

    const int D = a.D;
    const int lane = threadIdx.x % kWave;
    const int col = lane % 32;   // point within the tile
    const int half = lane / 32;  // which 8 of each 16 K elements this lane holds
    const int nchunks = (K_pad / 32 + KB - 1) / KB;
    unsigned my_rescored = 0;  // this lane's rescored points (under 2^32 per lane)

    // approximate values of chunk ch for this lane's point: value i of block
    // b is centre row 8*(i/4) + 4*half + i%4 of the block (the 32x32 MFMA
    // output layout).  The A fragments are read a few K-steps ahead of the
    // MFMA that uses them.
    // Blocks past the last centre row (when K_pad is not a multiple of
    // KB*32) are computed from block 0's rows -- the block index is clamped
    // on the scalar unit -- and skipped by the scans.
    const int kblocks = K_pad / 32;
    const int keep = key_mask();
    auto chunk_values = [&](int ch, const u32x4 (&bx)[NF], f32x16 (&acc)[KB]) {
        constexpr int T = KB * NS, P = 3;
        const u32x4 *ab = cbs + lane;
        int again = 0;  // where the high parts, read twice, would not fit in registers
        if (F16 && KS > 2) asm volatile("" : "+s"(again));
        auto frag = [&](int t) {
            // F16: high, low, high parts, norm
            const int st = t % NS, f = !F16 || st < 2 * KS ? st : (st < 3 * KS ? st - 2 * KS : 2 * KS);
            const int at = (F16 && st >= 2 * KS ? again : 0) + f * kWave;
            if (GC) return ab[t / NS * NF * kWave + at];  // the staged chunk
            const int blk = ch * KB + t / NS;
            return ab[(blk < kblocks ? blk : 0) * NF * kWave + at];
        };
        u32x4 fr[P];
#pragma unroll
        for (int t = 0; t < P; t++) fr[t] = frag(t);
#pragma unroll
        for (int t = 0; t < T; t++) {
            const int b = t / NS, st = t % NS;
            const u32x4 av = fr[t % P];
            if (t + P < T) fr[t % P] = frag(t + P);
            if (st == 0) acc[b] = f32x16{};
            // F16: high.low(x), low.high(x), high.high, norm: the small terms first
            const u32x4 bv = bx[!F16 ? st : (st < KS ? KS + st : (st < 3 * KS ? (st - KS) % KS : 2 * KS))];
            if constexpr (F16)
                acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, av),
                                                                __builtin_bit_cast(f16x8, bv), acc[b], 0, 0, 0);
            else
                acc[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, av),
                                                                 __builtin_bit_cast(bf16x8, bv), acc[b], 0, 0, 0);
        }
    };
    auto centre_of = [&](int ch, int idx) {
        const int b = idx >> 4, i = idx & 15;
        return (ch * KB + b) * 32 + 8 * (i >> 2) + 4 * half + (i & 3);
    };
    // GC: chunk ch's blocks into the LDS chunk buffer (blocks past the last
    // centre row are not copied; their values are never scanned).  Called
    // by every thread of the workgroup.
    auto stage_chunk = [&](int ch) {
        __syncthreads();  // every wavefront is done with the previous chunk
        const int nblk = min(KB, kblocks - ch * KB);
        const int n16 = nblk * NF * kWave;
        const u32x4 *src = (const u32x4 *)cb + (int64_t)ch * KB * NF * kWave;
        for (int i = threadIdx.x; i < n16; i += blockDim.x) cbs[i] = src[i];
        __syncthreads();
    };

    const int64_t ntiles = (a.N + 31) / 32;
    const int64_t nw = (int64_t)gridDim.x * (blockDim.x / kWave);
    // this lane's half of tile t's point row (dimensions 16s + 8*half + e);
    // dead lanes read a valid row (their values reach no result)
    auto load_half_row = [&](int64_t t, float (&xo)[8 * KS]) {
        const int64_t p = t * 32 + col;
        const bool live = p < a.N;
        const float *xp = a.x + (live ? p : a.N - 1) * D;
#pragma unroll
        for (int s = 0; s < KS; s++) {
            const int d0 = 16 * s + 8 * half;
            if (!TAIL) {
                const float4 lo = *(const float4 *)(xp + d0), hi = *(const float4 *)(xp + d0 + 4);
                xo[8 * s] = lo.x; xo[8 * s + 1] = lo.y; xo[8 * s + 2] = lo.z; xo[8 * s + 3] = lo.w;
                xo[8 * s + 4] = hi.x; xo[8 * s + 5] = hi.y; xo[8 * s + 6] = hi.z; xo[8 * s + 7] = hi.w;
            } else {
#pragma unroll
                for (int e = 0; e < 8; e += 4) {
                    const float4u q = ragged_4(xp, d0 + e, D);
                    xo[8 * s + e] = q.x; xo[8 * s + e + 1] = q.y; xo[8 * s + e + 2] = q.z; xo[8 * s + e + 3] = q.w;
                }
            }
        }
    };
    // With the centre fragments in LDS the next tile's rows are loaded
    // while this tile computes (its loads return during the MFMAs); the
    // global-fragment form loads them in place, since vector loads complete
    // in order and the fragment loads would wait behind them, and so do rows
    // of more than 64 dimensions or in workgroups over 512 threads (the
    // extra registers would spill).
    constexpr bool PF = !GC && KS <= 4 && BS <= 512;
    // software-pipelined chunk scan (one more accumulator of KB x 16 values)
    constexpr bool PIPE = !GC && KB == 1;
    const int64_t tile0 = (int64_t)blockIdx.x * (blockDim.x / kWave) + threadIdx.x / kWave;
    float xnext[8 * KS];
    if (PF && tile0 < ntiles) load_half_row(tile0, xnext);
    // GC: the workgroup's loop ends when its first wavefront's tile does
    const int64_t block_tile0 = (int64_t)blockIdx.x * (blockDim.x / kWave);
    for (int64_t tile = tile0; (GC ? block_tile0 + (tile - tile0) : tile) < ntiles; tile += nw) {
        const int64_t p = tile * 32 + col;
        const bool live = p < a.N;
        const float *xp = a.x + (live ? p : a.N - 1) * D;  // dead lanes read a valid row

        float xo[8 * KS];
        if (!PF) {
            load_half_row(tile, xo);
        } else {
#pragma unroll
            for (int i = 0; i < 8 * KS; i++) xo[i] = xnext[i];
            if (tile + nw < ntiles) load_half_row(tile + nw, xnext);
        }
        // B operand: point p, K elements [16s + 8*half, +8): x and ones for the
        // norm's three parts, or high and low parts of 2^a x and its ones;
        // pairs of elements, one packed conversion each
        u32x4 bx[NF];
        float xx = 0.0f;
#pragma unroll
        for (int s = 0; s < KS; s++) {
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                const f32x2 q = F16 ? (f32x2){xo[8 * s + e] * wb.sx, xo[8 * s + e + 1] * wb.sx}
                                    : (f32x2){xo[8 * s + e], xo[8 * s + e + 1]};
                xx = __builtin_fmaf(q[0], q[0], xx);  // a bound input only (used with slack)
                xx = __builtin_fmaf(q[1], q[1], xx);
                if constexpr (F16) {
                    const f16x2 h = __builtin_convertvector(q, f16x2);
                    const f32x2 r = {q[0] - (float)h[0], q[1] - (float)h[1]};
                    bx[s][e / 2] = __builtin_bit_cast(unsigned, h);
                    bx[KS + s][e / 2] = __builtin_bit_cast(unsigned, __builtin_convertvector(r, f16x2));
                } else {
                    bx[s][e / 2] = bf16_pair(q[0], q[1]);
                }
            }
        }
        // 2^15 or 1 three times
        bx[NF - 1] = half == 0 ? (F16 ? (u32x4){0x78007800u, 0x7800u, 0u, 0u} : (u32x4){0x3f803f80u, 0x3f80u, 0u, 0u})
                               : (u32x4){0u, 0u, 0u, 0u};
        xx = xx + __shfl_xor(xx, 32, kWave);  // ||x||^2 of point p (both halves)
        // an upper bound of ||x|| only: the hardware square root (within an
        // ulp or two for normal inputs, 0 for flushed subnormals, whose
        // root lies below 2^-63) with relative and absolute slack, in place
        // of the correctly rounded sequence
        const float xn = __builtin_amdgcn_sqrtf(xx) * 1.0001f + 0x1p-40f;
        const float E = F16 ? wb.c_dot * xn * C + wb.c_sum * (xn + C) + wb.c_cc * C * C + wb.c_abs
                            : bd.c_dot * xn * cmax + bd.c_norm * (cc_max + xx);

        f32x16 acc[KB];
        // The three smallest keys of this half.  With three terms, when the pairs
        // of a lane's values in all chunks fit the 7 index bits (gidx: at most
        // 128), a key is the smaller of two adjacent centres' values with the
        // pair's index (values i and i + 1 of block blk -> 8 blk + i / 2): five
        // instructions for two values, and the halves rescore one centre of a
        // pair each.  With one term, whose bound leaves many points several
        // candidates, a key is a value (16 blk + i, while those fit): 5 M x 32, K
        // 32: 405 us an iteration, 565 with pairs.  One sorted triple runs over
        // all chunks.  Otherwise the keys are single values, each chunk's two
        // smallest are merged with their chunk recorded and k3 stays unknown
        // (kFar, never used).
        const bool gidx = nchunks * KB <= (F16 ? 16 : 8);  // uniform
        float k1 = kFar, k2 = kFar, k3 = kFar;
        int ch1 = 0;
        auto scan3 = [&](int ch, const f32x16 (&v)[KB]) {
            constexpr int STEP = F16 ? 2 : 1;
#pragma unroll
            for (int b = 0; b < KB; b++) {
                if (b > 0 && ch * KB + b >= kblocks) break;  // uniform; block 0 of a chunk always exists
#pragma unroll
                for (int i = 0; i < 16; i += STEP) {
                    const float lo = F16 ? __builtin_amdgcn_fmed3f(v[b][i], v[b][i + STEP - 1], -kFar) : v[b][i];  // min (finite)
                    const float key = pack_key(lo, scalar_or((ch * KB + b) * (16 / STEP), i / STEP), keep);
                    k3 = __builtin_amdgcn_fmed3f(k2, k3, key);
                    k2 = __builtin_amdgcn_fmed3f(k1, k2, key);
                    k1 = __builtin_amdgcn_fmed3f(k1, key, -kFar);
                }
            }
        };
        if (PIPE && gidx) {
            // the next chunk's MFMAs are issued before this chunk's keys are
            // scanned, so one wavefront keeps the matrix cores and the vector
            // ALU busy together; two accumulators take the roles in turn
            // (no branch between a chunk's MFMAs and the other's scan, so the
            // scheduler can interleave them)
            f32x16 acc2[KB];
            chunk_values(0, bx, acc);
            int ch = 0;
            for (; ch + 2 < nchunks; ch += 2) {
                chunk_values(ch + 1, bx, acc2);
                scan3(ch, acc);
                chunk_values(ch + 2, bx, acc);
                scan3(ch + 1, acc2);
            }
            if (ch + 1 < nchunks) {
                chunk_values(ch + 1, bx, acc2);
                scan3(ch, acc);
                scan3(ch + 1, acc2);
            } else {
                scan3(ch, acc);
            }
        }
        for (int ch = 0; ch < (PIPE && gidx ? 0 : nchunks); ch++) {
            if (GC) stage_chunk(ch);
            chunk_values(ch, bx, acc);
            if (gidx) {
                scan3(ch, acc);
                continue;
            }
            float c1 = kFar, c2 = kFar;
#pragma unroll
            for (int b = 0; b < KB; b++) {
                if (ch * KB + b >= kblocks) break;  // uniform
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const float key = pack_key(acc[b][i], b * 16 + i, keep);
                    c2 = __builtin_amdgcn_fmed3f(c1, c2, key);
                    c1 = __builtin_amdgcn_fmed3f(c1, key, -kFar);  // min (keys are finite)
                }
            }
            if (c1 < k1) {
                k2 = fminf(k1, c2);
                k1 = c1;
                ch1 = ch;
            } else {
                k2 = fminf(k2, c1);
            }
        }
        // both halves: overall smallest and second smallest
        const float o1 = __shfl_xor(k1, 32, kWave), o2 = __shfl_xor(k2, 32, kWave), o3 = __shfl_xor(k3, 32, kWave);
        const float m1 = fminf(k1, o1);
        const float m2 = fminf(fmaxf(k1, o1), fminf(k2, o2));
        // candidates: keys within the margin of the minimum.  The packing
        // moves a value by 2^-16 of itself: at most ||c||^2 + 2 ||x|| ||c||,
        // or (F16) at most the larger of ||x||^2 / 2 and the smallest key, for
        // every centre that matters
        float dp, dhi;
        if (F16) {
            const float H = 0.5f * xx;
            dp = 0x1p-16f * 1.02f * (fmaxf(H, fabsf(m1)) * 1.01f + 4.0f * E) + 0x1p-126f;
            dhi = (H + m1 + 4.0f * E + 4.0f * dp) * 1.001f + wb.ref_abs;
        } else {
            dp = 0x1p-16f * (cc_max + 2.0f * xn * cmax) * 1.01f + 0x1p-126f;
            dhi = (xx + m1 + 4.0f * E + 4.0f * dp) * 1.001f + 1e-30f;
        }
        const float thr = m1 + 2.0f * E + 2.0f * dp + 2.0f * (F16 ? wb.c_ref : bd.c_ref) * dhi;
        const bool multi = !(m2 > thr);
        // points whose candidates may lie beyond the keys they kept: every
        // value under the threshold is then visited again (full)
        const bool full = multi && (!gidx || !((F16 ? fminf(k3, o3) : k3) > thr));
        // the whole point row in registers (full K-steps) where the form has
        // the registers to spare (the others would spill: they reload it)
        constexpr bool ROW = !TAIL && !GC && KB == 1 && (KS <= 2 || (KS == 4 && BS <= 512));
        float row[16 * KS];
        if (ROW) point_row<KS>(xo, row);

        float best_d = kInitMin;
        int best_k = 0x7fffffff;
        // exact distance to centre k
        auto rescore = [&](int k) {
            if (k < a.K) {
                const float *ck = a.c + (int64_t)k * D;
                const float dk = ROW ? exact_dist_row<KS>(row, ck) : exact_dist(xp, ck, D);
                if (dk < best_d || (dk == best_d && k < best_k)) {
                    best_d = dk;
                    best_k = k;
                }
            }
        };
        // this half's centre of the pair that key stands for, held by half h
        auto pair_centre = [&](float key, int h) {
            const int id = __float_as_int(key) & 127, i = 2 * (id & 7);
            return (id >> 3) * 32 + 8 * (i >> 2) + 4 * h + (i & 3) + half;
        };
        if (F16 && gidx) {
            // the kept pairs under the threshold are all of its candidates
            // (the third smallest of each half lies above it): the smallest,
            // and of several the other three as far as they are under it
            const bool first = half ? k1 < o1 : k1 <= o1;  // the halves agree on ties
            const bool second = half ? k2 < o2 : k2 <= o2;
            if (live && !full) rescore(pair_centre(m1, first ? half : 1 - half));
            const bool more = live && multi && !full;
            if (__any(more)) {
                const float t = fmaxf(k1, o1), u = fminf(k2, o2), w = fmaxf(k2, o2);
                if (more && !(t > thr)) rescore(pair_centre(t, first ? 1 - half : half));
                if (more && !(u > thr)) rescore(pair_centre(u, second ? half : 1 - half));
                if (more && !(w > thr)) rescore(pair_centre(w, second ? 1 - half : half));
            }
        } else if (live && !full) {
            // one candidate: rescored by the half that holds it; several (gidx
            // only): each half rescores its kept keys under the threshold, which
            // are all of its candidates since its third lies above it
            if (multi ? !(k1 > thr) : k1 < o1) rescore(centre_of(gidx ? 0 : ch1, __float_as_int(k1) & 127));
            if (multi && !(k2 > thr)) rescore(centre_of(0, __float_as_int(k2) & 127));
        }
        // Every value under the threshold for the full lanes.  Taken by the
        // whole wavefront (a vote), because recomputing a chunk's values
        // needs every lane's operands.
        if (GC ? __syncthreads_or(full && live) != 0 : __any(full)) {
            for (int ch = 0; ch < nchunks; ch++) {
                if (GC) {
                    stage_chunk(ch);
                    chunk_values(ch, bx, acc);
                } else if (nchunks > 1) {
                    chunk_values(ch, bx, acc);
                }
                if (!full) continue;
                uint64_t w0 = 0, w1 = 0;
#pragma unroll
                for (int b = 0; b < KB; b++) {
                    if (ch * KB + b >= kblocks) break;  // uniform
#pragma unroll
                    for (int i = 0; i < 16; i++)
                        if (pack_key(acc[b][i], b * 16 + i, keep) <= thr) {
                            if (b < 4) w0 |= 1ULL << (b * 16 + i);
                            else w1 |= 1ULL << ((b - 4) * 16 + i);
                        }
                }
                for (int w = 0; w < 2; w++) {
                    uint64_t mw = w ? w1 : w0;
                    while (mw) {
                        const int bit = __builtin_ctzll(mw);
                        mw &= mw - 1;
                        if (live) rescore(centre_of(ch, 64 * w + bit));
                    }
                }
            }
        }
        // merge the two half-waves' exact winners (same tie rule)
        const float od = __shfl_xor(best_d, 32, kWave);
        const int ok = __shfl_xor(best_k, 32, kWave);
        if (od < best_d || (od == best_d && ok < best_k)) {
            best_d = od;
            best_k = ok;
        }
        if (best_k == 0x7fffffff) best_k = 0;  // unreachable for live points
        if (live && a.defer_acc) {
            if (half == 0) {
                a.assign[p] = best_k;
                a.mindist[p] = best_d;
                if (multi) my_rescored++;
            }
        } else if (live) {
            if (half == 0) {
                a.assign[p] = best_k;
                if (a.mindist) a.mindist[p] = best_d;
                if (multi) my_rescored++;
            }
            // the point (count, distance, this half-wave's dimensions) into
            // the reduction object; the LDS form addresses the shared array
            // itself, so that its adds compile to LDS atomics
            auto add_point = [&](unsigned long long *acc, unsigned long long *cnt, unsigned long long *dsum) {
                if (half == 0) {
                    atomicAdd(&cnt[best_k], 1ULL);
                    atomicAdd(&dsum[best_k], to_fixed(best_d, a.dscale));
                }
                unsigned long long *row = acc + best_k * a.rs;
#pragma unroll
                for (int s = 0; s < KS; s++)
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        const int d = 16 * s + 8 * half + e;
                        if (!TAIL || d < D) atomicAdd(&row[d], to_fixed(xo[8 * s + e], a.scale));
                    }
            };
            if (a.use_lds_acc) add_point(smem, smem + a.K * a.rs, smem + a.K * a.rs + a.K);
            else add_point(a.gsum, a.gcnt, a.gdsum);
        }
    }
    // rescored-point counter
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) my_rescored += __shfl_xor(my_rescored, o, kWave);
    if (lane == 0 && my_rescored) atomicAdd(rescored, (unsigned long long)my_rescored);
    if (a.use_lds_acc) {
        __syncthreads();
        flush_lds_object(a, acc_o, cnt_o, dsum_o);
    }
}

// ------------------------------------------------------------ wide MFMA path
//
// Assignment where the reduction object does not fit in LDS (the bucketed
// reduction sums it afterwards, and computes min_dist on its way over the
// rows, so that this kernel only has to find the centre).
//
// The bound decides the cost here: with BF16 terms and the norm accumulated
// first, 58% of the points of a 1,000-centre mixture at D = 128 had another
// centre inside the margin, and nearly every workgroup went through the
// centres twice.  So the operands are split into FP16 high and low parts (u =
// 2^-11, the dropped terms O(u^2)), scaled by a power of two that puts the
// largest coordinate just below 2^10, and each value is accumulated with the
// small terms first: lo.hi and hi.lo, then hi.hi, then the norm, so that
// only 16 KS + 16 of the additions round at the size of the result.  In units
// of half the scaled squared distance, with x^ = 2^a x, c^ = -2^a c, X = ||x^||,
// C = max ||c^||, e = 2^-14 (an FP16 subnormal may be taken as zero) and
// g = 2^-23 per addition (twice the FP32 roundoff, for any rounding inside the
// MFMA), the value n^ + x^.c^ (n^ = ||c^||^2 / 2) is off by at most
//     3 u^2 X C + e sqrt(D) (X + C) + D e^2           the split
//   + g 32 KS (2 u X C + 2 e sqrt(D) (X + C))         the small terms
//   + g 16 KS (X C (1 + 2 u) + ...)                   hi.hi
//   + g 16 (X C + C^2 / 2) + u^3 C^2 / 2 + 2          the norm (FP16 parts of n^ / 2^15)
// (wide_bound, with 2% over it).  A key's packed index costs 2^-16 of its own
// magnitude, which for every centre that matters is at most max(X^2 / 2, |smallest
// key|) and not the sum of the largest norms.
//
// A wavefront takes TILES tiles of 32 points, so that a centre fragment read
// from LDS feeds TILES MFMAs, and steps through the centres in chunks of NB
// blocks of 32 with its workgroup; the next chunk is copied into the other LDS
// buffer meanwhile (16-byte loads straight to LDS).  Keys carry seven index
// bits, so eight blocks make a group: the three smallest keys of each group
// are merged into the lane's three with their places.  At the end every lane
// finishes one point: it gets the other half's keys of its point, and when
// only the smallest key lies under the threshold that is the centre.
// Otherwise its kept keys under the threshold (at most four centres) are left
// to km_rescore, in the point's assign and mindist words, and the point in a
// list: rescoring here, by one or two lanes of a wavefront that its whole
// workgroup waits for at the next barrier, took more than half the time.
// Only when a half's third key lies under the threshold too does the workgroup
// go through the centres again and rescore every one under the threshold.
//
// Bound by the matrix cores: 3 KS + 1 MFMAs per 32 x 32 values, issued at 1.03
// PFLOP/s at D = 128 (a large library product reaches 1.18 on this card); the
// scan takes 4 vector instructions a value.  1 M x 128, K 1,000: 0.80-0.84 ms a pass,
// 0.7% of the points rescored (2.66 ms with BF16 terms and a second pass over
// the centres in nearly every workgroup).
template <int KS, int NB, int TILES, bool TAIL>
__global__ __launch_bounds__(512) void km_wide(KmArgs a, const _Float16 *__restrict__ cb,
                                               const float *__restrict__ cnorm, int K_pad, WideBound bd,
                                               int *__restrict__ list, int *__restrict__ listed,
                                               unsigned long long *__restrict__ rescored)
{
    constexpr int NS = 2 * KS + 1;  // fragments per block: high, low, norm
    constexpr int BW = 512 / kWave;
    static_assert(8 % NB == 0, "a group of eight blocks is a whole number of chunks");
    extern __shared__ __align__(16) unsigned char wide_lds[];  // two chunks of NB x NS KiB
    __shared__ float red[BW];
    const int lane = threadIdx.x % kWave, col = lane % 32, half = lane / 32, wv = pat::wave_in_block();
    float cm = 0.0f;
    for (int i = threadIdx.x; i < a.K; i += 512) cm = fmaxf(cm, cnorm[i]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) cm = fmaxf(cm, __shfl_xor(cm, o, kWave));
    if (lane == 0) red[wv] = cm;
    __syncthreads();
    float cmax = 0.0f;
    for (int w = 0; w < BW; w++) cmax = fmaxf(cmax, red[w]);
    const float C = cmax * bd.sx;

    const int D = a.D, kblocks = K_pad / 32, nchunks = (kblocks + NB - 1) / NB;
    const int keep = key_mask();
    unsigned my_rescored = 0;

    // chunk ch into LDS buffer b, one KiB per wavefront instruction
    auto stage = [&](int ch, int b) {
        const int n = min(NB, kblocks - ch * NB) * NS;
        const unsigned char *src = (const unsigned char *)cb + (int64_t)ch * NB * NS * 1024 + lane * 16;
        unsigned char *dst = wide_lds + b * (NB * NS * 1024);
        for (int f = wv; f < n; f += BW)
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(src + f * 1024),
                                             (__attribute__((address_space(3))) void *)(dst + f * 1024), 16, 0, 0);
    };
    auto staged = [&] {  // the loads to LDS have landed, for every wavefront
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    };
    f16x8 ones;
#pragma unroll
    for (int e = 0; e < 8; e++) ones[e] = (_Float16)((half == 0 && e < 3) ? kWideOne : 0.0f);

    stage(0, 0);
    const int64_t per_block = (int64_t)BW * 32 * TILES;
    for (int64_t base0 = (int64_t)blockIdx.x * per_block; base0 < a.N; base0 += (int64_t)gridDim.x * per_block) {
        const int64_t base = base0 + (int64_t)wv * 32 * TILES;  // this wavefront's points
        // operands: point col of each tile, dimensions 16 s + 8 half + e, scaled and split
        f16x8 xh[TILES][KS], xl[TILES][KS];
        float xx[TILES];
#pragma unroll
        for (int t = 0; t < TILES; t++) {
            const int64_t p = base + 32 * t + col;
            const bool live = p < a.N;
            const float *xp = a.x + (live ? p : a.N - 1) * D;
            xx[t] = 0.0f;
#pragma unroll
            for (int s = 0; s < KS; s++) {
                const int d0 = 16 * s + 8 * half;
                float v[8];
                if (!TAIL) {
                    const float4 lo = *(const float4 *)(xp + d0), hi = *(const float4 *)(xp + d0 + 4);
                    v[0] = lo.x; v[1] = lo.y; v[2] = lo.z; v[3] = lo.w;
                    v[4] = hi.x; v[5] = hi.y; v[6] = hi.z; v[7] = hi.w;
                } else {
#pragma unroll
                    for (int e = 0; e < 8; e += 4) {
                        const float4u q = ragged_4(xp, d0 + e, D);
                        v[e] = q.x; v[e + 1] = q.y; v[e + 2] = q.z; v[e + 3] = q.w;
                    }
                }
                u32x4 wh, wl;
#pragma unroll
                for (int e = 0; e < 8; e += 2) {
                    const f32x2 q = {v[e] * bd.sx, v[e + 1] * bd.sx};
                    xx[t] = __builtin_fmaf(q[0], q[0], xx[t]);
                    xx[t] = __builtin_fmaf(q[1], q[1], xx[t]);
                    const f16x2 h = __builtin_convertvector(q, f16x2);
                    const f32x2 r = {q[0] - (float)h[0], q[1] - (float)h[1]};
                    wh[e / 2] = __builtin_bit_cast(unsigned, h);
                    wl[e / 2] = __builtin_bit_cast(unsigned, __builtin_convertvector(r, f16x2));
                }
                // the sum of squares follows the operands (left to the end it
                // would keep every coordinate in a register, and spill)
                asm volatile("" : "+v"(xx[t]), "+v"(wl[3]));
                xh[t][s] = __builtin_bit_cast(f16x8, wh);
                xl[t][s] = __builtin_bit_cast(f16x8, wl);
            }
        }
        // values of block b of LDS buffer 'buf' for every tile: value i of a
        // lane is centre row 8 (i / 4) + 4 half + i % 4 of the block
        auto block_values = [&](int buf, int b, f32x16 (&acc)[TILES]) {
            constexpr int T = 3 * KS + 1, P = 4;
            int at = (buf * NB + b) * (NS * 1024) + lane * 16, again = at;
            asm volatile("" : "+v"(again));  // the high parts are read twice: kept, they would spill
            auto frag = [&](int t) {
                const int f = t < 2 * KS ? t : (t < 3 * KS ? t - 2 * KS : 2 * KS);
                return *(const f16x8 *)(wide_lds + (t < 2 * KS ? at : again) + f * 1024);
            };
            f16x8 fr[P];
#pragma unroll
            for (int t = 0; t < P; t++) fr[t] = frag(t);
#pragma unroll
            for (int u = 0; u < TILES; u++) acc[u] = f32x16{};
#pragma unroll
            for (int t = 0; t < T; t++) {
                const f16x8 av = fr[t % P];
                if (t + P < T) fr[t % P] = frag(t + P);
#pragma unroll
                for (int u = 0; u < TILES; u++) {
                    // hi.lo(x), lo.hi(x), hi.hi, norm
                    const f16x8 bv = t < KS ? xl[u][t < KS ? t : 0]
                                            : (t < 2 * KS ? xh[u][t < 2 * KS ? (t - KS) & (KS - 1) : 0]
                                                          : (t < 3 * KS ? xh[u][t & (KS - 1)] : ones));
                    acc[u] = __builtin_amdgcn_mfma_f32_32x32x16_f16(av, bv, acc[u], 0, 0, 0);
                }
            }
            // P reads ahead of the MFMAs that use them, all the way (the
            // scheduler would bunch them, and wait for a read just issued)
            __builtin_amdgcn_sched_group_barrier(0x100, P, 0);
#pragma unroll
            for (int t = 0; t < T; t++) {
                __builtin_amdgcn_sched_group_barrier(0x008, TILES, 0);
                if (t + P < T) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            }
        };
        auto centre_of = [&](int id, int h) {  // id: block << 4 | value
            const int i = id & 15;
            return (id >> 4) * 32 + 8 * (i >> 2) + 4 * h + (i & 3);
        };

        // the three smallest keys of this half, sorted, and their places
        float g[TILES][3];
        int gi[TILES][3];
        float k[TILES][3];  // of the group
#pragma unroll
        for (int t = 0; t < TILES; t++)
#pragma unroll
            for (int q = 0; q < 3; q++) {
                g[t][q] = kFar;
                gi[t][q] = 0;
                k[t][q] = kFar;
            }
        f32x16 acc[TILES];
        for (int ch = 0; ch < nchunks; ch++) {
            staged();  // chunk ch is in buffer ch & 1, and every wavefront is done with the other
            if (ch + 1 < nchunks) stage(ch + 1, (ch + 1) & 1);
#pragma unroll 1
            for (int b = 0; b < NB; b++) {
                const int blk = ch * NB + b;
                if (blk >= kblocks) break;  // uniform
                block_values(ch & 1, b, acc);
                const int at = (blk & 7) * 16;
#pragma unroll
                for (int t = 0; t < TILES; t++)
#pragma unroll
                    for (int i = 0; i < 16; i++) {
                        const float key = pack_key(acc[t][i], scalar_or(at, i), keep);
                        k[t][2] = __builtin_amdgcn_fmed3f(k[t][1], k[t][2], key);
                        k[t][1] = __builtin_amdgcn_fmed3f(k[t][0], k[t][1], key);
                        k[t][0] = __builtin_amdgcn_fmed3f(k[t][0], key, -kFar);  // min (keys are finite)
                    }
                if ((blk & 7) == 7 || blk == kblocks - 1) {  // the group's keys into the lane's
#pragma unroll
                    for (int t = 0; t < TILES; t++)
#pragma unroll
                        for (int q = 0; q < 3; q++) {
                            float v = k[t][q];
                            int id = (blk >> 3) * 128 + (__float_as_int(v) & 127);
#pragma unroll
                            for (int r = 0; r < 3; r++) {
                                const bool less = v < g[t][r];
                                const float w = g[t][r];
                                const int wi = gi[t][r];
                                g[t][r] = less ? v : w;
                                gi[t][r] = less ? id : wi;
                                v = less ? w : v;
                                id = less ? wi : id;
                            }
                            k[t][q] = kFar;
                        }
                }
            }
        }

        // Every lane finishes a point: lane l point l (of the half's tile).
        // The partner's part of it: what the partner holds of this lane's tile.
        const int64_t p = base + lane;
        const bool live = p < a.N && (TILES == 2 || half == 0);
        auto own = [&](const auto &v0, const auto &v1) { return TILES == 2 && half ? v1 : v0; };
        auto theirs = [&](const auto &v0, const auto &v1) {
            return __shfl_xor(TILES == 2 && !half ? v1 : v0, 32, kWave);
        };
        constexpr int L = TILES - 1;
        const float A1 = own(g[0][0], g[L][0]), A2 = own(g[0][1], g[L][1]), A3 = own(g[0][2], g[L][2]);
        const float B1 = theirs(g[0][0], g[L][0]), B2 = theirs(g[0][1], g[L][1]), B3 = theirs(g[0][2], g[L][2]);
        const float X2 = own(xx[0], xx[L]) + theirs(xx[0], xx[L]);
        const int other = 1 - half;
        const int a1 = centre_of(own(gi[0][0], gi[L][0]), half), a2 = centre_of(own(gi[0][1], gi[L][1]), half);
        const int b1 = centre_of(theirs(gi[0][0], gi[L][0]), other), b2 = centre_of(theirs(gi[0][1], gi[L][1]), other);
        const float m1 = fminf(A1, B1), m2 = fminf(fmaxf(A1, B1), fminf(A2, B2));
        const float X = __builtin_amdgcn_sqrtf(X2) * 1.0001f + 0x1p-40f, H = 0.5f * X2;
        const float E = bd.c_dot * X * C + bd.c_sum * (X + C) + bd.c_cc * C * C + bd.c_abs;
        const float dp = 0x1p-16f * 1.02f * (fmaxf(H, fabsf(m1)) * 1.01f + 4.0f * E) + 0x1p-126f;
        const float dhi = (H + m1 + 4.0f * E + 4.0f * dp) * 1.001f + bd.ref_abs;
        const float thr = m1 + 2.0f * E + 2.0f * dp + 2.0f * bd.c_ref * dhi;
        // (comparisons that a value that is not a number fails)
        const bool multi = !(m2 > thr) || !(dhi < bd.far);
        const bool full = live && multi && !(A3 > thr && B3 > thr);
        const bool again = __syncthreads_or(full) != 0;  // and every wavefront is done with the last chunk
        if (!again) stage(0, 0);                         // the next round's first chunk

        float best_d = kInitMin;
        int best_k = 0x7fffffff;
        auto rescore = [&](const float *x, int c, float &bd_, int &bk) {
            if (c < a.K) {
                const float dk = exact_dist(x, a.c + (int64_t)c * D, D);
                if (dk < bd_ || (dk == bd_ && c < bk)) {
                    bd_ = dk;
                    bk = c;
                }
            }
        };
        if (live && !multi) best_k = A1 < B1 ? a1 : b1;
        const bool part = live && multi && !full;
        const unsigned long long parts = __ballot(part);
        if (parts) {
            int at = 0;
            if (lane == 0) at = atomicAdd(listed, __popcll(parts));
            at = __shfl(at, 0, kWave) + __popcll(parts & ((1ull << lane) - 1ull));
            if (part) {
                // up to four places; unused ones hold the smallest key's
                // centre again (rows past K are never under the threshold:
                // their keys are above every other's)
                const int c0 = A1 < B1 ? a1 : b1;
                const int c1 = A1 < B1 ? (!(B1 > thr) ? b1 : c0) : (!(A1 > thr) ? a1 : c0);
                const int c2 = !(A2 > thr) ? a2 : c0, c3 = !(B2 > thr) ? b2 : c0;
                list[at] = (int)p;
                a.assign[p] = c0 | c1 << 16;
                a.mindist[p] = __int_as_float(c2 | c3 << 16);
            }
        }
        if (again) {
            // every value under the threshold of the full points, rescored by
            // the half that holds it
            float bdist[TILES], tt[TILES];
            int bk[TILES], ff[TILES];
#pragma unroll
            for (int t = 0; t < TILES; t++) {
                const int mine = TILES == 2 ? half : 0;
                const float ot = __shfl_xor(thr, 32, kWave);
                const int of = __shfl_xor((int)full, 32, kWave);
                tt[t] = TILES == 1 ? (half ? ot : thr) : (t == mine ? thr : ot);
                ff[t] = TILES == 1 ? (half ? of : (int)full) : (t == mine ? (int)full : of);
                bdist[t] = kInitMin;
                bk[t] = 0x7fffffff;
            }
            for (int ch = 0; ch < nchunks; ch++) {
                stage(ch, 0);
                staged();
#pragma unroll 1
                for (int b = 0; b < NB; b++) {
                    const int blk = ch * NB + b;
                    if (blk >= kblocks) break;
                    block_values(0, b, acc);
#pragma unroll
                    for (int t = 0; t < TILES; t++) {
                        if (!ff[t]) continue;
                        unsigned w = 0;
#pragma unroll
                        for (int i = 0; i < 16; i++)
                            if (pack_key(acc[t][i], (blk & 7) * 16 + i, keep) <= tt[t]) w |= 1u << i;
                        const float *x = a.x + min(base + 32 * t + col, a.N - 1) * D;
                        while (w) {
                            const int i = __builtin_ctz(w);
                            w &= w - 1;
                            rescore(x, centre_of(blk * 16 + i, half), bdist[t], bk[t]);
                        }
                    }
                }
                __syncthreads();  // the buffer is free
            }
            stage(0, 0);
            const float ad = own(bdist[0], bdist[L]), od = theirs(bdist[0], bdist[L]);
            const int ak = own(bk[0], bk[L]), ok = theirs(bk[0], bk[L]);
            if (full) {
                const bool take = od < ad || (od == ad && ok < ak);
                best_d = take ? od : ad;
                best_k = take ? ok : ak;
            }
        }
        if (live && !part) a.assign[p] = best_k == 0x7fffffff ? 0 : best_k;
        if (live && multi) my_rescored++;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load to LDS outlives the workgroup
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) my_rescored += __shfl_xor(my_rescored, o, kWave);
    if (lane == 0 && my_rescored) atomicAdd(rescored, (unsigned long long)my_rescored);
}

// The listed points of km_wide: four lanes a point, one candidate each, with
// map1's exact arithmetic and tie rule.
__global__ __launch_bounds__(256) void km_rescore(KmArgs a, const int *__restrict__ list,
                                                  const int *__restrict__ listed)
{
    const int n = *listed, q = threadIdx.x % 4;
    for (int i = blockIdx.x * 64 + threadIdx.x / 4; i < n; i += gridDim.x * 64) {
        const int p = list[i];
        const unsigned w = q < 2 ? (unsigned)a.assign[p] : __float_as_uint(a.mindist[p]);
        int k = (int)(q & 1 ? w >> 16 : w & 0xffffu);
        float d = kInitMin;
        if (k < a.K) {
            const float v = exact_dist(a.x + (int64_t)p * a.D, a.c + (int64_t)k * a.D, a.D);
            if (v < d) d = v;
            else k = 0x7fffffff;
        } else {
            k = 0x7fffffff;
        }
#pragma unroll
        for (int o = 1; o < 4; o <<= 1) {
            const float od = __shfl_xor(d, o, kWave);
            const int ok = __shfl_xor(k, o, kWave);
            if (od < d || (od == d && ok < k)) {
                d = od;
                k = ok;
            }
        }
        if (q == 0) a.assign[p] = k == 0x7fffffff ? 0 : k;
    }
}

// ------------------------------------------------------------ update

// Centre k's part of the reduction object, by its wavefront: an update keeps
// it in snap (K x D sums, K counts, K distance sums), then it is cleared for
// the next pass (a fill, not a memset, so that the sequence can be captured).
// Ten iterations of 20,000 x 8, K 16: 256 us, 281 with three copies (a graph
// node each) before the update kernel.
__device__ __forceinline__ void retire_object(int k, int lane, int K, int D, unsigned long long *__restrict__ gsum,
                                              unsigned long long *__restrict__ gcnt,
                                              unsigned long long *__restrict__ gdsum, int update,
                                              unsigned long long *__restrict__ snap)
{
    const int64_t KD = (int64_t)K * D;
    for (int d = lane; d < D; d += kWave) {
        const int64_t i = (int64_t)k * D + d;
        if (update) snap[i] = gsum[i];
        gsum[i] = 0;
    }
    if (lane == 0) {
        if (update) {
            snap[KD + k] = gcnt[k];
            snap[KD + K + k] = gdsum[k];
        }
        gcnt[k] = 0;
        gdsum[k] = 0;
    }
}

// One wavefront per centre: applies the Lloyd update from the reduction
// object (c = (sum * 2^-s) / count in FP64, rounded to FP32; empty clusters
// keep their centre), writes the BF16 MFMA row and the norm, and clears the
// object for the next pass.  With update == 0 only the rows are prepared.  A
// centre with a coordinate that is not finite is never map1's nearest: its row
// is far, as the padding rows are.  So is that of one whose squared norm FP32
// does not hold, but its norm then makes every bound infinite, so that every
// centre is rescored.
template <int KS>
__global__ __launch_bounds__(256) void km_finalize(float *__restrict__ c, int K, int K_pad, int D,
                                                   unsigned long long *__restrict__ gsum,
                                                   unsigned long long *__restrict__ gcnt,
                                                   unsigned long long *__restrict__ gdsum, double inv_scale,
                                                   int update, __bf16 *__restrict__ cb, float *__restrict__ cnorm,
                                                   unsigned long long *__restrict__ snap)
{
    constexpr int KW = 16 * (KS + 1);
    constexpr int NB = 16 * KS;  // first norm column
    const int k = blockIdx.x * 4 + threadIdx.x / kWave;
    const int lane = threadIdx.x % kWave;
    if (k >= K_pad) return;
    if (k >= K) {  // padding row: never the minimum
        for (int e = lane; e < KW; e += kWave)
            cb[frag_index(k, e, KW / 16)] = (__bf16)((e == NB) ? 1.0e30f : 0.0f);  // far, finite
        return;
    }
    const long long n = (long long)gcnt[k];
    double ss = 0.0;
    for (int d = lane; d < D; d += kWave) {
        float v = c[(int64_t)k * D + d];
        if (update && n > 0) v = (float)(((double)(long long)gsum[(int64_t)k * D + d] * inv_scale) / (double)n);
        if (update) c[(int64_t)k * D + d] = v;
        ss += (double)v * (double)v;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o, kWave);
    const bool fine = isfinite((float)ss);
    for (int d = lane; d < 16 * KS; d += kWave) {
        const float v = fine && d < D ? -2.0f * c[(int64_t)k * D + d] : 0.0f;  // exact
        cb[frag_index(k, d, KW / 16)] = (__bf16)v;
    }
    if (lane < 16) {
        const double nn = fine ? ss : 1.0e30;
        const __bf16 n1 = (__bf16)(float)nn;
        const double r1 = nn - (double)(float)n1;
        const __bf16 n2 = (__bf16)(float)r1;
        const double r2 = r1 - (double)(float)n2;
        const __bf16 n3 = (__bf16)(float)r2;
        __bf16 v = (__bf16)0.0f;
        if (lane == 0) v = n1;
        if (lane == 1) v = n2;
        if (lane == 2) v = n3;
        cb[frag_index(k, NB + lane, KW / 16)] = v;
    }
    if (lane == 0) cnorm[k] = fine ? (float)sqrt(ss) * 1.0001f : (isfinite(ss) ? INFINITY : 0.0f);
    retire_object(k, lane, K, D, gsum, gcnt, gdsum, update, snap);
}

// The same update with FP16 rows: 2 KS + 1 fragments of 16
// elements per centre: high parts of c^ = -2^a c, low parts, and n^ / 2^15 in
// three parts.  A centre with a coordinate that is not finite is never map1's
// nearest: its row is far, as the padding rows are.
template <int KS>
__global__ __launch_bounds__(256) void km_finalize_wide(float *__restrict__ c, int K, int K_pad, int D,
                                                        unsigned long long *__restrict__ gsum,
                                                        unsigned long long *__restrict__ gcnt,
                                                        unsigned long long *__restrict__ gdsum, double inv_scale,
                                                        int update, _Float16 *__restrict__ cb,
                                                        float *__restrict__ cnorm, float sx,
                                                        unsigned long long *__restrict__ snap)
{
    constexpr int NS = 2 * KS + 1;
    const int k = blockIdx.x * 4 + threadIdx.x / kWave;
    const int lane = threadIdx.x % kWave;
    if (k >= K_pad) return;
    long long n = 0;
    double ss = 0.0;
    bool fine = k < K;
    if (k < K) {
        n = (long long)gcnt[k];
        for (int d = lane; d < D; d += kWave) {
            float v = c[(int64_t)k * D + d];
            if (update && n > 0) v = (float)(((double)(long long)gsum[(int64_t)k * D + d] * inv_scale) / (double)n);
            if (update) c[(int64_t)k * D + d] = v;
            ss += (double)v * (double)v;
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) ss += __shfl_xor(ss, o, kWave);
        fine = isfinite(ss);  // (also where FP32 does not hold it: it is scaled below)
    }
    for (int d = lane; d < 16 * KS; d += kWave) {
        const float v = fine && d < D ? -(c[(int64_t)k * D + d] * sx) : 0.0f;
        const _Float16 h = (_Float16)v;
        cb[frag_index(k, d, NS)] = h;
        cb[frag_index(k, 16 * KS + d, NS)] = (_Float16)(v - (float)h);
    }
    if (lane < 16) {
        const double nn = fine ? ss * (double)sx * (double)sx * (0.5 / kWideOne) : (double)kWideFar;
        const _Float16 n1 = (_Float16)(float)nn;
        const double r1 = nn - (double)(float)n1;
        const _Float16 n2 = (_Float16)(float)r1;
        const double r2 = r1 - (double)(float)n2;
        _Float16 v = (_Float16)0.0f;
        if (lane == 0) v = n1;
        if (lane == 1) v = n2;
        if (lane == 2) v = (_Float16)(float)r2;
        cb[frag_index(k, 32 * KS + lane, NS)] = v;
    }
    if (k >= K) return;
    if (lane == 0) cnorm[k] = fine ? (float)sqrt(ss) * 1.0001f : 0.0f;
    retire_object(k, lane, K, D, gsum, gcnt, gdsum, update, snap);
}

// 256 threads per workgroup.  Sixteen-byte loads, four in flight per thread,
// when x is 16-byte aligned (else one float at a time); the workgroup's
// maximum reaches *out by one atomic (atomics from every wavefront to one
// word serialise).  The maximum does not depend on the order.
__global__ __launch_bounds__(256) void km_maxabs(const float *__restrict__ x, int64_t n,
                                                 unsigned int *__restrict__ out)
{
    __shared__ float part[4];
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    const int64_t gid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    float m = 0.0f;
    if (((uintptr_t)x & 15) == 0) {
        auto mx = [](const float4 v) { return fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))); };
        const float4 *__restrict__ x4 = (const float4 *)x;
        const int64_t n4 = n / 4;
        int64_t i = gid;
        for (; i + 3 * stride < n4; i += 4 * stride) {
            const float4 v0 = x4[i], v1 = x4[i + stride], v2 = x4[i + 2 * stride], v3 = x4[i + 3 * stride];
            m = fmaxf(m, fmaxf(fmaxf(mx(v0), mx(v1)), fmaxf(mx(v2), mx(v3))));
        }
        for (; i < n4; i += stride) m = fmaxf(m, mx(x4[i]));
        if (gid < n - 4 * n4) m = fmaxf(m, fabsf(x[4 * n4 + gid]));  // the last n % 4 values
    } else {
        for (int64_t i = gid; i < n; i += stride) m = fmaxf(m, fabsf(x[i]));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, kWave));
    if (threadIdx.x % kWave == 0) part[threadIdx.x / kWave] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        const float b = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
        if (b > 0.0f) atomicMax(out, __float_as_uint(b));
    }
}

// ------------------------------------------------------------ bucketed reduction
//
// For a reduction object too large for LDS the assignment kernels only find
// the centres, and the object is summed afterwards bucket by bucket: points
// are counted per centre (each workgroup reserving its part of every bucket),
// the counts scanned, the point indices scattered into their centre's bucket,
// and wavefronts walk the buckets in runs of kRun positions, summing each
// centre's rows in registers (the same fixed-point integers as the direct
// path, so the sums are the same bit for bit) and adding them to the object
// once per centre run -- about (N / kRun + K) * D atomics instead of
// N * (D + 2).  The same walk computes min_dist, map1's exact distance to the
// assigned centre.

constexpr int kRun = 256;

// Points [blockIdx.x * chunk, + chunk) of one workgroup: their number per
// centre, and (lds_hist) where they start within the centre's bucket.
__global__ __launch_bounds__(512) void km_bucket_count(const int32_t *__restrict__ assign, int64_t N, int K,
                                                       int64_t chunk, int *__restrict__ cnt, int *__restrict__ part,
                                                       int lds_hist)
{
    extern __shared__ int hist[];
    const int64_t p0 = (int64_t)blockIdx.x * chunk, p1 = min<int64_t>(N, p0 + chunk);
    if (!lds_hist) {
        for (int64_t p = p0 + threadIdx.x; p < p1; p += blockDim.x) atomicAdd(&cnt[assign[p]], 1);
        return;
    }
    for (int k = threadIdx.x; k < K; k += blockDim.x) hist[k] = 0;
    __syncthreads();
    for (int64_t p = p0 + threadIdx.x; p < p1; p += blockDim.x) atomicAdd(&hist[assign[p]], 1);
    __syncthreads();
    for (int k = threadIdx.x; k < K; k += blockDim.x)
        part[(int64_t)blockIdx.x * K + k] = hist[k] ? atomicAdd(&cnt[k], hist[k]) : 0;
}

// One workgroup of 1024 threads: off[k] = exclusive prefix sum of cnt
// (K <= 65536 entries; off has K + 1), and cur = off (scatter cursors).
__global__ __launch_bounds__(1024) void km_bucket_scan(const int *__restrict__ cnt, int K, int *__restrict__ off,
                                                       int *__restrict__ cur)
{
    __shared__ int part[1024];
    const int per = (K + 1023) / 1024;
    const int k0 = threadIdx.x * per, k1 = min(K, k0 + per);
    int sum = 0;
    for (int k = k0; k < k1; k++) sum += cnt[k];
    part[threadIdx.x] = sum;
    __syncthreads();
    for (int d = 1; d < 1024; d <<= 1) {  // inclusive Hillis-Steele scan
        const int v = threadIdx.x >= d ? part[threadIdx.x - d] : 0;
        __syncthreads();
        part[threadIdx.x] += v;
        __syncthreads();
    }
    int run = part[threadIdx.x] - sum;
    for (int k = k0; k < k1; k++) {
        off[k] = run;
        cur[k] = run;
        run += cnt[k];
    }
    if (threadIdx.x == 1023) off[K] = part[1023];
}

// idx[slot] = p, each point into its centre's bucket (order within a bucket
// is arbitrary: the sums are integers).  With the workgroups' parts the
// cursors are in LDS; one returning global atomic per point took 0.24 ms for
// 1 M points of 1,000 centres.
__global__ __launch_bounds__(512) void km_bucket_scatter(const int32_t *__restrict__ assign, int64_t N, int K,
                                                         int64_t chunk, const int *__restrict__ off,
                                                         const int *__restrict__ part, int *__restrict__ cur,
                                                         int *__restrict__ idx, int lds_hist)
{
    extern __shared__ int at[];
    const int64_t p0 = (int64_t)blockIdx.x * chunk, p1 = min<int64_t>(N, p0 + chunk);
    if (!lds_hist) {
        for (int64_t p = p0 + threadIdx.x; p < p1; p += blockDim.x) idx[atomicAdd(&cur[assign[p]], 1)] = (int)p;
        return;
    }
    for (int k = threadIdx.x; k < K; k += blockDim.x) at[k] = off[k] + part[(int64_t)blockIdx.x * K + k];
    __syncthreads();
    for (int64_t p = p0 + threadIdx.x; p < p1; p += blockDim.x) idx[atomicAdd(&at[assign[p]], 1)] = (int)p;
}

// One wavefront per run of kRun bucket positions, 64 points at a time and 32
// dimensions of them: the rows go through LDS (eight lanes read 128 bytes of a
// row), then each lane takes its point's 32 dimensions for the distance (FP32
// in dimension order, as map1) and each half-wavefront's lane a dimension of
// every other point for the sums.  The wavefronts of a workgroup do not wait
// for each other.  One pass over the rows: bound by HBM (128 dimensions,
// rows in bucket order).  Reading them with the lanes over the dimensions, one
// point after another, took 0.52 ms for 1 M x 128, and the distances were
// computed by the assignment kernel.
constexpr int kRowsStride = 36;  // words per point: 16-byte aligned rows that spread over the banks

template <int DP>
__global__ __launch_bounds__(256) void km_bucket_rows(const float *__restrict__ x, const int *__restrict__ idx,
                                                      const int32_t *__restrict__ assign, const float *__restrict__ c,
                                                      float *__restrict__ mindist, int64_t N, int D, float scale,
                                                      float dscale, unsigned long long *__restrict__ gsum,
                                                      unsigned long long *__restrict__ gcnt,
                                                      unsigned long long *__restrict__ gdsum)
{
    __shared__ float4 rows_[4][kWave * kRowsStride / 4];
    const int lane = threadIdx.x % kWave, wv = pat::wave_in_block();
    float *rows = (float *)rows_[wv];
    const int64_t j0 = ((int64_t)blockIdx.x * 4 + wv) * kRun;
    if (j0 >= N) return;  // whole wavefronts, no barrier below
    const int64_t j1 = min<int64_t>(N, j0 + kRun);
    const bool vec = (D % 4) == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)c % 16) == 0;
    const int half = lane / 32, dim = lane % 32, sub = lane % 8;
    unsigned long long acc[DP];
#pragma unroll
    for (int q = 0; q < DP; q++) acc[q] = 0;
    auto flush = [&](int k, int q) {  // panel q's sums of centre k
        const unsigned long long v = acc[q] + __shfl_xor(acc[q], 32, kWave);
        const int d = 32 * q + dim;
        if (half == 0 && d < D && v) atomicAdd(&gsum[(int64_t)k * D + d], v);
        acc[q] = 0;
    };
    int kc = __builtin_amdgcn_readfirstlane(assign[idx[j0]]);  // the centre the sums belong to
    for (int64_t j = j0; j < j1; j += kWave) {
        const bool live = j + lane < j1;
        const int p = idx[live ? j + lane : j1 - 1];
        const int k = assign[p];
        const unsigned long long have = __ballot(live);
        float dist = 0.0f;
        int kend = kc;
#pragma unroll
        for (int q = 0; q < DP; q++) {
            float4 v[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const int64_t r = __shfl(p, 8 * i + lane / 8, kWave);
                const int d = 32 * q + 4 * sub;
                const float *xr = x + r * D + d;
                v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (vec) {
                    if (d < D) v[i] = *(const float4 *)xr;
                } else {
                    if (d < D) v[i].x = xr[0];
                    if (d + 1 < D) v[i].y = xr[1];
                    if (d + 2 < D) v[i].z = xr[2];
                    if (d + 3 < D) v[i].w = xr[3];
                }
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int i = 0; i < 8; i++) *(float4 *)(rows + (8 * i + lane / 8) * kRowsStride + 4 * sub) = v[i];
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            // past D both the row and the centre give 0, and (0 - 0)^2 = +0
            // changes no bit of the sum
            const float *ck = c + (int64_t)k * D + 32 * q;
#pragma unroll
            for (int e = 0; e < 32; e += 4) {
                if (32 * q + e < D) {
                    const float4 xv = *(const float4 *)(rows + lane * kRowsStride + e);
                    float4 cv = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (vec) {
                        cv = *(const float4 *)(ck + e);
                    } else {
                        cv.x = ck[e];
                        if (32 * q + e + 1 < D) cv.y = ck[e + 1];
                        if (32 * q + e + 2 < D) cv.z = ck[e + 2];
                        if (32 * q + e + 3 < D) cv.w = ck[e + 3];
                    }
                    float t = cv.x - xv.x;
                    dist = dist + t * t;
                    t = cv.y - xv.y;
                    dist = dist + t * t;
                    t = cv.z - xv.z;
                    dist = dist + t * t;
                    t = cv.w - xv.w;
                    dist = dist + t * t;
                }
            }
            // the points of one centre lie together
            int kcur = kc;
            for (unsigned long long rem = have; rem;) {
                const int r0 = __ffsll((long long)rem) - 1;
                const int kr = __shfl(k, r0, kWave);
                const unsigned long long m = __ballot(k == kr) & rem;
                const int r1 = r0 + __popcll(m);
                if (kr != kcur) {
                    flush(kcur, q);
                    kcur = kr;
                }
                for (int r = r0 + ((r0 ^ half) & 1); r < r1; r += 2)
                    acc[q] += to_fixed(rows[r * kRowsStride + dim], scale);
                rem &= ~m;
            }
            kend = kcur;
        }
        kc = __builtin_amdgcn_readfirstlane(kend);
        dist = sqrtf(dist);
        const float md = dist < kInitMin ? dist : kInitMin;  // map1 starts from kInitMin
        if (live) mindist[p] = md;
        for (unsigned long long rem = have; rem;) {
            const int kr = __shfl(k, __ffsll((long long)rem) - 1, kWave);
            const unsigned long long m = __ballot(k == kr) & rem;
            unsigned long long v = m >> lane & 1 ? to_fixed(md, dscale) : 0ull;
#pragma unroll
            for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, kWave);
            if (lane == 0) {
                atomicAdd(&gcnt[kr], (unsigned long long)__popcll(m));
                atomicAdd(&gdsum[kr], v);
            }
            rem &= ~m;
        }
    }
#pragma unroll
    for (int q = 0; q < DP; q++) flush(kc, q);
}

__global__ void km_zero_u64(unsigned long long *__restrict__ p, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

__global__ void km_zero_i32(int *__restrict__ p, int64_t n)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

}  // namespace

namespace pat {

// Fixed-point shift for n values of magnitude < maxabs: each value times
// 2^s stays within 2^30 (so it converts to int32) and the largest possible
// sum n * maxabs * 2^s below 2^62.  Same formula as the oracle's.
int kmeans_fixed_shift(int64_t n, float maxabs)
{
    int eN = 0, eM = 0;
    while ((1LL << eN) < n) eN++;
    double m = maxabs > 0 ? maxabs : 1.0f;
    frexp(m, &eM);
    int s = std::min(62 - eN - eM, 30 - eM);
    if (s > 60) s = 60;
    return s;
}

int kmeans_ks_for(int D)
{
    if (D <= 16) return 1;
    if (D <= 32) return 2;
    if (D <= 64) return 4;
    if (D <= 128) return 8;
    return 0;
}

// 32-centre blocks per chunk (accumulator registers: 16 per block).
int kmeans_kb_for(int ks) { return ks <= 2 ? 8 : (ks == 4 ? 4 : 2); }

// LDS bytes of the reduction object and the staged centres.
static int64_t object_bytes(int K, int D) { return 8LL * object_words(K, D); }

int kmeans_maxabs(const float *x, int64_t n, unsigned int *out_bits, hipStream_t st)
{
    hipLaunchKernelGGL(km_zero_u64, dim3(1), dim3(1), 0, st, (unsigned long long *)out_bits, 1);
    PAT_LAUNCH_CHECK();
    hipLaunchKernelGGL(km_maxabs, dim3(1024), dim3(256), 0, st, x, n, out_bits);
    PAT_LAUNCH_CHECK();
    return PAT_OK;
}


// Largest dynamic LDS a workgroup may request on this device (queried once).
static int64_t g_lds_limit = 64 * 1024;

static KmArgs make_args(const KmDev &d)
{
    KmArgs a;
    a.x = d.x;
    a.c = d.c;
    a.N = d.N;
    a.D = d.D;
    a.K = d.K;
    a.scale = ldexpf(1.0f, d.shift);
    a.dscale = ldexpf(1.0f, d.dshift);
    a.assign = d.assign;
    a.mindist = d.mindist;
    a.gsum = d.gsum;
    a.gcnt = d.gcnt;
    a.gdsum = d.gdsum;
    a.use_lds_acc = kmeans_object_in_lds(d.K, d.D);
    a.defer_acc = d.bucketed;
    a.rs = a.use_lds_acc ? object_stride(d.D) : d.D;
    return a;
}


// The MFMA forms that kmeans_assign_mfma chooses from.  One block of centres per
// chunk for three terms with the rows in LDS, at three wavefronts per SIMD; but
// at 64 dimensions a full row stays in registers for the exact distances, at
// two (1 M x 64, K 150: 142 us a pass, 196 with three and the row read again),
// while a row with a tail is read again in any case (1 M x 50, K 100: 131 us
// with three, 148 with two).
using MfmaKernel = void (*)(KmArgs, const void *, const float *, int, MfmaBound, WideBound, unsigned long long *);
struct MfmaForm {
    int ks, nt;
    bool tail, gc;
    int threads;
    MfmaKernel kernel;
};
template <int KS, int KB, int NT, bool TAIL, bool GC, int BS>
constexpr MfmaForm mfma_form()
{
    return {KS, NT, TAIL, GC, BS, km_mfma<KS, KB, NT, TAIL, GC, BS>};
}
static const MfmaForm kMfmaForms[] = {
    // one term
    mfma_form<1, 8, 1, true, false, 512>(), mfma_form<1, 8, 1, false, false, 512>(),
    mfma_form<2, 8, 1, true, false, 512>(), mfma_form<2, 8, 1, false, false, 512>(),
    mfma_form<4, 4, 1, true, false, 512>(), mfma_form<4, 4, 1, false, false, 512>(),
    mfma_form<8, 2, 1, true, false, 512>(), mfma_form<8, 2, 1, false, false, 512>(),
    // three terms, rows in LDS
    mfma_form<1, 1, 3, true, false, 768>(), mfma_form<1, 1, 3, false, false, 768>(),
    mfma_form<2, 1, 3, true, false, 768>(), mfma_form<2, 1, 3, false, false, 768>(),
    mfma_form<4, 1, 3, true, false, 768>(), mfma_form<4, 1, 3, false, false, 512>(),
    mfma_form<8, 1, 3, true, false, 512>(), mfma_form<8, 1, 3, false, false, 512>(),
    // three terms, rows staged chunk by chunk (kmeans_kb_for)
    mfma_form<1, 8, 3, true, true, 512>(), mfma_form<1, 8, 3, false, true, 512>(),
    mfma_form<2, 8, 3, true, true, 512>(), mfma_form<2, 8, 3, false, true, 512>(),
    mfma_form<4, 4, 3, true, true, 512>(), mfma_form<4, 4, 3, false, true, 512>(),
    mfma_form<8, 2, 3, true, true, 512>(), mfma_form<8, 2, 3, false, true, 512>()};

// Those of assign_wide: NB blocks of 32 centres per LDS chunk (two chunks of up
// to 72 KiB).
using WideKernel = void (*)(KmArgs, const _Float16 *, const float *, int, WideBound, int *, int *, unsigned long long *);
struct WideForm {
    int ks, nb, tiles;
    bool tail;
    WideKernel kernel;
};
template <int KS, int NB, int TILES, bool TAIL>
constexpr WideForm wide_form()
{
    return {KS, NB, TILES, TAIL, km_wide<KS, NB, TILES, TAIL>};
}
static const WideForm kWideForms[] = {
    wide_form<1, 8, 1, true>(), wide_form<1, 8, 1, false>(), wide_form<1, 8, 2, true>(), wide_form<1, 8, 2, false>(),
    wide_form<2, 8, 1, true>(), wide_form<2, 8, 1, false>(), wide_form<2, 8, 2, true>(), wide_form<2, 8, 2, false>(),
    wide_form<4, 8, 1, true>(), wide_form<4, 8, 1, false>(), wide_form<4, 8, 2, true>(), wide_form<4, 8, 2, false>(),
    wide_form<8, 4, 1, true>(), wide_form<8, 4, 1, false>(), wide_form<8, 4, 2, true>(), wide_form<8, 4, 2, false>()};

// Raises every kmeans kernel's dynamic-LDS limit to what the device allows
// per workgroup (160 KB on gfx950).  Best effort: the per-block limit the
// device reports is what the launch checks use.  Called once before any
// launch (outside graph capture).
int kmeans_prepare_kernels()
{
    static int done = 0;
    if (done) return PAT_OK;
    int dev = 0, lim = 0;
    PAT_HIP(hipGetDevice(&dev));
    PAT_HIP(hipDeviceGetAttribute(&lim, hipDeviceAttributeMaxSharedMemoryPerBlock, dev));
    g_lds_limit = lim - 256;  // room for the kernels' static LDS
    std::vector<const void *> fns = {(const void *)km_plain<8, 1024>, (const void *)km_plain<16, 1024>,
                                     (const void *)km_plain<32, 1024>, (const void *)km_plain<64, 1024>,
                                     (const void *)km_plain<128, 512>};
    for (const MfmaForm &f : kMfmaForms) fns.push_back((const void *)f.kernel);
    for (const WideForm &f : kWideForms) fns.push_back((const void *)f.kernel);
    for (const void *f : fns)
        if (hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)g_lds_limit) != hipSuccess)
            (void)hipGetLastError();
    done = 1;
    return PAT_OK;
}

// Whether the reduction object (K x D sums, counts, distance sums) is kept
// in LDS by the assignment kernels; otherwise a handle with fewer than 2^31
// points sums it with the bucketed reduction.
bool kmeans_object_in_lds(int K, int D)
{
    return object_bytes(K, D) <= std::min<int64_t>(96 * 1024, g_lds_limit - 32 * 1024);
}

// Largest K counted and placed in LDS by the bucketed reduction (32 KB).
constexpr int kBucketLdsK = 8192;

// Workgroups that count and place the points: one per 4,096 up to two per CU.
static int bucket_wgs(int64_t N, int cus)
{
    return (int)std::max<int64_t>(1, std::min<int64_t>((N + 4095) / 4096, 2LL * cus));
}

int64_t kmeans_bucket_part_words(int64_t N, int K, int cus)
{
    return K <= kBucketLdsK ? (int64_t)bucket_wgs(N, cus) * K : 1;
}

// The bucketed reduction after an assignment pass (see km_bucket_rows).
static int bucket_reduce(const KmDev &d, hipStream_t st)
{
    const int K = d.K;
    // the counts, and km_wide's list for the next pass
    hipLaunchKernelGGL(km_zero_i32, dim3((unsigned)(K / 256 + 1)), dim3(256), 0, st, d.bcnt, (int64_t)K + 1);
    PAT_LAUNCH_CHECK();
    const int wgs = bucket_wgs(d.N, d.cus);
    const int64_t chunk = (d.N + wgs - 1) / wgs;
    const int lds_hist = K <= kBucketLdsK;
    const size_t lds = lds_hist ? (size_t)4 * K : 0;
    hipLaunchKernelGGL(km_bucket_count, dim3((unsigned)wgs), dim3(512), lds, st, (const int32_t *)d.assign, d.N, K, chunk,
                       d.bcnt, d.bpart, lds_hist);
    PAT_LAUNCH_CHECK();
    hipLaunchKernelGGL(km_bucket_scan, dim3(1), dim3(1024), 0, st, (const int *)d.bcnt, K, d.boff, d.bcur);
    PAT_LAUNCH_CHECK();
    hipLaunchKernelGGL(km_bucket_scatter, dim3((unsigned)wgs), dim3(512), lds, st, (const int32_t *)d.assign, d.N, K,
                       chunk, (const int *)d.boff, (const int *)d.bpart, d.bcur, d.bidx, lds_hist);
    PAT_LAUNCH_CHECK();
    const unsigned gs = (unsigned)((d.N + 4 * kRun - 1) / (4 * kRun));
    const float scale = ldexpf(1.0f, d.shift), dscale = ldexpf(1.0f, d.dshift);
    auto rows = d.D <= 32 ? km_bucket_rows<1>
                          : (d.D <= 64 ? km_bucket_rows<2> : (d.D <= 96 ? km_bucket_rows<3> : km_bucket_rows<4>));
    hipLaunchKernelGGL(rows, dim3(gs), dim3(256), 0, st, d.x, (const int *)d.bidx, (const int32_t *)d.assign,
                       (const float *)d.c, d.mindist, d.N, d.D, scale, dscale, d.gsum, d.gcnt, d.gdsum);
    PAT_LAUNCH_CHECK();
    return PAT_OK;
}

static int check_lds(int64_t bytes)
{
    PAT_REQUIRE(bytes <= g_lds_limit, PAT_ERR_UNSUPPORTED, "kmeans: %lld bytes of LDS requested, device allows %lld",
                (long long)bytes, (long long)g_lds_limit);
    return PAT_OK;
}

int kmeans_finalize(const KmDev &d, int update, hipStream_t st)
{
    const double inv = ldexp(1.0, -d.shift);
    const dim3 g((unsigned)((d.K_pad + 3) / 4)), b(256);
    if (d.wide || d.NT == 3) {
        auto f = d.KS == 1 ? km_finalize_wide<1>
                           : (d.KS == 2 ? km_finalize_wide<2> : (d.KS == 4 ? km_finalize_wide<4> : km_finalize_wide<8>));
        hipLaunchKernelGGL(f, g, b, 0, st, d.c, d.K, d.K_pad, d.D, d.gsum, d.gcnt, d.gdsum, inv, update,
                           (_Float16 *)d.cb, d.cnorm, ldexpf(1.0f, d.wexp), d.snap);
        PAT_LAUNCH_CHECK();
        return PAT_OK;
    }
#define PAT_KF(KS_)                                                                                                    \
    hipLaunchKernelGGL((km_finalize<KS_>), g, b, 0, st, d.c, d.K, d.K_pad, d.D, d.gsum, d.gcnt, d.gdsum, inv, update,  \
                       (__bf16 *)d.cb, d.cnorm, d.snap)
    switch (d.KS) {
    case 1: PAT_KF(1); break;
    case 2: PAT_KF(2); break;
    case 4: PAT_KF(4); break;
    case 8: PAT_KF(8); break;
    default: pat::set_error("kmeans: D = %d or terms %d not supported", d.D, d.NT); return PAT_ERR_UNSUPPORTED;
    }
#undef PAT_KF
    PAT_LAUNCH_CHECK();
    return PAT_OK;
}

int kmeans_assign_plain(const KmDev &d, hipStream_t st)
{
    KmArgs a = make_args(d);
    const int64_t cbytes = 4LL * d.K * ((d.D + 3) & ~3);  // rows padded to 4 floats
    int64_t lds = a.use_lds_acc ? object_bytes(d.K, d.D) : 0;
    int in_lds = lds + cbytes <= g_lds_limit;
    if (in_lds) lds += cbytes;
    const int64_t want = (d.N + 1023) / 1024;
    const unsigned grid = (unsigned)std::max<int64_t>(1, std::min<int64_t>(want, (int64_t)d.cus));
#define PAT_KP(DM)                                                                                                     \
    do {                                                                                                               \
        constexpr int bs = DM <= 64 ? 1024 : 512;                                                                      \
        PAT_TRY(check_lds(lds));                                                                                       \
        hipLaunchKernelGGL((km_plain<DM, bs>), dim3(grid), dim3(bs), (size_t)lds, st, a, in_lds);                      \
    } while (0)
    if (d.D <= 8) PAT_KP(8);
    else if (d.D <= 16) PAT_KP(16);
    else if (d.D <= 32) PAT_KP(32);
    else if (d.D <= 64) PAT_KP(64);
    else if (d.D <= 128) PAT_KP(128);
    else {
        pat::set_error("kmeans: D = %d above 128", d.D);
        return PAT_ERR_UNSUPPORTED;
    }
#undef PAT_KP
    PAT_LAUNCH_CHECK();
    return d.bucketed ? bucket_reduce(d, st) : PAT_OK;
}

// LDS bytes of the MFMA kernel with nt terms (staged rows plus the reduction
// object when it is kept in LDS).
static int64_t mfma_lds_bytes(int K, int D, int nt, bool gc = false)
{
    const int ks = kmeans_ks_for(D);
    const int K_pad = (K + 31) / 32 * 32;
    // all rows, or (gc) one chunk: KB blocks of 32 rows (KB = 8, 8, 4, 2 for
    // KS = 1, 2, 4, 8)
    const int kb = kmeans_kb_for(ks);
    const int64_t cbb = 2LL * (gc ? 32 * kb : K_pad) * 16 * mfma_fragments(ks, nt);
    const int64_t obj = object_bytes(K, D) <= std::min<int64_t>(96 * 1024, g_lds_limit - 32 * 1024)
                            ? object_bytes(K, D) : 0;
    return cbb + obj;
}

// Terms of the MFMA path for this shape: 3 (FP16 high and low parts) when its
// rows fit in LDS, else 1 (BF16), 0 when neither fits.
int kmeans_nt_for(int K, int D)
{
    if (!kmeans_ks_for(D)) return 0;
    if (mfma_lds_bytes(K, D, 3) <= g_lds_limit) return 3;
    if (mfma_lds_bytes(K, D, 1) <= g_lds_limit) return 1;
    return 0;
}

// Whether the MFMA path reads its rows from global memory: when neither
// LDS form fits (it then uses three terms).
bool kmeans_gc_for(int K, int D) { return kmeans_ks_for(D) != 0 && kmeans_nt_for(K, D) == 0; }

bool kmeans_mfma_fits(int K, int D) { return kmeans_ks_for(D) != 0 && K <= 65536; }

// Words (FP16) of the wide path's rows.
int64_t kmeans_wide_row_words(int K_pad, int D) { return (int64_t)K_pad * 16 * mfma_fragments(kmeans_ks_for(D), 3); }

// Exponent a of the wide path's scale: 2^a times the largest coordinate lies
// below 2^10 (2^126 is the largest FP32 power of two with an FP32 inverse).
int kmeans_wide_exp(float maxabs)
{
    int e = 0;
    if (maxabs > 0) (void)frexpf(maxabs, &e);
    return std::min(126, 10 - e);
}

// The error bound of km_wide's values (derived there).
static WideBound wide_bound(const KmDev &d)
{
    const double u = ldexp(1.0, -11), e = ldexp(1.0, -14), g = ldexp(1.0, -23), sd = sqrt((double)d.D), KS = d.KS;
    const double over = 1.02;
    WideBound b;
    b.sx = ldexpf(1.0f, d.wexp);
    b.c_dot = (float)(over * (3 * u * u + g * 32 * KS * 2 * u + g * 16 * KS * (1 + 4 * u) + g * 16 * (1 + 4 * u)));
    b.c_sum = (float)(over * (e * sd * (1 + 2 * u) * (1 + g * (48 * KS + 16) * 2)));
    b.c_cc = (float)(over * 0.5 * (u * u * u + g * 16 * (1 + u)));
    b.c_abs = (float)(over * (d.D * e * e + 2.0));
    b.c_ref = (float)((3.0 + d.D + 16.0) * ldexp(1.0, -24) * 1.01);
    b.ref_abs = (float)std::min(1e30, ldexp(1e-30, 2 * d.wexp - 1));
    b.far = (float)std::min(1e38, ldexp(0.98 * kInitMin * kInitMin, 2 * d.wexp - 1));
    return b;
}

static int assign_wide(const KmDev &d, hipStream_t st)
{
    const KmArgs a = make_args(d);
    const WideBound bd = wide_bound(d);
    // two tiles per wavefront (each centre fragment feeds two MFMAs) where
    // that leaves every CU a workgroup, else one
    const bool two = d.N >= 512LL * d.cus;
    const int64_t per = two ? 512 : 256;
    const unsigned grid = (unsigned)std::min<int64_t>((d.N + per - 1) / per, d.cus);
    const bool tail = d.D != 16 * d.KS || ((uintptr_t)d.x % 16) != 0;
    const WideForm *f = std::find_if(std::begin(kWideForms), std::end(kWideForms), [&](const WideForm &w) {
        return w.ks == d.KS && w.tiles == (two ? 2 : 1) && w.tail == tail;
    });
    PAT_REQUIRE(f != std::end(kWideForms), PAT_ERR_UNSUPPORTED, "kmeans: D too large");
    const size_t lds = 2 * (size_t)f->nb * (2 * d.KS + 1) * 1024;
    PAT_TRY(check_lds((int64_t)lds));
    hipLaunchKernelGGL(f->kernel, dim3(grid), dim3(512), lds, st, a, (const _Float16 *)d.cb, (const float *)d.cnorm,
                       d.K_pad, bd, d.bidx, d.bcnt + d.K, d.rescored);
    PAT_LAUNCH_CHECK();
    hipLaunchKernelGGL(km_rescore, dim3((unsigned)std::min<int64_t>((d.N + 63) / 64, 4LL * d.cus)), dim3(256), 0, st, a,
                       (const int *)d.bidx, (const int *)(d.bcnt + d.K));
    PAT_LAUNCH_CHECK();
    return bucket_reduce(d, st);
}

int kmeans_assign_mfma(const KmDev &d, hipStream_t st)
{
    if (d.wide) return assign_wide(d, st);
    KmArgs a = make_args(d);
    PAT_REQUIRE(d.NT == 1 || d.NT == 3, PAT_ERR_UNSUPPORTED, "kmeans: K=%d, D=%d too large for the MFMA path", d.K,
                d.D);
    PAT_REQUIRE(!d.gc || d.NT == 3, PAT_ERR_STATE, "kmeans: global-row MFMA form needs three terms");
    const int64_t lds = mfma_lds_bytes(d.K, d.D, d.NT, d.gc != 0);
    PAT_REQUIRE(lds <= g_lds_limit, PAT_ERR_UNSUPPORTED, "kmeans: K=%d, D=%d too large for the MFMA path", d.K, d.D);
    // Error-bound constants of the one-term form.  u = 2^-8 (BF16 unit
    // roundoff); g = FP32 accumulation over every term of the MFMA chain, with
    // a factor 2 of slack for any internal rounding mode.
    // |x.c - bf(x).bf(c)| <= (2u + u^2) sum |x_d c_d|, scaled by 2 for the -2
    // factor; the norm split leaves u^3 ||c||^2.
    const double u = ldexp(1.0, -8), g = 2.0 * (16.0 * (d.KS + 1)) * ldexp(1.0, -24);
    MfmaBound bd;
    bd.c_dot = (float)((4 * u + 2 * u * u + 4 * g * (1 + u) * (1 + u)) * 1.01);
    bd.c_norm = (float)((u * u * u + 2 * g * (1 + 2 * u)) * 1.01);
    bd.c_ref = (float)((3.0 + d.D + 16.0) * ldexp(1.0, -24) * 1.01);
    const WideBound wb = wide_bound(d);
    // no tail: every K-step full and 16-byte aligned rows
    const bool tail = d.D != 16 * d.KS || ((uintptr_t)d.x % 16) != 0;
    const MfmaForm *f = std::find_if(std::begin(kMfmaForms), std::end(kMfmaForms), [&](const MfmaForm &m) {
        return m.ks == d.KS && m.nt == d.NT && m.gc == (d.gc != 0) && m.tail == tail;
    });
    PAT_REQUIRE(f != std::end(kMfmaForms), PAT_ERR_UNSUPPORTED, "kmeans: D too large");
    // one workgroup per CU (the LDS holds one).  While
    // the points do not fill the chip every wavefront takes one tile (rounded
    // down, a few took two, and 10 iterations of 3,000 x 4, K 8 took 165 us, not 137).  Smaller
    // workgroups on more CUs are slower: each stages the rows and flushes its
    // object (10 iterations of 20,000 x 8, K 16: 158 us with 256 threads, 149
    // with 768; of 100,000 x 16, K 32: 275 and 253).
    const int64_t tiles = (d.N + 31) / 32, waves = f->threads / 64;
    const unsigned grid = (unsigned)std::max<int64_t>(1, std::min<int64_t>((tiles + waves - 1) / waves, d.cus));
    hipLaunchKernelGGL(f->kernel, dim3(grid), dim3((unsigned)f->threads), (size_t)lds, st, a, (const void *)d.cb,
                       (const float *)d.cnorm, d.K_pad, bd, wb, d.rescored);
    PAT_LAUNCH_CHECK();
    return d.bucketed ? bucket_reduce(d, st) : PAT_OK;
}

int kmeans_zero(unsigned long long *p, int64_t n, hipStream_t st)
{
    if (n <= 0) return PAT_OK;
    hipLaunchKernelGGL(km_zero_u64, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, p, n);
    PAT_LAUNCH_CHECK();
    return PAT_OK;
}

}  // namespace pat
