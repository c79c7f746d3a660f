// Device state of one kmeans problem, shared by the kernels and the handle.
#pragma once

#include <cstdint>

#include <hip/hip_runtime.h>

namespace pat {

struct KmDev {
    const float *x;  // N x D points (device)
    float *c;        // K x D centres (FP32)
    int64_t N;
    int D, K, K_pad, KS;  // K_pad: K rounded up to 32; KS: 16-wide K-steps of the data
    int NT;               // MFMA data terms: 3 (FP16 high and low parts), 1 (BF16), 0 (no MFMA path)
    int wide;             // FP16 rows and km_wide instead of the NT forms (bucketed handles)
    int wexp;             // its scale 2^wexp
    int gc;               // MFMA rows read from global memory (K x D too large for LDS)
    int shift, dshift;    // fixed-point scales 2^shift (coordinates), 2^dshift (distances)
    int32_t *assign;      // N
    float *mindist;       // N
    unsigned long long *gsum, *gcnt, *gdsum;  // reduction object (K x D, K, K)
    unsigned long long *snap;                 // last pass's reduction object (K x D + 2 K)
    void *cb;             // MFMA rows: FP16, K_pad x 16*(2*KS+1) (wide, three terms), or BF16, K_pad x 16*(KS+1)
    float *cnorm;         // ||c_k|| (rounded up)
    unsigned long long *rescored;  // points with more than one candidate
    int cus;              // compute units
    int bucketed;         // reduction object too large for LDS: assignments first, then bucket sums
    int *bidx, *bcnt, *boff, *bcur;  // N bucketed point indices (km_wide: its list); K counts and the list's
                                     // length, K+1 offsets, K cursors
    int *bpart;  // bucket starts per workgroup (kmeans_bucket_part_words)
};

int kmeans_fixed_shift(int64_t n, float maxabs);
int kmeans_ks_for(int D);
bool kmeans_mfma_fits(int K, int D);
int kmeans_nt_for(int K, int D);
bool kmeans_gc_for(int K, int D);
bool kmeans_object_in_lds(int K, int D);
int64_t kmeans_bucket_part_words(int64_t N, int K, int cus);
int64_t kmeans_wide_row_words(int K_pad, int D);
int kmeans_wide_exp(float maxabs);
int kmeans_maxabs(const float *x, int64_t n, unsigned int *out_bits, hipStream_t st);
int kmeans_finalize(const KmDev &d, int update, hipStream_t st);
int kmeans_assign_plain(const KmDev &d, hipStream_t st);
int kmeans_assign_mfma(const KmDev &d, hipStream_t st);
int kmeans_zero(unsigned long long *p, int64_t n, hipStream_t st);
int kmeans_prepare_kernels();

}  // namespace pat
