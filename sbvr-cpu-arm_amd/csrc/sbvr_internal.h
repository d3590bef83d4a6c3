// What the translation units of libsbvr_hip.so call of each other (host side).
#ifndef SBVR_INTERNAL_H
#define SBVR_INTERNAL_H

#include <hip/hip_runtime.h>
#include <stdint.h>

typedef uint32_t v4u_image __attribute__((ext_vector_type(4)));

// The product of two encoded operands on the matrix cores (mm_ops.hip).
struct MmArgs {
    const uint32_t *l_bvr;       // (K / 32, M, Sl)
    const void *l_idx;           // (K / G, M)
    const uint16_t *l_cache;     // (Ll, Sl)
    const uint32_t *r_bvr;       // (K / 32, N, Sr)
    const void *r_idx;
    const uint16_t *r_cache;
    const uint16_t *bias;
    uint16_t *out;
    int M, N, K, Sl, Ll, Lr;
    int spg;                     // sub-groups of 128 elements per coefficient group
    int l_idx16, r_idx16;
    int m_per_wg;                // left rows of a workgroup
};
// Whether that kernel covers the shape (pointers: r_bvr and r_cache 16-byte aligned).
bool mm_T_mfma_ok(int M, int N, int K, int Sl, int Sr, int G, const void *r_bvr, const void *r_cache);
hipError_t launch_mm_T_mfma(int Sr, int G, MmArgs a, int cus, hipStream_t st);

// Activations encoded on the fly: which of the exponent's five bits (0 the lowest) of an fp16 number bit i of a plane word's half is
// put on.  Alone there it is the normal number 2^(2^b - 15).
__host__ __device__ constexpr int online_bit(int i) { return i == 15 ? 4 : i % 5; }

// The same product with a left operand encoded on the fly (mm_ops.hip, encoder_ops.hip).  image: per sub-group of 128 k and row
// tile of 16 the A operands of eight v_mfma_f32_16x16x32_f16, [u = 0..3][part][lane] of 16 bytes, dword e of lane (row r,
// block b) the pair k = 32 b + 4 u + e, + 16, each the sum of its selected coefficients times the group's power of two (below
// 2^15) in two parts, part 0 the nearest multiple of 2^4, part 1 what is left, both times 2^(1 - 2^online_bit(4 u + e)).  scales: per
// group 2^14 over that power of two.
struct OnlineArgs {
    const uint32_t *l_bvr;       // (K / 32, M, Sl)
    const uint16_t *lines;       // (K / G, Sl)
    const uint32_t *r_bvr;       // (K / 32, N, Sr)
    const void *r_idx;
    const uint16_t *r_cache;
    const uint16_t *bias;
    uint16_t *out;
    const v4u_image *image;
    const float *scales;
    int M, N, K, Sl, Lr;
    int spg, r_idx16;
};
bool online_product_ok(int M, int N, int K, int Sl, int Sr, int G, const void *r_bvr, const void *r_cache, int cus);
hipError_t launch_online_product(int Sr, int G, OnlineArgs a, int cus, hipStream_t st);

// The prefill kernels (sbvr_hip.hip, prefill_ops.hip).
struct GemmArgs {
    const uint16_t *x;
    const uint32_t *bvr;
    const void *idx;
    const uint16_t *cache;
    const uint16_t *bias;
    uint16_t *out;
    int M, N, K, L;
    int steps_per_group;   // G / 64
    int idx16;
    int ksplit;            // workgroups along K (blockIdx.z); 1: results go straight to out
    int part_steps;        // steps of 64 along K of a part (the last one's may be fewer)
    float *part;           // ksplit > 1: (ksplit, M, N) fp32 partial results, all zero between launches
};

// Floats from one part's partial results to the next's: M * N, and up to a multiple of 4, so that every part starts on
// 16 bytes and the second pass takes four outputs at a time whatever N is.
__host__ __device__ inline size_t part_floats(int M, int N) { return (static_cast<size_t>(M) * N + 3) & ~static_cast<size_t>(3); }

// Five to eight row blocks of 32 a workgroup (prefill_ops.hip).
hipError_t launch_gemm_lut_pipelined(int S, int rb, const GemmArgs &a, hipStream_t st);

#endif
