// The q4 GEMM kernels' host entry points (prompt-length and batched rows).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace fh {

// q4_gemm_rows.hip: rows / 16 and columns / 16 per block, and the estimated
// time; ct = 0 where the kernel does not take the shape.
struct RowsPlan {
    uint32_t rt = 0, ct = 0;
    double us = 0;
};
RowsPlan plan_q4_gemm_rows(uint32_t cus, uint32_t x_ld, const uint16_t *s, const uint16_t *b, uint32_t m, uint32_t n,
                           uint32_t k);
void launch_q4_gemm_rows(hipStream_t stream, const RowsPlan &plan, const uint16_t *x, uint32_t x_ld,
                         const uint32_t *wq, const uint16_t *s, const uint16_t *b, uint32_t m, uint32_t n, uint32_t k,
                         void *y, int y_is_f32);

// q4_gemm.hip: that plan where the dispatch of a shape takes it (ct = 0: one
// of the 256-row kernels).
RowsPlan q4_gemm_rows_plan(uint32_t cus, uint32_t x_ld, const uint16_t *s, const uint16_t *b, uint32_t m, uint32_t n,
                           uint32_t k, bool area);

// q4_gemm_direct.hip: the K ranges the direct-weight GEMM takes for the shape
// (0: it does not apply).
uint32_t direct_gemm_splits(uint32_t cus, uint32_t x_ld, uint32_t m, uint32_t n, uint32_t k, bool area);
uint32_t launch_q4_gemm_direct(hipStream_t stream, uint32_t cus, const uint16_t *x, uint32_t x_ld,
                               const uint32_t *wq, const uint16_t *s, const uint16_t *b, uint32_t m, uint32_t n,
                               uint32_t k, void *y, int y_is_f32, void *area);
// Whether launch_q4_gemm_direct_silu takes the [gate; up] GEMM of f pairs.
bool direct_silu_applies(uint32_t cus, uint32_t x_ld, uint32_t m, uint32_t f, uint32_t k, const uint16_t *act);
void launch_q4_gemm_direct_silu(hipStream_t stream, const uint16_t *x, uint32_t x_ld, const uint32_t *wq,
                                const uint16_t *s, const uint16_t *b, uint32_t m, uint32_t f, uint32_t k,
                                uint16_t *act);

}  // namespace fh
