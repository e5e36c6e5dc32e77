/*
 * tpk_counting.h - the three extra entry points of libtpk_hip_counting.so.
 *
 * libtpk_hip_counting.so is libtpk_hip.so (same sources, same C ABI: tpk.h) with the distance
 * scans compiled -DTPK_COUNT_WORK: furthest point sampling, the ball queries, three_nn and the
 * Chamfer forward pass count the pair evaluations their lanes EXECUTE (one count = one lane
 * forming one squared distance; for furthest point sampling one running minimum updated).  Chamfer's
 * search also counts the pairs it forms in matrix products of halves, to choose those it evaluates,
 * by themselves: one count per pair of a tile of 32 x 32 that is multiplied.  It is
 * a measuring instrument for benchmarks - executed work divided by time, for kernels that skip
 * most of the pairs a brute-force scan would test - and slower than the shipping library (an
 * atomic add per lane at the end of every kernel).  It has no counterpart in the reference.
 */
#ifndef TPK_COUNTING_H
#define TPK_COUNTING_H

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Waits for the device, stores the pair evaluations counted on the current device since the last
 * call in *pairs and sets the counters back to zero.  Returns TPK_OK or a hipError_t. */
int tpk_work_read_reset(unsigned long long* pairs);

/* The same, and in *products the pairs formed by matrix products since the last call of either. */
int tpk_work_read_reset_both(unsigned long long* pairs, unsigned long long* products);

/* `count` (at most 2^20) products of 32 x 16 halves by 16 x 32 on the matrix cores, for a test of the error that Chamfer's search
 * allows them: of product i, a holds row r's slots 8 h .. 8 h + 7 as its vector of 8 halves number 64 i + 32 h + r, b column c's
 * likewise (16-byte aligned), d (count, 32, 32) the float32 sums. */
int tpk_matrix_product(int64_t count, const void* a, const void* b, float* d, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* TPK_COUNTING_H */
