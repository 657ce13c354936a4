/* edenhip_diag.h -- self-tests of device arithmetic used by libedenhip's kernels.
 *
 * No counterpart in the reference: these entry points check, on the GPU, arithmetic that
 * the kernels rely on to reproduce the reference's fp32 results bit for bit. */
#ifndef EDENHIP_DIAG_H
#define EDENHIP_DIAG_H
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* Compare the kernels' division (through double where the operands are of moderate size) with the
 * compiler's fp32 division on `count` hashed operand pairs, half of them moderate, and on every
 * pair of the `n_special` given values. *mismatches gets the number of pairs whose results
 * differ in any bit (NaNs compare equal). Returns 0, or -1 for bad arguments, -2 for a
 * device error. */
int edenhip_diag_divide(uint64_t seed, int64_t count, const float *special, int32_t n_special, int64_t *mismatches);

/* The same for the divisions by a known reciprocal: mismatches[0] by 1 / d rounded to double, pairs
 * whose quotient is no denormal float; [1] by the reciprocal of a float from the double that it was
 * rounded from, moderate d; [2] by 1 / d as two doubles, finite operands, d not zero (zeros of
 * either sign compare equal). */
int edenhip_diag_reciprocals(uint64_t seed, int64_t count, const float *special, int32_t n_special,
                             int64_t mismatches[3]);

#ifdef __cplusplus
}
#endif
#endif /* EDENHIP_DIAG_H */
