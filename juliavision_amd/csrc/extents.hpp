// Whole pieces of an extent, and the extent they cover; the K up to which sums keep one order.
#pragma once
#include <stddef.h>
#include <stdint.h>

static inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
static inline size_t round_up(size_t a, size_t b) { return (a + b - 1) / b * b; }

constexpr int MI_LNA_KMAX = 512;         // deepest K of the layer-norm prologue; up to it an unsplit GEMM keeps one chain of sums
