// Whole pieces of an extent, and the extent they cover.
#pragma once
#include <stddef.h>
#include <stdint.h>

static inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }
static inline size_t round_up(size_t a, size_t b) { return (a + b - 1) / b * b; }
