// Index arithmetic of the kernels in plain constexpr functions, which the host's tests
// compile as they stand.
#pragma once
#include <stdint.h>

// Byte offset of point i of a chunk, from the chunk's first point; last: the index of the
// dataset's last point from there, which lanes past it load again.  The chunk's own offset,
// which passes 32 bits from 2^30 points on, stays out of it: it goes to the base address.
constexpr uint32_t gpr_point_offset(int i, int last) { return 4u * (uint32_t)(i < last ? i : last); }

// Most workgroups of a launch of `threads` threads each.  A launch's size in threads has 32
// bits: HIP starts what is left of a larger one modulo 2^32, and reports no error.
constexpr int gpr_max_groups(int threads) { return (int)(0xffffffffu / (unsigned)threads); }

// `groups` workgroups of `threads` in as many launches as that takes: launch(first, count),
// which returns 0 or an error, starts `count` of them from `first` on.
template <class F>
inline int gpr_launches(int groups, int threads, F launch) {
    for (int first = 0, count; first < groups; first += count) {
        count = groups - first < gpr_max_groups(threads) ? groups - first : gpr_max_groups(threads);
        if (const int e = launch(first, count)) return e;
    }
    return 0;
}

// A token of the adjoint's plan: op code (5 bits; every code past the table's is 31, an unknown op
// as they are, since its low bits alone may be another's), row of its value, and its left
// and right operands (a unary token's operand on the right), eight bits each.
constexpr int gpr_gtok(int op, int row, int left, int right) {
    return (op < 31 ? op : 31) | (row & 255) << 5 | (left & 255) << 13 | (right & 255) << 21;
}
constexpr int gpr_gtok_op(int w) { return w & 31; }
constexpr int gpr_gtok_row(int w) { return (w >> 5) & 255; }
constexpr int gpr_gtok_left(int w) { return (w >> 13) & 255; }
constexpr int gpr_gtok_right(int w) { return (w >> 21) & 255; }
