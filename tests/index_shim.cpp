// The kernels' index arithmetic for the CPU tests.
#include "../gpuropolis_amd/csrc/gpr_index.h"

extern "C" uint32_t shim_point_offset(int i, int last) { return gpr_point_offset(i, last); }
extern "C" int shim_max_groups(int threads) { return gpr_max_groups(threads); }
// the launches of `groups` workgroups: pairs of first and count into out, their number returned;
// the launch that starts at `fail` returns error 5
extern "C" int shim_launches(int groups, int threads, int fail, int *out, int room) {
    int n = 0;
    const int e = gpr_launches(groups, threads, [&](int first, int count) {
        if (first == fail || n == room) return 5;
        out[2 * n] = first;
        out[2 * n++ + 1] = count;
        return 0;
    });
    return e ? -e : n;
}
extern "C" void shim_gtok(int op, int row, int left, int right, int *out) {
    const int w = gpr_gtok(op, row, left, right);
    out[0] = gpr_gtok_op(w);
    out[1] = gpr_gtok_row(w);
    out[2] = gpr_gtok_left(w);
    out[3] = gpr_gtok_right(w);
}
