// The kernels' index arithmetic for the CPU tests.
#include "../gpuropolis_amd/csrc/gpr_index.h"

extern "C" uint32_t shim_point_offset(int i, int last) { return gpr_point_offset(i, last); }
extern "C" int shim_max_groups(int threads) { return gpr_max_groups(threads); }
