// The kernels' index arithmetic for the CPU tests.
#include "../gpuropolis_amd/csrc/gpr_index.h"

extern "C" uint32_t shim_point_offset(int i, int last) { return gpr_point_offset(i, last); }
