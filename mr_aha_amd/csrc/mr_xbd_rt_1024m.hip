// Run-time-length fused x pass, 1024 work-items, masked kernel, ranks 1 to 16.

#include "mr_xbd_rt_kernels.hpp"

mr_xbd_rt_fn mr_xbd_rt_1024m(int L) { return mr_rt_pick<true, 1024>(L); }
