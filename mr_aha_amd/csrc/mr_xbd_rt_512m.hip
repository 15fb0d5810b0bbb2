// Run-time-length fused x pass, 512 work-items, masked kernel, ranks 1 to 16.

#include "mr_xbd_rt_kernels.hpp"

mr_xbd_rt_fn mr_xbd_rt_512m(int L) { return mr_rt_pick<true, 512>(L); }
