// Run-time-length fused x pass, 1024 work-items, unmasked kernel, ranks 1 to 16.

#include "mr_xbd_rt_kernels.hpp"

mr_xbd_rt_fn mr_xbd_rt_1024(int L) { return mr_rt_pick<false, 1024>(L); }
