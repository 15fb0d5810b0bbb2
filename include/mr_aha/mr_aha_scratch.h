/*
 * mr_aha_scratch.h — device memory that libmr_aha_c keeps between calls. No
 * counterpart in the reference's C ABI.
 */
#ifndef MR_AHA_MR_AHA_SCRATCH_H
#define MR_AHA_MR_AHA_SCRATCH_H

#include "mr_aha/mr_aha.h"

#ifdef __cplusplus
extern "C" {
#endif

/* Scratch that the kernel builds keep between calls (at most 4 GiB idle in a
 * process). mr_scratch_idle: bytes idle on `device` (negative: the current
 * one). mr_scratch_release: gives them back to the device and reports how many
 * (bytes may be NULL); blocks in use stay, and the next build takes new ones.
 * The library does this by itself when one of its own allocations fails; it
 * cannot see other allocators fail. */
MR_EXPORT int mr_scratch_idle(int device, int64_t *bytes);
MR_EXPORT int mr_scratch_release(int device, int64_t *bytes);

#ifdef __cplusplus
}
#endif

#endif
