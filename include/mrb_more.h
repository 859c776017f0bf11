/*
 * mrb_more.h - entry points of libmrb.so beyond the replacement of the reference's primitives (mrb.h): what this
 * library's own Python classes need besides. Conventions as in mrb.h; not part of its ABI version.
 */
#ifndef MRB_MORE_H_
#define MRB_MORE_H_

#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

/* The gradient of mrb_discounted_return: grad_out is the gradient of `out`, grad_reward ([timesteps, batch, inner])
 * receives the gradient of `reward` and grad_last ([batch, inner], may be NULL) that of `last_value`. With c_t =
 * (1 - done_t) * gamma it is the same recurrence forwards in time, A_t = grad_out_t + c_{t-1} * A_{t-1} (A_0 = grad_out_0):
 * grad_reward_t = A_t, grad_last = c_{T-1} * A_{T-1}. One launch; neither waits nor allocates. */
int mrb_discounted_return_grad(const float *grad_out, const uint8_t *done, float *grad_reward, float *grad_last,
                               int64_t timesteps, int64_t batch, int64_t inner, float gamma, void *stream);

/* Staging memory for rows that lie in host memory: `bytes` (at most 512 KiB) of page-locked memory of buffer `h` (any
 * kind), which the caller fills and hands to the handle's next push or append on `stream` as if it were device memory:
 * the kernels read it where it is. Valid for that one call. The memory, 2 MiB per buffer that is pushed host rows in four
 * segments, is allocated by the first call (no device memory) and freed with the buffer. It is handed out in turn. A
 * segment is read by work on ONE stream: a call on another stream goes on to the next segment. An event on that stream is
 * recorded when the segment is left, and a call that comes around to it waits for the event (for the whole device, if the
 * stream is gone by then). Refused (MRB_ESTATE) while `stream` is recorded into a HIP graph. Calls on one handle are
 * ordered by the caller, as those that change it are. */
int mrb_stage(int64_t h, int64_t bytes, void **ptr, void *stream);

/* Before the host reads rows at `rows` (n host addresses, NULLs among them are skipped): where one of them is page-locked
 * memory, waits for the work on `stream`, which may still be writing it (a non-blocking copy from the device). Pageable
 * memory is not written by queued work, and nothing is waited for (0.1 us an address). */
int mrb_host_settled(const void *const *rows, int n, void *stream);

#ifdef __cplusplus
}
#endif
#endif /* MRB_MORE_H_ */
