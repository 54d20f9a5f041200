// The ticket order of a persistent workgroup with two row buffers (ew_persistent2 in
// mg_elementwise.h), apart from the GPU: host and device, over a workgroup `Wg` that gives
//   first()      thread 0 takes the first ticket and shares it with the epoch;
//   next(e)      thread 0 takes another (0 in the other threads, and not shared yet);
//   share(t)     thread 0 writes the shared ticket;
//   ticket(), epoch()   what was shared;
//   barrier()    every thread.
#pragma once

#include <hip/hip_runtime.h>

// load(ticket, rows) issues a chunk's loads, finish(ticket, epoch, rows, mid) runs the chunk;
// it calls mid() in every thread and passes a barrier after it (so every wave has read the
// ticket that mid() shared before the next mid() replaces it).
template <typename Rows, typename Wg, typename Load, typename Finish>
__host__ __device__ __forceinline__ void ew_two_buffers(Wg& wg, unsigned chunks, Load&& load,
                                                        Finish&& finish) {
  wg.first();
  wg.barrier();
  unsigned t = wg.ticket();
  const unsigned e = wg.epoch();
  // Every wave has read the first ticket: without this the first mid() could replace it
  // under a late wave, which would then run another chunk than its workgroup.
  wg.barrier();
  Rows r0, r1;
  if (t < chunks) load(t, r0);
  auto step = [&](unsigned tk, Rows& r, Rows& nr) {
    const unsigned next = wg.next(e);
    unsigned tn = 0u;
    finish(tk, e, r, [&] {
      wg.share(next);
      wg.barrier();
      tn = wg.ticket();
      if (tn < chunks) load(tn, nr);
    });
    return tn;
  };
  while (t < chunks) {
    t = step(t, r0, r1);
    if (t >= chunks) break;
    t = step(t, r1, r0);
  }
}
