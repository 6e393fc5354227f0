// hostio.h -- raw host arrays <-> device, in chunks of sites (hostio.hip).
#pragma once
#include "common.h"
#include "host_chunks.h"

#include <functional>

namespace qphix {

// One raw host array of a transfer: `bytes` per site, site 0 at `p`.
struct HostArray {
  char *p;
  size_t bytes;
};

// A transfer covers `halves` parities of `half` sites each, one after the other
// in the arrays; a chunk of it lies within one of them.

// stage: device staging of host_stage_bytes() (host_chunks.h), `per_site` bytes a
// site over all its arrays (allocated by the caller, so that running out of
// memory is its to report).

// na (<= 4) arrays to the device: for every chunk, use(d, first, n) queues what
// consumes sites [first, first + n), the chunk of array k at d[k].  The host
// arrays have been read and what use() queued has finished on return.
using HostUse = std::function<void(char *const *d, size_t first, size_t n)>;
void host_to_device(const HostArray *a, int na, size_t half, int halves, char *stage, const HostUse &use);

// The other way: fill(d, first, n) queues what writes the chunk of array k at
// d[k].  The host arrays are complete on return.
void device_to_host(const HostArray *a, int na, size_t half, int halves, char *stage, const HostUse &fill);

// Gives back the pinned buffers, events and copy threads (at finalize).
void host_io_release();

} // namespace qphix
