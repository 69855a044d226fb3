// Copies from device memory to pageable host arrays (the C ABI's borrowed result pointers).
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace ovl {

// Ordered after the work queued on `st`; returns when the copy is complete.  Arrays of at least HOSTCOPY_MIN
// bytes whose pages do not exist yet go through a ring of pinned buffers that a few host threads empty
// while the DMA engine fills the next ones; all others (memory that the HIP runtime knows among them), and
// copies that find the ring in use by another host thread, are a plain hipMemcpyAsync and a
// synchronisation.
hipError_t copy_to_host(void *host, const void *dev, size_t bytes, hipStream_t st);

// The ring and its threads belong to the process: made by the first copy that wants them, given back when
// the last holder lets go (every context holds it from its creation to its end).
void hostcopy_hold();
void hostcopy_release();

// The line: below it the threads' start costs what they save (fresh arrays, plain and ring: 1 MiB 298 and
// 357 us, 1.7 MiB 460 and 467, 2 MiB 577 and 570, 3 MiB 900 and 656, 4 MiB 1202 and 796).
constexpr size_t HOSTCOPY_MIN = (size_t)2 << 20;

}  // namespace ovl

// copies of this process that took the ring (not in ovl.h: which way a copy goes does not show in its result,
// the tests ask here)
extern "C" long ovl_hostcopy_ring_copies();

// the CPUs this process may keep busy: those of its affinity mask, or fewer by the CPU quota of its control
// group (cgroup_root: where the hierarchy is mounted; null: /sys/fs/cgroup)
extern "C" int ovl_hostcopy_cpus(const char *cgroup_root);
