// device_pool.hpp -- device memory kept between owners.
#pragma once

#include "swift_common.hpp"

namespace swift {

// hipMalloc maps memory and hipFree unmaps it behind a device synchronisation:
// 20-60 us and up to 0.7 ms a call, 3 ms of the 6.8 that indexing 50 Mbp and
// aligning 20,000 reads took, from a process's second run on (its first finds
// nothing kept).  Freed blocks are kept instead (at most kPoolBytes a device,
// none above kPoolBlock, none left unused for kPoolAge frees) and given back when
// an allocation of this library fails, or by pool_trim (swift_device_trim), which
// another allocator of the process may need.  A block is handed out once the device
// has been waited for since its owner let it go, as hipFree waits, so the next
// owner may use it on any stream.  Safe from any thread.
//
// `wait`: the wait is at the free (swift_device_free's, as hipFree's is); without
// it, at the first allocation that needs the block and may wait.  The library's
// own arrays leave it to that: 16 of them in the run above, one wait.
constexpr size_t kPoolBytes = (size_t)1 << 30;
constexpr size_t kPoolBlock = (size_t)256 << 20;
constexpr uint64_t kPoolAge = 256;
hipError_t pool_alloc(void **ptr, size_t bytes, bool may_wait);
// ptr: null, or what pool_alloc or hipMalloc returned
hipError_t pool_free(void *ptr, bool wait);
hipError_t pool_trim();  // gives back what is kept on the current device
// hipMalloc, for memory that the pool does not keep (workspaces): gives back
// what the pool keeps before it fails
hipError_t device_malloc(void **ptr, size_t bytes);

}  // namespace swift
