// Reads of device memory into a caller's ordinary (pageable) host memory.
//
// The runtime's own copy of pageable memory takes 130 us for 300 KB, 0.96 ms for 16.8 MB and 5.8 ms for
// 100 MB into mapped pages, and four times as long into fresh ones, against 13 us, 0.30 and 1.8 ms of
// transfer (57 GB/s). Here a copy runs in chunks through a pinned ring, the transfer of the next chunks
// under the host copy of the last; a long read is copied out by a few short-lived threads, because
// what then bounds it is the destination's page faults.
#pragma once

#include <cstddef>
#include <memory>
#include <mutex>

#include "common.h"

namespace cgp {

// The pinned ring: one per process while some handle that used it lives, used by one copy at a time (a
// copy that finds it taken goes through the runtime instead).
struct HostRing;

class HostCopier {
public:
	HostCopier() = default;
	HostCopier(const HostCopier &) = delete;
	HostCopier &operator=(const HostCopier &) = delete;
	~HostCopier();
	// Returns when the copy is complete (and so is all earlier work on the stream).
	void read(void *host, const void *device, size_t bytes, hipStream_t stream);

private:
	std::unique_lock<std::mutex> take_ring(size_t bytes);
	hipEvent_t event(size_t slot);
	std::shared_ptr<HostRing> mRing;
	std::vector<hipEvent_t> mEvents;  // one per slot, of the handle's device
};

}  // namespace cgp
