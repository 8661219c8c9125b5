// nrc_scratch.hpp -- device scratch that the stateless gradient keeps between its calls.
// Host code on the HIP runtime alone, so that a test can build it against a stand-in runtime.
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>
#include <mutex>

namespace nrc {

// A few blocks per GPU kept between calls, each guarded by the event of its last use.  A call
// takes a block of its stream's GPU that no other host thread holds and that its own stream
// used last, or whose last use is over; it makes its stream wait for that event and records
// the event again after its last kernel, so calls on several streams and threads never share
// a block in use, nor wait for each other.  With no such block, on a stream of another GPU
// than the current one (whose memory the current GPU's runtime calls would not give), or under
// stream capture, the scratch is stream-ordered as a library's is (hipMallocAsync,
// hipFreeAsync).  Those two cost 25-40 us of host time a call: a forward and a gradient of
// 16,384 rows took 109 us a pass with them, 33 us of it in kernels (38 us a pass with a kept
// block).
class ScratchPool {
public:
	explicit constexpr ScratchPool(size_t block_bytes) : block_bytes_(block_bytes) {}

private:
	static constexpr int kMaxDevices = 64, kBlocks = 2;
	struct Block {
		void *p = nullptr;
		hipEvent_t done = nullptr;
		hipStream_t last = nullptr; // compared only: a reused handle still waits for `done`
		bool held = false;
	};

public:
	class Lease {
	public:
		void *p = nullptr;

	private:
		friend class ScratchPool;
		Block *block = nullptr; // null: stream-ordered
	};

	hipError_t take(Lease &l, size_t bytes, hipStream_t s) {
		if (s == hipStreamLegacy) s = nullptr; // the same stream; not every call takes this handle
		int dev = 0;
		const hipError_t e = hipGetDevice(&dev);
		if (e != hipSuccess) return e;
		hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
		const bool captured = hipStreamIsCapturing(s, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone;
		if (!captured && bytes <= block_bytes_ && dev >= 0 && dev < kMaxDevices && on_device(s, dev)) {
			std::lock_guard<std::mutex> lock(mu_);
			// relaxed: a capture that another stream has under way neither forbids nor sees
			// the allocation and the queries
			hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
			const bool swapped = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
			Block *b = find(blocks_[dev], s);
			if (swapped) (void)hipThreadExchangeStreamCaptureMode(&mode);
			if (b && hipStreamWaitEvent(s, b->done, 0) == hipSuccess) {
				b->held = true;
				l.block = b;
				l.p = b->p;
				return hipSuccess;
			}
		}
		(void)hipGetLastError();
		hipError_t m = hipMallocAsync(&l.p, bytes, s);
		if (m == hipErrorOutOfMemory && !captured) {
			trim();
			(void)hipGetLastError();
			m = hipMallocAsync(&l.p, bytes, s);
		}
		return m;
	}

	// after the last kernel that uses the scratch was launched, whatever failed
	hipError_t give(Lease &l, hipStream_t s) {
		if (s == hipStreamLegacy) s = nullptr;
		if (!l.block) return hipFreeAsync(l.p, s);
		std::lock_guard<std::mutex> lock(mu_);
		const hipError_t e = hipEventRecord(l.block->done, s);
		l.block->last = s;
		if (e == hipSuccess) l.block->held = false; // a block whose use cannot be marked is never handed out again
		return e;
	}

	// Frees the kept blocks of this GPU that no call holds (hipFree waits for their last use);
	// a capture that is under way elsewhere is not disturbed.
	void trim() {
		int dev = 0;
		if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return;
		std::lock_guard<std::mutex> lock(mu_);
		hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
		const bool swapped = hipThreadExchangeStreamCaptureMode(&mode) == hipSuccess;
		for (Block &b : blocks_[dev])
			if (b.p && !b.held) {
				(void)hipFree(b.p);
				(void)hipEventDestroy(b.done);
				b = Block{};
			}
		if (swapped) (void)hipThreadExchangeStreamCaptureMode(&mode);
	}

	// hipMalloc for the library's other allocations: the kept blocks go before one is refused
	hipError_t malloc(void **p, size_t bytes) {
		hipError_t e = hipMalloc(p, bytes);
		if (e != hipErrorOutOfMemory) return e;
		trim();
		(void)hipGetLastError();
		return hipMalloc(p, bytes);
	}

private:
	// The default streams are the current GPU's (hipStreamGetDevice does not take their handles).
	static bool on_device(hipStream_t s, int dev) {
		hipDevice_t own = -1;
		return s == nullptr || s == hipStreamPerThread || (hipStreamGetDevice(s, &own) == hipSuccess && own == dev);
	}

	Block *find(Block (&blocks)[kBlocks], hipStream_t s) {
		for (Block &b : blocks)
			if (b.p && !b.held && b.last == s) return &b;
		for (Block &b : blocks) {
			if (b.held) continue;
			if (b.p) {
				if (hipEventQuery(b.done) == hipSuccess) return &b;
				continue;
			}
			if (hipEventCreateWithFlags(&b.done, hipEventDisableTiming) != hipSuccess) return nullptr;
			if (hipMalloc(&b.p, block_bytes_) == hipSuccess) return &b;
			(void)hipEventDestroy(b.done);
			b = Block{};
			return nullptr;
		}
		return nullptr;
	}

	size_t block_bytes_;
	std::mutex mu_;
	Block blocks_[kMaxDevices][kBlocks];
};

} // namespace nrc
