// hostexport.hpp — particle records in canonical order to the caller's host arrays.
#pragma once

#include "device_common.hpp"
#include "internal.hpp"

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace mmd {

// The caller's arrays (any of them may be NULL) and one piece of the staging memory.
struct ParticleRecords {
	float4 *pos, *mom, *force;
	int32_t *type, *id;
};

// Records [first, first + count) of the canonical order from the slot-order state.
static __global__ void k_export(const float4* __restrict__ pos, const float4* __restrict__ mom,
								const float4* __restrict__ force, const int32_t* __restrict__ ids,
								const uint32_t* __restrict__ slot_of_canon, uint64_t first, uint64_t count,
								ParticleRecords out) {
	const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if (i >= count)
		return;
	const uint32_t s = slot_of_canon[first + i];
	const float4 p = pos[s];
	out.pos[i] = make_float4(p.x, p.y, p.z, 0.0f);
	out.mom[i] = mom[s];
	out.force[i] = force[s];
	out.type[i] = int32_t(meta_type(__float_as_uint(p.w)));
	out.id[i] = ids[s];
}

// The records go out in pieces: a kernel writes a piece straight into pinned memory, over
// the link, while worker threads copy earlier pieces into the caller's arrays. The copies
// are the larger part (fresh arrays are faulted in and cleared page by page by the thread
// that first writes them), so they are shared by several threads. The staging memory, at
// most kSlots pieces (14.7 MB), stays with the object and serves one call at a time (host
// threads that read one object take turns). A call into fresh arrays, against a kernel into
// five device arrays allocated for it and their copies into pageable memory: 500 particles
// 97 -> 18 us, 10^5 428 -> 335 us, 10^6 4.4 -> 2.5 ms, 2.6 10^6 16.0 -> 5.6 ms
// (147 MB: 26 GB/s). With 1, 2, 4, 6, 8 threads the last took 12.8, 8.1, 5.6, 5.0, 5.3 ms
// and 10^6 particles 4.0, 3.5, 2.7, 3.1, 3.5 ms.
class HostExport {
public:
	static constexpr uint64_t kPiece = 16384; // particles
	static constexpr uint64_t kRecord = 3 * sizeof(float4) + 2 * sizeof(int32_t);
	static constexpr uint64_t kSlots = 16;
	static constexpr unsigned kWorkers = 4;

	HostExport() = default;
	HostExport(const HostExport&) = delete;
	HostExport& operator=(const HostExport&) = delete;
	~HostExport() {
		for (hipEvent_t e : events)
			(void)hipEventDestroy(e);
		if (staging)
			(void)hipHostFree(staging);
	}

	// Particles [0, n) to `out`; launch(first, count, records) writes those of one piece to
	// staging records on the null stream.
	template<class Launch>
	void copy(uint64_t n, const ParticleRecords& out, Launch&& launch) {
		const std::lock_guard<std::mutex> one_call(calls);
		const uint64_t pieces = (n + kPiece - 1) / kPiece, slots = std::min(pieces, kSlots);
		reserve(std::min(n, kPiece), slots);
		const auto count = [&](uint64_t i) { return std::min(kPiece, n - i * kPiece); };
		const auto copy_out = [&](uint64_t i) {
			const ParticleRecords from = slot(i % slots);
			const uint64_t first = i * kPiece, c = count(i);
			const auto part = [&](auto* dst, const auto* src) {
				if (dst)
					std::memcpy(dst + first, src, c * sizeof(*src));
			};
			part(out.pos, from.pos);
			part(out.mom, from.mom);
			part(out.force, from.force);
			part(out.type, from.type);
			part(out.id, from.id);
		};
		Team team(pieces);
		if (pieces > 1)
			team.start(unsigned(std::min<uint64_t>(pieces, kWorkers)), copy_out);
		uint64_t launched = 0;
		for (uint64_t i = 0; i < pieces; ++i) {
			// as many pieces under way as there are free slots, at least piece i
			while (launched < pieces && (launched < slots || team.finished(launched - slots, launched == i))) {
				launch(launched * kPiece, count(launched), slot(launched % slots));
				MMD_HIP(hipEventRecord(events[launched % slots], nullptr));
				++launched;
			}
			MMD_HIP(hipEventSynchronize(events[i % slots]));
			if (!team.post(i))
				copy_out(i);
		}
	} // the team's end waits for the copies

private:
	// Worker threads that copy the posted pieces, in order of posting.
	struct Team {
		std::mutex m;
		std::condition_variable cv;
		std::vector<uint8_t> done;
		uint64_t ready = 0, taken = 0;
		bool stop = false;
		std::vector<std::thread> threads;

		explicit Team(uint64_t pieces) : done(pieces, 0) {}
		~Team() {
			{
				const std::lock_guard<std::mutex> lock(m);
				stop = true;
			}
			cv.notify_all();
			for (std::thread& t : threads)
				t.join();
		}
		template<class Copy>
		void start(unsigned workers, const Copy& copy_out) {
			threads.reserve(workers);
			try {
				for (unsigned w = 0; w < workers; ++w)
					threads.emplace_back([this, &copy_out] { work(copy_out); });
			} catch (const std::system_error&) { // fewer threads, or none
			}
		}
		template<class Copy>
		void work(const Copy& copy_out) {
			std::unique_lock<std::mutex> lock(m);
			for (;;) {
				cv.wait(lock, [this] { return taken < ready || stop; });
				if (taken == ready)
					return;
				const uint64_t i = taken++;
				lock.unlock();
				copy_out(i);
				lock.lock();
				done[i] = 1;
				cv.notify_all();
			}
		}
		// Piece i (the next one) is in its slot; false: there is no thread to copy it.
		bool post(uint64_t i) {
			{
				const std::lock_guard<std::mutex> lock(m);
				if (threads.empty()) {
					done[i] = 1;
					return false;
				}
				ready = i + 1;
			}
			cv.notify_all();
			return true;
		}
		// Whether piece i has been copied; `wait` until it is.
		bool finished(uint64_t i, bool wait) {
			std::unique_lock<std::mutex> lock(m);
			if (wait)
				cv.wait(lock, [this, i] { return done[i] != 0; });
			return done[i] != 0;
		}
	};

	std::mutex calls;
	char* staging = nullptr;
	uint64_t piece = 0, have = 0; // particles of a slot, slots
	std::vector<hipEvent_t> events;

	void reserve(uint64_t particles, uint64_t slots) {
		if (particles > piece || slots > have) {
			const uint64_t p = std::max(particles, piece), k = std::max(slots, have);
			if (staging)
				MMD_HIP(hipHostFree(staging));
			staging = nullptr;
			piece = have = 0;
			MMD_HIP(hipHostMalloc(reinterpret_cast<void**>(&staging), p * k * kRecord));
			piece = p;
			have = k;
		}
		while (events.size() < slots) {
			hipEvent_t e;
			MMD_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
			events.push_back(e);
		}
	}
	ParticleRecords slot(uint64_t k) const {
		ParticleRecords r;
		r.pos = reinterpret_cast<float4*>(staging + k * piece * kRecord);
		r.mom = r.pos + piece;
		r.force = r.mom + piece;
		r.type = reinterpret_cast<int32_t*>(r.force + piece);
		r.id = r.type + piece;
		return r;
	}
};

} // namespace mmd
