// segsort.hpp — a stable LSD radix sort of up to kSegSortMax 32-bit keys by one workgroup.
#pragma once

#include "internal.hpp"

namespace mmd {

constexpr int kSegWaves = 16;
constexpr int kSegThreads = kSegWaves * 64;
constexpr int kSegPerLane = 20;
constexpr uint32_t kSegSortMax = uint32_t(kSegThreads) * kSegPerLane; // 20480: 159.8 KB of LDS
constexpr int kSegStride = kSegWaves / 2 + 1;                          // words per digit, padded
constexpr uint32_t kSegSpare = 1024u * kSegStride;                      // the bin of idle lanes
constexpr uint32_t kSegHistWords = kSegSpare + 1u;

// Sorts keys[0, n) (n <= kSegThreads PER_LANE, as the LDS arrays) by bits [0, key_bits) in digits of 10 bits: on return
// s_pos holds the sorted order's positions and, with KEYS, s_key the sorted keys. Called by
// all kSegThreads threads. Wave w takes the run [w C, w C + C) of the range (C = ceil(n /
// kSegWaves)) in batches of 64 held in registers, counts its digits, and after the
// block's exclusive scan (digit-major, wave-minor) scatters each batch in order: the
// entries of one batch with one digit rank by lane (their peer mask from 10 ballots) and
// the lowest of them moves the wave's offset for that digit on. Equal digits therefore
// keep wave, batch and lane order. A pass reads the whole range into registers before
// its first barrier and scatters it back after the scan, so one LDS copy suffices; the
// entries carry their position (16 bits). Counts and offsets stay below 2^16, so two waves
// share a histogram word (wave 2k in the low half, 2k + 1 in the high half).
template<bool KEYS, int PER_LANE>
__device__ __forceinline__ void seg_sort(const uint32_t* __restrict__ keys, uint32_t n, int key_bits, uint32_t* s_key,
										 uint16_t* s_pos, uint32_t* hist, uint32_t* wsum) {
	const int passes = (key_bits + 9) / 10;
	const int wv = int(threadIdx.x >> 6), lane = int(threadIdx.x & 63);
	const uint32_t half = 16u * uint32_t(wv & 1), col = uint32_t(wv >> 1);
	const uint32_t C = (n + kSegWaves - 1) / kSegWaves; // <= 64 * kSegPerLane
	const uint32_t w0_ = min(n, uint32_t(wv) * C), w1_ = min(n, w0_ + C);
	const uint64_t lt = (uint64_t(1) << lane) - 1;
	uint32_t key[PER_LANE], at[PER_LANE];
	if (w1_ > w0_) { // the first pass's entries, from global memory (reads clamped into the run)
		const uint32_t nb = (w1_ - w0_ + 63u) / 64u;
#pragma unroll
		for (int j = 0; j < PER_LANE; ++j) {
			if (uint32_t(j) < nb) { // wave-uniform
				const uint32_t e = min(w0_ + uint32_t(j) * 64u + uint32_t(lane), w1_ - 1u);
				key[j] = keys[e];
				at[j] = e;
			}
		}
	}
#pragma unroll 1
	for (int pass = 0; pass < passes; ++pass) {
		const int shift = 10 * pass;
		const uint32_t mask = (1u << min(10, key_bits - shift)) - 1u;
		// the run's bounds, opaque to the compiler each pass: otherwise it hoists every
		// batch's address and mask out of the pass loop (64 SGPRs and 32 VGPRs)
		uint32_t w0 = w0_, w1 = w1_;
		asm volatile("" : "+v"(w0), "+v"(w1));
		const uint32_t nb = (w1 - w0 + 63u) / 64u; // batches of this wave
		for (uint32_t i = threadIdx.x; i <= kSegSpare; i += kSegThreads)
			hist[i] = 0u;
		__syncthreads();
		if (w1 > w0) { // reads clamped into the run, a lane past its end counted in the spare bin
			if (pass > 0) {
#pragma unroll
				for (int j = 0; j < PER_LANE; ++j) {
					if (uint32_t(j) < nb) { // wave-uniform
						const uint32_t e = min(w0 + uint32_t(j) * 64u + uint32_t(lane), w1 - 1u);
						key[j] = s_key[e];
						at[j] = s_pos[e];
					}
				}
			}
#pragma unroll
			for (int j = 0; j < PER_LANE; ++j) {
				if (uint32_t(j) < nb) {
					const bool live = w0 + uint32_t(j) * 64u + uint32_t(lane) < w1;
					atomicAdd(&hist[live ? ((key[j] >> shift) & mask) * kSegStride + col : kSegSpare],
							  live ? 1u << half : 1u);
				}
			}
		}
		__syncthreads();
		{ // thread t owns digit t: its waves' counts become their first destinations
			const uint32_t row = threadIdx.x * kSegStride;
			uint32_t c[kSegWaves / 2], s = 0;
#pragma unroll
			for (int k = 0; k < kSegWaves / 2; ++k) {
				c[k] = hist[row + uint32_t(k)];
				s += (c[k] & 0xFFFFu) + (c[k] >> 16);
			}
			const uint32_t incl = wave_inclusive_scan(s);
			if (lane == 63)
				wsum[wv] = incl;
			__syncthreads();
			uint32_t run = incl - s;
			for (int w = 0; w < wv; ++w)
				run += wsum[w];
#pragma unroll
			for (int k = 0; k < kSegWaves / 2; ++k) {
				const uint32_t lo = run;
				run += c[k] & 0xFFFFu;
				hist[row + uint32_t(k)] = lo | (run << 16);
				run += c[k] >> 16;
			}
		}
		__syncthreads();
#pragma unroll
		for (int j = 0; j < PER_LANE; ++j) {
			if (uint32_t(j) >= nb) // wave-uniform
				continue;
			const bool live = w0 + uint32_t(j) * 64u + uint32_t(lane) < w1;
			const uint32_t d = (key[j] >> shift) & mask;
			// the peer mask on 32-bit halves, sx all ones where the lane's bit is set: the
			// lanes that agree on every bit stay (4 VALU a bit instead of 10 on 64-bit masks)
			const uint64_t lv = __ballot(live);
			uint32_t plo = uint32_t(lv), phi = uint32_t(lv >> 32);
#pragma unroll
			for (int b = 0; b < 10; ++b) {
				const int32_t sx = int32_t(d << (31 - b)) >> 31;
				const uint64_t ones = __ballot(sx != 0);
				plo &= ~(uint32_t(ones) ^ uint32_t(sx));
				phi &= ~(uint32_t(ones >> 32) ^ uint32_t(sx));
			}
			const uint64_t peers = uint64_t(plo) | (uint64_t(phi) << 32);
			if (live) {
				// the other half of the word is the sibling wave's: it moves by atomic adds
				uint32_t* h = &hist[d * kSegStride + col];
				const uint32_t first = (*h >> half) & 0xFFFFu;
				const uint32_t rank = uint32_t(__popcll(peers & lt));
				if (rank == 0u)
					atomicAdd(h, uint32_t(__popcll(peers)) << half);
				const uint32_t dst = first + rank;
				if (KEYS || pass + 1 < passes)
					s_key[dst] = key[j];
				s_pos[dst] = uint16_t(at[j]);
			}
		}
		__syncthreads();
	}
}

} // namespace mmd
