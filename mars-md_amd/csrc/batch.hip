// batch.hip — many independent replicas of a periodic nonbonded system, each one the
// reference's Patch, stepped together on one GPU: one persistent launch per step over
// every replica's particles and one batched rebuild (sort, cell tables, home-cell walk,
// one capacity read-back) for all replicas.
//
// Each replica follows the Patch / SimManager sequence (Patch.cpp:85-121, 238-352,
// 456-480; ReorderManager.cpp:8-25) exactly: its id is the patch id of the seed mix
// (Patch.cpp:252-254); its canonical index (Philox counter, exported order) is
// relabelled at every reorder as Patch::reorder_particles does, by a sort whose ties
// fall to the canonical index as the reference's stable sort; its pair set is its own
// ZOrderPairlist's. Only the scheduling is shared: replica r owns slots
// [off_r, off_r + n_r), every sort is stable within replicas (each replica's range
// sorted by Morton key in one workgroup; above 20480 particles a global sort by key,
// then by replica id), and each kernel serves all replicas.
//
// Cadence: at a reorder step every replica reorders and rebuilds, as each Patch does.
// At a rebuild-period step that is not a reorder step the displacements of all
// replicas are reduced in one kernel and, if any replica has moved more than skin/2,
// every replica gets a new list (forces are those of the same pairs within the cutoff;
// only the FP32 summation order of a replica that would have kept its list changes).
// With the reference's default reorderPeriod (= decompPeriod) the two coincide.
//
// Scope: the replicas share particle types and pair tables and carry no bonded
// topology, exclusions or grids (the workload of many independent nonbonded systems);
// every box is periodic on all axes and particles must lie inside their box.
#include "batch.hpp"

#include "homewalk.hpp"
#include "nbforce.hpp"
#include "segsort.hpp"
#include "step.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>

namespace mmd {

namespace {

constexpr int kBatchBlock = 256;

// Per-replica geometry of the batched build and step.
struct RepGeom {
	DevBox box;
	float lo[3], hi[3]; // Morton domain = the periodic box
	float cw[3], margin[3];
	uint32_t slot0, n;
	int h, mf, reach[3], full[3];
	uint32_t home_off, fine_off;
	uint64_t pid;
	// the reference grid's stencil, when it misses seam pairs (see HomeParams)
	int ref_filter, ref_shift, ref_cells, ref_r[3], ref_full[3];
	// the home-frame prefilter of the walk (see HomeParams)
	int pre;
	float pre_lo2, pre_hi2;
	// the replica's fine-cell stencil in the batch's table (count 0: none), one list for each
	// position under the mask (see HomeParams)
	uint32_t stencil_off, stencil_n, stencil_lists;
};

// A wrapped coordinate lies in [lo, hi] up to the rounding of PeriodicBox::wrap_scalar
// (x - floor((x - o) inv_L) L can end an ulp or two below lo or above hi; the Morton
// quantisation clamps such a coordinate, as the reference's does). One more than 2^-20
// of the box length outside, or NaN, has left the box.
__device__ __forceinline__ bool beyond_box(float x, float lo, float hi) {
	const float tol = (hi - lo) * 0x1p-20f;
	return !(x >= lo - tol && x <= hi + tol);
}

// keys / vals in canonical position: global canonical g = off_r + canon.
__global__ void k_b_encode(const float4* __restrict__ pos, uint64_t total, const uint32_t* __restrict__ rep_of_slot,
						   const RepGeom* __restrict__ geom, uint32_t* __restrict__ keys,
						   uint32_t* __restrict__ vals, uint32_t* __restrict__ outside) {
	const uint64_t s = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if (s >= total)
		return;
	const float4 p = pos[s];
	const RepGeom& G = geom[rep_of_slot[s]];
	const uint32_t g = G.slot0 + meta_canon(__float_as_uint(p.w));
	bool out = false;
	const uint32_t qx = morton_quantize(p.x, G.lo[0], G.hi[0], out);
	const uint32_t qy = morton_quantize(p.y, G.lo[1], G.hi[1], out);
	const uint32_t qz = morton_quantize(p.z, G.lo[2], G.hi[2], out);
	// stored at the canonical index, so the stable sort breaks ties by it; the value is
	// the particle's current slot, which the gather reads from
	keys[g] = split_by3(qz) | (split_by3(qy) << 1) | (split_by3(qx) << 2);
	vals[g] = uint32_t(s);
	if (beyond_box(p.x, G.lo[0], G.hi[0]) || beyond_box(p.y, G.lo[1], G.hi[1]) || beyond_box(p.z, G.lo[2], G.hi[2]))
		atomicOr(outside, 1u);
}

// Second pass key of the global sort (replicas above the per-replica sort's size): the
// replica of each Morton-sorted entry (a slot of that replica), carrying the entry's
// current slot along.
__global__ void k_b_rep_keys(const uint32_t* __restrict__ vals_s, uint64_t total,
							 const uint32_t* __restrict__ rep_of_slot, uint32_t* __restrict__ rkeys,
							 uint32_t* __restrict__ rvals) {
	const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if (i >= total)
		return;
	const uint32_t old = vals_s[i];
	rkeys[i] = rep_of_slot[old];
	rvals[i] = old;
}

// The same order in one launch when every replica has at most kSegSortMax particles:
// each replica's Morton keys sorted by one workgroup (seg_sort). The encode leaves replica
// r's entries at [slot0, slot0 + n) in canonical order, so sorting each such range
// stably by key gives the order of the global stable sort by key followed by the stable
// sort by replica. The old slots are read once, in order, at the end.
__global__ __launch_bounds__(kSegThreads) void k_b_seg_sort(const RepGeom* __restrict__ geom,
															const uint32_t* __restrict__ order,
															const uint32_t* __restrict__ keys,
															const uint32_t* __restrict__ vals,
															uint32_t* __restrict__ out_vals) {
	__shared__ uint32_t s_key[kSegSortMax];
	__shared__ uint16_t s_pos[kSegSortMax];
	__shared__ uint32_t hist[kSegHistWords];
	__shared__ uint32_t wsum[kSegWaves];
	const uint32_t r = order[blockIdx.x];
	const uint32_t base = geom[r].slot0, n = geom[r].n;
	seg_sort<false, kSegPerLane>(keys + base, n, 30, s_key, s_pos, hist, wsum);
#pragma unroll
	for (int k = 0; k < kSegPerLane; ++k) { // every load in flight at once
		const uint32_t i = threadIdx.x + uint32_t(k) * kSegThreads;
		if (i < n)
			out_vals[base + i] = vals[base + s_pos[i]];
	}
}

// New slot i holds the particle of current slot old_slot[i], its Morton code computed
// again from the same position with the same operations as k_b_encode.
__global__ void k_b_gather(const uint32_t* __restrict__ old_slot, uint64_t total,
						   const uint32_t* __restrict__ rep_of_slot, const RepGeom* __restrict__ geom,
						   const float4* __restrict__ pos_in, const float4* __restrict__ mom_in,
						   const int32_t* __restrict__ ids_in, bool relabel, float4* __restrict__ pos_out,
						   float4* __restrict__ snap, float4* __restrict__ mom_out, int32_t* __restrict__ ids_out,
						   uint32_t* __restrict__ codes, uint32_t* __restrict__ slot_of_canon_out) {
	const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if (i >= total)
		return;
	const uint32_t old = old_slot[i];
	const RepGeom& G = geom[rep_of_slot[i]];
	float4 p = pos_in[old];
	bool out = false;
	const uint32_t qx = morton_quantize(p.x, G.lo[0], G.hi[0], out);
	const uint32_t qy = morton_quantize(p.y, G.lo[1], G.hi[1], out);
	const uint32_t qz = morton_quantize(p.z, G.lo[2], G.hi[2], out);
	const uint32_t m = __float_as_uint(p.w);
	const uint32_t canon = relabel ? uint32_t(i) - G.slot0 : meta_canon(m);
	p.w = __uint_as_float(make_meta(meta_type(m), canon));
	pos_out[i] = p;
	snap[i] = p;
	mom_out[i] = mom_in[old];
	ids_out[i] = ids_in[old];
	codes[i] = split_by3(qz) | (split_by3(qy) << 1) | (split_by3(qx) << 2);
	slot_of_canon_out[G.slot0 + canon] = uint32_t(i);
}

// Fine and home cell ranges of every replica (BuildCellRangesKernel, ZOrderNeighbor.h:27-43,
// per replica) as {begin, end} in global slots.
__global__ void k_b_cell_ranges(const uint32_t* __restrict__ codes, uint64_t total,
								const uint32_t* __restrict__ rep_of_slot, const RepGeom* __restrict__ geom,
								uint2* __restrict__ fine, uint2* __restrict__ home, uint32_t* __restrict__ flags) {
	const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if (i >= total)
		return;
	const RepGeom& G = geom[rep_of_slot[i]];
	const bool first = i == G.slot0;
	const bool last = i + 1 == uint64_t(G.slot0) + G.n;
	const uint32_t c = codes[i];
	const uint32_t cp = first ? ~c : codes[i - 1], cn = last ? ~c : codes[i + 1];
	// the gather recomputes each code from the position it moves: codes out of order
	// within a replica (a mismatch with the sort's keys) would give wrong cell ranges
	if (!first && cp > c && flags)
		atomicOr(flags, 2u);
	const int fs = 3 * (10 - G.mf), hs = 3 * (10 - G.h);
	const uint32_t fc = c >> fs, hc = c >> hs;
	if (first || (cp >> fs) != fc)
		fine[G.fine_off + fc].x = uint32_t(i);
	if (last || (cn >> fs) != fc)
		fine[G.fine_off + fc].y = uint32_t(i + 1);
	if (first || (cp >> hs) != hc)
		home[G.home_off + hc].x = uint32_t(i);
	if (last || (cn >> hs) != hc)
		home[G.home_off + hc].y = uint32_t(i + 1);
}

// The stencils' lists in row order, one a workgroup (see stencil_list).
__global__ __launch_bounds__(256) void k_b_stencil_lists(const StencilList* __restrict__ lists,
														 const int4* __restrict__ offsets,
														 uint32_t* __restrict__ codes) {
	__shared__ uint64_t keys[kStencilMax];
	const StencilList l = lists[blockIdx.x];
	stencil_list(offsets + l.first, l.n, int(l.level), l.position, l.by_slot != 0u, codes + l.out, keys);
}

// The home-cell walk over the work items of all replicas (item_off[r] = first item of
// replica r, one item per home cell).
__global__ __launch_bounds__(256, 6) void k_b_walk(const RepGeom* __restrict__ geom, const uint32_t* __restrict__ item_off,
												uint32_t R, uint32_t num_items, const float4* __restrict__ spos,
												const uint2* __restrict__ home, const uint2* __restrict__ fine,
												float rc2, uint32_t cap, const uint32_t* __restrict__ stencils,
												uint32_t* __restrict__ counts,
												uint32_t* __restrict__ nbr) {
	__shared__ WalkLds lds[kHomeWaves];
	const int wv = threadIdx.x >> 6;
	const TileRange TR = xcd_tiles((num_items + kHomeWaves - 1) / kHomeWaves);
	for (uint32_t gidx = TR.tile; gidx < TR.end; gidx += TR.stride) {
		const uint32_t item = uint32_t(__builtin_amdgcn_readfirstlane(int(gidx * kHomeWaves + uint32_t(wv))));
		if (item >= num_items)
			continue;
		uint32_t lo = 0, hi = R; // item_off[lo] <= item < item_off[hi]
		while (hi - lo > 1) {
			const uint32_t mid = (lo + hi) >> 1;
			if (item_off[mid] <= item)
				lo = mid;
			else
				hi = mid;
		}
		const uint32_t r = uint32_t(__builtin_amdgcn_readfirstlane(int(lo)));
		const RepGeom& G = geom[r];
		HomeParams P{};
		P.spos = spos;
		P.home = home + G.home_off;
		P.fine = fine + G.fine_off;
		P.num_home = uint32_t(1) << (3 * G.h);
		P.h = G.h;
		P.s = G.mf - G.h;
		for (int a = 0; a < 3; ++a) {
			P.reach[a] = G.reach[a];
			P.full[a] = G.full[a];
			P.cw[a] = G.cw[a];
			P.margin[a] = G.margin[a];
		}
		P.rc2 = rc2;
		P.box = G.box;
		P.ex = marsmd_exclusion_view{};
		P.cap = cap;
		P.ref_filter = G.ref_filter;
		P.ref_shift = G.ref_shift;
		P.ref_cells = G.ref_cells;
		for (int a = 0; a < 3; ++a) {
			P.ref_r[a] = G.ref_r[a];
			P.ref_full[a] = G.ref_full[a];
			P.dom_lo[a] = G.lo[a];
			P.dom_hi[a] = G.hi[a];
		}
		P.pre = G.pre;
		P.pre_lo2 = G.pre_lo2;
		P.pre_hi2 = G.pre_hi2;
		P.stencil_code = G.stencil_n ? stencils + G.stencil_off : nullptr;
		P.stencil_n = G.stencil_n;
		P.stencil_lists = G.stencil_lists;
		const uint32_t cell = item - item_off[r];
		const uint2 hr = P.home[cell];
		const uint32_t from = uint32_t(__builtin_amdgcn_readfirstlane(int(hr.x)));
		const uint32_t to = uint32_t(__builtin_amdgcn_readfirstlane(int(hr.y)));
		if (walk_mode(P) == kWalkPlain)
			walk_home_cell<kWalkPlain>(P, cell, from, to, lds[wv], counts, nbr);
		else
			walk_home_cell<kWalkGeneral>(P, cell, from, to, lds[wv], counts, nbr);
	}
}

// max over particles of |min_image(pos - snapshot)|^2, per batch (the largest replica
// displacement decides): DisplacementKernel (AdaptiveKernels.h:48-101).
// The largest squared displacement since the build (as float bits) to the host's pinned
// word. Bound by the 36 bytes read a particle and the atomics, one pair per workgroup; the
// last workgroup writes the word and clears acc (two words): 29 us at 2.6 10^6 beads (64 with
// one atomic per wave and the word copied).
constexpr int kDispBlock = 1024;
__global__ __launch_bounds__(kDispBlock) void k_b_max_disp(const float4* __restrict__ cur,
														   const float4* __restrict__ snap, uint64_t total,
														   const uint32_t* __restrict__ rep_of_slot,
														   const RepGeom* __restrict__ geom,
														   uint32_t* __restrict__ acc,
														   unsigned long long* __restrict__ out) {
	__shared__ float wmax[kDispBlock / 64];
	float m = 0.0f;
	for (uint64_t s = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x; s < total;
		 s += uint64_t(gridDim.x) * blockDim.x) {
		const float4 a = cur[s];
		const float4 b = snap[s];
		const RepGeom& G = geom[rep_of_slot[s]];
		float d[3] = {a.x - b.x, a.y - b.y, a.z - b.z};
#pragma unroll
		for (int k = 0; k < 3; ++k) {
			const float L = G.box.L[k];
			int guard = 0;
			while (d[k] > 0.5f * L && guard++ < 8)
				d[k] -= L;
			while (d[k] < -0.5f * L && guard++ < 16)
				d[k] += L;
		}
		m = fmaxf(m, d[0] * d[0] + d[1] * d[1] + d[2] * d[2]);
	}
	for (int o = 32; o > 0; o >>= 1)
		m = fmaxf(m, __shfl_xor(m, o, 64));
	if ((threadIdx.x & 63) == 0)
		wmax[threadIdx.x >> 6] = m;
	__syncthreads();
	if (threadIdx.x == 0) {
		for (int w = 1; w < kDispBlock / 64; ++w)
			m = fmaxf(m, wmax[w]);
		atomicMax(&acc[0], __float_as_uint(m)); // non-negative floats order as uints
		__threadfence(); // before the ticket
		if (atomicAdd(&acc[1], 1u) == gridDim.x - 1u) {
			*out = atomicExch(&acc[0], 0u);
			acc[1] = 0u;
		}
	}
}

// The step kernels' constants in device memory (as kernel arguments they were 3.4 KB read
// back by every workgroup of every launch).
struct BatchConsts {
	alignas(16) NbTables nb;
	alignas(16) marsmd_particle_types types;
};
constexpr int kBatchSplitBlock = 512;

// The rest of slot t's step once its nonbonded force f is summed.
template<int INTEG, bool ENERGY>
__device__ __forceinline__ void b_step_finish(uint64_t t, const float4 p, float4 f, const RepGeom& G, uint32_t step,
											  float4* __restrict__ pos_next, float4* __restrict__ mom,
											  float4* __restrict__ force, const marsmd_particle_types& types,
											  const TypeStep* steps, const StepParams& S, uint64_t base_seed,
											  int store_force) {
	StepParams P = S;
	P.box = G.box;
	P.step = step;
	P.seed = mix_seed(base_seed, G.pid, uint64_t(step));
	float4 pn;
	if (INTEG == MARSMD_INTEGRATOR_BROWNIAN) {
		const float4 pmf =
			position_dependent_force(p.x, p.y, p.z, int(meta_type(fb(p.w))), types, nullptr, P.ef, P.scheme);
		pn = bd_update(p, f, steps[meta_type(fb(p.w))], pmf, P);
	} else {
		float4 mo = mom[t];
		pn = baoab_update(p, mo, f, steps[meta_type(fb(p.w))], P);
		mom[t] = mo;
	}
	pos_next[t] = pn;
	if (ENERGY || store_force)
		force[t] = f;
}

template<int INTEG>
__device__ __forceinline__ void b_stage_step(const BatchConsts& C, const StepParams& S, marsmd_particle_types& types,
											 TypeStep* steps) {
	stage_types(C.types, types);
	if (threadIdx.x < uint32_t(C.types.num_types))
		steps[threadIdx.x] = INTEG == MARSMD_INTEGRATOR_BROWNIAN ? bd_type_step(C.types, int(threadIdx.x), S)
																 : baoab_type_step(C.types, int(threadIdx.x), S);
}

// The fused step over every replica's particles, persistent over XCD-local tiles: the
// replica of a slot gives its box and its seed mix. Bounded to 96 VGPRs (5 waves per
// SIMD; the analytical instances spill 16-21): 160 -> 156.5 us at 512 replicas against 4
// waves with 123 VGPRs; with analytical terms 13 replicas of 40k beads take 188 us and 209
// at 4 waves, 16 of them 246 and 243.
template<int INTEG, bool ENERGY, bool ANALYTIC>
__global__ __launch_bounds__(kBatchBlock, 5) void k_b_step(const float4* __restrict__ pos, float4* __restrict__ pos_next,
														  float4* __restrict__ mom, float4* __restrict__ force,
														  uint64_t total, const uint32_t* __restrict__ rep_of_slot,
														  const RepGeom* __restrict__ geom, NbrList L,
														  const BatchConsts* __restrict__ C,
														  const float* __restrict__ knots_g, StepParams S,
														  uint64_t base_seed, int store_force,
														  const uint32_t* __restrict__ step_base, uint32_t, uint32_t) {
	extern __shared__ float lds_knots[];
	__shared__ NbLds lds_nb;
	__shared__ marsmd_particle_types lds_types;
	__shared__ TypeStep lds_steps[MARSMD_MAX_TYPES]; // the integrator's per-type constants
	const NbTables& T = C->nb;
	b_stage_step<INTEG>(*C, S, lds_types, lds_steps);
	stage_tables(T, knots_g, lds_knots, lds_nb);
	// a replayed segment carries the step's offset in S.step and its first step in memory
	const uint32_t step = S.step + (step_base ? step_base[0] : 0u);
	const TileRange R = xcd_tiles(uint32_t((total + kBatchBlock - 1) / kBatchBlock));
	for (uint32_t tile = R.tile; tile < R.end; tile += R.stride) {
		const uint64_t t = uint64_t(tile) * kBatchBlock + threadIdx.x;
		if (t >= total)
			continue;
		const RepGeom& G = geom[rep_of_slot[t]];
		const float4 p = pos[t];
		const DevBox box = G.box;
		const float4 f =
			nb_force<ANALYTIC>(uint32_t(t), p, pos, L, T, lds_knots, knots_g, lds_nb, box, S.cut_d, ENERGY);
		b_step_finish<INTEG, ENERGY>(t, p, f, G, step, pos_next, mom, force, lds_types, lds_steps, S, base_seed,
									 store_force);
	}
}

// The same step with 1 << split lanes to a slot's row (row_split, nb_force_split), for
// batches whose slots do not fill the chip: the serial walk along a row bounds them. A
// tile is 512 >> split slots; the sums change hands in LDS (two tiles' buffers in turn)
// and one lane per slot finishes the step. 24 replicas, 45k beads (4 lanes a row): 13.4 -> 9.8 us.
template<int INTEG, bool ENERGY, bool ANALYTIC>
__global__ __launch_bounds__(kBatchSplitBlock, 4) void k_b_step_split(
	const float4* __restrict__ pos, float4* __restrict__ pos_next, float4* __restrict__ mom, float4* __restrict__ force,
	uint64_t total, const uint32_t* __restrict__ rep_of_slot, const RepGeom* __restrict__ geom, NbrList L,
	const BatchConsts* __restrict__ C, const float* __restrict__ knots_g, StepParams S, uint64_t base_seed,
	int store_force, const uint32_t* __restrict__ step_base, uint32_t split, uint32_t knot_words) {
	extern __shared__ float lds_knots[]; // knot_words words (a multiple of 4), then the handed-over forces
	__shared__ NbLds lds_nb;
	__shared__ marsmd_particle_types lds_types;
	__shared__ TypeStep lds_steps[MARSMD_MAX_TYPES];
	__shared__ float terms[kBatchSplitBlock / 64][split_terms(ENERGY)];
	const NbTables& T = C->nb;
	const uint32_t per = uint32_t(kBatchSplitBlock) >> split; // slots of a tile
	const uint32_t mine = threadIdx.x >> split, sub = threadIdx.x & ((1u << split) - 1u);
	float4* lds_force = reinterpret_cast<float4*>(lds_knots + knot_words);
	const uint32_t lane = threadIdx.x & 63u;
	const uint32_t first = (threadIdx.x - lane) >> split; // the wave's first slot of a tile
	const TileRange R = xcd_tiles(uint32_t((total + per - 1) / per));
	RowHead h{};
	if (R.tile < R.end)
		h = row_head(R.tile * per + mine, uint32_t(total), sub, pos, L);
	b_stage_step<INTEG>(*C, S, lds_types, lds_steps);
	stage_tables(T, knots_g, lds_knots, lds_nb);
	const uint32_t step = S.step + (step_base ? step_base[0] : 0u);
	float* const wt = terms[threadIdx.x >> 6];
	uint32_t turn = 0;
	for (uint32_t tile = R.tile; tile < R.end; tile += R.stride, turn ^= 1u) {
		const DevBox box = geom[rep_of_slot[min(tile * per + mine, uint32_t(total) - 1u)]].box;
		const float f = T.lds ? nb_force_split<ANALYTIC>(h, sub, split, pos, T, lds_knots, lds_nb, box, S.cut_d, ENERGY, wt)
							  : nb_force_split<ANALYTIC>(h, sub, split, pos, T, knots_g, lds_nb, box, S.cut_d, ENERGY, wt);
		if ((lane >> 2) < (64u >> split))
			reinterpret_cast<float*>(lds_force)[4u * (turn * per + first + (lane >> 2)) + (lane & 3u)] = f;
		if (tile + R.stride < R.end)
			h = row_head((tile + R.stride) * per + mine, uint32_t(total), sub, pos, L);
		__syncthreads(); // (the other buffer's readers finished before it)
		const uint32_t u = tile * per + threadIdx.x;
		if (threadIdx.x < per && u < total)
			b_step_finish<INTEG, ENERGY>(u, pos[u], lds_force[turn * per + threadIdx.x], geom[rep_of_slot[u]], step,
										 pos_next, mom, force, lds_types, lds_steps, S, base_seed, store_force);
	}
}

__global__ void k_b_import(const float4* __restrict__ pos_h, const float4* __restrict__ mom_h,
						   const int32_t* __restrict__ types, uint64_t total, const uint32_t* __restrict__ rep_of_slot,
						   const RepGeom* __restrict__ geom, float4* __restrict__ pos, float4* __restrict__ mom,
						   int32_t* __restrict__ ids, uint32_t* __restrict__ slot_of_canon,
						   float4* __restrict__ force) {
	const uint64_t g = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if (g >= total)
		return;
	const uint32_t c = uint32_t(g) - geom[rep_of_slot[g]].slot0;
	const float4 p = pos_h[g];
	pos[g] = make_float4(p.x, p.y, p.z, __uint_as_float(make_meta(uint32_t(types[g]), c)));
	mom[g] = mom_h ? make_float4(mom_h[g].x, mom_h[g].y, mom_h[g].z, 0.0f) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
	ids[g] = int32_t(c);
	slot_of_canon[g] = uint32_t(g);
	force[g] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
}

__global__ void k_b_half_counts(NbrList L, uint64_t slot0, uint64_t n, uint32_t* __restrict__ half) {
	const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	const uint32_t t = uint32_t(slot0 + i);
	const uint64_t base = L.tile_base[t >> 6];
	uint32_t h = 0;
	for (uint32_t k = 0; k < L.count[t]; ++k)
		h += L.nbr[nbr_slot_index(base, t, k)] > t ? 1u : 0u;
	half[i] = h;
}

__global__ void k_b_write_pairs(NbrList L, const float4* __restrict__ pos, uint64_t slot0, uint64_t n,
								const uint32_t* __restrict__ half_off, int32_t* __restrict__ pairs) {
	const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if (i >= n)
		return;
	const uint32_t t = uint32_t(slot0 + i);
	uint64_t w = half_off[i];
	const uint64_t base = L.tile_base[t >> 6];
	const int32_t a = int32_t(meta_canon(__float_as_uint(pos[t].w)));
	for (uint32_t k = 0; k < L.count[t]; ++k) {
		const uint32_t j = L.nbr[nbr_slot_index(base, t, k)];
		if (j > t) {
			const int32_t b = int32_t(meta_canon(__float_as_uint(pos[j].w)));
			pairs[2 * w] = a < b ? a : b;
			pairs[2 * w + 1] = a < b ? b : a;
			++w;
		}
	}
}

// Full-list entries of each replica (twice its pair count): one workgroup per replica
// sums the counts of its slots, which are one contiguous range.
// Each replica's entries and longest row to the host's pinned words out[1 + r] and
// out[1 + R + r], and the build's flags to out[0] (cleared for the next build).
__global__ __launch_bounds__(256) void k_b_rep_stats(const uint32_t* __restrict__ counts,
													 const RepGeom* __restrict__ geom, uint32_t* __restrict__ flags,
													 unsigned long long* __restrict__ out) {
	__shared__ unsigned long long wsum[4];
	__shared__ uint32_t wmax[4];
	const uint32_t b = geom[blockIdx.x].slot0;
	const uint32_t e = b + geom[blockIdx.x].n;
	unsigned long long sum = 0;
	uint32_t m = 0;
	for (uint32_t i = b + threadIdx.x; i < e; i += 1024u) { // four loads in flight
		const uint32_t c0 = counts[i];
		const uint32_t c1 = i + 256u < e ? counts[i + 256u] : 0u;
		const uint32_t c2 = i + 512u < e ? counts[i + 512u] : 0u;
		const uint32_t c3 = i + 768u < e ? counts[i + 768u] : 0u;
		sum += (unsigned long long)c0 + c1 + c2 + c3;
		m = max(max(m, c0), max(c1, max(c2, c3)));
	}
	for (int o = 32; o > 0; o >>= 1) {
		sum += __shfl_xor(sum, o, 64);
		m = max(m, uint32_t(__shfl_xor(int(m), o, 64)));
	}
	if ((threadIdx.x & 63) == 0) {
		wsum[threadIdx.x >> 6] = sum;
		wmax[threadIdx.x >> 6] = m;
	}
	__syncthreads();
	if (threadIdx.x == 0) {
		out[1 + blockIdx.x] = wsum[0] + wsum[1] + wsum[2] + wsum[3];
		out[1 + gridDim.x + blockIdx.x] = max(max(wmax[0], wmax[1]), max(wmax[2], wmax[3]));
		if (blockIdx.x == 0) {
			out[0] = flags[0];
			flags[0] = 0u;
		}
	}
}

// BAOAB_LastUpdate (BAOAB.h:151-172) on every replica's particles.
__global__ void k_b_last_update(float4* __restrict__ mom, const float4* __restrict__ force, uint64_t total, float dt) {
	const uint64_t t = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if (t >= total)
		return;
	const float4 f = force[t];
	float4 m = mom[t];
	const float hdt = 0.5f * dt;
	const float FCF = 4.18679994e4f;
	m.x += hdt * f.x * FCF;
	m.y += hdt * f.y * FCF;
	m.z += hdt * f.z * FCF;
	mom[t] = m;
}

// The first step of a replayed segment, written by the stream before the replay.
__global__ void k_b_set_word(uint32_t* __restrict__ word, uint32_t value) {
	if (threadIdx.x == 0)
		word[0] = value;
}

using StepKernel = void (*)(const float4*, float4*, float4*, float4*, uint64_t, const uint32_t*, const RepGeom*,
							NbrList, const BatchConsts*, const float*, StepParams, uint64_t, int, const uint32_t*,
							uint32_t, uint32_t);

template<int INTEG, bool ENERGY, bool ANALYTIC>
StepKernel b_step_kernel(bool split) {
	return split ? k_b_step_split<INTEG, ENERGY, ANALYTIC> : k_b_step<INTEG, ENERGY, ANALYTIC>;
}
StepKernel pick_b_step(bool split, bool bd, bool energy, bool analytic) {
	constexpr int B = MARSMD_INTEGRATOR_BROWNIAN, L = MARSMD_INTEGRATOR_LANGEVIN;
	if (bd)
		return energy ? (analytic ? b_step_kernel<B, true, true>(split) : b_step_kernel<B, true, false>(split))
					  : (analytic ? b_step_kernel<B, false, true>(split) : b_step_kernel<B, false, false>(split));
	return energy ? (analytic ? b_step_kernel<L, true, true>(split) : b_step_kernel<L, true, false>(split))
				  : (analytic ? b_step_kernel<L, false, true>(split) : b_step_kernel<L, false, false>(split));
}

// What a captured segment bakes in besides the step offsets: the graph cache's key.
struct SegmentKey {
	const void* kernel;
	unsigned grid, lds;
	uint32_t split, knot_words;
	uint64_t count, total, base_seed;
	const void* ptr[9];
	StepParams S;
};

} // namespace

BatchImpl::BatchImpl(const marsmd_batch_desc& d) : tables(new NbTables{}) {
	R = d.num_replicas;
	if (R == 0)
		raise(MARSMD_ERR_VALUE, "batch: no replicas");
	if (!d.num_particles || !d.boxes)
		raise(MARSMD_ERR_VALUE, "batch: num_particles and boxes are required");
	types = d.types;
	if (types.num_types < 1 || types.num_types > MARSMD_MAX_TYPES)
		raise(MARSMD_ERR_VALUE, "batch: num_types must be in [1, 16]");
	for (int t = 0; t < types.num_types; ++t)
		if (types.pmf_grid_count[t] != 0)
			raise(MARSMD_ERR_VALUE, "batch: grids are not on the batched path");
	off.assign(R + 1, 0);
	for (uint64_t r = 0; r < R; ++r) {
		const marsmd_box& b = d.boxes[r];
		for (int a = 0; a < 3; ++a)
			if (!(b.periodic[a] && b.size[a] > 0.0f))
				raise(MARSMD_ERR_VALUE, "batch: every replica box must be periodic with a positive size");
		if (d.num_particles[r] >= kMaxParticles)
			raise(MARSMD_ERR_VALUE, "batch: a replica holds at most 2^24 particles");
		boxes.push_back(b);
		count.push_back(d.num_particles[r]);
		pid.push_back(d.patch_ids ? d.patch_ids[r] : r);
		off[r + 1] = off[r] + d.num_particles[r];
	}
	total = off[R];
	if (total == 0 || total >= (uint64_t(1) << 28)) // position records addressed by 32-bit byte offsets
		raise(MARSMD_ERR_VALUE, "batch: total particle count must be in [1, 2^28)");
	while ((uint64_t(1) << rep_bits) < R)
		++rep_bits;
	// pair tables (as PatchImpl)
	NbTables& T = *tables;
	T.num_types = types.num_types;
	T.enabled = d.enabled_terms;
	T.coef = make_pair_coeffs(types, d.pair_params);
	for (int i = 0; i < types.num_types * types.num_types; ++i)
		T.tag[i] = d.term_matrix ? d.term_matrix[i] : 0u;
	if (d.num_nb_tables < 0 || d.num_nb_tables > kMaxTables)
		raise(MARSMD_ERR_VALUE, "batch: too many nonbonded tables");
	T.num_tables = d.num_nb_tables;
	std::vector<float> kn;
	for (int k = 0; k < d.num_nb_tables; ++k) {
		const marsmd_table& t = d.nb_tables[k];
		if (t.size < 2 || t.is_periodic)
			raise(MARSMD_ERR_VALUE, "batch: nonbonded tables need >= 2 knots and are not periodic");
		T.start[k] = t.start;
		T.step_inv[k] = t.step_inv;
		T.size[k] = int(t.size);
		T.offset[k] = int(kn.size());
		kn.insert(kn.end(), t.pot, t.pot + t.size);
	}
	for (int i = 0; i < types.num_types * types.num_types; ++i)
		if ((T.tag[i] & MARSMD_PAIR_TERM_TABULATED) && int(T.tag[i] >> MARSMD_PAIR_TABLE_SHIFT) >= d.num_nb_tables)
			raise(MARSMD_ERR_VALUE, "batch: a pair tag names a missing table");
	T.total_knots = int(kn.size());
	T.lds = T.total_knots <= kLdsKnots ? 1 : 0;
	{
		BatchConsts c;
		std::memset(&c, 0, sizeof(c));
		c.nb = T;
		c.types = types;
		consts.resize(sizeof(c));
		MMD_HIP(hipMemcpy(consts.data(), &c, sizeof(c), hipMemcpyHostToDevice));
	}
	knots.resize(std::max<uint64_t>(kn.size(), 1));
	if (!kn.empty())
		MMD_HIP(hipMemcpy(knots.data(), kn.data(), kn.size() * 4, hipMemcpyHostToDevice));
	// slot -> replica
	std::vector<uint32_t> rep(total);
	for (uint64_t r = 0; r < R; ++r)
		std::fill(rep.begin() + long(off[r]), rep.begin() + long(off[r + 1]), uint32_t(r));
	rep_of_slot.resize(total);
	MMD_HIP(hipMemcpy(rep_of_slot.data(), rep.data(), 4 * total, hipMemcpyHostToDevice));
	// the per-replica sort's workgroups, largest replica first (the dispatcher hands the
	// later, smaller ones to the CUs that free up first)
	std::vector<uint32_t> order(R);
	for (uint64_t r = 0; r < R; ++r)
		order[r] = uint32_t(r);
	std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) { return count[a] > count[b]; });
	sort_order.resize(R);
	MMD_HIP(hipMemcpy(sort_order.data(), order.data(), 4 * R, hipMemcpyHostToDevice));
	for (int b = 0; b < 2; ++b)
		pos[b].resize(total);
	mom.resize(total);
	mom_tmp.resize(total);
	force.resize(total);
	snap.resize(total);
	ids.resize(total);
	ids_tmp.resize(total);
	slot_of_canon.resize(total);
	slot_of_canon_tmp.resize(total);
	ref_max_pairs.resize(R);
	for (uint64_t r = 0; r < R; ++r)
		ref_max_pairs[r] = std::max<uint64_t>(count[r], 1);
	rep_pairs_host.resize(R);
}

BatchImpl::~BatchImpl() {
	clear_graphs();
	if (readback)
		(void)hipHostFree(readback);
	if (staging)
		(void)hipHostFree(staging);
	if (capture_stream)
		(void)hipStreamDestroy(capture_stream);
	for (hipEvent_t e : timing_events)
		(void)hipEventDestroy(e);
	for (hipEvent_t e : t_events)
		if (e)
			(void)hipEventDestroy(e);
	delete tables;
}

void BatchImpl::clear_graphs() {
	for (SegmentGraph& g : graphs)
		if (g.exec)
			(void)hipGraphExecDestroy(g.exec);
	graphs.clear();
}

void BatchImpl::copy_from_host(const float* pos4, const float* mom4, const int32_t* type_ids, uint64_t n) {
	if (n != total)
		raise(MARSMD_ERR_VALUE, "batch: copy_particles_from_host takes every replica's particles (" +
									std::to_string(total) + ")");
	for (uint64_t r = 0; r < R; ++r)
		for (uint64_t g = off[r]; g < off[r + 1]; ++g) {
			if (type_ids[g] < 0 || type_ids[g] >= types.num_types)
				raise(MARSMD_ERR_VALUE, "batch: particle type out of range");
			for (int a = 0; a < 3; ++a) {
				const float x = pos4[4 * g + uint64_t(a)];
				const float lo = boxes[r].origin[a];
				if (!(x >= lo && x <= lo + boxes[r].size[a]))
					raise(MARSMD_ERR_VALUE, "batch: particle " + std::to_string(g - off[r]) + " of replica " +
												std::to_string(r) + " lies outside its box");
			}
		}
	DevArray<float4> hp(total), hm(mom4 ? total : 0);
	DevArray<int32_t> ht(total);
	MMD_HIP(hipMemcpy(hp.data(), pos4, 16 * total, hipMemcpyHostToDevice));
	if (mom4)
		MMD_HIP(hipMemcpy(hm.data(), mom4, 16 * total, hipMemcpyHostToDevice));
	MMD_HIP(hipMemcpy(ht.data(), type_ids, 4 * total, hipMemcpyHostToDevice));
	// the import needs only the boxes: the next build uploads the planned geometry again
	geom_uploaded = false;
	std::vector<RepGeom> G(R);
	for (uint64_t r = 0; r < R; ++r) {
		G[r].box = make_devbox(boxes[r]);
		G[r].slot0 = uint32_t(off[r]);
		G[r].n = uint32_t(count[r]);
		G[r].pid = pid[r];
	}
	geom.resize(R * sizeof(RepGeom));
	MMD_HIP(hipMemcpy(geom.data(), G.data(), R * sizeof(RepGeom), hipMemcpyHostToDevice));
	k_b_import<<<grid_for(total, 256), 256>>>(hp.data(), mom4 ? hm.data() : nullptr, ht.data(), total,
											  rep_of_slot.data(), reinterpret_cast<const RepGeom*>(geom.data()),
											  pos[0].data(), mom.data(), ids.data(), slot_of_canon.data(),
											  force.data());
	MMD_LAUNCH_CHECK();
	MMD_HIP(hipDeviceSynchronize());
	cur = 0;
	built = false;
	prepared = false;
	deferred_kick = false;
}

void BatchImpl::copy_to_host(float* pos4, float* mom4, float* force4, int32_t* type_ids, int32_t* id_out,
							 uint64_t n) {
	if (n != total)
		raise(MARSMD_ERR_VALUE, "batch: copy_particles_to_host returns every replica's particles");
	MMD_HIP(hipDeviceSynchronize());
	const ParticleRecords out{reinterpret_cast<float4*>(pos4), reinterpret_cast<float4*>(mom4),
							  reinterpret_cast<float4*>(force4), type_ids, id_out};
	host_export.copy(total, out, [this](uint64_t first, uint64_t count, const ParticleRecords& to) {
		k_export<<<grid_for(count, 256), 256>>>(pos[cur].data(), mom.data(), force.data(), ids.data(),
												slot_of_canon.data(), first, count, to);
		MMD_LAUNCH_CHECK();
	});
}

// Sort every replica (stable by Morton key of its box, ties by canonical index), move
// the state into the new slot order (relabelling canonical indices when reordering),
// then cell tables and the home-cell walk of all replicas, with one read-back.
int batch_size_bucket(uint64_t n) {
	int b = 0;
	while (b + 1 < kBatchBuckets && (uint64_t(1) << (b + 1)) <= n)
		++b;
	return b;
}

// Per-replica geometry of a build with the cell configuration of each replica's size
// bucket (walk_grid; left to the library, the home cells of all replicas together occupy
// the chip, and a replica's rows are in the order that its own size gives, as a Patch's).
void BatchImpl::plan_geometry(float rc, std::vector<uint8_t>& gh, std::vector<uint32_t>& items,
							  uint64_t& fine_total, uint64_t& home_total, hipStream_t s) {
	const float rc2 = rc * rc;
	gh.assign(R * sizeof(RepGeom), 0);
	RepGeom* G = reinterpret_cast<RepGeom*>(gh.data());
	items.assign(R + 1, 0);
	fine_total = 0;
	home_total = 0;
	for (uint64_t r = 0; r < R; ++r) {
		RepGeom& g = G[r];
		const uint64_t n = count[r];
		g.box = make_devbox(boxes[r]);
		g.slot0 = uint32_t(off[r]);
		g.n = uint32_t(n);
		g.pid = pid[r];
		const int bucket = batch_size_bucket(n);
		int m = 0;
		while (m < 10 && (uint64_t(1) << (3 * (m + 1))) <= 2 * std::max<uint64_t>(n, 1))
			++m;
		for (int a = 0; a < 3; ++a) {
			g.lo[a] = boxes[r].origin[a];
			g.hi[a] = boxes[r].origin[a] + boxes[r].size[a];
		}
		const bool per[3] = {true, true, true};
		const WalkGrid w = walk_grid(n, m, cell_target[size_t(bucket)], cell_fine[size_t(bucket)],
									 kWalkFill * double(n) / double(total), 0.0, 4, g.lo, g.hi, per, double(rc), rc2);
		const int h = w.h;
		g.h = h;
		g.mf = w.mf;
		g.stencil_lists = w.lists - 1u;
		for (int a = 0; a < 3; ++a) {
			g.reach[a] = w.reach[a];
			g.full[a] = w.full[a];
			g.cw[a] = w.cw[a];
			g.margin[a] = w.margin[a];
		}
		// the reference grid of this replica: when it misses seam pairs, the walk keeps
		// exactly the pairs its stencil reaches
		const float ext[3] = {boxes[r].size[0], boxes[r].size[1], boxes[r].size[2]};
		const CellGrid ref = select_cell_grid(rc, n, ext, ref_max_pairs[r]);
		const int rcells = 1 << ref.m;
		bool complete = true;
		for (int a = 0; a < 3; ++a) {
			g.ref_r[a] = ref.r[a];
			g.ref_full[a] = 2 * ref.r[a] + 1 >= rcells ? 1 : 0;
			if (g.ref_full[a])
				continue;
			const double W = double(ext[a]) / 1023.0;
			if ((double(ref.r[a]) * (1024 / rcells) - 1.0) * W < double(rc) * (1.0 + 1e-6) + 1e-3)
				complete = false;
		}
		g.ref_filter = complete ? 0 : 1;
		g.pre = home_prefilter_band(boxes[r], g.lo, g.hi, h, rc, &g.pre_lo2, &g.pre_hi2) ? 1 : 0;
		// the walk's stencil, shared by the replicas of one geometry
		const std::vector<float> key = {float(h),		   float(g.mf - h),	   float(g.reach[0]),
										float(g.reach[1]), float(g.reach[2]),  float(g.full[0]),
										float(g.full[1]),  float(g.full[2]),   g.cw[0],
										g.cw[1],		   g.cw[2],			   g.margin[0],
										g.margin[1],	   g.margin[2],		   rc2,
										float(w.lists),	   w.by_slot ? 1.0f : 0.0f};
		auto it = stencil_index.find(key);
		if (it == stencil_index.end()) {
			const std::vector<int4> st = g.mf < h ? std::vector<int4>{make_int4(0, 0, 0, 0)}
												  : home_stencil(h, g.mf - h, g.reach, g.full, g.cw, g.margin, rc2, kStencilMax);
			const uint32_t cells = uint32_t(st.size());
			if (stencil_codes + uint64_t(cells) * w.lists >= (uint64_t(1) << 32))
				raise(MARSMD_ERR_VALUE, "batch: stencils exceed 2^32 entries");
			it = stencil_index.emplace(key, std::make_pair(uint32_t(stencil_codes), cells)).first;
			for (uint32_t b = 0; b < (cells > 0 ? w.lists : 0u); ++b) {
				stencil_lists_host.push_back(StencilList{uint32_t(stencil_cells_host.size()), cells,
														 uint32_t(stencil_codes), uint32_t(g.mf), b,
														 w.by_slot ? 1u : 0u});
				stencil_codes += cells;
			}
			stencil_cells_host.insert(stencil_cells_host.end(), st.begin(), st.end());
		}
		g.stencil_off = it->second.first;
		g.stencil_n = it->second.second;
		g.ref_shift = 10 - ref.m;
		g.ref_cells = rcells;
		g.fine_off = uint32_t(fine_total);
		g.home_off = uint32_t(home_total);
		fine_total += uint64_t(1) << (3 * g.mf);
		home_total += uint64_t(1) << (3 * h);
		items[r + 1] = items[r] + (uint32_t(1) << (3 * h));
	}
	if (fine_total >= (uint64_t(1) << 32))
		raise(MARSMD_ERR_VALUE, "batch: cell tables exceed 2^32 entries");
	if (stencil_lists_host.size() > stencils_made) { // new geometries (synchronous uploads, rare)
		stencils_made = 0; // until all are made
		stencils.resize(stencil_codes);
		stencil_cells.resize(stencil_cells_host.size());
		stencil_lists.resize(stencil_lists_host.size());
		MMD_HIP(hipMemcpy(stencil_cells.data(), stencil_cells_host.data(), sizeof(int4) * stencil_cells_host.size(),
						  hipMemcpyHostToDevice));
		MMD_HIP(hipMemcpy(stencil_lists.data(), stencil_lists_host.data(),
						  sizeof(StencilList) * stencil_lists_host.size(), hipMemcpyHostToDevice));
		k_b_stencil_lists<<<unsigned(stencil_lists_host.size()), 256, 0, s>>>(stencil_lists.data(),
																			  stencil_cells.data(), stencils.data());
		MMD_LAUNCH_CHECK();
		stencils_made = stencil_lists_host.size();
	}
}

void BatchImpl::build(float pairlist_cutoff, bool relabel, hipStream_t s) {
	const float rc = pairlist_cutoff;
	const float rc2 = rc * rc;
	std::vector<uint32_t>& items = items_host;
	// the plan depends on the cutoff, the cell configuration and the pair bookkeeping
	// (boxes and sizes are fixed): planned again only when one of them changed, which
	// keeps it off the GPU's idle time when a run starts with a rebuild
	if (!(plan.valid && plan.rc == rc && plan.target == cell_target && plan.fine == cell_fine &&
		  plan.ref == ref_max_pairs)) {
		plan.valid = geom_uploaded = false; // until planned whole and uploaded
		plan_geometry(rc, geom_host, items, plan.fine_total, plan.home_total, s);
		plan.valid = true;
		plan.rc = rc;
		plan.target = cell_target;
		plan.fine = cell_fine;
		plan.ref = ref_max_pairs;
	}
	const uint64_t fine_total = plan.fine_total, home_total = plan.home_total;
	num_fine = fine_total;
	num_home = home_total;
	num_items = items[R];
	if (!geom_uploaded) {
		// both uploads from pinned memory, so that they queue behind the running steps
		// without the host waiting for them (the last build's copies ended before its wait)
		const size_t gbytes = R * sizeof(RepGeom);
		if (!staging)
			MMD_HIP(hipHostMalloc(reinterpret_cast<void**>(&staging), gbytes + 4 * (R + 1), hipHostMallocDefault));
		std::memcpy(staging, geom_host.data(), gbytes);
		std::memcpy(staging + gbytes, items.data(), 4 * (R + 1));
		geom.resize(gbytes);
		MMD_HIP(hipMemcpyAsync(geom.data(), staging, gbytes, hipMemcpyHostToDevice, s));
		item_off.resize(R + 1);
		MMD_HIP(hipMemcpyAsync(item_off.data(), staging + gbytes, 4 * (R + 1), hipMemcpyHostToDevice, s));
	}
	const RepGeom* gd = reinterpret_cast<const RepGeom*>(geom.data());
	// sort: Morton key (stable; ties by canonical index), then replica (stable)
	keys.resize(total);
	vals.resize(total);
	keys_s.resize(total);
	vals_s.resize(total);
	rkeys.resize(total);
	rvals.resize(total);
	rkeys_s.resize(total);
	rvals_s.resize(total);
	codes.resize(total);
	if (!scalars.data()) { // zero between builds and checks: their kernels leave them so
		scalars.resize(4);
		fill_u32(scalars.data(), 0u, 4, s);
	}
	k_b_encode<<<grid_for(total, 256), 256, 0, s>>>(pos[cur].data(), total, rep_of_slot.data(), gd, keys.data(),
													vals.data(), scalars.data());
	MMD_LAUNCH_CHECK();
	if (*std::max_element(count.begin(), count.end()) <= kSegSortMax) {
		k_b_seg_sort<<<unsigned(R), kSegThreads, 0, s>>>(gd, sort_order.data(), keys.data(), vals.data(),
														 rvals_s.data());
		MMD_LAUNCH_CHECK();
	} else {
		sort_scratch.resize(radix_sort_scratch_bytes(total));
		radix_sort_pairs(keys.data(), vals.data(), keys_s.data(), vals_s.data(), total, 30, sort_scratch.data(),
						 sort_scratch.count, s);
		k_b_rep_keys<<<grid_for(total, 256), 256, 0, s>>>(vals_s.data(), total, rep_of_slot.data(), rkeys.data(),
														  rvals.data());
		MMD_LAUNCH_CHECK();
		radix_sort_pairs(rkeys.data(), rvals.data(), rkeys_s.data(), rvals_s.data(), total, rep_bits,
						 sort_scratch.data(), sort_scratch.count, s);
	}
	const int nxt = 1 - cur;
	k_b_gather<<<grid_for(total, 256), 256, 0, s>>>(rvals_s.data(), total, rep_of_slot.data(), gd, pos[cur].data(),
													mom.data(), ids.data(), relabel, pos[nxt].data(), snap.data(),
													mom_tmp.data(), ids_tmp.data(), codes.data(),
													slot_of_canon_tmp.data());
	MMD_LAUNCH_CHECK();
	cur = nxt;
	mom.swap(mom_tmp);
	ids.swap(ids_tmp);
	slot_of_canon.swap(slot_of_canon_tmp);
	// cell tables
	cells.resize(num_fine + num_home);
	uint2* const fine = cells.data();
	uint2* const home = fine + num_fine;
	// walk with uniform rows of `cap` entries; once more with larger rows if needed
	const uint64_t tiles = (total + 63) / 64;
	counts.resize(total);
	tile_base.resize(tiles + 1);
	if (cap == 0) {
		double vol = 0.0;
		for (uint64_t r = 0; r < R; ++r)
			vol += double(boxes[r].size[0]) * boxes[r].size[1] * boxes[r].size[2];
		const double mean = double(total) / vol * 4.0 / 3.0 * 3.141592653589793 * double(rc) * rc * rc;
		cap = uint32_t(std::min(1.6 * mean + 16.0, 4096.0) + 3) & ~3u;
	}
	k_walk_setup<<<grid_for(std::max(num_fine + num_home, tiles + 1), 256), 256, 0, s>>>(
		fine, num_fine + num_home, tile_base.data(), tiles, 64u * cap);
	MMD_LAUNCH_CHECK();
	k_b_cell_ranges<<<grid_for(total, 256), 256, 0, s>>>(codes.data(), total, rep_of_slot.data(), gd, fine, home,
														 scalars.data());
	MMD_LAUNCH_CHECK();
	const unsigned groups = unsigned((num_items + kHomeWaves - 1) / kHomeWaves);
	const unsigned grid = std::max(8u, (groups + 7u) / 8u * 8u);
	for (int attempt = 0; attempt < 2; ++attempt) {
		const uint64_t storage = tiles * 64 * uint64_t(cap);
		if (storage >= (uint64_t(1) << 32))
			raise(MARSMD_ERR_CAPACITY, "batch: neighbour storage exceeds 2^32 entries");
		if (storage > nbr.count)
			nbr.resize(storage + storage / 8 + 1024);
		if (attempt > 0) { // larger rows
			k_walk_setup<<<grid_for(tiles + 1, 256), 256, 0, s>>>(nullptr, 0, tile_base.data(), tiles, 64u * cap);
			MMD_LAUNCH_CHECK();
		}
		k_b_walk<<<grid, 256, 0, s>>>(gd, item_off.data(), uint32_t(R), uint32_t(num_items), pos[cur].data(),
									  home, fine, rc2, cap, stencils.data(), counts.data(), nbr.data());
		MMD_LAUNCH_CHECK();
		// Pairlist::grow_pair_capacity (Pairlist.h:244-251) bookkeeping per replica with the
		// walk's statistics: one wait for both (in pinned memory)
		if (!readback)
			MMD_HIP(hipHostMalloc(reinterpret_cast<void**>(&readback), 8 * (1 + 2 * R), hipHostMallocDefault));
		k_b_rep_stats<<<unsigned(R), 256, 0, s>>>(counts.data(), gd, scalars.data(),
												  reinterpret_cast<unsigned long long*>(readback));
		MMD_LAUNCH_CHECK();
		MMD_HIP(hipStreamSynchronize(s));
		geom_uploaded = true;
		if (readback[0] & 1u)
			raise(MARSMD_ERR_VALUE, "batch: a particle left its replica's box (positions must stay wrapped)");
		if (readback[0] & 2u)
			raise(MARSMD_ERR_RUNTIME, "batch: Morton codes after the sort were not in order");
		nbr_entries = 0;
		max_neighbors = 0;
		for (uint64_t r = 0; r < R; ++r) {
			nbr_entries += readback[1 + r];
			max_neighbors = std::max(max_neighbors, uint32_t(readback[1 + R + r]));
		}
		if (max_neighbors <= cap)
			break;
		cap = (max_neighbors + max_neighbors / 8 + 4 + 3) & ~3u;
	}
	// the pair counts set the reference grid of the next build
	std::memcpy(rep_pairs_host.data(), readback + 1, 8 * R);
	for (uint64_t r = 0; r < R; ++r) {
		const uint64_t np = rep_pairs_host[r] / 2;
		if (np > ref_max_pairs[r])
			ref_max_pairs[r] = np + np / 4;
	}
	built = true;
	built_cutoff = pairlist_cutoff;
}

bool BatchImpl::needs_rebuild(float skin, hipStream_t s) {
	// (a build has allocated both)
	k_b_max_disp<<<std::min<unsigned>(grid_for(total, kDispBlock), 256), kDispBlock, 0, s>>>(
		pos[cur].data(), snap.data(), total, rep_of_slot.data(), reinterpret_cast<const RepGeom*>(geom.data()),
		scalars.data() + 1, reinterpret_cast<unsigned long long*>(readback));
	MMD_LAUNCH_CHECK();
	MMD_HIP(hipStreamSynchronize(s));
	const uint32_t bits = uint32_t(readback[0]);
	float d2;
	std::memcpy(&d2, &bits, 4);
	return std::sqrt(d2) > skin * 0.5f;
}

BatchImpl::StepShape BatchImpl::step_shape() const {
	const unsigned words = tables->lds ? unsigned(std::max(tables->total_knots, 2)) : 0u;
	StepShape sh;
	sh.split = row_split(total, max_neighbors, nbr_entries);
	if (sh.split == 0) {
		sh.tiles = (total + kBatchBlock - 1) / kBatchBlock;
		sh.block = kBatchBlock;
		sh.lds = 4u * words;
	} else {
		const unsigned per = unsigned(kBatchSplitBlock) >> sh.split;
		sh.tiles = (total + per - 1) / per;
		sh.block = kBatchSplitBlock;
		sh.knot_words = (words + 3u) & ~3u;
		sh.lds = 4u * sh.knot_words + 32u * per; // the knots, then the handed-over forces of two tiles
	}
	return sh;
}

// Workgroups per CU of a step kernel (its instances hold different LDS and registers).
int BatchImpl::step_occupancy(const void* kernel, const StepShape& sh) {
	auto it = occupancy.find(kernel);
	if (it == occupancy.end() || it->second.first != sh.lds) {
		int occ = 0;
		MMD_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kernel, int(sh.block), sh.lds));
		it = occupancy.insert_or_assign(kernel, std::make_pair(sh.lds, std::max(occ, 1))).first;
	}
	return it->second.second;
}

unsigned BatchImpl::step_grid(const void* kernel, const StepShape& sh) {
	const int occ = step_occupancy(kernel, sh);
	if (num_cus == 0) {
		int dev = 0;
		MMD_HIP(hipGetDevice(&dev));
		MMD_HIP(hipDeviceGetAttribute(&num_cus, hipDeviceAttributeMultiprocessorCount, dev));
		num_cus = std::max(num_cus, 1);
	}
	const int per_cu = blocks_per_cu > 0 ? std::min(blocks_per_cu, occ) : occ;
	uint64_t g = std::min<uint64_t>(uint64_t(per_cu) * uint64_t(num_cus), (sh.tiles + 7) / 8 * 8);
	return unsigned(std::max<uint64_t>((g + 7) / 8 * 8, 8));
}

void BatchImpl::set_launch(int bpc, bool graph) {
	if (bpc < 0)
		raise(MARSMD_ERR_VALUE, "batch: blocks_per_cu must be >= 0");
	blocks_per_cu = bpc;
	use_graph = graph;
}

hipGraphExec_t BatchImpl::segment_graph(const void* kernel, unsigned grid, const StepShape& sh, const StepParams& S,
										uint64_t count) {
	SegmentKey k;
	std::memset(&k, 0, sizeof(k));
	k.kernel = kernel;
	k.grid = grid;
	k.lds = sh.lds;
	k.split = sh.split;
	k.knot_words = sh.knot_words;
	k.count = count;
	k.total = total;
	k.base_seed = base_seed;
	const void* ptrs[9] = {pos[cur].data(), pos[1 - cur].data(), mom.data(), force.data(), rep_of_slot.data(),
						   geom.data(), counts.data(), tile_base.data(), nbr.data()};
	std::memcpy(k.ptr, ptrs, sizeof(ptrs));
	k.S = S;
	k.S.step = 0;
	const uint8_t* kb = reinterpret_cast<const uint8_t*>(&k);
	std::vector<uint8_t> key(kb, kb + sizeof(k));
	for (const SegmentGraph& g : graphs)
		if (g.key == key)
			return g.exec;
	if (!capture_stream)
		MMD_HIP(hipStreamCreateWithFlags(&capture_stream, hipStreamNonBlocking));
	step_word.resize(1);
	const StepKernel kern = reinterpret_cast<StepKernel>(const_cast<void*>(kernel));
	const NbrList L{counts.data(), tile_base.data(), nbr.data()};
	MMD_HIP(hipStreamBeginCapture(capture_stream, hipStreamCaptureModeThreadLocal));
	hipError_t err = hipSuccess;
	for (uint64_t j = 0; j < count && err == hipSuccess; ++j) {
		StepParams Sj = S;
		Sj.step = uint32_t(j);
		const int c = (cur + int(j & 1)) & 1;
		kern<<<grid, sh.block, sh.lds, capture_stream>>>(
			pos[c].data(), pos[1 - c].data(), mom.data(), force.data(), total, rep_of_slot.data(),
			reinterpret_cast<const RepGeom*>(geom.data()), L, reinterpret_cast<const BatchConsts*>(consts.data()),
			knots.data(), Sj, base_seed, 0, step_word.data(), sh.split, sh.knot_words);
		err = hipGetLastError();
	}
	hipGraph_t graph = nullptr;
	const hipError_t end = hipStreamEndCapture(capture_stream, &graph);
	if (err != hipSuccess || end != hipSuccess) {
		if (graph)
			(void)hipGraphDestroy(graph);
		raise(MARSMD_ERR_DEVICE, std::string("batch: capturing a step segment failed: ") +
								  hipGetErrorString(err != hipSuccess ? err : end));
	}
	hipGraphExec_t exec = nullptr;
	const hipError_t inst = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
	(void)hipGraphDestroy(graph);
	if (inst != hipSuccess)
		raise(MARSMD_ERR_DEVICE, std::string("batch: instantiating a step segment failed: ") + hipGetErrorString(inst));
	if (graphs.size() >= 8) { // segments of other lengths or of an older list
		(void)hipGraphExecDestroy(graphs.front().exec);
		graphs.erase(graphs.begin());
	}
	graphs.push_back(SegmentGraph{std::move(key), exec});
	return exec;
}

void BatchImpl::launch_steps(const marsmd_run_params& P, uint64_t first, uint64_t count, bool store,
							 hipStream_t s) {
	const bool bd = P.integrator == MARSMD_INTEGRATOR_BROWNIAN;
	const bool energy = count == 1 && P.energy_period > 0 && first % P.energy_period == 0;
	const bool an = (tables->enabled & kAnalyticTerms) != 0;
	const StepShape sh = step_shape();
	const StepKernel kern = pick_b_step(sh.split > 0, bd, energy, an);
	const unsigned grid = step_grid(reinterpret_cast<const void*>(kern), sh);
	StepParams S{};
	S.cut_d = cutoff_threshold(P.cutoff > 0.0f ? P.cutoff * P.cutoff : 0.0f);
	S.dt = P.timestep;
	S.kT = P.kT;
	S.ctr = 0;
	S.scheme = MARSMD_INTERP_LINEAR;
	S.has_grids = 0;
	S.deferred = deferred_kick ? 1 : 0;
	// a segment replays when the launches differ only in their step: no forces kept,
	// and the deferred-kick state settled (Langevin defers from its first step on)
	const bool replay = use_graph && count >= 2 && !store && (bd || deferred_kick);
	hipGraphExec_t exec = replay ? segment_graph(reinterpret_cast<const void*>(kern), grid, sh, S, count) : nullptr;
	if (timing) {
		while (timing_events.size() < timing_used + 2) {
			hipEvent_t e;
			MMD_HIP(hipEventCreate(&e));
			timing_events.push_back(e);
		}
		MMD_HIP(hipEventRecord(timing_events[timing_used], s));
	}
	if (exec) {
		k_b_set_word<<<1, 64, 0, s>>>(step_word.data(), uint32_t(first));
		MMD_LAUNCH_CHECK();
		MMD_HIP(hipGraphLaunch(exec, s));
		if (count & 1)
			cur = 1 - cur;
	} else {
		const NbrList L{counts.data(), tile_base.data(), nbr.data()};
		for (uint64_t j = 0; j < count; ++j) {
			S.step = uint32_t(first + j);
			S.deferred = deferred_kick ? 1 : 0;
			const int keep = store && j + 1 == count ? 1 : 0;
			kern<<<grid, sh.block, sh.lds, s>>>(pos[cur].data(), pos[1 - cur].data(), mom.data(), force.data(), total,
												rep_of_slot.data(), reinterpret_cast<const RepGeom*>(geom.data()), L,
												reinterpret_cast<const BatchConsts*>(consts.data()), knots.data(), S,
												base_seed, keep, nullptr, sh.split, sh.knot_words);
			MMD_LAUNCH_CHECK();
			if (!bd)
				deferred_kick = true;
			cur = 1 - cur;
		}
	}
	if (timing) {
		MMD_HIP(hipEventRecord(timing_events[timing_used + 1], s));
		timing_used += 2;
		timing_steps.push_back(count);
	}
}

void BatchImpl::run(const marsmd_run_params& P, uint64_t first_step, uint64_t num_steps, hipStream_t s) {
	if (P.integrator != MARSMD_INTEGRATOR_BROWNIAN && P.integrator != MARSMD_INTEGRATOR_LANGEVIN)
		raise(MARSMD_ERR_VALUE, "Unsupported integrator type: " + std::to_string(P.integrator));
	const uint64_t rp = P.reorder_period > 0 ? uint64_t(P.reorder_period) : P.rebuild_period;
	const uint64_t last = first_step + num_steps;
	// a step needs the host when it may reorder or rebuild or sums energies
	auto host_step = [&](uint64_t step) {
		return (rp > 0 && (step - 1) % rp == 0) || P.rebuild_period == 0 ||
			   (step - 1) % P.rebuild_period == 0 || (P.energy_period > 0 && step % P.energy_period == 0);
	};
	uint64_t step = first_step + 1;
	while (step <= last) {
		// maybe_reorder (ReorderManager.cpp:8-25): the reorder forces a rebuild
		const bool reorder = rp > 0 && (step - 1) % rp == 0 && prepared;
		prepared = true;
		// rebuild policy (Patch.cpp:85-121), over all replicas
		bool rebuild = !built || reorder || built_cutoff != P.pairlist_cutoff;
		if (!rebuild && (P.rebuild_period == 0 || (step - 1) % P.rebuild_period == 0)) {
			const float skin = P.pairlist_cutoff - P.cutoff;
			rebuild = P.rebuild_period == 0 || skin <= 0.0f || needs_rebuild(skin, s);
		}
		if (rebuild)
			build(P.pairlist_cutoff, reorder, s);
		launch_steps(P, step, 1, step == last, s);
		++step;
		// then every step up to the next one the host decides on, and not the run's last
		// (which keeps its forces): the same list, no reorder, no energies
		uint64_t end = step;
		while (end < last && !host_step(end))
			++end;
		if (end > step) {
			launch_steps(P, step, end - step, false, s);
			step = end;
		}
	}
}

void BatchImpl::autotune(const marsmd_run_params& P, uint64_t first_step, uint64_t num_steps, hipStream_t s,
						 double* best_ms) {
	// candidates: workgroups per CU from the occupancy down, each with and without
	// segment replay; results do not depend on them (each particle's sums are
	// taken in one order, and a replay launches the same kernels with the same arguments)
	const StepShape sh = step_shape();
	const bool bd = P.integrator == MARSMD_INTEGRATOR_BROWNIAN;
	const bool an = (tables->enabled & kAnalyticTerms) != 0;
	const int occ = step_occupancy(reinterpret_cast<const void*>(pick_b_step(sh.split > 0, bd, false, an)), sh);
	std::vector<int> per_cu = {occ};
	for (int v : {occ - 1, occ / 2, 1})
		if (v >= 1 && std::find(per_cu.begin(), per_cu.end(), v) == per_cu.end())
			per_cu.push_back(v);
	struct Cand {
		int bpc;
		bool graph;
		double ms = 1e300;
	};
	std::vector<Cand> cands;
	for (int v : per_cu)
		for (bool g : {false, true})
			cands.push_back(Cand{v, g});
	const bool was_timing = timing;
	const uint64_t passes = 2;
	const uint64_t chunk = num_steps / (passes * cands.size());
	uint64_t step = first_step;
	if (chunk >= 2) {
		for (uint64_t pass = 0; pass < passes; ++pass)
			for (Cand& c : cands) {
				set_launch(c.bpc, c.graph);
				set_kernel_timing(true);
				run(P, step, chunk, s);
				step += chunk;
				// the runs of steps without host decisions; every launch if there are none
				double ms = 0.0, ms_all = 0.0;
				uint64_t n = 0, n_all = 0;
				for (size_t k = 0; k + 1 < timing_used; k += 2) {
					MMD_HIP(hipEventSynchronize(timing_events[k + 1]));
					float t = 0.0f;
					MMD_HIP(hipEventElapsedTime(&t, timing_events[k], timing_events[k + 1]));
					const uint64_t steps = timing_steps[k / 2];
					ms_all += t;
					n_all += steps;
					if (steps >= 2) {
						ms += t;
						n += steps;
					}
				}
				const double per = n ? ms / double(n) : (n_all ? ms_all / double(n_all) : 1e300);
				c.ms = std::min(c.ms, per);
			}
	}
	const Cand* best = &cands.front();
	for (const Cand& c : cands)
		if (c.ms < best->ms)
			best = &c;
	set_launch(best->bpc, best->graph);
	set_kernel_timing(was_timing);
	if (step < first_step + num_steps)
		run(P, step, first_step + num_steps - step, s);
	*best_ms = best->ms < 1e300 ? best->ms : 0.0;
}

void BatchImpl::set_cells(const marsmd_batch_cells& c) {
	for (int b = 0; b < kBatchBuckets; ++b) {
		if (c.home_target[b] < 1 || c.home_target[b] > 4096)
			raise(MARSMD_ERR_VALUE, "batch: home_target must be in [1, 4096]");
		if (c.fine_offset[b] < 1 || c.fine_offset[b] > 4)
			raise(MARSMD_ERR_VALUE, "batch: fine_offset must be in [1, 4]");
	}
	for (int b = 0; b < kBatchBuckets; ++b) {
		cell_target[size_t(b)] = c.home_target[b];
		cell_fine[size_t(b)] = c.fine_offset[b];
	}
}

void BatchImpl::get_cells(marsmd_batch_cells* c) const {
	for (int b = 0; b < kBatchBuckets; ++b) {
		c->home_target[b] = cell_target[size_t(b)];
		c->fine_offset[b] = cell_fine[size_t(b)];
	}
}

double BatchImpl::walk_ms(hipStream_t s) {
	std::vector<uint8_t> gh;
	std::vector<uint32_t> items;
	uint64_t ft = 0, ht = 0;
	plan_geometry(built_cutoff, gh, items, ft, ht, s);
	t_geom.resize(R * sizeof(RepGeom));
	MMD_HIP(hipMemcpyAsync(t_geom.data(), gh.data(), R * sizeof(RepGeom), hipMemcpyHostToDevice, s));
	t_items.resize(R + 1);
	MMD_HIP(hipMemcpyAsync(t_items.data(), items.data(), 4 * (R + 1), hipMemcpyHostToDevice, s));
	t_cells.resize(ft + ht);
	uint2* const fine = t_cells.data();
	uint2* const home = fine + ft;
	t_counts.resize(total);
	const uint64_t storage = (total + 63) / 64 * 64 * uint64_t(cap);
	t_nbr.resize(std::max<uint64_t>(storage, 1));
	if (!t_events[0]) {
		MMD_HIP(hipEventCreate(&t_events[0]));
		MMD_HIP(hipEventCreate(&t_events[1]));
	}
	const RepGeom* gd = reinterpret_cast<const RepGeom*>(t_geom.data());
	const uint64_t nitems = items[R];
	const unsigned groups = unsigned((nitems + kHomeWaves - 1) / kHomeWaves);
	const unsigned grid = std::max(8u, (groups + 7u) / 8u * 8u);
	MMD_HIP(hipEventRecord(t_events[0], s));
	fill_u32(reinterpret_cast<uint32_t*>(fine), 0u, 2 * (ft + ht), s);
	k_b_cell_ranges<<<grid_for(total, 256), 256, 0, s>>>(codes.data(), total, rep_of_slot.data(), gd, fine, home,
														 nullptr);
	MMD_LAUNCH_CHECK();
	k_b_walk<<<grid, 256, 0, s>>>(gd, t_items.data(), uint32_t(R), uint32_t(nitems), snap.data(), home, fine,
								  built_cutoff * built_cutoff, cap, stencils.data(), t_counts.data(), t_nbr.data());
	MMD_LAUNCH_CHECK();
	MMD_HIP(hipEventRecord(t_events[1], s));
	MMD_HIP(hipEventSynchronize(t_events[1]));
	float ms = 0.0f;
	MMD_HIP(hipEventElapsedTime(&ms, t_events[0], t_events[1]));
	return double(ms);
}

void BatchImpl::autotune_cells(const marsmd_run_params& P, uint64_t first_step, uint64_t num_steps, hipStream_t s,
							   double* walk_out) {
	uint64_t step = first_step;
	if (!built && num_steps > 0) { // the first build
		run(P, step, 1, s);
		++step;
	}
	if (!built)
		raise(MARSMD_ERR_RUNTIME, "batch: the cell autotuner needs a first build (num_steps >= 1)");
	std::vector<int> present;
	for (uint64_t r = 0; r < R; ++r) {
		const int b = batch_size_bucket(count[r]);
		if (std::find(present.begin(), present.end(), b) == present.end())
			present.push_back(b);
	}
	std::sort(present.begin(), present.end());
	// the fastest of three timings of one configuration
	const auto measure = [&]() {
		double best = 1e300;
		for (int k = 0; k < 3; ++k)
			best = std::min(best, walk_ms(s));
		return best;
	};
	(void)walk_ms(s); // warm the scratch buffers and stencils
	double best = measure();
	const int targets[] = {8, 16, 24, 48, 96};
	const int fines[] = {1, 2, 3};
	// one bucket at a time, the others held; a candidate must beat the incumbent by 1%
	for (int b : present) {
		int bt = cell_target[size_t(b)], bf = cell_fine[size_t(b)];
		for (int t : targets)
			for (int f : fines) {
				if (t == bt && f == bf)
					continue;
				cell_target[size_t(b)] = t;
				cell_fine[size_t(b)] = f;
				const double ms = measure();
				if (ms < 0.99 * best) {
					best = ms;
					bt = t;
					bf = f;
				}
			}
		cell_target[size_t(b)] = bt;
		cell_fine[size_t(b)] = bf;
	}
	*walk_out = best < 1e300 ? best : 0.0;
	if (step < first_step + num_steps)
		run(P, step, first_step + num_steps - step, s);
}

void BatchImpl::finish_deferred_kick(float dt, hipStream_t s) {
	if (!deferred_kick)
		return;
	deferred_kick = false;
	k_b_last_update<<<grid_for(total, 256), 256, 0, s>>>(mom.data(), force.data(), total, dt);
	MMD_LAUNCH_CHECK();
}

const int32_t* BatchImpl::neighbor_pairs(uint64_t replica, uint64_t* np_out, hipStream_t s) {
	if (replica >= R)
		raise(MARSMD_ERR_VALUE, "batch: replica index out of range");
	if (!built)
		raise(MARSMD_ERR_RUNTIME, "batch: no pairlist has been built yet");
	const uint64_t n = count[replica], slot0 = off[replica];
	half_counts.resize(n + 1);
	half_offsets.resize(n + 1);
	scan_scratch.resize(scan_scratch_bytes(n + 1));
	const NbrList L{counts.data(), tile_base.data(), nbr.data()};
	uint32_t np = 0;
	if (n) {
		k_b_half_counts<<<grid_for(n, 256), 256, 0, s>>>(L, slot0, n, half_counts.data());
		MMD_LAUNCH_CHECK();
		exclusive_scan_u32(half_counts.data(), half_offsets.data(), n, scan_scratch.data(), s);
		MMD_HIP(hipMemcpyAsync(&np, half_offsets.data() + n, 4, hipMemcpyDeviceToHost, s));
		MMD_HIP(hipStreamSynchronize(s));
		pairs.resize(2 * uint64_t(np) + 2);
		k_b_write_pairs<<<grid_for(n, 256), 256, 0, s>>>(L, pos[cur].data(), slot0, n, half_offsets.data(),
														 pairs.data());
		MMD_LAUNCH_CHECK();
	} else {
		pairs.resize(2);
	}
	*np_out = np;
	return pairs.data();
}

void BatchImpl::set_kernel_timing(bool enable) {
	timing = enable;
	timing_used = 0;
	timing_steps.clear();
}

void BatchImpl::kernel_timing(double* total_ms, uint64_t* steps) {
	double sum = 0.0;
	uint64_t n = 0;
	for (size_t k = 0; k + 1 < timing_used; k += 2) {
		MMD_HIP(hipEventSynchronize(timing_events[k + 1]));
		float ms = 0.0f;
		MMD_HIP(hipEventElapsedTime(&ms, timing_events[k], timing_events[k + 1]));
		sum += double(ms);
		n += timing_steps[k / 2];
	}
	*total_ms = sum;
	*steps = n;
}

} // namespace mmd
