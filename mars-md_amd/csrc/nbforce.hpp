// nbforce.hpp — the nonbonded pair term over the wave-tiled neighbour list, shared by
// the Patch kernels (patch.hip), the replica batch (batch.hip) and force matching
// (fm.hip).
#pragma once

#include "analytic.hpp"
#include "pairlist.hpp"

namespace mmd {

constexpr int kMaxTables = 32;
constexpr int kLdsKnots = 15360; // 60 KB of table knots staged in LDS

struct NbTables {
	int num_tables;
	int num_types;
	uint32_t enabled;
	int lds; // knots staged in LDS
	int total_knots;
	float start[kMaxTables];
	float step_inv[kMaxTables];
	int size[kMaxTables];
	int offset[kMaxTables];
	uint32_t tag[MARSMD_MAX_TYPES * MARSMD_MAX_TYPES];
	PairCoeffs coef; // read by the analytical terms only
};

// What a pair term reads besides positions and knots, staged in LDS once per
// workgroup: parameters indexed per lane (table index, particle type) would otherwise
// be vector loads from the kernel-argument block on every pair.
struct NbLds {
	uint32_t tag[MARSMD_MAX_TYPES * MARSMD_MAX_TYPES]; // [x type << 4 | y type]
	float4 tab[kMaxTables];        // {start, step_inv, size, offset} (size, offset as int bits)
	float4 coef[MARSMD_MAX_TYPES]; // {charge, softcore radius, softcore eps, 0}
	// per type pair: {start, step_inv, last, offset} of its enabled table, last = size - 2
	// (int bits; -2 when the pair has no enabled tabulated term): one read per pair on
	// the tabulated-only path. Indexed from one end of the pair, both orientations:
	// [o << 8 | own type << 4 | other type], o = 1 when the own end is the pair's x
	// (lower canonical index), so no type selects are needed per pair
	float4 pairtab[2 * MARSMD_MAX_TYPES * MARSMD_MAX_TYPES];
};

__device__ __forceinline__ uint32_t fb(float f) { return __float_as_uint(f); }

// One pair term on slot t (PairNonbondedComputer, Pairwise.h:184-305) in canonical
// orientation: r = wrap_diff(pos[higher canon] - pos[lower canon]), the lower takes -F.
// ANALYTIC adds the analytical terms enabled by the pair's tag; without it only the
// tabulated term is evaluated (the kernels are instantiated per case, so the
// tabulated-only path carries none of the analytical code). `knots` points into LDS or
// global memory, as the caller's instantiation says: a pointer that might be either
// would be read with flat loads, whose waits also drain the position gathers in flight.
// Calls add(x, y, z, e) with what the pair adds to the slot's force and energy, unless it is
// skipped (without ANALYTIC a skipped pair adds +-0, which leaves the sums' bits unchanged:
// they start at +0 and can never become -0). The additions stand in the analytical terms'
// branches: as a value merged behind them they cost the one-lane steps 9-12 VGPRs, at 5
// waves 14-42 spilled ones instead of 4-9 (the batch's 54 instead of 16-21). Step, us, merged
// and in the branches: 300k beads 139 and 137, with energies 153.5 and 147; 1M 379 and 376,
// 417 and 404; 16 replicas of 40k 261 and 245, 280 and 268.
template<bool ANALYTIC, class Add>
__device__ __forceinline__ void nb_pair_add(const float4& p, uint32_t tt, const float4& q, const NbTables& T,
											const float* __restrict__ knots, const NbLds& S, const DevBox& box,
											float cut_d, bool energy, Add&& add) {
	const uint32_t mj = fb(q.w);
	const uint32_t tj = meta_type(mj);
	// ct < cj, from the meta words (canonical index in the high bits; a pad entry is the
	// slot itself: equal words, not lower)
	const bool t_is_x = fb(p.w) < mj;
	const float4 px = t_is_x ? p : q;
	const float4 py = t_is_x ? q : p;
	const uint32_t tx = t_is_x ? tt : tj;
	const uint32_t ty = t_is_x ? tj : tt;
	if constexpr (!ANALYTIC) {
		// Tabulated term only, without branches: every quantity is computed for every
		// pair (table reads clamped into the table) and a pair that the reference would
		// skip adds +-0, which leaves the sums' bits unchanged (they start at +0 and can
		// never become -0). Straight-line code lets the four pairs of a group overlap
		// their LDS reads.
		const float4 tp = S.pairtab[(t_is_x ? 256u : 0u) + ((tt << 4) | tj)];
		const int last = __float_as_int(tp.z); // table size - 2
		const bool tab = last >= 0;
		// py - px is q - p or its negation, exactly (rounding is sign-symmetric)
		const float dx = q.x - p.x, dy = q.y - p.y, dz = q.z - p.z;
		const float3 r = wrap_diff_uniform(box, t_is_x ? make_float3(dx, dy, dz) : make_float3(-dx, -dy, -dz));
		// correctly rounded (d picks the table bin); distances below 1e-6 are skipped
		const float d = sqrt_rn_nonneg(len2(r));
		// the unit vector only scales the force: the hardware reciprocal (1 ulp) in place
		// of the correctly rounded division moves the force by ~1e-7 relative
		// (floored at 1e-6, so the zero-distance pads give a finite product with +0)
		const float inv = __builtin_amdgcn_rcpf(fmaxf(d, 1e-6f));
		// the pairs the reference evaluates (d >= 1e-6, within the cutoff); at d == 1e-6
		// exactly its unit vector is 0, so the force needs d > 1e-6
		const bool in_cut = tab && !(d > cut_d);
		// TabulatedPotential::compute (TabulatedPotential.h:19-52), non-periodic; a pair
		// without the term reads knots 0 and 1 (last -2 clamps the bin to 0) and adds 0
		const float* pot = knots + __float_as_int(tp.w);
		float w = (d - tp.x) * tp.y;
		const int home = int(floorf(w));
		w = w - float(home);
		const int hc = max(min(home, last), 0);
		const float U0 = pot[hc];
		const float U1 = pot[hc + 1];
		const float dU = U1 - U0;
		const bool beyond = home > last;
		// (the reference adds these to a +0 accumulator; without that add a -0 can reach
		// the sums only as a product, and adding -0 to a sum leaves its bits unchanged)
		const float fm = beyond ? 0.0f : -dU * tp.y;
		const float en = beyond ? U1 : dU * w + U0;
		// the lower canonical end takes -F: -(fm u) = (-fm) u exactly
		// (force over distance once, then per axis: the product rounds in another order
		// than fm * (r / d), a relative change of about 1e-7)
		const float g = ((in_cut && d > 1e-6f) ? (t_is_x ? -fm : fm) : 0.0f) * inv;
		add(g * r.x, g * r.y, g * r.z, energy && in_cut && !(d < 1e-6f) ? en * 0.5f : 0.0f);
		return;
	}
	const uint32_t tag = S.tag[(tx << 4) | ty];
	const uint32_t terms = tag & T.enabled;
	if (terms == 0u)
		return;
	const float3 r = wrap_diff(box, sub3(py, px));
	const float r2 = len2(r);
	const float d = sqrtf(r2);
	float ux = 0.0f, uy = 0.0f, uz = 0.0f;
	if (d > 1e-6f) {
		const float inv = 1.0f / d;
		ux = inv * r.x;
		uy = inv * r.y;
		uz = inv * r.z;
	}
	if (d < 1e-6f || d > cut_d)
		return;
	float fm = 0.0f, en = 0.0f;
	if (ANALYTIC && (terms & kAnalyticTerms)) {
		const float4 cx = S.coef[tx], cy = S.coef[ty];
		analytic_terms(terms, d, r2, cx.x, cy.x, cx.y, cy.y, cx.z, cy.z, T.coef.prm, fm, en);
	}
	if (terms & MARSMD_PAIR_TERM_TABULATED) {
		const float4 tp = S.tab[tag >> MARSMD_PAIR_TABLE_SHIFT];
		const FE v = table_compute(d, knots + __float_as_int(tp.w), __float_as_int(tp.z), tp.x, tp.y, false);
		fm += v.f;
		en += v.e;
	}
	const float gx = fm * ux, gy = fm * uy, gz = fm * uz;
	const float half = energy ? en * 0.5f : 0.0f;
	if (t_is_x)
		add(-gx, -gy, -gz, half);
	else
		add(gx, gy, gz, half);
}
template<bool ANALYTIC>
__device__ __forceinline__ float4 nb_pair_term(const float4& p, uint32_t tt, const float4& q, const NbTables& T,
											   const float* __restrict__ knots, const NbLds& S, const DevBox& box,
											   float cut_d, bool energy) {
	float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
	nb_pair_add<ANALYTIC>(p, tt, q, T, knots, S, box, cut_d, energy,
						  [&](float x, float y, float z, float e) { v = make_float4(x, y, z, e); });
	return v;
}
template<bool ANALYTIC>
__device__ __forceinline__ void nb_pair(const float4& p, uint32_t tt, const float4& q, const NbTables& T,
										const float* __restrict__ knots, const NbLds& S, const DevBox& box,
										float cut_d, bool energy, float4& sum) {
	nb_pair_add<ANALYTIC>(p, tt, q, T, knots, S, box, cut_d, energy, [&](float x, float y, float z, float e) {
		sum.x += x;
		sum.y += y;
		sum.z += z;
		if (energy)
			sum.w += e;
	});
}

// Position record of slot j, addressed by a 32-bit byte offset from the array base
// (scalar base + vector offset addressing; every caller holds fewer than 2^28 slots).
__device__ __forceinline__ float4 pos_at(const float4* __restrict__ pos, uint32_t j) {
	return *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(pos) + (j << 4));
}

// Sum of the nonbonded pair terms on slot t over its neighbour list, in list order.
// A lane's list is read in groups of 4 indices (one 16-byte load) and pipelined three
// deep: while group g is evaluated, the positions of group g+1 and the indices of
// group g+2 are in flight. The padding entries of a row are t itself (skipped as d = 0).
template<bool ANALYTIC = false>
__device__ __forceinline__ float4 nb_force_list(uint32_t t, const float4& p, const float4* __restrict__ pos,
											   const NbrList& L, const NbTables& T, const float* __restrict__ knots,
											   const NbLds& S, const DevBox& box, float cut_d, bool energy) {
	const uint32_t mt = fb(p.w);
	const uint32_t tt = meta_type(mt);
	float4 sum = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
	const uint32_t ng = (L.count[t] + 3u) >> 2;
	if (ng == 0)
		return sum;
	const uint4* __restrict__ row = reinterpret_cast<const uint4*>(L.nbr + L.tile_base[t >> 6]) + (t & 63u);
	// two register sets (a, b) take turns: while one group is evaluated the positions
	// of the next are in flight in the other set, and the indices of the one after;
	// each index register is reloaded in place once its gathers are issued
	uint4 ja = row[0];
	float4 a0 = pos_at(pos, ja.x), a1 = pos_at(pos, ja.y), a2 = pos_at(pos, ja.z), a3 = pos_at(pos, ja.w);
	float4 b0, b1, b2, b3;
	uint4 jb = ng > 1 ? row[64] : ja;
	for (uint32_t g = 0;; g += 2) {
		if (g + 1 < ng) {
			b0 = pos_at(pos, jb.x);
			b1 = pos_at(pos, jb.y);
			b2 = pos_at(pos, jb.z);
			b3 = pos_at(pos, jb.w);
			if (g + 2 < ng)
				ja = row[uint64_t(g + 2) * 64u];
		}
		nb_pair<ANALYTIC>(p, tt, a0, T, knots, S, box, cut_d, energy, sum);
		nb_pair<ANALYTIC>(p, tt, a1, T, knots, S, box, cut_d, energy, sum);
		nb_pair<ANALYTIC>(p, tt, a2, T, knots, S, box, cut_d, energy, sum);
		nb_pair<ANALYTIC>(p, tt, a3, T, knots, S, box, cut_d, energy, sum);
		if (g + 1 >= ng)
			break;
		if (g + 2 < ng) {
			a0 = pos_at(pos, ja.x);
			a1 = pos_at(pos, ja.y);
			a2 = pos_at(pos, ja.z);
			a3 = pos_at(pos, ja.w);
			if (g + 3 < ng)
				jb = row[uint64_t(g + 3) * 64u];
		}
		nb_pair<ANALYTIC>(p, tt, b0, T, knots, S, box, cut_d, energy, sum);
		nb_pair<ANALYTIC>(p, tt, b1, T, knots, S, box, cut_d, energy, sum);
		nb_pair<ANALYTIC>(p, tt, b2, T, knots, S, box, cut_d, energy, sum);
		nb_pair<ANALYTIC>(p, tt, b3, T, knots, S, box, cut_d, energy, sum);
		if (g + 2 >= ng)
			break;
	}
	return sum;
}

// The same sum with each slot's row dealt to m = 2^split adjacent lanes (4 or 8; this one's
// index `sub`): a round takes m groups of 4 entries, lane k evaluates group k's
// pairs and leaves their terms in LDS, and then four lanes per slot, one a component, add
// the round's 4 m terms to their running sums one by one. The additions are
// nb_force_list's, in its order, so the bits do not depend on the split. A row of g groups
// takes ceil(g / m) rounds instead of g, which is what bounds a step whose slots do not
// fill the chip; the serial additions are about a quarter of a round's instructions
// (handing the sum from lane to lane instead: the step of 10k beads with 115 neighbours
// 14.6 us instead of 11.2).
// log2 of the lanes that share a slot's row (0: one), from the slots, the longest row and
// the entries of all rows: 8 lanes up to 2^15 slots and 4 up to 7 2^14 (7 waves on each of
// the chip's 1024 SIMDs), of which each has a group of the longest row to take; with long
// rows (12 groups on average) beyond that while a lane keeps 6 groups of the longest one,
// whose tail bounds uneven rows. Step kernel, us at 1, 4, 8, 16 lanes: 10k beads of 115
// neighbours 39, 16, 11.2, 11.4; 60k of 22 (trilinear grid) 18, 14.6, 18, 27; 100k polymer
// beads 92, 44, 41, 45; 100k of 22 (tricubic) 32, 27, 29, 47; 120k of 22 (trilinear) 23, 24,
// 32; 200k of 108 74, 64, 67, 77; 1M of 22 (tricubic) 140, 165, 213.
inline uint32_t row_split(uint64_t n, uint32_t max_neighbors, uint64_t entries) {
	const uint32_t groups = (max_neighbors + 3u) >> 2;
	const bool long_rows = entries >= 48 * n;
	for (uint32_t s : {3u, 2u})
		if ((groups >> s) >= 1 && (n <= (s == 3 ? 1u << 15 : 7u << 14) || (long_rows && (groups >> s) >= 6)))
			return s;
	return 0;
}

struct RowHead { // what a lane reads before its first pair term
	float4 p;
	uint32_t ng;
	const uint4* row;
	uint4 j, self; // its first group's entries; the slot itself four times
};
// The head of lane position `at`: its slot is lane_slot[at] (NULL: the position itself) and
// its row is L's at the position (`placed`: rows in lane order) or at the slot. A position
// past the end stands in as the last one with an empty row.
__device__ __forceinline__ RowHead row_head(uint32_t at, uint32_t n, uint32_t sub, const float4* __restrict__ pos,
											const NbrList& L, const uint32_t* __restrict__ lane_slot = nullptr,
											bool placed = true) {
	const uint32_t l = min(at, n - 1u);
	const uint32_t t = lane_slot ? lane_slot[l] : l, r = placed ? l : t;
	RowHead h;
	h.p = pos[t];
	h.ng = at < n ? (L.count[r] + 3u) >> 2 : 0u;
	h.row = reinterpret_cast<const uint4*>(L.nbr + L.tile_base[r >> 6]) + (r & 63u);
	h.self = make_uint4(t, t, t, t);
	h.j = h.self;
	if (sub < h.ng)
		h.j = h.row[uint64_t(sub) * 64u];
	return h;
}
// Floats of LDS per wave: three components (with energies four) of 64 / m rows of 4 m terms
// (and 4 spare against bank conflicts).
constexpr uint32_t split_terms(bool energy) { return (energy ? 4u : 3u) * (256u + 64u); }
// The wave's slots' sums: lane 4 s + c (s < 64 >> split) returns component c of the wave's
// slot s (x, y, z, energy). Called by every lane of the wave.
template<bool ANALYTIC>
__device__ __forceinline__ float nb_force_split(const RowHead& h, uint32_t sub, uint32_t split,
												const float4* __restrict__ pos, const NbTables& T,
												const float* __restrict__ knots, const NbLds& S, const DevBox& box,
												float cut_d, bool energy, float* terms) {
	const float4 p = h.p;
	const uint32_t mt = fb(p.w);
	const uint32_t tt = meta_type(mt);
	const uint32_t m = 1u << split, ng = h.ng, lane = threadIdx.x & 63u;
	const uint32_t row = 4u * m + 4u, comp = (64u >> split) * row;
	float* const mine = terms + (lane >> split) * row + 4u * sub;
	const uint32_t slot = lane >> 2, c = lane & 3u;
	const bool adds = slot < (64u >> split) && (c < 3u || energy);
	const float* const theirs = terms + c * comp + slot * row;
	float sum = 0.0f;
	uint4 j = h.j; // past the row: the slot itself, whose terms are +0
	for (uint32_t g0 = 0; __ballot(g0 < ng) != 0; g0 += m) {
		const float4 q0 = pos_at(pos, j.x), q1 = pos_at(pos, j.y), q2 = pos_at(pos, j.z), q3 = pos_at(pos, j.w);
		j = h.self;
		if (g0 + m + sub < ng)
			j = h.row[uint64_t(g0 + m + sub) * 64u];
		const float4 t0 = nb_pair_term<ANALYTIC>(p, tt, q0, T, knots, S, box, cut_d, energy);
		const float4 t1 = nb_pair_term<ANALYTIC>(p, tt, q1, T, knots, S, box, cut_d, energy);
		const float4 t2 = nb_pair_term<ANALYTIC>(p, tt, q2, T, knots, S, box, cut_d, energy);
		const float4 t3 = nb_pair_term<ANALYTIC>(p, tt, q3, T, knots, S, box, cut_d, energy);
		wave_lds_sync(); // (the last round's reads)
		*reinterpret_cast<float4*>(mine) = make_float4(t0.x, t1.x, t2.x, t3.x);
		*reinterpret_cast<float4*>(mine + comp) = make_float4(t0.y, t1.y, t2.y, t3.y);
		*reinterpret_cast<float4*>(mine + 2u * comp) = make_float4(t0.z, t1.z, t2.z, t3.z);
		if (energy)
			*reinterpret_cast<float4*>(mine + 3u * comp) = make_float4(t0.w, t1.w, t2.w, t3.w);
		wave_lds_sync();
		if (adds) {
			for (uint32_t k = 0; k < m; k += 4) {
				float4 v[4];
#pragma unroll
				for (uint32_t u = 0; u < 4; ++u)
					v[u] = *reinterpret_cast<const float4*>(theirs + 4u * (k + u));
#pragma unroll
				for (uint32_t u = 0; u < 4; ++u)
					sum = sum + v[u].x + v[u].y + v[u].z + v[u].w;
			}
		}
	}
	return sum;
}

// Stage the tag matrix, the table parameters and the per-type coefficients in LDS (the
// caller synchronises).
__device__ __forceinline__ void stage_params(const NbTables& T, NbLds& S) {
	const int nt2 = T.num_types * T.num_types;
	for (int i = threadIdx.x; i < nt2; i += blockDim.x) {
		const uint32_t tag = T.tag[i];
		const int x = i / T.num_types, y = i % T.num_types;
		S.tag[(x << 4) | y] = tag;
		const int ti = int(tag >> MARSMD_PAIR_TABLE_SHIFT);
		const float4 v = (tag & T.enabled & MARSMD_PAIR_TERM_TABULATED) && ti < T.num_tables
							 ? make_float4(T.start[ti], T.step_inv[ti], __int_as_float(T.size[ti] - 2),
										   __int_as_float(T.offset[ti]))
							 : make_float4(0.0f, 0.0f, __int_as_float(-2), __int_as_float(0));
		S.pairtab[256 + ((x << 4) | y)] = v; // seen from x
		S.pairtab[(y << 4) | x] = v;         // seen from y
	}
	for (int i = threadIdx.x; i < T.num_tables; i += blockDim.x)
		S.tab[i] = make_float4(T.start[i], T.step_inv[i], __int_as_float(T.size[i]), __int_as_float(T.offset[i]));
	if (T.num_tables == 0 && threadIdx.x == 0) // pairs without the tabulated term read table 0
		S.tab[0] = make_float4(0.0f, 0.0f, __int_as_float(2), __int_as_float(0));
	for (int i = threadIdx.x; i < T.num_types; i += blockDim.x)
		S.coef[i] = make_float4(T.coef.charge[i], T.coef.radius[i], T.coef.eps[i], 0.0f);
}

// Copy the particle-type record into LDS: the integrators and the PMF index it per
// lane (mass, damping, diffusion, charge, grid terms), which from the kernel-argument
// block would be vector loads (the caller synchronises).
__device__ __forceinline__ void stage_types(const marsmd_particle_types& src, marsmd_particle_types& dst) {
	static_assert(sizeof(marsmd_particle_types) % 4 == 0, "4-byte fields");
	const uint32_t* a = reinterpret_cast<const uint32_t*>(&src);
	uint32_t* b = reinterpret_cast<uint32_t*>(&dst);
	for (int i = threadIdx.x; i < int(sizeof(marsmd_particle_types) / 4); i += blockDim.x)
		b[i] = a[i];
}

// Stage table knots (when they fit) and the pair parameters in LDS.
__device__ __forceinline__ void stage_tables(const NbTables& T, const float* __restrict__ knots_g, float* lds_knots,
											 NbLds& S) {
	stage_params(T, S);
	if (T.lds) {
		// 16 bytes a lane (a caller's knots may be only 4-byte aligned: GridRun4), then the rest
		const int quads = T.total_knots >> 2;
		for (int i = threadIdx.x; i < quads; i += blockDim.x) {
			const GridRun4 v = reinterpret_cast<const GridRun4*>(knots_g)[i];
			reinterpret_cast<float4*>(lds_knots)[i] = make_float4(v.v[0], v.v[1], v.v[2], v.v[3]);
		}
		for (int i = 4 * quads + int(threadIdx.x); i < T.total_knots; i += blockDim.x)
			lds_knots[i] = knots_g[i];
	}
	__syncthreads();
}

// nb_force_list with the knots read from LDS when staged there, else from global
// memory: each branch sees one address space.
template<bool ANALYTIC = false>
__device__ __forceinline__ float4 nb_force(uint32_t t, const float4& p, const float4* __restrict__ pos,
										   const NbrList& L, const NbTables& T, const float* lds_knots,
										   const float* __restrict__ knots_g, const NbLds& S, const DevBox& box,
										   float cut_d, bool energy) {
	if (T.lds)
		return nb_force_list<ANALYTIC>(t, p, pos, L, T, lds_knots, S, box, cut_d, energy);
	return nb_force_list<ANALYTIC>(t, p, pos, L, T, knots_g, S, box, cut_d, energy);
}

} // namespace mmd
