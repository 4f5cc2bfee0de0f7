// homewalk.hpp — the home-cell pairlist walk (see k_walk_home) and the reference's
// canonical pair predicate, shared by the pairlist (pairlist.hip) and the replica batch
// (batch.hip).
#pragma once

#include "pairlist.hpp"

#include <algorithm>
#include <cmath>
#include <vector>

namespace mmd {

namespace {

// Not excluded by lo's CSR row or a shared rigid body.
__device__ __forceinline__ bool pair_unexcluded(const marsmd_exclusion_view& ex, const float4& plo,
												const float4& phi) {
	const int a = int(meta_canon(__float_as_uint(plo.w)));
	const int b = int(meta_canon(__float_as_uint(phi.w)));
	if (ex.rigid_body_id) {
		const int body = ex.rigid_body_id[a];
		if (body >= 0 && ex.rigid_body_id[b] == body)
			return false;
	}
	if (ex.offsets && a >= 0 && uint64_t(a) < ex.num_particles) {
		const int e0 = ex.offsets[a], e1 = ex.offsets[a + 1];
		for (int e = e0; e < e1; ++e)
			if (ex.excluded[e] == b)
				return false;
	}
	return true;
}

// Canonical pair predicate of ZOrderCellNeighborKernel for sorted lo < hi
// (ZOrderNeighbor.h:204-221): wrap_diff(pos_hi - pos_lo)^2 <= rc^2, and not excluded.
__device__ __forceinline__ bool pair_predicate(const DevBox& box, float rc2, const marsmd_exclusion_view& ex,
											   const float4& plo, const float4& phi) {
	const float3 dr = wrap_diff(box, sub3(phi, plo));
	return len2(dr) <= rc2 && pair_unexcluded(ex, plo, phi);
}

// ------------------------------------------------------------ home-cell walk
// One wave per home cell: a Morton cell of the home level h, whose particles are
// contiguous in sorted order. The wave enumerates the fine cells (level m = h + s)
// within `reach` fine cells of the home cell whose box can lie within rc of the home
// cell's box (both widened by the quantisation margin, so the test is conservative
// across the periodic seam), 64 cells at a time, spreads their particles over its lanes,
// drops those farther than rc from the bounding box of the home particles, queues the
// rest in LDS and tests each full queue of 64 against the home particles one by one (a
// home particle is wave-uniform: scalar loads). The hits of a home particle are one
// 64-bit mask; each hit lane writes its slot at the row's end plus its rank in the mask.
// Predicate and orientation are k_walk's (the reference's), so the pair set is the
// same; a particle's list is in candidate order. Entries past `cap` are not written
// (the host sees the count and walks again with a larger cap).
//
// What bounds it: with thousands of cells per SIMD the VALU instructions of the tests
// (17 a home particle and 64 candidates), with few the chain of one wave: cell ranges ->
// positions -> queue -> tests. Both want cells with few particles while the chip is not
// full (walk_level), and no search per candidate: the earlier form kept the cells of the
// whole stencil as LDS segments, found each candidate's by bisection (9 dependent LDS
// reads) and appended each home particle's hits in a per-lane loop.
constexpr int kHomeWaves = 4;
// home cells that occupy the chip: four waves on each of its 1024 SIMDs
constexpr double kWalkFill = 4096.0;
// candidates of one 64-cell step mapped to lanes at a time (start bits in LDS)
constexpr uint32_t kWalkWindow = 1024;

struct HomeParams {
	const float4* spos;
	const uint2* home; // {begin, end} of every home cell
	const uint2* fine; // {begin, end} of every fine cell
	uint32_t num_home;
	int h;         // home level
	int s;         // fine level m = h + s
	int reach[3];  // fine cells enumerated beyond the home cell's span
	int full[3];   // periodic axis enumerated whole at the fine level
	float cw[3];   // fine cell width (quantised)
	float margin[3];
	float rc2;
	DevBox box;
	marsmd_exclusion_view ex;
	// the sorted slot of every canonical index, when the exclusion rows are symmetric (a
	// in b's row exactly when b is in a's): a home particle's own row then decides all of
	// its pairs and is read once, as slots; null: each pair looks at its lower end's row
	const uint32_t* ex_slot;
	uint32_t cap;  // entries per slot the uniform tile rows hold
	// When the reference cell grid misses pairs at the periodic seam, only the pairs its
	// stencil reaches are kept: cells (quantised coordinate >> ref_shift) within
	// ref_r per axis, wrapped on periodic axes; ref_full marks axes it enumerates whole.
	int ref_filter;
	int ref_shift;
	int ref_cells;
	int ref_r[3];
	int ref_full[3];
	float dom_lo[3], dom_hi[3];
	// Home-frame prefilter (pre != 0): each candidate is moved by whole box lengths next
	// to the wave's first home particle, and its plain squared distance d2' to a home
	// particle decides the pair when it is below pre_lo2 (in) or above pre_hi2 (out);
	// between the two, which are rc^2 -+ a bound on |d2' - d2| over pairs near the
	// cutoff, the reference's predicate decides. Set only where the box is wide enough
	// for that move to give the minimum image of every pair within the cutoff.
	int pre;
	float pre_lo2, pre_hi2;
	// The fine cells the walk enumerates, when given: their offsets from the home cell's
	// first fine cell (the absolute cell on an axis enumerated whole) that pass the gap
	// test, in enumeration order. In a box periodic on every axis an offset is the Morton
	// code of its three components modulo the cells (stencil_code, added to the home
	// cell's code axis by axis on the interleaved bits, which wraps by itself); else three
	// integers (stencil). Neither: every cell of the reach is enumerated and gap-tested.
	const uint32_t* stencil_code;
	const int4* stencil;
	uint32_t stencil_n;
	// rows in the order of a coarser level's cells: one list of codes for each position of a
	// home cell within its cell of that level, the home code's bits under this mask
	uint32_t stencil_lists;
};

// f(offset) for the fine cells of the walk's enumeration that pass its gap test, as offsets
// (see HomeParams::stencil), until it returns false. The test is the walk's own: per axis
// not enumerated whole, the number of cells between the cell and the home cell's span times
// the cell width, less twice the margin, floored at 0, squared and summed, against rc^2.
template<class F>
inline void for_each_stencil_cell(int h, int s, const int reach[3], const int full[3], const float cw[3],
								  const float margin[3], float rc2, F&& f) {
	const int fine_cells = 1 << (h + s), span = 1 << s;
	int lo[3], nax[3];
	for (int a = 0; a < 3; ++a) {
		lo[a] = full[a] ? 0 : -reach[a];
		nax[a] = full[a] ? fine_cells : span + 2 * reach[a];
	}
	for (int z = 0; z < nax[2]; ++z)
		for (int y = 0; y < nax[1]; ++y)
			for (int x = 0; x < nax[0]; ++x) {
				const int o[3] = {lo[0] + x, lo[1] + y, lo[2] + z};
				float gap2 = 0.0f;
				for (int a = 0; a < 3; ++a) {
					if (full[a])
						continue;
					const int apart = o[a] < 0 ? -o[a] - 1 : (o[a] >= span ? o[a] - span : 0);
					const float g = std::fmax(0.0f, float(apart) * cw[a] - 2.0f * margin[a]);
					gap2 += g * g;
				}
				if (gap2 <= rc2 && !f(make_int4(o[0], o[1], o[2], 0)))
					return;
			}
}
// All of them in Morton order; empty when there are more than max_cells.
inline std::vector<int4> home_stencil(int h, int s, const int reach[3], const int full[3], const float cw[3],
									  const float margin[3], float rc2, size_t max_cells) {
	std::vector<int4> out;
	bool fits = true;
	for_each_stencil_cell(h, s, reach, full, cw, margin, rc2, [&](const int4& o) {
		fits = out.size() < max_cells;
		if (fits)
			out.push_back(o);
		return fits;
	});
	if (!fits)
		return {};
	// Morton order of the offsets: 64 consecutive candidates then come from a compact
	// cluster of cells
	auto key = [](const int4& c) {
		uint64_t k = 0;
		const uint32_t v[3] = {uint32_t(c.x + 1024), uint32_t(c.y + 1024), uint32_t(c.z + 1024)};
		for (int b = 10; b >= 0; --b)
			for (int a = 0; a < 3; ++a)
				k = (k << 1) | ((v[a] >> b) & 1u);
		return k;
	};
	std::stable_sort(out.begin(), out.end(), [&](const int4& a, const int4& b) { return key(a) < key(b); });
	return out;
}
// The walk's home level h and its fine cells' depth s below it. target > 0: the finest
// level below m holding `target` particles per home cell on average, and `offset`. Else
// the library's own choice for n particles (fine cells = home cells, which the candidates'
// bounding-box test prunes more cheaply than a larger stencil does): a level finer while
// its cells hold per_cell particles on average or there are fewer of them than occupy the
// chip (`fill`). Walk times (us; one bead type, cutoff 35): 10k beads at 6.4e-4 per A^3:
// level 2 (156 a cell) 642, 3 (20) 54, 4 (2.4) 21; 60k at 1.25e-4: 3 (117) 240, 4 (15) 31,
// 5 (1.8) 44; 250k: 4 (61) 150, 5 (7.6) 67; 1M: 5 (30) 261, 6 (3.8) 375.
struct WalkLevel {
	int h, s;
};
inline WalkLevel walk_level(uint64_t n, int m, int target, int offset, double fill, uint64_t per_cell = 4) {
	int h = 0;
	if (target > 0) {
		while (h + 1 <= m - 1 && (n >> (3 * (h + 1))) >= uint64_t(target))
			++h;
		return WalkLevel{h, offset};
	}
	while (h + 1 <= m && ((n >> (3 * (h + 1))) >= per_cell || double(uint64_t(1) << (3 * h)) < fill))
		++h;
	return WalkLevel{h, 0};
}
// Rows list a particle's neighbours by the Morton order of their offsets from the
// particle's cell at the level that holds kRowTarget particles per cell on average (by slot
// where that level's stencil wraps onto itself on every axis), whatever level the walk runs
// at: the FP32 sum over a row is then the same bits. Where the cells were set, in boxes with
// an open axis and where that stencil wraps on one or two axes only (which the order level
// walks slowly: a build of 60k in 300 x 300 x 60 at cutoff 28 takes 6360 us there, 1060 here),
// a row is in the order of the walk's own cells.
constexpr int kRowTarget = kCellsTarget, kRowOffset = kCellsOffset;
// cells of a stencil; a larger one is not listed, the walk then tests every cell of its reach
constexpr uint32_t kStencilMax = 8192;

// home levels at which a stencil may have a list for every home cell (512 of a few hundred)
constexpr int kSlotListLevel = 3;

// The cells of a walk: home cells of level h; fine cells of level mf with their enumeration
// (mf < h: one fine cell, the whole box); the lists its stencil has
// (HomeParams::stencil_lists + 1), by_slot: in the order of the cells themselves.
struct WalkGrid {
	int h, mf;
	uint32_t lists;
	bool by_slot;
	int reach[3], full[3];
	float cw[3], margin[3];
};
// The grid for n particles in the Morton domain [lo, hi), periodic where `per`, with build
// levels up to m and the cell configuration given (see walk_level for fill and per_cell;
// own_fill: the fill where rows follow the walk's own cells).
inline WalkGrid walk_grid(uint64_t n, int m, int home_target, int fine_offset, double fill, double own_fill,
						  uint64_t per_cell, const float lo[3], const float hi[3], const bool per[3], double rc,
						  float rc2) {
	const auto extent = [&](int a) { return std::fmax(hi[a] - lo[a], 1e-6f); };
	// fine cells of level `mf` beyond a home cell that cover rc with the seam slack of the
	// quantised top cell, and whether such a stencil wraps onto itself on the axis
	const auto reach_of = [&](int mf, int a) {
		const double W = double(extent(a)) / 1023.0;
		const double need = (rc * (1.0 + 1e-6) + 1e-3) / W + (per[a] ? 1.0 : 0.0);
		return std::max(1, int(std::min(std::ceil(need / double(1024 >> mf)), double(1 << mf))));
	};
	const auto full_of = [&](int h, int mf, int a) {
		return per[a] && (1 << (mf - h)) + 2 * reach_of(mf, a) >= (1 << mf);
	};
	const auto grid_of = [&](const WalkLevel& lv) {
		WalkGrid g{};
		g.h = lv.h;
		g.mf = std::min(10, lv.h + lv.s);
		g.lists = 1;
		for (int a = 0; a < 3; ++a) {
			const double W = double(extent(a)) / 1023.0;
			g.reach[a] = reach_of(g.mf, a);
			g.full[a] = g.mf < g.h || full_of(g.h, g.mf, a) ? 1 : 0;
			g.cw[a] = float(double(extent(a)) * (1024 >> g.mf) / 1023.0);
			g.margin[a] = float(W * 1.001 + 1e-5 * double(extent(a)) + 1e-3);
		}
		return g;
	};
	// whether the home frame of a cell of level h gives minimum images (home_prefilter_band)
	const auto frames = [&](int h) {
		for (int a = 0; a < 3; ++a)
			if (per[a] && !(0.5f * extent(a) > extent(a) / float(1 << h) + float(rc) + 0.01f * extent(a) + 1.0f))
				return false;
		return true;
	};
	// The library's own level. Without the home frame each test takes the whole predicate and
	// no candidate is dropped before, so one level finer where that has the frame and the
	// cells to choose from (a build of 120k in 300 x 300 x 60 at cutoff 25: 2440 -> 725 us),
	// or where its cells still hold 2 particles and leave out some of the box (the same at
	// cutoff 27: 2440 -> 1510 us; 128 replicas of 900 that test all their particles anyway:
	// 340 -> 432 us a step with a build, and with 0.6 particles a cell 512 of 300: 157 -> 288).
	const auto own_level = [&](double f, bool prunes) {
		WalkLevel l = walk_level(n, m, 0, 0, f, per_cell);
		if (l.h < m && !frames(l.h) &&
			((frames(l.h + 1) && double(uint64_t(1) << (3 * l.h)) <= f) || (prunes && (n >> (3 * l.h)) >= 16)))
			++l.h;
		return l;
	};
	if (!cells_auto(home_target, fine_offset))
		return grid_of(walk_level(n, m, home_target, fine_offset, fill, per_cell));
	if (!(per[0] && per[1] && per[2]))
		return grid_of(own_level(own_fill, true));
	const WalkGrid order = grid_of(walk_level(n, m, kRowTarget, kRowOffset, 0.0));
	const int full_axes = order.full[0] + order.full[1] + order.full[2];
	WalkLevel lv = own_level(full_axes == 1 || full_axes == 2 ? own_fill : fill, full_axes < 3);
	WalkGrid g = grid_of(lv);
	if (full_axes == 3) {
		// rows by slot: every particle is a candidate, in slot order; where the walk fills the
		// chip and its stencil does not wrap, the stencil's cells in their own order, a list
		// for each home cell (2000 replicas of 500: a step with its build 488 -> 456 us)
		if (lv.h <= kSlotListLevel && double(uint64_t(1) << (3 * lv.h)) > fill && !g.full[0] && !g.full[1] &&
			!g.full[2]) {
			g.lists = 1u << (3 * lv.h);
			g.by_slot = true;
			return g;
		}
		lv.s = -lv.h;
		return grid_of(lv);
	}
	if (full_axes > 0)
		return g;
	if (g.full[0] || g.full[1] || g.full[2])
		return order; // (offsets and absolute cells mixed)
	if (g.h > order.h) {
		uint64_t reached = 1;
		for (int a = 0; a < 3; ++a)
			reached *= uint64_t(1 << (g.mf - g.h)) + 2u * uint64_t(g.reach[a]);
		uint32_t cells = 0;
		if (reached > kStencilMax)
			for_each_stencil_cell(g.h, g.mf - g.h, g.reach, g.full, g.cw, g.margin, rc2,
								  [&](const int4&) { return ++cells <= kStencilMax; });
		if (cells > kStencilMax)
			return order;
		g.lists = 1u << (3 * (g.h - order.h));
	}
	return g;
}

// An offset of home_stencil as the Morton code of its components modulo 2^level cells.
__host__ __device__ inline uint32_t stencil_offset_code(const int4& o, int level) {
	const uint32_t mask = (1u << level) - 1u;
	return split_by3(uint32_t(o.z) & mask) | (split_by3(uint32_t(o.y) & mask) << 1) |
		   (split_by3(uint32_t(o.x) & mask) << 2);
}

// List b of a stencil in row order: its n offsets (relative to a home cell of `level`) in the
// Morton order of the cells' offsets from the home cell's ancestor of the order level,
// within which the home cell lies at the position whose Morton code is b, as codes
// (stencil_offset_code); by_slot: b is the home cell, and the cells are in their own Morton
// order. Ranks by counting (a few hundred cells; no two keys are equal), by a workgroup with
// `keys` in LDS.
__device__ inline void stencil_list(const int4* __restrict__ offsets, uint32_t n, int level, uint32_t b, bool by_slot,
									uint32_t* __restrict__ codes, uint64_t* keys) {
	const int p[3] = {int(compact_by3(b >> 2)), int(compact_by3(b >> 1)), int(compact_by3(b))};
	for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
		const int4 o = offsets[i];
		if (by_slot) {
			keys[i] = stencil_offset_code(make_int4(p[0] + o.x, p[1] + o.y, p[2] + o.z, 0), level);
			continue;
		}
		const uint32_t v[3] = {uint32_t(p[0] + o.x + 1024), uint32_t(p[1] + o.y + 1024), uint32_t(p[2] + o.z + 1024)};
		keys[i] = (uint64_t(((v[0] >> 10) & 1u) << 2 | ((v[1] >> 10) & 1u) << 1 | ((v[2] >> 10) & 1u)) << 30) |
				  (split_by3(v[0]) << 2 | split_by3(v[1]) << 1 | split_by3(v[2]));
	}
	__syncthreads();
	for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) {
		const uint64_t k = keys[i];
		uint32_t rank = 0;
		for (uint32_t j = 0; j < n; ++j)
			rank += keys[j] < k ? 1u : 0u;
		codes[rank] = stencil_offset_code(offsets[i], level);
	}
}

// The prefilter's band for a domain [lo, hi) whose home cells (level h) have width
// extent / 2^h: false when a periodic axis is too short for the home frame to give
// minimum images (half the box must exceed a home cell plus the cutoff, with slack).
// The bound on |d2' - d2|: the two differences of an axis differ by a few roundings at
// the coordinates' magnitude C (|x| <= C), i.e. a few ulp(C), over |d| <= rc + 1, plus
// the roundings of the squares and sums at rc^2.
inline bool home_prefilter_band(const marsmd_box& box, const float lo[3], const float hi[3], int h, float rc,
								float* lo2, float* hi2) {
	float C = 0.0f;
	for (int a = 0; a < 3; ++a) {
		const float w = (hi[a] - lo[a]) / float(1 << h);
		C = std::fmax(C, std::fmax(std::fabs(lo[a]), std::fabs(hi[a])));
		if (box.periodic[a] && !(0.5f * box.size[a] > w + rc + 0.01f * box.size[a] + 1.0f))
			return false;
		C = std::fmax(C, box.size[a]);
	}
	const float rc2 = rc * rc;
	const float ulp_c = std::nextafter(C, INFINITY) - C;
	const float ulp_r = std::nextafter(rc2 + 1.0f, INFINITY) - (rc2 + 1.0f);
	const float eps = 64.0f * ulp_c * (rc + 1.0f) + 16.0f * ulp_r;
	if (!(eps < 0.01f * rc2))
		return false;
	*lo2 = rc2 - eps;
	*hi2 = rc2 + eps;
	return true;
}

// Whether the reference grid's stencil (BuildCellNeighborsKernel, ZOrderNeighbor.h:
// 55-139) links the cells of a and b. The relation is symmetric, so it is the pair
// set of ZOrderCellNeighborKernel whichever of the two emits.
__device__ __forceinline__ bool in_reference_stencil(const HomeParams& P, const float4& a, const float4& b) {
	const float pa[3] = {a.x, a.y, a.z}, pb[3] = {b.x, b.y, b.z};
	bool clamped = false;
#pragma unroll
	for (int k = 0; k < 3; ++k) {
		if (P.ref_full[k])
			continue;
		const int ca = int(morton_quantize(pa[k], P.dom_lo[k], P.dom_hi[k], clamped) >> P.ref_shift);
		const int cb = int(morton_quantize(pb[k], P.dom_lo[k], P.dom_hi[k], clamped) >> P.ref_shift);
		int d = ca > cb ? ca - cb : cb - ca;
		if (P.box.periodic[k])
			d = min(d, P.ref_cells - d);
		if (d > P.ref_r[k])
			return false;
	}
	return true;
}

__device__ __forceinline__ float bcast_f32(float v, uint32_t lane) {
	return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), int(lane)));
}
template<int CTRL, int ROWS>
__device__ __forceinline__ float dpp_min(float v) {
	const int x = __float_as_int(v);
	return fminf(v, __int_as_float(__builtin_amdgcn_update_dpp(x, x, CTRL, ROWS, 0xf, false)));
}
__device__ __forceinline__ float wave_min(float v) {
	v = dpp_min<0x111, 0xf>(v);
	v = dpp_min<0x112, 0xf>(v);
	v = dpp_min<0x114, 0xf>(v);
	v = dpp_min<0x118, 0xf>(v);
	v = dpp_min<0x142, 0xa>(v);
	v = dpp_min<0x143, 0xc>(v);
	return bcast_f32(v, 63);
}
__device__ __forceinline__ float wave_max(float v) { return -wave_min(-v); }
__device__ __forceinline__ uint32_t bcast_u32(uint32_t v, uint32_t lane) {
	return uint32_t(__builtin_amdgcn_readlane(int(v), int(lane)));
}
// Number of set bits of the wave-uniform mask m below this lane.
__device__ __forceinline__ uint32_t bits_below(uint64_t m) {
	return uint32_t(__builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u)));
}
// Lane i (wave-uniform) of v takes the wave-uniform x.
__device__ __forceinline__ void set_lane(uint32_t& v, uint32_t x, uint32_t i) {
	asm("v_writelane_b32 %0, %1, %2" : "+v"(v) : "s"(x), "{m0}"(i));
}

// LDS of one wave of the walk.
struct WalkLds {
	float4 keep[128];                    // queued candidates {position, slot}
	uint32_t delta[64];                  // slot less index of each nonempty cell's candidates
	uint32_t start[kWalkWindow / 32];    // bit q: a cell's candidates start at index q of the window
};

typedef float walk_f4 __attribute__((ext_vector_type(4)));

// The distance part of the reference's predicate for home particle pi (slot ti) and this
// lane's candidate j: the difference of the higher slot's position less the lower's is
// q - pi or its exact negation (rounding is sign-symmetric).
__device__ __forceinline__ bool pair_within(const HomeParams& P, const walk_f4& pi, uint32_t ti, uint32_t j,
											const float4& q) {
	const float dx = q.x - pi.x, dy = q.y - pi.y, dz = q.z - pi.z;
	return len2(wrap_diff(P.box, j > ti ? make_float3(dx, dy, dz) : make_float3(-dx, -dy, -dz))) <= P.rc2;
}

// The pairs of home particle i with the candidates of one block that pass everything but
// the distance: exclusions and rigid bodies by the lower end's row, the reference's stencil.
__device__ __forceinline__ bool pair_allowed(const HomeParams& P, uint32_t ti, uint32_t j) {
	const float4 pi = P.spos[ti], q = P.spos[j];
	if ((P.ex.rigid_body_id || P.ex.offsets) && !pair_unexcluded(P.ex, j > ti ? pi : q, j > ti ? q : pi))
		return false;
	return !P.ref_filter || in_reference_stencil(P, pi, q); // symmetric in its two ends
}

// The exclusion row of this lane's home particle as slots, the first four in registers.
struct HomeExcl {
	uint32_t begin, count, slot[4];
};
__device__ __forceinline__ HomeExcl home_exclusions(const HomeParams& P, bool valid, const float4& p) {
	HomeExcl x{0u, 0u, {0u, 0u, 0u, 0u}};
	const uint32_t c = meta_canon(__float_as_uint(p.w));
	if (valid && c < P.ex.num_particles) {
		x.begin = uint32_t(P.ex.offsets[c]);
		x.count = uint32_t(P.ex.offsets[c + 1]) - x.begin;
	}
	uint32_t e[4];
#pragma unroll
	for (uint32_t k = 0; k < 4; ++k)
		e[k] = k < x.count ? uint32_t(P.ex.excluded[x.begin + k]) : 0u;
#pragma unroll
	for (uint32_t k = 0; k < 4; ++k)
		x.slot[k] = k < x.count ? P.ex_slot[e[k]] : 0u;
	return x;
}

// The walk's instances. Fast ones: a box periodic on every axis, the prefilter, the
// stencil as codes, no rigid bodies and no reference stencil, without exclusions or with
// symmetric rows (ex_slot); the parameters of the rest would otherwise hold, and spill,
// scalar registers throughout.
constexpr int kWalkPlain = 0, kWalkOwnRows = 1, kWalkGeneral = 2;
__host__ __device__ inline int walk_mode(const HomeParams& P) {
	if (!P.pre || !P.stencil_code || P.ref_filter || P.ex.rigid_body_id || (P.ex.offsets && !P.ex_slot))
		return kWalkGeneral;
	return P.ex.offsets ? kWalkOwnRows : kWalkPlain;
}

// One block of up to 64 candidates (slot j, position q: in the home frame with the
// prefilter; dead lanes have j = ~0 and, with the prefilter, q = +inf) against the wave's
// nh home particles, the first at slot c0: each one's hits go to the end of its row
// (cnt: this lane's home particle's entries so far).
template<int MODE>
__device__ __forceinline__ void test_block(const HomeParams& P, uint32_t c0, uint32_t nh, uint32_t j, float qx,
										   float qy, float qz, const HomeExcl& X, bool own_rows, bool filter,
										   uint32_t& cnt, uint32_t* __restrict__ nbr) {
	const walk_f4 MMD_CONST_AS* home = (const walk_f4 MMD_CONST_AS*)(uint64_t(P.spos) + 16ull * c0);
	const uint32_t self = j - c0; // this candidate's index among the home particles
	// rows: slot t's entries lie 16 t bytes into its tile of 64 slots, the home particles in
	// at most two tiles (byte offsets from the first one's fit 32 bits: a tile's rows do)
	char* const rows = reinterpret_cast<char*>(nbr + uint64_t(c0 >> 6) * 64u * P.cap);
	const uint64_t alive = __ballot(j != ~0u);
	walk_f4 hp[4], hn[4];
#pragma unroll
	for (uint32_t u = 0; u < 4; ++u)
		hn[u] = home[min(u, nh - 1u)];
	for (uint32_t i0 = 0; i0 < nh; i0 += 4) {
#pragma unroll
		for (uint32_t u = 0; u < 4; ++u) {
			hp[u] = hn[u];
			hn[u] = home[min(i0 + 4u + u, nh - 1u)]; // the next four, in flight
		}
#pragma unroll
		for (uint32_t u = 0; u < 4; ++u) {
			const uint32_t i = i0 + u, ti = c0 + i;
			// keeps the unused fourth word of each load alive: its register would otherwise be
			// taken at once, with a wait for the load in flight
			asm volatile("" ::"s"(hp[u].w));
			if (i < nh) {
				const uint64_t other = __ballot(self != i);
				uint64_t hits;
				if (MODE != kWalkGeneral || P.pre) {
					const float dx = qx - hp[u].x, dy = qy - hp[u].y, dz = qz - hp[u].z;
					const float d2 = fmaf(dx, dx, fmaf(dy, dy, dz * dz));
					hits = __ballot(d2 <= P.pre_lo2) & other;
					// between the two bounds the reference's predicate decides
					if ((__ballot(d2 <= P.pre_hi2) & other) != hits)
						hits = __ballot(j != ~0u && pair_within(P, hp[u], ti, j, P.spos[j])) & other;
				} else {
					hits = __ballot(pair_within(P, hp[u], ti, j, make_float4(qx, qy, qz, 0.0f))) & other & alive;
				}
				if (own_rows) {
					const uint32_t nx = bcast_u32(X.count, i);
#pragma unroll
					for (uint32_t k = 0; k < 4; ++k)
						if (k < nx)
							hits &= ~__ballot(j == bcast_u32(X.slot[k], i));
					for (uint32_t k = 4; k < nx; ++k)
						hits &= ~__ballot(j == P.ex_slot[P.ex.excluded[bcast_u32(X.begin, i) + k]]);
				}
				if (filter)
					hits = __ballot(__builtin_amdgcn_inverse_ballot_w64(hits) && pair_allowed(P, ti, j));
				const uint32_t base = bcast_u32(cnt, i);
				// this home particle's rows: entry e of slot t (nbr_slot_index)
				const uint32_t at = ((ti >> 6) - (c0 >> 6)) * 256u * P.cap + (ti & 63u) * 16u;
				if (__builtin_amdgcn_inverse_ballot_w64(hits)) {
					const uint32_t e = uint32_t(__builtin_amdgcn_mbcnt_hi(
						uint32_t(hits >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(hits), base)));
					const uint32_t off = ((e << 8) & ~1023u) | ((e & 3u) << 2);
					if (e < P.cap)
						*reinterpret_cast<uint32_t*>(rows + (off + at)) = j;
				}
				set_lane(cnt, base + uint32_t(__popcll(hits)), i);
			}
		}
	}
}

// Fine cell k of the enumeration around home cell `home` (its particle range; empty when
// there is none or the gap test drops it).
template<int MODE>
struct WalkCells {
	const HomeParams& P;
	uint32_t home, total;
	const uint32_t* codes; // this home cell's list
	uint32_t base[3], mask[3]; // home code with every bit outside the axis set, axis bits
	int hc[3], lo[3], nax[3];
	__device__ __forceinline__ WalkCells(const HomeParams& P_, uint32_t home_) : P(P_), home(home_) {
		const uint32_t all = uint32_t((uint64_t(1) << (3 * (P.h + P.s))) - 1u);
		const uint32_t code = all ? home << (3 * P.s) : 0u; // (fine level 0: one cell, the whole box)
		codes = P.stencil_code + uint64_t(home & P.stencil_lists) * P.stencil_n;
#pragma unroll
		for (int a = 0; a < 3; ++a) {
			mask[a] = (0x24924924u >> a) & all;
			base[a] = (P.full[a] ? 0u : code & mask[a]) | ~mask[a];
		}
		total = P.stencil_n;
		if (MODE == kWalkGeneral && !P.stencil_code) {
			const int fine_cells = 1 << (P.h + P.s), span = 1 << P.s;
			hc[0] = int(compact_by3(home >> 2));
			hc[1] = int(compact_by3(home >> 1));
			hc[2] = int(compact_by3(home));
#pragma unroll
			for (int a = 0; a < 3; ++a) {
				lo[a] = P.full[a] ? 0 : hc[a] * span - P.reach[a];
				int hgh = P.full[a] ? fine_cells - 1 : hc[a] * span + span - 1 + P.reach[a];
				if (!P.full[a] && !P.box.periodic[a]) { // open axis: only cells that exist (the reach
					lo[a] = max(lo[a], 0);               // can be huge when the extent is degenerate)
					hgh = min(hgh, fine_cells - 1);
				}
				nax[a] = hgh - lo[a] + 1;
			}
			if (!P.stencil)
				total = uint32_t(nax[0] * nax[1] * nax[2]);
		}
	}
	__device__ __forceinline__ uint32_t offset(uint32_t k) const { // the stencil word, loaded ahead
		return (MODE != kWalkGeneral || P.stencil_code) && k < total ? codes[k] : 0u;
	}
	__device__ __forceinline__ uint2 range(uint32_t k, uint32_t off) const {
		uint2 none = make_uint2(0u, 0u);
		if (k >= total)
			return none;
		uint32_t code = 0;
		if (MODE != kWalkGeneral || P.stencil_code) {
#pragma unroll
			for (int a = 0; a < 3; ++a)
				code |= (base[a] + (off & mask[a])) & mask[a];
			return P.fine[code];
		}
		const int fine_cells = 1 << (P.h + P.s), span = 1 << P.s;
		int iv[3];
		if (P.stencil) {
			const int4 o = P.stencil[k];
			iv[0] = o.x;
			iv[1] = o.y;
			iv[2] = o.z;
#pragma unroll
			for (int a = 0; a < 3; ++a)
				iv[a] += P.full[a] ? 0 : hc[a] * span;
		} else {
			iv[0] = lo[0] + int(k) % nax[0];
			iv[1] = lo[1] + (int(k) / nax[0]) % nax[1];
			iv[2] = lo[2] + int(k) / (nax[0] * nax[1]);
		}
		float gap2 = 0.0f;
#pragma unroll
		for (int a = 0; a < 3; ++a) {
			int u = iv[a];
			if (!P.full[a]) {
				const int h0 = hc[a] * span;
				const int apart = u < h0 ? h0 - u - 1 : (u >= h0 + span ? u - h0 - span : 0);
				const float g = fmaxf(0.0f, float(apart) * P.cw[a] - 2.0f * P.margin[a]);
				gap2 += g * g;
				if (P.box.periodic[a])
					u = (u + fine_cells) & (fine_cells - 1);
				else if (u < 0 || u >= fine_cells)
					return none;
			}
			code |= split_by3(uint32_t(u) & 1023u) << (2 - a);
		}
		return gap2 <= P.rc2 ? P.fine[code] : none;
	}
};

// A candidate at q moved by whole box lengths next to the home frame's anchor (so the
// image is exact).
template<int MODE>
__device__ __forceinline__ float frame_axis(const HomeParams& P, int a, float q, float p0) {
	return MODE != kWalkGeneral || P.box.periodic[a] ? q - P.box.L[a] * rintf((q - p0) * P.box.inv_L[a]) : q;
}

// Particles [from, to) of home cell `home`, 64 at a time.
template<int MODE>
__device__ __forceinline__ void walk_home_cell(const HomeParams& P, uint32_t home, uint32_t from, uint32_t to,
											   WalkLds& S, uint32_t* __restrict__ counts, uint32_t* __restrict__ nbr) {
	const uint32_t lane = threadIdx.x & 63u;
	const WalkCells<MODE> cells(P, home);
	const bool own_rows = MODE == kWalkOwnRows || (MODE == kWalkGeneral && P.ex_slot);
	const bool filter = MODE == kWalkGeneral && (P.ref_filter || P.ex.rigid_body_id || (P.ex.offsets && !own_rows));
	for (uint32_t c0 = from; c0 < to; c0 += 64) {
		const uint32_t nh = min(to - c0, 64u);
		const bool valid = lane < nh;
		const float4 p = P.spos[c0 + min(lane, nh - 1u)];
		HomeExcl X{};
		if (own_rows)
			X = home_exclusions(P, valid, p);
		const float ox = bcast_f32(p.x, 0), oy = bcast_f32(p.y, 0), oz = bcast_f32(p.z, 0); // the frame's anchor
		// (lanes past the end repeat the last home particle)
		const float lox = wave_min(p.x), hix = wave_max(p.x);
		const float loy = wave_min(p.y), hiy = wave_max(p.y);
		const float loz = wave_min(p.z), hiz = wave_max(p.z);
		uint32_t cnt = 0;
		uint32_t nk = 0; // queued candidates (wave-uniform), fewer than 64 between blocks
		const auto block = [&](bool live, const float4& c) {
			test_block<MODE>(P, c0, nh, live ? __float_as_uint(c.w) : ~0u, live ? c.x : INFINITY, c.y, c.z, X, own_rows,
					   filter, cnt, nbr);
		};
		// the next step's cells and the stencil words of the one after are in flight while a
		// step's candidates are tested
		uint32_t off = cells.offset(lane);
		uint2 rg = cells.range(lane, off);
		off = cells.offset(64u + lane);
		for (uint32_t k0 = 0; k0 < cells.total; k0 += 64) {
			const uint32_t b = rg.x, n = rg.y > rg.x ? rg.y - rg.x : 0u;
			if (k0 + 64 < cells.total) {
				rg = cells.range(k0 + 64 + lane, off);
				off = cells.offset(k0 + 128 + lane);
			}
			const uint64_t some = __ballot(n > 0);
			if (some == 0)
				continue;
			// candidate q of this step (q < total, cells in lane order) is slot q + delta of its
			// cell; a cell's rank is the number of cells starting at or before q
			const uint32_t incl = wave_inclusive_scan(n), excl = incl - n;
			const uint32_t total = bcast_u32(incl, 63);
			wave_lds_sync(); // (reads of the last step's words)
			if (n > 0)
				S.delta[bits_below(some)] = b - excl;
			for (uint32_t w0 = 0; w0 < total; w0 += kWalkWindow) {
				if (w0 > 0)
					wave_lds_sync();
				if (lane < kWalkWindow / 32)
					S.start[lane] = 0u;
				wave_lds_sync();
				if (n > 0 && excl - w0 < kWalkWindow)
					atomicOr(&S.start[(excl - w0) >> 5], 1u << (excl & 31u));
				uint32_t before = uint32_t(__popcll(__ballot(n > 0 && excl < w0)));
				wave_lds_sync();
				const uint32_t end = min(total, w0 + kWalkWindow);
				const auto load = [&](uint32_t q0, uint32_t& j, float4& q) {
					const uint32_t at = (q0 - w0) >> 5;
					const uint32_t lo = uint32_t(__builtin_amdgcn_readfirstlane(int(S.start[at])));
					const uint32_t hi = uint32_t(__builtin_amdgcn_readfirstlane(int(S.start[at + 1])));
					const uint64_t bits = uint64_t(lo) | (uint64_t(hi) << 32);
					const uint32_t rank = before + bits_below(bits) + uint32_t((bits >> lane) & 1u) - 1u;
					before += uint32_t(__popcll(bits));
					// past the end: the last cell's last candidate, dropped by `live`
					j = min(q0 + lane, total - 1u) + S.delta[rank];
					q = P.spos[j];
				};
				uint32_t j;
				float4 q;
				load(w0, j, q);
				for (uint32_t q0 = w0; q0 < end; q0 += 64) {
					uint32_t jn = j;
					float4 qn = q;
					if (q0 + 64 < end)
						load(q0 + 64, jn, qn);
					bool kept = q0 + lane < total;
					if (MODE != kWalkGeneral || P.pre) {
						q.x = frame_axis<MODE>(P, 0, q.x, ox);
						q.y = frame_axis<MODE>(P, 1, q.y, oy);
						q.z = frame_axis<MODE>(P, 2, q.z, oz);
						// farther than the cutoff from the home particles' bounding box: its d2' to
						// every home particle is at least this, by the same monotone operations, so
						// the prefilter would drop it for each of them
						const float ax = fmaxf(fmaxf(lox - q.x, q.x - hix), 0.0f);
						const float ay = fmaxf(fmaxf(loy - q.y, q.y - hiy), 0.0f);
						const float az = fmaxf(fmaxf(loz - q.z, q.z - hiz), 0.0f);
						kept = kept && !(fmaf(ax, ax, fmaf(ay, ay, az * az)) > P.pre_hi2);
					}
					const uint64_t km = __ballot(kept);
					if (kept)
						S.keep[nk + bits_below(km)] = make_float4(q.x, q.y, q.z, __uint_as_float(j));
					nk += uint32_t(__popcll(km));
					wave_lds_sync();
					if (nk >= 64) {
						const float4 c = S.keep[lane], rest = S.keep[64 + lane];
						wave_lds_sync();
						nk -= 64;
						if (lane < nk)
							S.keep[lane] = rest;
						wave_lds_sync();
						block(true, c);
					}
					j = jn;
					q = qn;
				}
			}
		}
		if (nk > 0) {
			const float4 c = S.keep[lane];
			wave_lds_sync();
			block(lane < nk, c);
		}
		if (valid) {
			const uint32_t t = c0 + lane;
			counts[t] = cnt;
			if (cnt <= P.cap) {
				const uint64_t row = (uint64_t(t) >> 6) * 64u * P.cap;
				for (uint32_t k = cnt; (k & 3u) != 0; ++k)
					nbr[nbr_slot_index(row, t, k)] = t;
			}
		}
	}
}

template<int MODE>
__global__ __launch_bounds__(256, 6) void k_walk_home(HomeParams P, uint32_t* __restrict__ counts,
													  uint32_t* __restrict__ nbr) {
	__shared__ WalkLds lds[kHomeWaves];
	static_assert(kHomeWaves == 4, "a group's four cells");
	const uint32_t wv = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)));
	const TileRange R = xcd_tiles((P.num_home + kHomeWaves - 1) / kHomeWaves);
	for (uint32_t g = R.tile; g < R.end; g += R.stride) {
		if constexpr (MODE == kWalkPlain) {
			const uint32_t home = g * kHomeWaves + wv;
			if (home < P.num_home) {
				const uint2 r = *(const uint2 MMD_CONST_AS*)(uint64_t(P.home) + 8ull * home);
				if (r.x < r.y)
					walk_home_cell<MODE>(P, home, r.x, r.y, lds[wv], counts, nbr);
			}
		} else {
			// systems with exclusions are crowded along their chains: the 64-particle chunks of
			// the group's cells are dealt to its waves in turn (polymers of 100k beads: 209 ->
			// 158 us; the plain walk's extra scalar registers cost it 6% at 1M beads)
			uint32_t chunk = 0; // chunks of the cells so far
			for (uint32_t k = 0; k < uint32_t(kHomeWaves); ++k) {
				const uint32_t home = g * kHomeWaves + k;
				if (home >= P.num_home)
					break;
				const uint2 r = *(const uint2 MMD_CONST_AS*)(uint64_t(P.home) + 8ull * home);
				const uint32_t chunks = r.y > r.x ? (r.y - r.x + 63u) / 64u : 0u;
				for (uint32_t c = (wv - chunk) & 3u; c < chunks; c += 4u)
					walk_home_cell<MODE>(P, home, r.x + 64u * c, min(r.y, r.x + 64u * c + 64u), lds[wv], counts, nbr);
				chunk += chunks;
			}
		}
	}
}

// Ready for a walk: the cell tables cleared and the uniform rows' bases
// (tile_base[w] = w * row for w in [0, tiles], rows of `row` entries per tile).
__global__ void k_walk_setup(uint2* __restrict__ cells, uint64_t num_cells, uint32_t* __restrict__ tile_base,
							 uint64_t tiles, uint32_t row) {
	const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
	if (i < num_cells)
		cells[i] = make_uint2(0u, 0u);
	if (i <= tiles)
		tile_base[i] = uint32_t(i * row);
}

} // namespace

} // namespace mmd
