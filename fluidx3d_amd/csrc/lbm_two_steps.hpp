// Two time steps per pass over memory (FP32 DDFs), for runs of several steps.
//
// One stream_collide step of FP32 DDFs waits on HBM (256^3 D3Q19: 153 bytes per cell, 6.4
// TB/s, the VALU 24 % busy).  This kernel reads the DDFs of step t once, keeps the
// populations between the steps t and t+1 in LDS, and writes those of step t+1 once, so a
// step costs half the bytes.  Per cell the arithmetic is that of the two single steps
// (collide_cell), so the DDFs come out the same, bit for bit.
//
// A block owns a tile of at most TX x TY columns (two_step_shape) and marches through a segment of planes.
// At plane k it takes step t for the tile extended by one cell on each side (phase 1), then
// step t+1 for the tile's own cells of plane k-1 (phase 2), whose inputs come from the
// planes k-2, k-1 and k.  Neighbouring blocks read each other's border cells, so the result
// goes to a second DDF array of the same layout: no block sees another one's stores, and
// the blocks need no order.
//
// - Waves have fixed roles: a wave is 64 columns of one row of the extended tile; the first
//   and the last row and one more wave with the two border columns of every row only take
//   phase 1, the others both.  Every wave runs a loop of its own with the same barriers,
//   in which the number of loads and stores between a load and its use is fixed: with
//   branches around the stores the wait for the next plane's loads has to wait for the
//   stores too (256^3: 322 against 278 us per step with buffer addressing).
// - Lanes past a clipped tile's last column repeat that column (same loads, same stores),
//   so there are no partial waves.
// - LDS holds, per cell of the extended tile, the populations that leave their column: those
//   with c_z = -1 are used in the same iteration (one plane), c_z = 0 one iteration later
//   and c_z = +1 two later.  Phase 2 reads the last two groups into registers before the
//   barrier that allows the new plane to overwrite them, so c_z = 0 needs one plane and
//   c_z = +1 two.  Populations that stay in their column (i = 0 and +-z) stay in registers.
//   D3Q19: 80 bytes per cell, 73 KB for 128 x 5 and 79 KB for 64 x 13; D3Q27: 128 bytes.
// - The loads of plane k+1 are issued before phase 2 of plane k-1.
//
// What bounds it: memory, in tile order.  256^3 D3Q19 SRT, 256 blocks of 128 x 4 columns and
// 128 planes, one per CU: 267 us per step against 399 us for single steps.  Two steps move
// the bytes of one (FETCH_SIZE +4 %, WRITE_SIZE the same; the border cells' reads hit L2).  A
// kernel that only copies 19 arrays takes 235 us per step's worth in the order of these
// tiles (5.4 TB/s) and 205 us in linear order (6.2 TB/s); without the collisions this one
// takes 256 us.  Loads two planes ahead (-1 to +2 %), two blocks of fewer rows per CU (-20 to
// -30 %), stores interleaved with the next plane's loads (-10 %), one barrier per plane with
// three planes in LDS (-10 %) and 2- or 3-row tiles (-15 to -20 %) measured no better.
#pragma once
#include "lbm_device.hpp"

namespace fx {

struct TwoStepArgs {
	LbmArgs a;                        // a.fi: DDFs before step t (parity a.odd)
	void* dst;                        // DDFs after step t+1
	uint32_t tiles_x, tiles_y, tiles; // tiles along x and y, and blocks with work in all
	uint32_t width, height, zlen;     // columns (<= TX) and rows (<= TY) of a tile and planes of a segment; the last ones are clipped
};

// f(integral constant) for I, I+S, ... below N: array indices are constants when the compiler
// first splits arrays into registers (with unrolled loops it kept whole planes of loaded
// values as one register tuple and copied it, waiting for the loads, in every iteration).
template<int I> struct Index { static constexpr int value = I; };
template<int I, int N, int S, class F> __device__ __forceinline__ void static_for(F&& f) {
	if constexpr(I < N) { f(Index<I>{}); static_for<I + S, N, S>(f); }
}

// Populations that stay in their column, and the position of population i among those with
// the same c_z that leave it (i < Q; count of them for i = Q).
template<int Q> constexpr bool stays(int i) { return VS<Q>::cx[i] == 0 && VS<Q>::cy[i] == 0; }
template<int Q> constexpr int plane_slot(int i, int cz) {
	int k = 0;
	for(int j = 0; j < i; j++) if(VS<Q>::cz[j] == cz && !stays<Q>(j)) k++;
	return k;
}

// Threads of a block with tiles of TX x height columns: a wave per 64 columns of every row of
// the extended tile, and one for the border columns.
constexpr uint32_t two_step_threads(uint32_t TX, uint32_t height) { return (height + 2u) * TX + 64u; }

template<int Q, bool TRT, uint32_t EXT, int TX, int TY, bool CACHED>
__global__ __launch_bounds__((two_step_threads(TX, TY))) void k_two_steps(TwoStepArgs g) {
	constexpr int ROWS = TY + 2, PITCH = TX + 2, CELLS = ROWS * PITCH;
	constexpr int NM = plane_slot<Q>(Q, -1), N0 = plane_slot<Q>(Q, 0), NP = plane_slot<Q>(Q, 1);
	__shared__ float lds[(NM + N0 + 2 * NP) * CELLS];
	float* const lm = lds; float* const l0 = lds + NM * CELLS; float* const lp = lds + (NM + N0) * CELLS;
	// consecutive blocks go to the 8 XCDs in turn: each XCD takes a run of neighbouring tiles
	const uint32_t per = gridDim.x >> 3, tile = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
	if(tile >= g.tiles) return;
	static_assert(!(EXT & EXT_UPDATE_FIELDS), "step t of a border cell would write rho and u beside the block that owns it");
	LbmArgs a = g.a;
	a.ext &= EXT;
	const uint32_t Nx = a.Nx, Ny = a.Ny, Nz = a.Nz;
	const uint32_t tx = tile % g.tiles_x, tr = tile / g.tiles_x, ty = tr % g.tiles_y, tz = tr / g.tiles_y;
	const uint32_t x0 = tx * g.width, y0 = ty * g.height, z0 = tz * g.zlen;
	const uint32_t wx = min(g.width, Nx - x0), wy = min(g.height, Ny - y0), wz = min(g.zlen, Nz - z0);
	// the column of this thread: (lx, lr) in the extended tile, the tile's own cells at 1 .. wx, 1 .. wy
	constexpr uint32_t WAVES = TX / 64; // per row
	const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63u;
	const bool border = wave == (g.height + 2u) * WAVES;
	const uint32_t wrow = wave / WAVES, wcol = (wave % WAVES) * 64u;
	const bool idle = !border && (wrow > wy + 1u || wcol >= wx);
	const bool inner = !border && !idle && wrow >= 1u && wrow <= wy;
	uint32_t lx, lr;
	if(border) { const uint32_t s = min(lane, 2u * wy + 3u); lr = s >> 1; lx = (s & 1u) ? wx + 1u : 0u; }
	else { lr = idle ? 0u : wrow; lx = min(wcol + lane, wx - 1u) + 1u; }
	uint32_t x = x0 + lx, y = y0 + lr; // one more than the coordinate, periodic
	x = x == 0u ? Nx - 1u : x - 1u; if(x >= Nx) x -= Nx;
	y = y == 0u ? Ny - 1u : y - 1u; if(y >= Ny) y -= Ny;
	const uint32_t e = lr * PITCH + lx;
	// byte offsets of the column and its neighbours in a plane (below 4 GiB), 64-bit offsets of the slots
	const uint32_t xs[3] = {x == 0u ? Nx - 1u : x - 1u, x, x + 1u == Nx ? 0u : x + 1u};
	const uint32_t ys[3] = {(y == 0u ? Ny - 1u : y - 1u) * Nx, y * Nx, (y + 1u == Ny ? 0u : y + 1u) * Nx};
	const uint32_t col = ys[1] + x;
	const uint64_t P = (uint64_t)Nx * Ny, Pb = P * 4u;
	uint64_t slot[Q]; // of population i as step t loads it; store_f of step t+1 writes it to the same slot
	slot[0] = 0u;
	static_for<1, Q, 2>([&](auto c) __attribute__((always_inline)) {
		constexpr int i = decltype(c)::value;
		slot[i] = (uint64_t)(a.odd ? i : i + 1) * a.N * 4u;
		slot[i + 1] = (uint64_t)(a.odd ? i + 1 : i) * a.N * 4u;
	});
	typedef __attribute__((address_space(1))) float gfloat;
	const auto put = [](auto* p, float v) __attribute__((always_inline)) {
		if constexpr(CACHED) *p = v;
		else __builtin_nontemporal_store(v, p);
	};
	const auto at = [](const void* p, uint64_t uniform_bytes, uint32_t cell) __attribute__((always_inline)) {
		return (gfloat*)((__attribute__((address_space(1))) char*)((uint64_t)p + uniform_bytes) + cell * 4u);
	};
	const auto plane = [&](int k) -> uint32_t { // z of plane k of the segment, -1 <= k, periodic
		const int v = (int)z0 + k;
		uint32_t z = v < 0 ? Nz - 1u : (uint32_t)v;
		while(z >= Nz) z -= Nz;
		return z;
	};
	struct Offsets { uint64_t z[3]; };
	const auto offsets = [&](uint32_t z) { return Offsets{{(z == 0u ? Nz - 1u : z - 1u) * Pb, z * Pb, (z + 1u == Nz ? 0u : z + 1u) * Pb}}; };
	float r[Q];       // loaded DDFs of the next plane
	uint32_t fl;      // its flags
	const auto load_plane = [&](int k) __attribute__((always_inline)) { // load_f at the parity of step t
		const uint32_t z = plane(k);
		const Offsets o = offsets(z);
		fl = (a.flags + z * P)[col];
		r[0] = *at(a.fi, o.z[1], col);
		static_for<1, Q, 2>([&](auto c) __attribute__((always_inline)) {
			constexpr int i = decltype(c)::value;
			r[i] = *at(a.fi, slot[i] + o.z[1], col);
			r[i + 1] = *at(a.fi, slot[i + 1] + o.z[VS<Q>::cz[i] + 1], ys[VS<Q>::cy[i] + 1] + xs[VS<Q>::cx[i] + 1]);
		});
	};
	// streamed-in populations -> post-collision populations of the cell (col, z).  Solid and
	// gas cells are mailboxes: every population goes back where it came from.
	const auto collide = [&](uint32_t z, uint32_t flagsn, const float* in, float* out) __attribute__((always_inline)) {
		if((flagsn & TYPE_BO) == TYPE_S || (flagsn & TYPE_SU) == TYPE_G) {
			out[0] = in[0];
			static_for<1, Q, 2>([&](auto c) __attribute__((always_inline)) { constexpr int i = decltype(c)::value; out[i] = in[i + 1]; out[i + 1] = in[i]; });
		} else {
			float f[Q];
			static_for<0, Q, 1>([&](auto c) __attribute__((always_inline)) { constexpr int i = decltype(c)::value; f[i] = in[i]; });
			if((a.ext & EXT_MOVING_BOUNDARIES) && (flagsn & TYPE_BO) == TYPE_MS) moving_boundaries<Q>(a, make_site(x, y, z, Nx, Ny, Nz), f);
			collide_cell<Q, TRT, EXT, false, false, shared_pair_difference(Q, EXT, false)>(a, z * P + col, flagsn & TYPE_BO, f, nullptr);
			static_for<0, Q, 1>([&](auto c) __attribute__((always_inline)) { constexpr int i = decltype(c)::value; out[i] = f[i]; });
		}
	};
	const auto publish = [&](int k, const float* out) __attribute__((always_inline)) {
		const int ring = (k & 1) * NP * CELLS;
		static_for<1, Q, 1>([&](auto c) __attribute__((always_inline)) {
			constexpr int i = decltype(c)::value, cz = VS<Q>::cz[i], s = plane_slot<Q>(i, cz);
			if constexpr(!stays<Q>(i)) {
				if constexpr(cz == 0) l0[s * CELLS + e] = out[i];
				else if constexpr(cz == 1) lp[ring + s * CELLS + e] = out[i];
				else lm[s * CELLS + e] = out[i];
			}
		});
	};
	const auto barrier = []() __attribute__((always_inline)) {
		__builtin_amdgcn_sched_barrier(0);
		__syncthreads();
		__builtin_amdgcn_sched_barrier(0);
	};
	// Every role passes two barriers per plane -1 .. wz.
	if(idle) {
		for(int k = -1; k <= (int)wz; k++) { barrier(); barrier(); }
		return;
	}
	load_plane(-1);
	if(!inner) {
		for(int k = -1; k <= (int)wz; k++) {
			float out[Q];
			collide(plane(k), fl, r, out);
			barrier();
			publish(k, out);
			load_plane(k + 1);
			barrier();
		}
		return;
	}
	// the populations that stay in their column: 0 of plane k-1, 5 (c_z = +1) of planes k-2 and k-1
	float s0 = 0.0f, s5a = 0.0f, s5b = 0.0f;
	uint32_t fl1 = 0u; // flags of plane k-1
	for(int k = -1; k < 1; k++) { // nothing to finish yet
		float out[Q];
		fl1 = fl;
		collide(plane(k), fl, r, out);
		s0 = out[0]; s5a = s5b; s5b = out[5];
		barrier();
		publish(k, out);
		load_plane(k + 1);
		barrier();
	}
	for(int k = 1; k <= (int)wz; k++) {
		float out[Q], in[Q];
		const uint32_t flk = fl;
		collide(plane(k), flk, r, out);
		__builtin_amdgcn_sched_barrier(0);
		// inputs of plane k-1 from the planes k-2 (c_z = 1) and k-1 (c_z = 0)
		const int ring = (k & 1) * NP * CELLS;
		static_for<1, Q, 1>([&](auto c) __attribute__((always_inline)) {
			constexpr int i = decltype(c)::value, cz = VS<Q>::cz[i], s = plane_slot<Q>(i, cz), d = -VS<Q>::cx[i] - VS<Q>::cy[i] * PITCH;
			if constexpr(!stays<Q>(i) && cz == 0) in[i] = l0[s * CELLS + (int)e + d];
			else if constexpr(!stays<Q>(i) && cz == 1) in[i] = lp[ring + s * CELLS + (int)e + d];
		});
		in[0] = s0; in[5] = s5a; in[6] = out[6];
		s0 = out[0]; s5a = s5b; s5b = out[5];
		barrier();
		publish(k, out);
		load_plane(k + 1);
		barrier();
		static_for<1, Q, 1>([&](auto c) __attribute__((always_inline)) {
			constexpr int i = decltype(c)::value, cz = VS<Q>::cz[i], s = plane_slot<Q>(i, cz), d = -VS<Q>::cx[i] - VS<Q>::cy[i] * PITCH;
			if constexpr(!stays<Q>(i) && cz == -1) in[i] = lm[s * CELLS + (int)e + d];
		});
		const uint32_t z = z0 + (uint32_t)k - 1u;
		collide(z, fl1, in, out);
		fl1 = flk;
		// store_f at the parity of step t+1
		const Offsets o = offsets(z);
		put(at(g.dst, o.z[1], col), out[0]);
		static_for<1, Q, 2>([&](auto c) __attribute__((always_inline)) {
			constexpr int i = decltype(c)::value;
			*at(g.dst, slot[i] + o.z[VS<Q>::cz[i] + 1], ys[VS<Q>::cy[i] + 1] + xs[VS<Q>::cx[i] + 1]) = out[i];
			put(at(g.dst, slot[i + 1] + o.z[1], col), out[i + 1]);
		});
	}
}

} // namespace fx
