// patch.h -- patch form of the slice stencil: a thread owns PX x PY sites of the lattice.
//
// Patch (bx, by) covers the sites (bx PX + x, by PY + y), coordinates modulo (l1, l2).  Where an
// extent is not a multiple of the patch's, the last patch of a row or column runs over the seam and
// holds ghost copies of the sites there; a ghost has its owner's bonds and neighbours, so it computes
// its owner's values, and only the owner's are stored to memory.  Inside a patch neighbours are the
// thread's own registers; the halo is
//   top[x], x = 0 .. PX: sites (x - 1, PY);   bot[x], x = 0 .. PX: sites (x, -1);
//   lft[y], rgt[y], y < PY: sites (-1, y) and (PX, y),
// 2 PX + 2 PY + 2 values per stencil instead of 6 PX PY.
//
// In LDS site (x, y) of patch p sits at slot (y PX + x) of tp places: place [slot][p].  Lanes hold
// consecutive patches, so writes and most reads touch consecutive places (no bank conflicts).
//
// A patch's bonds, each once: R, U (up) and T (up-left) of its sites, then those that enter from
// outside: R of (-1, y), U of (x, -1), T of (x + 1, -1), T of (PX, y) for y < PY - 1:
// 3 PX PY + 2 PX + 2 PY - 1 coefficients.  Memory holds them [slice][bond][patch].
#pragma once
#include "internal.h"

namespace ephmc {

constexpr int patch_halo(int px, int py){ return 2 * px + 2 * py + 2; }
constexpr int patch_bonds(int px, int py){ return 3 * px * py + 2 * px + 2 * py - 1; }

// index of a bond in the patch's list
template <int PX, int PY>
struct PatchBond {
	static constexpr int S = PX * PY;
	static constexpr int right(int x, int y){ return x >= 0 ? 3 * (y * PX + x) : 3 * S + y; }
	static constexpr int up(int x, int y){ return y >= 0 ? 3 * (y * PX + x) + 1 : 3 * S + PY + x; }
	// up-left bond of (x, y): y = -1 (x = 1 .. PX) or x = PX (y = 0 .. PY - 2) lie outside
	static constexpr int upl(int x, int y)
	{
		return y < 0 ? 3 * S + PY + PX + x - 1 : (x == PX ? 3 * S + PY + 2 * PX + y : 3 * (y * PX + x) + 2);
	}
};

// out = A v for a patch of C columns: own values v, halo h, bonds cf; the sum over the neighbours in
// the order R, L, up, down, up-left, down-right of the site form, so both give the same bits
template <typename R, int C, int PX, int PY>
__device__ __forceinline__ void patch_stencil(const R (&v)[PX * PY][C], const R (&h)[patch_halo(PX, PY)][C],
		const R (&cf)[patch_bonds(PX, PY)], R mu, R (&out)[PX * PY][C])
{
	using B = PatchBond<PX, PY>;
	constexpr int TOP = 0, BOT = PX + 1, LFT = 2 * PX + 2, RGT = LFT + PY;
#pragma unroll
	for(int y = 0; y < PY; y++)
#pragma unroll
		for(int x = 0; x < PX; x++)
#pragma unroll
			for(int c = 0; c < C; c++){
				const int s = y * PX + x;
				const R r = x < PX - 1 ? v[x < PX - 1 ? s + 1 : s][c] : h[RGT + y][c];
				const R l = x > 0 ? v[x > 0 ? s - 1 : s][c] : h[LFT + y][c];
				const R u = y < PY - 1 ? v[y < PY - 1 ? s + PX : s][c] : h[TOP + x + 1][c];
				const R d = y > 0 ? v[y > 0 ? s - PX : s][c] : h[BOT + x][c];
				const R ul = y < PY - 1 ? (x > 0 ? v[y < PY - 1 && x > 0 ? s + PX - 1 : s][c] : h[LFT + (y < PY - 1 ? y + 1 : y)][c]) : h[TOP + x][c];
				const R dr = y > 0 ? (x < PX - 1 ? v[y > 0 && x < PX - 1 ? s - PX + 1 : s][c] : h[RGT + (y > 0 ? y - 1 : y)][c]) : h[BOT + x + 1][c];
				R o = mu * v[s][c];
				o = fmac(cf[B::right(x, y)], r, o);
				o = fmac(cf[B::right(x - 1, y)], l, o);
				o = fmac(cf[B::up(x, y)], u, o);
				o = fmac(cf[B::up(x, y - 1)], d, o);
				o = fmac(cf[B::upl(x, y)], ul, o);
				o = fmac(cf[B::upl(x + 1, y - 1)], dr, o);
				out[s][c] = o;
			}
}

} // namespace ephmc
