// Row addressing of the level-0 strips (k_mg0_strip), shared by the kernel and
// by the CPU test that checks it.
//
// An access goes through a buffer descriptor of n bytes with a lane's byte
// offset v and the row's scalar offset at.  It is carried out where
// v < n - at and dropped (a load returns 0) elsewhere, the difference taken
// without a sign: at must never exceed n, also in a row that is not to be
// touched.  Such a row has n = at = 0; a lane that is not to touch its row
// has v = M0_OFF, which no n - at reaches.
#pragma once
#include "sp_gs.h"

constexpr int M0_NU = 5, M0_HALO = 2 * M0_NU, M0_TX = 128 - 2 * M0_HALO, M0_TY = 44;
constexpr int M0_BA = 4, M0_CA = 7;      // rows that b / codes are ahead
constexpr unsigned M0_OFF = 0xfffffff0u; // beyond every buffer

struct M0Row { unsigned n, at; };        // bytes of the descriptor, scalar offset

// the rows of one strip: row r is image row jt + r
struct M0Rows {
	unsigned w, h, cw, ch;               // the plane and the next coarser level
	int jt;

	// the row's first pixel; outside the image, where every lane's code is 0,
	// that of the nearest row
	SP_HD unsigned at(int r) const { return clamp(jt + r, h) * w; }
	SP_HD unsigned coarse_at(int r) const { return clamp((jt + r) >> 1, ch) * cw; }
	static SP_HD M0Row row(bool in, unsigned n, unsigned at)
	{
		return {in ? n : 0u, in ? at : 0u};
	}
	// what a step reads: the codes of row r; b and zd of row r, by lanes with a
	// code; the coarse correction of row r
	SP_HD M0Row code(int r, unsigned n) const
	{
		return row((unsigned)(jt + r) < h, n, at(r));
	}
	SP_HD M0Row values(int r, unsigned n) const { return {n, 4u * at(r)}; }
	SP_HD M0Row coarse(int r, unsigned n) const { return {n, 4u * coarse_at(r)}; }
	// what step t writes: z or zd of the row it finishes (none of the halo
	// above the tile), by lanes with a code; the coarse b of that row and the
	// one above
	SP_HD M0Row out(int t, unsigned n) const
	{
		return row(t >= 2 * M0_HALO, n, 4u * at(t - M0_HALO));
	}
	SP_HD M0Row coarse_out(int t, unsigned n) const
	{
		return row(t >= 2 * M0_HALO && (jt + t - M0_HALO) >> 1 < (int)ch, n,
				4u * coarse_at(t - M0_HALO));
	}
	static SP_HD unsigned clamp(int v, unsigned n)
	{
		return v < 0 ? 0u : (unsigned)v >= n ? n - 1 : (unsigned)v;
	}
};

// steps of a tile whose first row is y0
SP_HD int m0_steps(int h, int y0)
{
	const int rows = h - y0 < M0_TY ? h - y0 : M0_TY;
	return ((rows + 3) & ~3) + 2 * M0_HALO;
}

// byte offsets of lane tid of the tile at column x0: its pair's codes, its b
// and zd to load, z to store, coarse values to load and to store.  lone: an
// odd width's last column, whose loads are of the pair one column to the left,
// of which it is the right cell, and which has a store of its own (vl).
struct M0Lane {
	unsigned vc, vb, vo, vl, vk, vko;
	bool mine, lone;
};
template <bool EVEN> SP_HD M0Lane m0_lane(int tid, int x0, int w)
{
	const int i0 = x0 - M0_HALO + 2 * tid;
	const bool ok = i0 >= 0 && i0 < w;
	M0Lane L;
	L.mine = tid >= M0_HALO / 2 && tid < (M0_HALO + M0_TX) / 2 && ok;
	L.lone = !EVEN && i0 == w - 1;
	const unsigned il = (unsigned)(i0 - (L.lone ? 1 : 0));
	L.vc = ok ? il : M0_OFF;
	L.vb = ok ? 4u * il : M0_OFF;
	L.vo = L.mine && !L.lone ? 4u * (unsigned)i0 : M0_OFF;
	L.vl = L.mine && L.lone ? 4u * (unsigned)i0 : M0_OFF;
	L.vk = ok ? 4u * (unsigned)(i0 >> 1) : M0_OFF;
	L.vko = L.mine ? 4u * (unsigned)(i0 >> 1) : M0_OFF;
	return L;
}
