// CPU check of the level-0 strips' addressing (imscript_amd/csrc/sp_strip.h):
// every access of every lane and step of every tile of a W x H plane, carried
// out by the rule of a raw buffer (lane offset v, scalar offset at, n bytes: in
// range where v < n - at, without a sign).
//
// usage: strip_rows W H
// prints "OK <accesses carried out>" or what is wrong, and exits 1
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "../../imscript_amd/csrc/sp_strip.h"

static long carried;

static void fail(const char *what, int x0, int y0, int lane, int t)
{
	printf("%s: tile %d,%d lane %d step %d\n", what, x0, y0, lane, t);
	exit(1);
}

template <bool EVEN> static void check(int W, int H)
{
	const unsigned w = W, h = H, cw = (w + 1) / 2, ch = (h + 1) / 2, n = w * h, nc = cw * ch;
	std::vector<int> stored(n, 0), cstored(nc, 0);
	for (int y0 = 0; y0 < H; y0 += M0_TY)
		for (int x0 = 0; x0 < W; x0 += M0_TX)
			for (int lane = 0; lane < 64; lane++) {
				const M0Rows R{w, h, cw, ch, y0 - M0_HALO};
				const M0Lane L = m0_lane<EVEN>(lane, x0, W);
				const int i0 = x0 - M0_HALO + 2 * lane, steps = m0_steps(H, y0);
				auto at = [&](M0Row r, unsigned v, unsigned size, const char *what, int t) {
					if (r.at > r.n) fail(what, x0, y0, lane, t);
					if (v >= r.n - r.at) return -1L;
					if (v + size > r.n - r.at) fail("past the end", x0, y0, lane, t);
					carried++;
					return (long)v + r.at;
				};
				auto want = [&](long got, long expect, const char *what, int t) {
					if (got != expect) fail(what, x0, y0, lane, t);
				};
				const bool col = i0 >= 0 && i0 < W;
				for (int t = 0; t < steps + M0_CA; t++) {
					// (what is read in row t; a row is asked for rows ahead)
					const int j = y0 - M0_HALO + t, i = i0 - L.lone;
					const bool in = j >= 0 && j < H && col;
					const long p = (long)j * W + i;
					want(at(R.code(t, n), L.vc, 2, "codes: scalar offset", t),
							in ? p : -1, "codes", t);
					const long b = at(R.values(t, 4 * n), in ? L.vb : M0_OFF, 8,
							"values: scalar offset", t);
					want(b, in ? 4 * p : -1, "values", t);
					const long c = at(R.coarse(t, 4 * nc), L.vk, 4, "coarse: scalar offset", t);
					if (in) want(c, 4 * ((long)(j >> 1) * cw + (i0 >> 1)), "coarse", t);
				}
				for (int t = 0; t < steps; t++) {
					// the row that step t finishes; lanes of no code drop out
					const int j = y0 - M0_HALO + t - M0_HALO;
					const bool any = j >= 0 && j < H && col;
					const bool own = t >= 2 * M0_HALO && j < H && i0 >= x0 && i0 < x0 + M0_TX && col;
					const long p = (long)j * W + i0;
					const M0Row r = R.out(t, 4 * n);
					const long s = at(r, any ? L.vo : M0_OFF, 8, "stores: scalar offset", t);
					want(s, own && !L.lone ? 4 * p : -1, "stores", t);
					const long s1 = EVEN ? -1 : at(r, any ? L.vl : M0_OFF, 4,
							"last column: scalar offset", t);
					want(s1, own && L.lone ? 4 * p : -1, "last column", t);
					if (s >= 0) { stored[p]++; stored[p + 1]++; }
					if (s1 >= 0) stored[p]++;
					if (!(t & 1)) continue;
					const long c = at(R.coarse_out(t, 4 * nc), L.vko, 4,
							"coarse stores: scalar offset", t);
					const bool cown = t >= 2 * M0_HALO && (j >> 1) < (int)ch && i0 >= x0
						&& i0 < x0 + M0_TX && col;
					const long cp = (long)(j >> 1) * cw + (i0 >> 1);
					want(c, cown ? 4 * cp : -1, "coarse stores", t);
					if (c >= 0) cstored[cp]++;
				}
			}
	for (int v : stored) if (v != 1) fail("a pixel not stored once", 0, 0, 0, v);
	for (int v : cstored) if (v != 1) fail("a coarse cell not stored once", 0, 0, 0, v);
}

int main(int argc, char **argv)
{
	if (argc != 3) return 2;
	const int W = atoi(argv[1]), H = atoi(argv[2]);
	if (W & 1) check<false>(W, H);
	else { check<true>(W, H); check<false>(W, H); }
	printf("OK %ld\n", carried);
	return 0;
}
