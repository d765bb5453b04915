// Streaming Gauss-Seidel sweeps of radius 1 (sp_stream.h).
//
// One task is a band of 64 skewed rows through a block of K NW sweeps: a
// work-group of NW wavefronts of K sweeps each, wavefront w one phase
// (SS_C steps) behind wavefront w-1 and fed by it through LDS, one wavefront
// that fetches what the band needs from other tasks, and one that publishes
// what other tasks need.  A task runs as soon as the tasks before it are a
// few phases ahead, not when they have ended, so the chain of a level is its
// hyperplanes plus a few microseconds per band and block of sweeps.
//
// Against the tiles (sp_gs.h, LDS values and a barrier per hyperplane step)
// an update costs 11 vector instructions and its share of a step's LDS
// accesses instead of 22 and 6: finest levels of 4096 x 4096 x 3 with 256
// sweeps 6.9 ms instead of 15, of 1920 x 1080 x 3 with 10 sweeps 0.55 ms
// instead of 1.6, of 512 x 512 with 2000 sweeps 2.2 ms instead of 6.  Bound:
// vector issue where there are tasks enough (4096 x 4096 x 3), else the
// phases of 1.0 (2 sweeps a wavefront) to 1.4 us (4) times the 10.5 of them
// that a band starts after the one above it.
#include <algorithm>
#include <limits.h>
#include <type_traits>
#include "sp_internal.h"
#include "sp_stream.h"

namespace spk {

constexpr unsigned SS_KNOWN0 = 0x80000000u;   // Laplace, AMLE: known pixel (holes hold t)

static __device__ __forceinline__ float ss_nan() { return __uint_as_float(SP_QNAN_BITS); }

template <class T>
static __device__ __forceinline__ T ss_ld(const __attribute__((address_space(1))) T *p)
{
	return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
template <class T>
static __device__ __forceinline__ void ss_st(__attribute__((address_space(1))) T *p, T v)
{
	__hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
typedef const __attribute__((address_space(1))) int *ss_flag;

// the same at a 32-bit byte offset from a base in scalar registers
static __device__ __forceinline__ float ss_ld_b(const float *base, unsigned off)
{
	asm("" : "+v"(off));
	return ss_ld((const __attribute__((address_space(1))) float *)(
			(const __attribute__((address_space(1))) char *)base + off));
}
static __device__ __forceinline__ void ss_st_b(float *base, unsigned off, float v)
{
	asm("" : "+v"(off));
	ss_st((__attribute__((address_space(1))) float *)(
			(__attribute__((address_space(1))) char *)base + off), v);
}

// the value of lane l-1, and of `first` in lane 0
static __device__ __forceinline__ float ss_shift(float first, float v)
{
	return __int_as_float(__builtin_amdgcn_update_dpp(__float_as_int(first),
			__float_as_int(v), 0x138 /* wave_shr:1 */, 0xf, 0xf, false));
}

// LDS written before is visible after; loads from memory stay in flight
static __device__ __forceinline__ void ss_barrier()
{
	asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

static __device__ __forceinline__ int ss_uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
template <class T> static __device__ __forceinline__ T *ss_uni(T *p)
{
	const unsigned long long v = (unsigned long long)p;
	const unsigned lo = (unsigned)ss_uni((int)(unsigned)v), hi = (unsigned)ss_uni((int)(v >> 32));
	return (T *)((unsigned long long)hi << 32 | lo);
}

// the phase in which step s0 - 2 falls
static __device__ __forceinline__ int ss_first(int s0)
{
	static_assert(SS_C == 8, "shift");
	return (s0 - 2) >> 3;
}

static __device__ __forceinline__ void ss_wait(ss_flag p, int need, int &seen, int spin_max,
		int *err)
{
	int n = 0;
	while (seen < need) {
		seen = __builtin_amdgcn_readfirstlane(ss_ld(p));
		if (seen >= need) break;
		if (++n > spin_max) {
			if ((threadIdx.x & 63) == 0) atomicOr(err, 1);
			seen = INT_MAX;   // goes on with what is there; the host reports it
		}
		__builtin_amdgcn_s_sleep(1);
	}
	asm volatile("" ::: "memory");
}

// The forms of an update.  SS_GENERAL is the reference's: the terms E, S, W, N
// in that order (simpois.c:72-90), a neighbour that is not finite skipped.
// Cells outside the image hold NaN and the coefficient of a known pixel, and
// so stay NaN.  The others need every value of the level finite and small
// enough that no sum overflows: then only cells outside the image are not
// finite, and SS_EDGE turns their NaN terms into zeros (the median of NaN,
// NaN and 0 is 0, of d, d and 0 it is d); SS_INNER reads none.  The sum
// starts from E - x instead of 0 + (E - x), which only moves the sign of a
// zero sum, which x + t (r - c) does not show.
enum { SS_GENERAL = 0, SS_EDGE = 1, SS_INNER = 2 };

template <int FORM>
static __device__ __forceinline__ float ss_term(float v, float x)
{
	const float d = v - x;
	return FORM == SS_EDGE ? __builtin_amdgcn_fmed3f(d, d, 0.0f) : d;
}

// AMLE of 4 neighbours (sp_amle.h): the mean of the first strict minimum and
// maximum in the order E, S, W, N.  With finite values those are the plain
// minimum and maximum, in which NaN cells outside the image drop out; only
// where they are equal does the order show, in the sign of a zero: then the
// result is the first neighbour in the image.  SS_GENERAL scans, from the
// first neighbour by its place (column i, row j), since a pixel may be NaN.
static __device__ __forceinline__ float ss_min3(float a, float b, float c)
{
	float r;
	asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
	return r;
}
static __device__ __forceinline__ float ss_max3(float a, float b, float c)
{
	float r;
	asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
	return r;
}
template <int FORM>
static __device__ __forceinline__ float ss_amle(float x, float e, float so, float w, float n,
		float c, int i, int j, int W, int H)
{
	float f = e, y;
	if (FORM == SS_GENERAL) {
		if (i + 1 >= W) f = j + 1 < H ? so : i > 0 ? w : n;
		float mn = f, mx = f;
		mn = so < mn ? so : mn;
		mx = so > mx ? so : mx;
		mn = w < mn ? w : mn;
		mx = w > mx ? w : mx;
		mn = n < mn ? n : mn;
		mx = n > mx ? n : mx;
		y = (mn + mx) * 0.5f;
	} else {
		const float mn = ss_min3(ss_min3(e, so, w), n, n), mx = ss_max3(ss_max3(e, so, w), n, n);
		if (FORM == SS_EDGE) f = e == e ? e : so == so ? so : w;
		y = mn == mx ? f : (mn + mx) * 0.5f;
	}
	return __float_as_int(c) < 0 ? x : y;
}

template <int OP, int FORM>
static __device__ __forceinline__ float ss_update(float x, float e, float so, float w,
		float n, float c, float t)
{
	if (FORM == SS_GENERAL) {
		float r = 0.0f;
		if (isfinite(e)) r = r + (e - x);
		if (isfinite(so)) r = r + (so - x);
		if (isfinite(w)) r = r + (w - x);
		if (isfinite(n)) r = r + (n - x);
		const bool known = OP == SS_LAPLACE ? sp_bits(c) == SS_KNOWN0 : sp_known(c);
		const float y = OP == SS_LAPLACE ? x + t * r : x + t * (r - c);
		return known ? x : y;
	}
	float r = ss_term<FORM>(e, x);
	r = r + ss_term<FORM>(so, x);
	r = r + ss_term<FORM>(w, x);
	r = r + ss_term<FORM>(n, x);
	// Laplace: c is t at a hole and -0 at a known pixel (x + -0 r = x, up to
	// the sign of a zero, which no neighbour shows)
	if (OP == SS_LAPLACE) return x + c * r;
	const float y = x + t * (r - c);
	return sp_known(c) ? x : y;
}

// a coefficient through a buffer resource: the lane's offset and the row's
// stay apart, without an addition per load
static __device__ __forceinline__ float ss_coef(__amdgpu_buffer_rsrc_t b, unsigned lane_off,
		unsigned row_off)
{
	return __int_as_float(__builtin_amdgcn_raw_buffer_load_b32(b, lane_off, row_off, 0));
}

template <int K> struct SsState {
	float Y[K], Z[K];   // values of the K sweeps and of lane l-1's, last step
	float Ym, Zm;       // the same of the sweep before them
};

// the LDS areas of a phase, the wavefront's own
struct SsLds {
	const float *line, *zin, *zinm;
	float *lout, *zout;
};

// SS_C steps from the coefficient row crow on.  cv: the coefficients of the next SS_C
// steps, each replaced after its use by the one SS_C steps on (crow + its offset).
template <int K, int OP, int FORM, bool SUM>
static __device__ __forceinline__ void ss_chunk(SsState<K> &q, float (&cv)[SS_C][K],
		__amdgpu_buffer_rsrc_t cbuf, unsigned crow, const unsigned (&voff)[K], const SsLds &l,
		int lane, float t, int i0, int jrow, int W, int H, __amdgpu_buffer_rsrc_t hbuf,
		unsigned hs4)
{
	constexpr int KP = K <= 4 ? 4 : 8;
	float zi[K], zm, ym;
#pragma unroll
	for (int k = 0; k < K; k++) zi[k] = l.zin[k];
	zm = l.zinm[K - 1];
	ym = l.line[lane];
#pragma unroll
	for (int c = 0; c < SS_C; c++) {
		float zn[K], yn[K], zi1[K], zm1 = 0, ym1 = 0;
		if (c + 1 < SS_C) {   // the next step's, before this step's stores
#pragma unroll
			for (int k = 0; k < K; k++) zi1[k] = l.zin[(c + 1) * KP + k];
			zm1 = l.zinm[(c + 1) * KP + K - 1];
			ym1 = l.line[(c + 1) * 64 + lane];
		}
		zm = ss_shift(zm, q.Ym);
#pragma unroll
		for (int k = 0; k < K; k++) zn[k] = ss_shift(zi[k], q.Y[k]);
#pragma unroll
		for (int k = K - 1; k >= 0; k--) {
			if (OP == SS_AMLE)
				yn[k] = ss_amle<FORM>(k ? q.Z[k - 1] : q.Zm, k ? zn[k - 1] : zm,
						k ? q.Y[k - 1] : q.Ym, q.Y[k], zn[k], cv[c][k], i0 + c - k,
						jrow - k, W, H);
			else yn[k] = ss_update<OP, FORM>(k ? q.Z[k - 1] : q.Zm, k ? zn[k - 1] : zm,
					k ? q.Y[k - 1] : q.Ym, q.Y[k], zn[k], cv[c][k], t);
		}
#pragma unroll
		for (int k = 0; k < K; k++) {
			cv[c][k] = ss_coef(cbuf, voff[k], crow + (c + SS_C) * 256);
			if (SUM)
				__builtin_amdgcn_raw_buffer_store_b32(__float_as_int(yn[k]), hbuf, voff[k],
						crow + c * 256 + k * hs4, 0);
			q.Y[k] = yn[k];
			q.Z[k] = zn[k];
		}
		q.Zm = zm;
		q.Ym = ym;
		l.lout[c * 64 + lane] = yn[K - 1];
		if (lane == 63) {
#pragma unroll
			for (int k = 0; k < K; k++) l.zout[c * KP + k] = yn[k];
		}
		if (c + 1 < SS_C) {
#pragma unroll
			for (int k = 0; k < K; k++) zi[k] = zi1[k];
			zm = zm1;
			ym = ym1;
		}
		__builtin_amdgcn_sched_barrier(0);   // steps do not mix: fewer registers
	}
}

template <int K, int NW, int OP, bool SUM>
__global__ __launch_bounds__((NW + 2) * 64) __attribute__((amdgpu_waves_per_eu(4))) void k_ss_run(const SsTask *tasks, int nt,
		const SsInst *insts, unsigned *claim, const unsigned *mx, int spin_max, int *err)
{
	constexpr int C = SS_C, KT = K * NW, KP = K <= 4 ? 4 : 8;
	static_assert(C * K <= 64 && KT < 64 && 64 % C == 0 && NW <= 8, "phase shape");
	__shared__ __align__(16) float line[NW + 1][2][C][64];   // [w]: into wavefront w
	__shared__ __align__(16) float zin[NW + 1][4][C][KP];    // [w + 1]: lane 0 of wavefront w
	__shared__ __align__(16) float zo[NW][2][C][KP];         // lane 63 of wavefront w
	__shared__ int s_k;
	// values bounded by these stay far from overflow: with 0 < t <= 1/4 a sweep
	// averages, and the data term adds at most t |c| (finite by the first test)
	const bool gen = !mx || !(mx[0] < __float_as_uint(1e33f) && mx[1] < __float_as_uint(1e28f));
	const int lane = threadIdx.x & 63;
	const int wv = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
	for (;;) {
		__syncthreads();   // the last task's LDS and s_k are free
		if (threadIdx.x == 0) s_k = (int)min(atomicAdd(claim, 1u), (unsigned)nt);
		__syncthreads();
		const int id = __builtin_amdgcn_readfirstlane(s_k);
		if (id >= nt) return;
		// the task and its plane, in scalar registers
		const int J = ss_uni(tasks[id].J), tb = ss_uni(tasks[id].tb);
		const SsInst *const ip = insts + ss_uni(tasks[id].inst);
		const int W = ss_uni(ip->w), H = ss_uni(ip->h), T = ss_uni(ip->T);
		const int pad = ss_uni(ip->pad), U = ss_uni(ip->U), nslot = ss_uni(ip->nslot);
		const unsigned BS = (unsigned)ss_uni((int)ip->BS);
		float *const pA = ss_uni(ip->A), *const pC = ss_uni(ip->C), *const pbz = ss_uni(ip->bz);
		int *const pprog = ss_uni(ip->prog);
		const float t = __int_as_float(ss_uni(__float_as_int(ip->t)));
		const float fv = ss_nan();   // the value of cells outside the image
		const int k0 = tb * KT, nwa = (min(KT, T - k0) + K - 1) / K, k1 = k0 + nwa * K - 1;
		const int j0 = 64 * J, jmin = k0 / 64, q = J - jmin;
		// phases gs on: the first update reads values of two steps before it
		const int gs = ss_first(j0 + k0), nch = (j0 + 63 + k1 + W - 1) / C - gs + 1;
		const int nph = nch + nwa - 1;
		// float offset of row j at sigma = -pad; of a row outside the plane
		// (or where known is set): in the band after the last, which holds
		// known pixels throughout
		const int nb = (H + 63) >> 6;
		auto rowoff = [&](int j, bool known = false) {
			const unsigned r = (unsigned)(j & 63) - 4096u * (unsigned)(j >> 6);
			return r + ((unsigned)j < (unsigned)H && !known ? (unsigned)(j >> 6) : (unsigned)nb) * BS;
		};
		if (wv < NW) {
			SsState<K> st;
			float cv[SS_C][K];
			unsigned voff[K];
			const int kw = k0 + wv * K, jrow = j0 + lane - kw;
#pragma unroll
			for (int k = 0; k < K; k++) {
				st.Y[k] = st.Z[k] = fv;
				// sweeps past the last leave every pixel: known pixels
				voff[k] = 4 * (rowoff(jrow - k, kw + k >= T) + 2 * (K - 1 - k) * 64);
			}
			st.Ym = st.Zm = fv;
			// row of the coefficients of the last sweep on step 0
			const unsigned cbase = 256u * (unsigned)(pad - 2 * (kw + K - 1));
			const __amdgpu_buffer_rsrc_t cbuf = __builtin_amdgcn_make_buffer_rsrc(pC, 0,
					4 * (nb + 1) * BS, 0x00027000);
			const bool rows = j0 - (kw + K - 1) >= 1 && j0 + 63 - kw <= H - 2;
			if (wv < nwa) {
#pragma unroll
				for (int c = 0; c < SS_C; c++)
#pragma unroll
					for (int k = 0; k < K; k++)
						cv[c][k] = ss_coef(cbuf, voff[k], cbase + 256u * (unsigned)(gs * C + c));
				__builtin_amdgcn_s_waitcnt(0);
			}
			ss_barrier();
			const unsigned hs4 = SUM ? 4u * (unsigned)(nb + 1) * BS : 0u;
			const __amdgpu_buffer_rsrc_t hbuf = __builtin_amdgcn_make_buffer_rsrc(
					SUM ? ss_uni(ip->hist) + (size_t)kw * (hs4 / 4) : pC, 0, (int)(K * hs4),
					0x00027000);
			auto run = [&](auto form, int pa, int pb) {
				for (int p = pa; p < pb; p++) {
					if (wv < nwa && p >= wv && p - wv < nch) {
						const SsLds l = {&line[wv][p & 1][0][0], &zin[wv + 1][p & 3][0][0],
							&zin[wv][(wv ? p - 1 : p) & 3][0][0],
							&line[wv + 1][(p + 1) & 1][0][0], &zo[wv][(p + 1) & 1][0][0]};
						const int s0 = (gs + p - wv) * C;
						ss_chunk<K, OP, decltype(form)::value, SUM>(st, cv, cbuf,
								cbase + 256u * (unsigned)s0, voff, l, lane, t,
								s0 - jrow - 2 * kw, jrow, W, H, hbuf, hs4);
					}
					ss_barrier();
				}
			};
			if (gen) {
				run(std::integral_constant<int, SS_GENERAL>(), 0, nph);
			} else {
				// phases [pa, pb) touch no cell beside the image's border: their
				// first column is at least 1, their last at most W - 2
				const int lo = (j0 + 63 + kw + K - 1) / C + 1, hi = (W - 2 + j0 + kw + 1) / C;
				int pa = sp_clamp(lo - gs + wv, 0, nph), pb = sp_clamp(hi - gs + wv, 0, nph);
				if (!rows || pb < pa) pa = pb = nph;
				run(std::integral_constant<int, SS_EDGE>(), 0, pa);
				run(std::integral_constant<int, SS_INNER>(), pa, pb);
				run(std::integral_constant<int, SS_EDGE>(), pb, nph);
			}
		} else if (wv == NW) {
			// fetches for phase p + 1 while phase p runs (two round trips to the
			// coherent memory, about 0.3 us each, are less than a phase)
			const ss_flag prog = (ss_flag)pprog;
			const int jmaxp = tb ? (H - 1 + k0 - 1) / 64 : -1, jminp = tb ? (k0 - KT) / 64 : 0;
			const bool up = q > 0, prev = tb > 0 && J <= jmaxp;
			const int gsu = ss_first(j0 - 64 + k0), gsp = ss_first(j0 + k0 - KT);
			ss_flag pu = up ? prog + ((ptrdiff_t)tb * nslot + q - 1) * SS_PS : prog;
			ss_flag pp = prev ? prog + ((ptrdiff_t)(tb - 1) * nslot + (J - jminp)) * SS_PS : prog;
			int su = up ? 0 : INT_MAX, sp = prev ? 0 : INT_MAX, sw = INT_MAX;
			// the band slot's reader two blocks of sweeps ago, which has to be
			// past what this task overwrites (its band starts 64 steps later)
			ss_flag pw = prog;   // (a word that is there, where none is asked for)
			if (tb > 1) {
				const int kk = k0 - 2 * KT;
				if (q + 1 <= (H - 1 + kk + KT - 1) / 64 - kk / 64) {
					pw = prog + ((ptrdiff_t)(tb - 2) * nslot + q + 1) * SS_PS;
					sw = 0;
				}
			}
			const int jr = j0 + lane - k0 + 1;   // row of the sweep before k0
			const unsigned arow = 4 * rowoff(jr);
			const bool jok = (unsigned)jr < (unsigned)H;
			const int ju = j0 - k0;              // the row of lane -1
			const unsigned aup = 4 * rowoff(ju) + (lane & (C - 1)) * 256;
			const float *A = pA;
			const float *bz = pbz + ((ptrdiff_t)(tb & 1) * nslot + max(q - 1, 0)) * U * KT;
			const int ec = lane / K, ek = lane - ec * K;
			struct Regs { float lv[C], uv, zv[NW]; } r;
			const unsigned zlane = 4u * ((ec < C ? ec : 0) * KT + ek);
			// every call loads the same, from addresses that exist; commit
			// puts fv where the value is no pixel's
			auto issue = [&](int p, Regs &r) {
				const float *a = A + (ptrdiff_t)(pad - 2 * k0 + 2 + (gs + min(p, nch - 1)) * C) * 64;
#pragma unroll
				for (int c = 0; c < C; c++) r.lv[c] = ss_ld_b(a + c * 64, arow);
				r.uv = ss_ld_b(a - 64, aup);
#pragma unroll
				for (int w = 0; w < NW; w++) {
					const int g = gs + sp_clamp(p - w, 0, nch - 1) - gsu;   // >= 0
					r.zv[w] = ss_ld_b(bz + (ptrdiff_t)max(g * C - 1, 0) * KT + w * K, zlane);
				}
			};
			// the phases [lo, hi) in which every value is a pixel's
			int lo = (j0 + k0 + KT + 63 + C * NW) / C + 1 - gs;
			const int hi = min((W - C - 2 + j0 + k0) / C + 1 - gs, nch);
			if (!(j0 - k0 - KT >= 0 && j0 + 64 - k0 <= H - 1)) lo = INT_MAX;
			auto commit = [&](int p, const Regs &r) {
				float lv[C], uv = r.uv, zv[NW];
#pragma unroll
				for (int c = 0; c < C; c++) lv[c] = r.lv[c];
#pragma unroll
				for (int w = 0; w < NW; w++) zv[w] = r.zv[w];
				if (p < lo || p >= hi) {
					int i = (gs + p) * C - 2 * k0 + 2 - jr;
#pragma unroll
					for (int c = 0; c < C; c++)
						lv[c] = jok && (unsigned)(i + c) < (unsigned)W ? lv[c] : fv;
					i = (gs + p) * C + (lane & (C - 1)) - 2 * k0 + 1 - ju;
					uv = (unsigned)ju < (unsigned)H && (unsigned)i < (unsigned)W ? uv : fv;
					i = (gs + p) * C + ec - j0 - k0 - ek;
#pragma unroll
					for (int w = 0; w < NW; w++) {
						const int iw = i - w * (C + K), j = j0 - 1 - k0 - w * K - ek;
						const bool on = up && w < nwa && p >= w && p - w < nch;
						zv[w] = on && (unsigned)iw < (unsigned)W && (unsigned)j < (unsigned)H
							? zv[w] : fv;
					}
				}
				if (p < nch) {
#pragma unroll
					for (int c = 0; c < C; c++) line[0][p & 1][c][lane] = lv[c];
					if (lane < C) zin[0][p & 3][lane][K - 1] = uv;
				}
				if (ec < C) {
#pragma unroll
					for (int w = 0; w < NW; w++) zin[w + 1][p & 3][ec][ek] = zv[w];
				}
			};
			auto fetch = [&](int p) {
				if (p >= nph) return;
				if (up) ss_wait(pu, p + gs - gsu + 1, su, spin_max, err);
				if (prev && p < nch) ss_wait(pp, p + gs - gsp + NW, sp, spin_max, err);
				ss_wait(pw, p + 2 - 64 / C, sw, spin_max, err);
				issue(p, r);
				commit(p, r);
			};
			fetch(0);
			ss_barrier();
			for (int p = 0; p < nph; p++) {
				fetch(p + 1);
				ss_barrier();
			}
		} else {
			// stores phase p - 1 while phase p runs
			auto *prog = (__attribute__((address_space(1))) int *)pprog
				+ ((ptrdiff_t)tb * nslot + q) * SS_PS;
			const bool down = J < (H - 1 + k1) / 64;
			const int jr = j0 + lane - k1;
			const unsigned arow = 4 * rowoff(jr);
			const bool jok = (unsigned)jr < (unsigned)H;
			float *bz = pbz + ((ptrdiff_t)(tb & 1) * nslot + q) * U * KT;
			const int ec = lane / K, ek = lane - ec * K;
			float *const A = pA;
			const bool rows = j0 - k1 >= 0 && j0 + 63 - k1 <= H - 1;
			const unsigned zlane = 4u * (ec * KT + ek);
			auto out = [&](int p) {
				const int pl = p - nwa;   // the last wavefront's phase
				const int s = (gs + pl) * C;
				const float *lp = &line[nwa][p & 1][0][lane];
				if (rows && pl >= 0 && pl < nch && s - j0 - 63 - k1 >= 0
						&& s + C - 1 - j0 - k1 <= W - 1) {
					float *a = A + (ptrdiff_t)(pad - 2 * k1 + s) * 64;
#pragma unroll
					for (int c = 0; c < C; c++) ss_st_b(a + c * 64, arow, lp[c * 64]);
				} else if (pl >= 0 && pl < nch) {
#pragma unroll
					for (int c = 0; c < C; c++) {
						const int i = s + c - 2 * k1 - jr;
						if (jok && (unsigned)i < (unsigned)W)
							ss_st_b(A + (ptrdiff_t)(pad - 2 * k1 + s + c) * 64, arow, lp[c * 64]);
					}
				}
				if (down && ec < C) {
					const float *zp = &zo[0][p & 1][ec][ek];
#pragma unroll
					for (int w = 0; w < NW; w++) {
						const int pw = p - 1 - w;
						if (w < nwa && pw >= 0 && pw < nch)
							ss_st_b(bz + (ptrdiff_t)pw * C * KT + w * K, zlane, zp[w * 2 * C * KP]);
					}
				}
				asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
				if (lane == 0) ss_st(prog, p < nph ? p : INT_MAX);
			};
			ss_barrier();
			for (int p = 0; p < nph; p++) {
				if (p) out(p);
				ss_barrier();
			}
			out(nph);
		}
	}
}

// the coefficients of known pixels everywhere (the cells outside the image
// keep them)
__global__ __launch_bounds__(256) void k_ss_clear(float *C, size_t n, float v)
{
	for (size_t i = blockIdx.x * (size_t)256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
		C[i] = v;
}

// image layout -> skewed layout, one 64 x 64 block through LDS; cells of the
// layout outside the image keep what they have
template <int OP>
__global__ __launch_bounds__(256) void k_ss_in(const SsInst *insts, const SsBlock *bw)
{
	__shared__ float su[64][65], sc[64][65];
	__shared__ unsigned m0, m1;
	const SsBlock b = bw[blockIdx.x];
	const SsInst in = insts[b.inst];
	const int lane = threadIdx.x & 63, r0 = threadIdx.x >> 6;
	if (threadIdx.x == 0) m0 = m1 = 0;
	float uv[16], cv[16];
#pragma unroll
	for (int r = 0; r < 16; r++) {
		const int jr = r0 + 4 * r, j = b.jb * 64 + jr, i = b.sb * 64 + lane - jr;
		const size_t p = (size_t)sp_clamp(j, 0, in.h - 1) * in.w + sp_clamp(i, 0, in.w - 1);
		uv[r] = gload<float>(in.u + p);
		cv[r] = gload<float>(in.c + p);
	}
	unsigned a0 = 0, a1 = 0;
#pragma unroll
	for (int r = 0; r < 16; r++) {
		const int jr = r0 + 4 * r, j = b.jb * 64 + jr, i = b.sb * 64 + lane - jr;
		const bool known = sp_known(cv[r]);
		if (j < in.h && i >= 0 && i < in.w) {
			a0 = max(a0, sp_bits(uv[r]) & 0x7fffffffu);
			if (!known) a1 = max(a1, sp_bits(cv[r]) & 0x7fffffffu);
		}
		su[jr][lane] = uv[r];
		sc[jr][lane] = OP != SS_POISSON ? (known ? __uint_as_float(SS_KNOWN0) : in.t) : cv[r];
	}
#pragma unroll
	for (int o = 32; o; o >>= 1) {
		a0 = max(a0, (unsigned)__shfl_xor((int)a0, o));
		a1 = max(a1, (unsigned)__shfl_xor((int)a1, o));
	}
	__syncthreads();
	if (lane == 0) {
		atomicMax(&m0, a0);
		atomicMax(&m1, a1);
	}
	const size_t base = (size_t)b.jb * in.BS + (size_t)(b.sb * 64 + in.pad) * 64 + lane;
#pragma unroll
	for (int r = 0; r < 16; r++) {
		const int x = r0 + 4 * r, j = b.jb * 64 + lane, i = b.sb * 64 + x - lane;
		if (j < in.h && i >= 0 && i < in.w) {
			in.A[base + x * 64] = su[lane][x];
			in.C[base + x * 64] = sc[lane][x];
		}
	}
	__syncthreads();
	if (threadIdx.x == 0) {
		if (m0 > in.mx[0]) atomicMax(in.mx, m0);
		if (m1 > in.mx[1]) atomicMax(in.mx + 1, m1);
	}
}

// acc += the values after each of the first nsum sweeps at the swept pixels,
// in that order
__global__ __launch_bounds__(256) void k_ss_sum(const SsInst *insts, const SsBlock *bw, int nsum)
{
	__shared__ float sa[64][65];
	const SsBlock b = bw[blockIdx.x];
	const SsInst in = insts[b.inst];
	const int lane = threadIdx.x & 63, r0 = threadIdx.x >> 6;
	float a[16];
#pragma unroll
	for (int r = 0; r < 16; r++) {
		const int jr = r0 + 4 * r, j = b.jb * 64 + jr, i = b.sb * 64 + lane - jr;
		a[r] = gload<float>(in.acc + (size_t)sp_clamp(j, 0, in.h - 1) * in.w
				+ sp_clamp(i, 0, in.w - 1));
	}
#pragma unroll
	for (int r = 0; r < 16; r++) sa[r0 + 4 * r][lane] = a[r];
	__syncthreads();
	const float *h = in.hist + (size_t)b.jb * in.BS + (size_t)(b.sb * 64 + in.pad + r0) * 64 + lane;
#pragma unroll
	for (int r = 0; r < 16; r++) a[r] = sa[lane][r0 + 4 * r];
	for (int k = 0; k < nsum; k++, h += in.hs)
#pragma unroll
		for (int r = 0; r < 16; r++) a[r] = a[r] + gload<float>(h + r * 256);
	__syncthreads();
#pragma unroll
	for (int r = 0; r < 16; r++) sa[lane][r0 + 4 * r] = a[r];
	__syncthreads();
#pragma unroll
	for (int r = 0; r < 16; r++) {
		const int jr = r0 + 4 * r, j = b.jb * 64 + jr, i = b.sb * 64 + lane - jr;
		if (j >= in.h || i < 0 || i >= in.w) continue;
		const size_t p = (size_t)j * in.w + i;
		if (!sp_known(in.c[p])) in.acc[p] = sa[jr][lane];
	}
}

// the swept pixels back to the image layout
// (and the words of the next run's synchronisation back to 0)
__global__ __launch_bounds__(256) void k_ss_out(const SsInst *insts, const SsBlock *bw,
		unsigned *words, int nwords)
{
	for (int i = blockIdx.x * 256 + threadIdx.x; i < nwords; i += gridDim.x * 256) words[i] = 0;

	__shared__ float su[64][65];
	const SsBlock b = bw[blockIdx.x];
	const SsInst in = insts[b.inst];
	const int lane = threadIdx.x & 63, r0 = threadIdx.x >> 6;
	const size_t base = (size_t)b.jb * in.BS + (size_t)(b.sb * 64 + in.pad) * 64 + lane;
	float uv[16], cv[16];
#pragma unroll
	for (int r = 0; r < 16; r++) {
		const int x = r0 + 4 * r, jr = r0 + 4 * r;
		const int j = b.jb * 64 + jr, i = b.sb * 64 + lane - jr;
		uv[r] = gload<float>(in.A + base + x * 64);   // inside the band's padding
		cv[r] = gload<float>(in.c + (size_t)sp_clamp(j, 0, in.h - 1) * in.w
				+ sp_clamp(i, 0, in.w - 1));
	}
#pragma unroll
	for (int r = 0; r < 16; r++) su[lane][r0 + 4 * r] = uv[r];
	__syncthreads();
#pragma unroll
	for (int r = 0; r < 16; r++) {
		const int jr = r0 + 4 * r, j = b.jb * 64 + jr, i = b.sb * 64 + lane - jr;
		if (j < in.h && i >= 0 && i < in.w && !sp_known(cv[r]))
			in.u[(size_t)j * in.w + i] = su[jr][lane];
	}
}

template <class F> static void ss_with(int form, int op, bool sum, F &&f)
{
	sp_with_form(form, [&](auto fm) {
		constexpr int K = decltype(fm)::K, NW = decltype(fm)::NW;
		if (sum) f(k_ss_run<K, NW, SS_LAPLACE, true>, (NW + 2) * 64);
		else if (op == SS_LAPLACE) f(k_ss_run<K, NW, SS_LAPLACE, false>, (NW + 2) * 64);
		else if (op == SS_AMLE) f(k_ss_run<K, NW, SS_AMLE, false>, (NW + 2) * 64);
		else f(k_ss_run<K, NW, SS_POISSON, false>, (NW + 2) * 64);
	});
}

int ss_blocks(int form, int op, bool sum)
{
	int nb = INT_MAX;
	auto ask = [&](auto *k, int threads) {
		int per = 0, dev = 0, ncu = 0;
		if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, k, threads, 0) != hipSuccess)
			per = 1;
		(void)hipGetDevice(&dev);
		if (hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev)
				!= hipSuccess || ncu <= 0)
			ncu = 256;
		nb = std::min(nb, std::max(1, per) * ncu);
	};
	ss_with(form, op, sum, ask);
	return nb;
}

void launch_ss_clear(int op, float *C, size_t n, hipStream_t s)
{
	k_ss_clear<<<1024, 256, 0, s>>>(C, n, sp_float(op == SS_POISSON ? SP_KNOWN_BITS : SS_KNOWN0));
}

void launch_ss_in(int op, const SsInst *in, const SsBlock *bw, int nb, hipStream_t s)
{
	if (op != SS_POISSON) k_ss_in<SS_LAPLACE><<<nb, 256, 0, s>>>(in, bw);
	else k_ss_in<SS_POISSON><<<nb, 256, 0, s>>>(in, bw);
}

void launch_ss_run(int form, int op, bool sum, bool small, const SsTask *tasks, int nt, int blocks,
		const SsInst *in, unsigned *claim, const unsigned *mx, int spin_max, int *err,
		hipStream_t s)
{
	auto run = [&](auto *k, int threads) {
		k<<<std::min(nt, blocks), threads, 0, s>>>(tasks, nt, in, claim, small ? mx : nullptr,
				spin_max, err);
	};
	ss_with(form, op, sum, run);
}

void launch_ss_sum(const SsInst *in, const SsBlock *bw, int nb, int nsum, hipStream_t s)
{
	if (nsum > 0) k_ss_sum<<<nb, 256, 0, s>>>(in, bw, nsum);
}

void launch_ss_out(const SsInst *in, const SsBlock *bw, int nb, unsigned *words,
		int nwords, hipStream_t s)
{
	k_ss_out<<<nb, 256, 0, s>>>(in, bw, words, nwords);
}

} // namespace spk
