// Streaming Gauss-Seidel sweeps of radius 1 (sp_stream.hip): descriptors
// shared by the kernels and the host driver.
//
// Sweep k of pixel (i, j) runs on step s = i + j + 2k (sp_gs.h).  With the
// row skewed by the sweep, j' = j + k, everything an update reads was
// computed one or two steps earlier in the same or the previous row j':
//
//   W (i-1, j, k)      row j',    step s-1     S (i, j+1, k-1)  row j',    step s-1
//   N (i, j-1, k)      row j'-1,  step s-1     E (i+1, j, k-1)  row j'-1,  step s-1
//   x (i, j, k-1)      row j'-1,  step s-2
//
// So a wavefront whose lane l holds row j' = 64 J + l for K consecutive
// sweeps advances one step at a time with its K values in registers: W and S
// are its own values, N, E and x come from lane l-1.  Only lane 0 needs
// another wavefront's values, those of lane 63 of band J-1, and only the
// first of its sweeps reads what an earlier block of sweeps left.
#pragma once
#include <hip/hip_runtime.h>
#include "sp_gs.h"

namespace spk {

constexpr int SS_C = 8;    // steps per phase (between two barriers)
constexpr int SS_PS = 32;  // words between two tasks' progress words

// the compiled forms: K sweeps per wavefront, NW wavefronts of sweeps
template <int K_, int NW_> struct SsForm { static constexpr int K = K_, NW = NW_; };
template <class F> inline void sp_with_form(int form, F &&f)
{
	if (form == 0) f(SsForm<4, 4>());
	else f(SsForm<2, 5>());
}
inline void ss_form_shape(int form, int &K, int &KT)
{
	sp_with_form(form, [&](auto f) { K = f.K; KT = f.K * f.NW; });
}

// one plane.  The values u and the coefficients are laid out by bands of 64
// rows and, inside a band, by sigma = i + j: pixel (i, j) at
//   (j / 64) BS + (i + j - 64 (j / 64) + pad) 64 + j % 64,
// the order in which the lanes of a step read them.  One more band and the
// cells outside the image hold the coefficients of known pixels.
struct SsInst {
	float *u;            // the level's values, image layout
	const float *c;      // its coefficients (sp_gs.h), image layout
	float *A, *C;        // values and coefficients, skewed layout
	float *bz;           // lane 63's values of every band, for the band below
	int *prog;           // phases done by each task (one word in SS_PS), INT_MAX: all
	unsigned *mx;        // the level's largest |value| and |data term| (float bits)
	int w, h, T;         // sweeps
	float t;
	unsigned BS;         // floats per band
	int pad;             // steps of padding before i = 0
	int U, nslot;        // bz: steps per band, bands per block of sweeps
	float *hist;         // the values after every sweep, hs floats each, or null
	size_t hs;
	float *acc;          // image layout: where they are added up
};
struct SsTask { int inst, tb, J; };   // band J of the tb-th block of sweeps
struct SsBlock { int inst, jb, sb; }; // 64 x 64 block of the skewed layout

enum { SS_LAPLACE = 0, SS_POISSON = 1, SS_AMLE = 2 };   // SS_AMLE: 4 neighbours

inline int ss_pad(int KT) { return 2 * (64 + KT) + 2 * SS_C + 8; }
// the most steps of a band, its own and those the band below asks for
inline int ss_steps(int w, int KT) { return w + KT + 2 * 64 + 5 * SS_C; }
inline int ss_bands(int h) { return (h + 63) / 64; }
inline size_t ss_band_floats(int w, int KT) { return (size_t)64 * (w + 63 + 2 * ss_pad(KT)); }

int ss_blocks(int form, int op, bool sum);   // work-groups that can be resident
void launch_ss_clear(int op, float *C, size_t n, hipStream_t s);
void launch_ss_in(int op, const SsInst *in, const SsBlock *bw, int nb, hipStream_t s);
// small: the step and the sweeps are such that values bounded by those the
// kernels test for stay small; mx: the level's largest |value| and |data term|
// sum (SS_LAPLACE): also writes hist
void launch_ss_run(int form, int op, bool sum, bool small, const SsTask *tasks, int nt, int blocks,
		const SsInst *in, unsigned *claim, const unsigned *mx, int spin_max, int *err,
		hipStream_t s);
// acc += the values after sweeps 0..nsum-1, one by one, at the swept pixels
void launch_ss_sum(const SsInst *in, const SsBlock *bw, int nb, int nsum, hipStream_t s);
// also sets words[0, nwords) (the progress words, claim and mx) to 0
void launch_ss_out(const SsInst *in, const SsBlock *bw, int nb, unsigned *words,
		int nwords, hipStream_t s);

} // namespace spk
