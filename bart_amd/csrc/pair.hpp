// pair.hpp -- FFT passes over the pairs of sub-grids that differ in the shift
// of one axis (gfx950), for any supported length.
//
// The 2x oversampled grid is decomposed into sub-grids s = (bit per active
// axis); the linear phase of sub-grid s is a product over the axes, so the
// transform along an axis needs only the bits of the axes done so far:
//   split: the column h of a volume is multiplied by l_b(k) and transformed,
//          for b = 0, 1, into two volumes (forward, one axis after the
//          other: 1 -> 2 -> 4 -> 8 volumes per coil);
//   merge: the columns of two volumes are transformed backward and
//          conj(l_b(k)) x result is summed (adjoint, 8 -> 4 -> 2 -> 1);
//   turn:  split, multiply by the PSFs of the two members, merge, in one
//          pass (last axis of the Toeplitz normal operator).
// Per coil a 2-D Toeplitz operator then moves 2 + 4 + 2 volumes between its
// passes and a 3-D one 2 + 6 + 8 + 6 + 2, where transforming every sub-grid
// on its own moves 4 + 8 + 4 and 8 + 16 + 16 + 16 + 8, with 2/3 of the
// transforms.
//
// A transform of length n = R0 R1 (R0 R1 R2) is held by NJ = max n / Ri lanes;
// a lane's R points j + r n / R are one butterfly of the first pass (inputs)
// and of the last (outputs), so the first pass runs on the loaded registers,
// the last one stores from registers, and one exchange through LDS lies between
// them (two with three radices).  Columns sit in LDS
// transform-fastest ([k][P], P adjacent columns: 128-byte global rows, no
// bank conflicts in any pass), rows point-fastest with one element of
// padding after eight.
#pragma once

#include <type_traits>

#include "fft.hpp"
#include "volume.hpp"

namespace bam {

#define BAM_INLINE __attribute__((always_inline))

constexpr int PF_MAXR = 16;       // largest radix
constexpr int PF_MAXN = 1024;     // longest transform of the pair kernels
// work-group limits: rows (two members of half the lanes); columns of at most
// two radices (n / Ri <= 16), of three.  n <= PF_MAXN never takes more than 256
// lanes.
constexpr int pf_threads(bool rows, bool three) { return (rows || three) ? 512 : 256; }

struct PairPlan {

	int n = 0;
	int nr = 0;            // radices (0: no pair kernel for this length)
	int rad[3] = { 1, 1, 1 };
	int NJ = 0;            // lanes per transform
	FastDiv fF, fB, fNJ;   // middle pass: division by rad[0] (forward) and rad[2]
	const float2* tw = nullptr;
};

// host: the balanced factorisation into at most three radices
PairPlan make_pair_plan(const AxisPlan& a);

// arguments of one pass over one plan
struct PairArgs {

	PairPlan pl;
	VolAxis va;              // the axis; nvol = volumes split or merged
	const int* skip;
	const float2* l[2];      // linear phase of the axis per bit
	float2* grid;
	long half;               // from a volume to its second member
	int cl;                  // kernel
	int P, logP, pitch;      // transforms per work-group; rows: LDS pitch
	int group;               // rows: threads per member (whole waves), twice as many in all
	int C;
	uint32_t ncg;            // columns: groups of P columns; rows: groups of P rows
	FastDiv f_ncg, f_outer, f_nvol, f_C;
	uint32_t nblk;

	// rows (image side)
	const float2* src;       // split: coil images [C][N] or one image (with sens)
	const float2* sens;      // [C][N] or null
	float2* dst;             // merge: coil images, or partial images per coil group
	int cc;                  // merge with sens: coils per group
	const float* roll[3];    // null: no rolloff
	// split of the last axis: fftmod tables (null: none)
	const float2* fm[3];
	// turn, split with PSFs
	const float2* psf;
	long psf_half;
};

// kernel of a length: general with two radices, with three, or with the radices
// in the code
enum { PF_TWO = 0, PF_THREE, PF_32, PF_64, PF_128, PF_256, PF_CLASSES };

constexpr int pf_class(int n, int nr)
{
	return (32 == n) ? PF_32 : (64 == n) ? PF_64 : (128 == n) ? PF_128 : (256 == n) ? PF_256 : (3 == nr) ? PF_THREE : PF_TWO;
}

constexpr int PF_FP = 16;  // columns per work-group of the latter: 128-byte rows

// the last of their two radices: the lanes of a transform
constexpr int pf_fixed_lanes(int cl) { return (PF_256 == cl) ? 16 : (PF_32 == cl) ? 4 : 8; }

// LDS pitch of a row
constexpr int pf_row_pitch(int n) { return (n + n / 8 + 1) | 1; }

size_t pair_lds_bytes(const PairArgs& a, bool rows);
unsigned pair_threads(const PairArgs& a, bool rows);
// fills P, logP, pitch, the block count and the divisions; `units`: row
// kernels only, the coils (or coil groups); `ncu`: the device's compute units
void pair_geometry(PairArgs& a, bool rows, uint32_t units, int ncu);

// ---------------------------------------------------------------------------
// DFTs of radix 2 .. 16 in registers, w = exp(SG 2 pi i / R)
// ---------------------------------------------------------------------------

constexpr double pf_sin_series(double x)
{
	double t = x, s = x;
	for (int i = 1; i < 20; i++) {
		t *= -x * x / ((2. * i) * (2. * i + 1.));
		s += t;
	}
	return s;
}

constexpr double pf_cos_series(double x)
{
	double t = 1., s = 1.;
	for (int i = 1; i < 20; i++) {
		t *= -x * x / ((2. * i - 1.) * (2. * i));
		s += t;
	}
	return s;
}

// exp(2 pi i k / n) as constants, the angle reduced to (-pi, pi]
template <int N, int K> struct PfW {
	static constexpr int k0 = ((K % N) + N) % N;
	static constexpr int k = (2 * k0 > N) ? k0 - N : k0;
	static constexpr double a = 6.283185307179586476925286766559 * k / N;
	static constexpr float c = (float)pf_cos_series(a);
	static constexpr float s = (float)pf_sin_series(a);
};

template <int I, int END, class F> __device__ __forceinline__ void pf_for(F&& f)
{
	if constexpr (I < END) {
		f(std::integral_constant<int, I>{});
		pf_for<I + 1, END>(f);
	}
}

template <int R, int SG> struct PfDft;

// odd primes: the pairs v[m] +- v[R - m] share their products
template <int R, int SG> struct PfPrime {
	__device__ __forceinline__ static void run(float2 (&v)[R])
	{
		constexpr int H = (R - 1) / 2;
		float2 t[H], d[H], o[R];
		float2 s = v[0];
#pragma unroll
		for (int m = 0; m < H; m++) {
			t[m] = cadd(v[m + 1], v[R - 1 - m]);
			d[m] = csub(v[m + 1], v[R - 1 - m]);
			s = cadd(s, t[m]);
		}
		o[0] = s;
		pf_for<1, H + 1>([&](auto kc) BAM_INLINE {
			constexpr int k = decltype(kc)::value;
			float2 a = v[0];
			float2 b = make_float2(0.f, 0.f);
			pf_for<1, H + 1>([&](auto mc) BAM_INLINE {
				constexpr int m = decltype(mc)::value;
				constexpr float c = PfW<R, m * k>::c, sn = SG * PfW<R, m * k>::s;
				a.x += c * t[m - 1].x;
				a.y += c * t[m - 1].y;
				// i sn d
				b.x -= sn * d[m - 1].y;
				b.y += sn * d[m - 1].x;
			});
			o[k] = cadd(a, b);
			o[R - k] = csub(a, b);
		});
#pragma unroll
		for (int m = 0; m < R; m++)
			v[m] = o[m];
	}
};

// R = A B: A-point DFTs over the points B apart, twiddles, B-point DFTs
template <int A, int B, int SG> struct PfComposite {
	__device__ __forceinline__ static void run(float2 (&v)[A * B])
	{
		float2 y[B][A];
		pf_for<0, B>([&](auto nc) BAM_INLINE {
			constexpr int n2 = decltype(nc)::value;
#pragma unroll
			for (int n1 = 0; n1 < A; n1++)
				y[n2][n1] = v[B * n1 + n2];
			PfDft<A, SG>::run(y[n2]);
			if constexpr (n2 > 0) {
				pf_for<1, A>([&](auto kc) BAM_INLINE {
					constexpr int k1 = decltype(kc)::value;
					using W = PfW<A * B, n2 * k1>;
					y[n2][k1] = cmul(y[n2][k1], make_float2(W::c, SG * W::s));
				});
			}
		});
#pragma unroll
		for (int k1 = 0; k1 < A; k1++) {
			float2 z[B];
#pragma unroll
			for (int n2 = 0; n2 < B; n2++)
				z[n2] = y[n2][k1];
			PfDft<B, SG>::run(z);
#pragma unroll
			for (int k2 = 0; k2 < B; k2++)
				v[k1 + A * k2] = z[k2];
		}
	}
};

template <int R, int SG> struct PfDft {
	__device__ __forceinline__ static void run(float2 (&v)[R])
	{
		if constexpr (2 == R || 3 == R || 4 == R || 5 == R || 8 == R || 16 == R)
			Dft<R>::run(v, (float)SG);
		else if constexpr (7 == R || 11 == R || 13 == R)
			PfPrime<R, SG>::run(v);
		else if constexpr (6 == R)
			PfComposite<2, 3, SG>::run(v);
		else if constexpr (9 == R)
			PfComposite<3, 3, SG>::run(v);
		else if constexpr (10 == R)
			PfComposite<2, 5, SG>::run(v);
		else if constexpr (12 == R)
			PfComposite<4, 3, SG>::run(v);
		else if constexpr (14 == R)
			PfComposite<2, 7, SG>::run(v);
		else
			PfComposite<3, 5, SG>::run(v);
	}
};

// The value recomputed here: keeps the addresses of the radix cases from
// being hoisted out of the loops around them (all fifteen cases' at once).
__device__ __forceinline__ int pf_fresh(int x)
{
	asm volatile("" : "+v"(x));
	return x;
}

__device__ __forceinline__ int pf_fresh_s(int x)
{
	asm volatile("" : "+s"(x));
	return x;
}

// f with the radix as a constant
template <class F> __device__ __forceinline__ void pf_switch(int r, F&& f)
{
#define BAM_PF(R) case R: f(std::integral_constant<int, R>{}); break
	switch (r) {
		BAM_PF(2);
		BAM_PF(3);
		BAM_PF(4);
		BAM_PF(5);
		BAM_PF(6);
		BAM_PF(7);
		BAM_PF(8);
		BAM_PF(9);
		BAM_PF(10);
		BAM_PF(11);
		BAM_PF(12);
		BAM_PF(13);
		BAM_PF(14);
		BAM_PF(15);
		BAM_PF(16);
	default:
		break;
	}
#undef BAM_PF
}

// ---------------------------------------------------------------------------
// One lane of a transform
// ---------------------------------------------------------------------------

template <bool ROWS> struct PfLane {

	float2* ls;          // the transform's points in LDS
	const float2* tw;    // exp(-2 pi i k / n), in LDS
	int n, logP;
	int j;               // the lane's butterfly
	bool in;             // the lane has a transform

	__device__ __forceinline__ int at(int k) const { return ROWS ? k + (k >> 3) : k << logP; }

	template <int SG> __device__ __forceinline__ float2 twiddle(float2 x, int i) const
	{
		const float2 w = tw[i];
		return (SG > 0) ? cmulc(x, w) : cmul(x, w);
	}

	// the butterfly of the first pass to LDS
	template <int R> __device__ __forceinline__ void put(const float2 (&v)[R]) const
	{
		const int jj = pf_fresh(j);
#pragma unroll
		for (int q = 0; q < R; q++)
			ls[at(jj * R + q)] = v[q];
	}

	// last pass: inputs with twiddles, DFT; v[q] is point j + q n / R
	template <int R, int SG> __device__ __forceinline__ void last(float2 (&v)[R]) const
	{
		const int nR = pf_fresh_s(n) / R;
		const int jj = pf_fresh(j);
#pragma unroll
		for (int r = 0; r < R; r++) {
			v[r] = ls[at(jj + r * nR)];
			if (r > 0)
				v[r] = twiddle<SG>(v[r], r * jj);
		}
		PfDft<R, SG>::run(v);
	}

	// middle pass of three, in place: sub-transforms of length Ns built, f
	// divides by Ns, n / (Ns R) = step
	template <int SG> __device__ __forceinline__ void middle(int radix, int Ns, const FastDiv& f, int step) const
	{
		pf_switch(radix, [&](auto rc) BAM_INLINE {
			constexpr int R = decltype(rc)::value;
			const int nR = pf_fresh_s(n) / R;
			const int j = pf_fresh(this->j);
			const bool act = in && j < nR;
			float2 v[R];
			int dst = 0;

			if (act) {
				uint32_t jb, k;
				f.divmod((uint32_t)j, jb, k);
				dst = (int)jb * Ns * R + (int)k;
				const int i0 = (int)k * step;
#pragma unroll
				for (int r = 0; r < R; r++) {
					v[r] = ls[at(j + r * nR)];
					if (r > 0)
						v[r] = twiddle<SG>(v[r], r * i0);
				}
				PfDft<R, SG>::run(v);
			}

			lds_barrier();

			if (act)
#pragma unroll
				for (int q = 0; q < R; q++)
					ls[at(dst + q * Ns)] = v[q];
		});

		lds_barrier();
	}
};

// LDS: the transforms, the twiddles, the two linear-phase tables (x rolloff of
// the axis: a real factor of both, of a split's input and a merge's output)
__device__ __forceinline__ void pf_tables(const PairArgs& a, float2* tw, float2* l, const float* roll)
{
	const int n = a.pl.n;

	for (int i = threadIdx.x; i < n; i += blockDim.x) {
		const float r = (nullptr != roll) ? roll[i] : 1.f;
		tw[i] = a.pl.tw[i];
		l[i] = cscale(a.l[0][i], r);
		l[n + i] = cscale(a.l[1][i], r);
	}
}

// PF_SPLIT_PSF: the split of a plan's only axis, x the PSFs (rows; a mode of its
// own: with the product as a branch in the split, the split of 128^3, 16 coils
// took 196 instead of 211 us but the two passes after it 327 and 305 instead of
// 310 and 294)
enum { PF_SPLIT = 0, PF_MERGE = 1, PF_TURN = 2, PF_SPLIT_PSF = 3 };

constexpr bool pf_is_split(int mode) { return PF_SPLIT == mode || PF_SPLIT_PSF == mode; }

// Rows: half of a work-group's waves take member b = 0, the other half b = 1,
// and a merge's second member hands its points over through LDS, at the
// positions the same lane has read last.  (Twice the waves in flight: the
// passes of a single 2-D problem have one to four waves per SIMD, which wait
// for a lane's chain of loads, DFTs and exchanges: merge of 256^2 with 8 coils
// 15.4 -> 12.1 us, of 96 x 80 x 60 with 6 coils 37.8 -> 36.2.)  Columns: one
// member after the other in the same lanes (as halves of a work-group, 256^2:
// turn 18.5 -> 16.0 us, but 96 x 80 x 60: turn 98 -> 136, merge 29 -> 45,
// split 28 -> 35 us).

// radix of the first or last pass as a constant, n / R and the lane's
// butterfly; `act`: the lane has one
#define BAM_PF_PASS(radix)                                                  \
	pf_switch(radix, [&](auto rc) BAM_INLINE {                          \
		constexpr int R = decltype(rc)::value;                      \
		const int nR = pf_fresh_s(a.pl.n) / R, j = pf_fresh(t.j);   \
		const bool act = t.in && j < nR;
#define BAM_PF_END })

// ---------------------------------------------------------------------------
// Strided axis: P adjacent columns of a volume per work-group, in place
// ---------------------------------------------------------------------------

// work-group -> column group, outer index, volume.  Turn: the volumes of a
// column group one after the other (coils share its PSF columns); otherwise
// neighbouring column groups
__device__ __forceinline__ void pf_column(int mode, const PairArgs& a, uint32_t w, uint32_t& cg, uint32_t& o,
					  uint32_t& v)
{
	uint32_t r;

	if (PF_TURN == mode) {
		a.f_nvol.divmod(w, r, v);
		a.f_ncg.divmod(r, o, cg);
	} else {
		a.f_ncg.divmod(w, r, cg);
		a.f_outer.divmod(r, v, o);
	}
}

template <int MODE, bool MID>
__device__ __forceinline__ void pair_cols_block(const PairArgs& a, uint32_t w, float2* lds)
{
	const int n = a.pl.n;
	const int size = a.P * n;
	float2* tw = lds + size;
	float2* lin = tw + n;

	uint32_t cg, o, v;
	pf_column(MODE, a, w, cg, o, v);

	const uint32_t inner = a.va.inner;
	const int p = threadIdx.x & (a.P - 1);
	const uint32_t i = cg * a.P + p;
	PfLane<false> t;
	t.ls = lds + p;
	t.tw = tw;
	t.n = n;
	t.logP = a.logP;
	t.j = threadIdx.x >> a.logP;
	t.in = i < inner;
	const long vol0 = (long)inner * n * o + i;  // of the column, in its volume
	float2* col = a.grid + (long)v * a.va.N + vol0;
	const int r0 = a.pl.rad[0];
	const int nr = a.pl.nr;
	const int rl = a.pl.rad[nr - 1];

	if constexpr (PF_SPLIT == MODE) {

		float2 h[PF_MAXR];

		BAM_PF_PASS(r0)
			if (act) {
				const float2* q = col + (long)inner * j;
				const long step = (long)inner * nR;
#pragma unroll
				for (int r = 0; r < R; r++)
					h[r] = q[r * step];
			}
		BAM_PF_END;

		pf_tables(a, tw, lin, nullptr);

		// fftmod of the other axes of this column
		float2 fo = make_float2(1.f, 0.f);
		const float2* fma = nullptr;

		if (nullptr != a.fm[0]) {
			int c[3];
			a.va.coords(t.in ? i : 0, o, 0, c);
#pragma unroll
			for (int d = 0; d < 3; d++) {
				if (d == a.va.axis)
					fma = a.fm[d];
				else
					fo = cmul(fo, a.fm[d][c[d]]);
			}
		}

		lds_barrier();

#pragma unroll 1
		for (int b = 0; b < 2; b++) {

			float2* out = col + b * a.half;
			const float2* lb = lin + b * n;

			auto store = [&](int k, float2 x) BAM_INLINE {
				if (nullptr != fma)
					x = cmul(x, cmul(fo, fma[k]));
				out[(long)inner * k] = x;
			};

			if (b > 0)
				lds_barrier();  // the first member's last pass has read LDS

			BAM_PF_PASS(r0)
				if (act) {
					float2 x[R];
#pragma unroll
					for (int r = 0; r < R; r++)
						x[r] = cmul(h[r], lb[j + r * nR]);
					PfDft<R, -1>::run(x);
					if (1 == nr) {
#pragma unroll
						for (int q = 0; q < R; q++)
							store(q, x[q]);
					} else {
						t.put(x);
					}
				}
			BAM_PF_END;

			if (1 == nr)
				continue;

			lds_barrier();

			if constexpr (MID)
				t.template middle<-1>(a.pl.rad[1], r0, a.pl.fF, rl);

			BAM_PF_PASS(rl)
				if (act) {
					float2 x[R];
					t.template last<R, -1>(x);
#pragma unroll
					for (int q = 0; q < R; q++)
						store(j + q * nR, x[q]);
				}
			BAM_PF_END;
		}

	} else {

		float2 acc[PF_MAXR];
#pragma unroll
		for (int q = 0; q < PF_MAXR; q++)
			acc[q] = make_float2(0.f, 0.f);

		// radix of the last backward pass
		const int re = (PF_TURN == MODE) ? r0 : rl;

		pf_tables(a, tw, lin, nullptr);
		lds_barrier();

#pragma unroll 1
		for (int b = 0; b < 2; b++) {

			const float2* lb = lin + b * n;

			const float2* in = (PF_MERGE == MODE) ? col + b * a.half : col;

			// first pass, forward or backward
			BAM_PF_PASS(r0)
				float2 x[R];
				if (act) {
					const float2* g = in + (long)inner * j;
					const long step = (long)inner * nR;
#pragma unroll
					for (int r = 0; r < R; r++)
						x[r] = g[r * step];
					if constexpr (PF_TURN == MODE)
#pragma unroll
						for (int r = 0; r < R; r++)
							x[r] = cmul(x[r], lb[j + r * nR]);
					PfDft<R, (PF_TURN == MODE) ? -1 : 1>::run(x);
				}
				if (nr > 1) {
					if (b > 0)
						lds_barrier();
					if (act)
						t.put(x);
				} else if (act) {
					if constexpr (PF_TURN == MODE) {
						const float2* q = a.psf + (long)a.f_C.div(v) * a.va.N + vol0 + b * a.psf_half;
#pragma unroll
						for (int r = 0; r < R; r++)
							x[r] = cmul(x[r], q[(long)inner * r]);
						PfDft<R, 1>::run(x);
					}
#pragma unroll
					for (int q = 0; q < R; q++)
						acc[q] = cadd(acc[q], cmulc(x[q], lb[q]));
				}
			BAM_PF_END;

			if (1 == nr)
				continue;

			if constexpr (PF_TURN == MODE) {

				// the PSF values of the lane's last-pass points, with two
				// radices in flight across the exchange (with three the
				// registers are short)
				float2 ps[PF_MAXR];
				const float2* psf = a.psf + (long)a.f_C.div(v) * a.va.N + vol0 + b * a.psf_half;

				auto load_psf = [&](auto rc, int j, int nR) BAM_INLINE {
					constexpr int R = decltype(rc)::value;
					const float2* q = psf + (long)inner * j;
					const long step = (long)inner * nR;
#pragma unroll
					for (int r = 0; r < R; r++)
						ps[r] = q[r * step];
				};

				if constexpr (!MID) {
					BAM_PF_PASS(rl)
						if (act)
							load_psf(rc, j, nR);
					BAM_PF_END;
				}

				lds_barrier();

				if constexpr (MID)
					t.template middle<-1>(a.pl.rad[1], r0, a.pl.fF, rl);

				// last forward pass, PSF, first backward pass (the radices
				// run backward from here)
				BAM_PF_PASS(rl)
					float2 x[R];
					if (act) {
						if constexpr (MID)
							load_psf(rc, j, nR);
						t.template last<R, -1>(x);
#pragma unroll
						for (int q = 0; q < R; q++)
							x[q] = cmul(x[q], ps[q]);
						PfDft<R, 1>::run(x);
					}
					lds_barrier();
					if (act)
						t.put(x);
				BAM_PF_END;
			}

			lds_barrier();

			if constexpr (MID) {
				if (PF_TURN == MODE)
					t.template middle<1>(a.pl.rad[1], rl, a.pl.fB, r0);
				else
					t.template middle<1>(a.pl.rad[1], r0, a.pl.fF, rl);
			}

			BAM_PF_PASS(re)
				if (act) {
					float2 x[R];
					t.template last<R, 1>(x);
#pragma unroll
					for (int q = 0; q < R; q++)
						acc[q] = cadd(acc[q], cmulc(x[q], lb[j + q * nR]));
				}
			BAM_PF_END;
		}

		BAM_PF_PASS(re)
			if (act) {
				float2* q = col + (long)inner * j;
				const long step = (long)inner * nR;
#pragma unroll
				for (int r = 0; r < R; r++)
					q[r * step] = acc[r];
			}
		BAM_PF_END;
	}
}

// ---------------------------------------------------------------------------
// Strided axis of a length n = RA RB with RB | RA (32, 64, 128, 256): RB lanes
// hold a column, RA points j + r RB each.  These are the inputs of one radix-RA
// butterfly of the first pass and, for the RA / RB radix-RB butterflies of the
// last pass, its outputs: every lane works in both passes, the points of a
// forward transform are those that the backward one starts from, and nothing
// but the exchange between the two passes goes through LDS.  With the radix in
// the code: the general kernel above switches on it around every pass, and n =
// 128 = 8 x 16 leaves half of its lanes idle in one of the two.
// Split and merge are bound by HBM (128^3, 16 coils, between 2 and 4 volumes
// per coil: 1.6 GB in 290 us), the turn by its vector instructions (4
// transforms per point: 999 us in the general kernel, 914 with the passes of
// the strided FFT, 665 here); 256^2, 8 coils: 16 -> 13.6 us.  One Toeplitz
// operator on coil images, against whole x-y slices in LDS (the z axis after
// them) for 128^3, 16 coils: 1842 -> 1665 us; 64^3: 232 -> 172; 32^3: 73 -> 68.
// ---------------------------------------------------------------------------

template <int MODE, int RA, int RB>
__device__ __forceinline__ void pair_cols_fixed(const PairArgs& a, uint32_t w, float2* lds)
{
	constexpr int N = RA * RB, K = RA / RB;
	static_assert(0 == RA % RB, "the last pass takes whole lanes");
	float2* tw = lds + PF_FP * N;
	float2* lin = tw + N;

	uint32_t cg, o, v;
	pf_column(MODE, a, w, cg, o, v);

	const uint32_t inner = a.va.inner;
	const int p = threadIdx.x & (PF_FP - 1);
	const int j = threadIdx.x / PF_FP;
	const uint32_t i = cg * PF_FP + p;
	const bool in = i < inner;
	float2* ls = lds + p;
	const long vol0 = (long)inner * N * o + i + (long)inner * j;  // the lane's first point
	float2* col = a.grid + (long)v * a.va.N + vol0;
	const long step = (long)inner * RB;

	auto load = [&](float2 (&x)[RA], const float2* q) BAM_INLINE {
#pragma unroll
		for (int r = 0; r < RA; r++)
			x[r] = in ? q[r * step] : make_float2(0.f, 0.f);
	};

	auto put = [&](const float2 (&x)[RA]) BAM_INLINE {
#pragma unroll
		for (int q = 0; q < RA; q++)
			ls[(j * RA + q) * PF_FP] = x[q];
	};

	// butterfly m of the last pass: f(r, point j + r RB)
	auto last = [&](auto sg, auto&& f) BAM_INLINE {
		constexpr int SG = decltype(sg)::value;
#pragma unroll
		for (int m = 0; m < K; m++) {
			const int jb = j + m * RB;
			float2 y[RB];
#pragma unroll
			for (int r = 0; r < RB; r++) {
				y[r] = ls[(jb + r * RA) * PF_FP];
				if (r > 0)
					y[r] = (SG > 0) ? cmulc(y[r], tw[r * jb]) : cmul(y[r], tw[r * jb]);
			}
			PfDft<RB, SG>::run(y);
#pragma unroll
			for (int q = 0; q < RB; q++)
				f(m + K * q, y[q]);
		}
	};

	using Fwd = std::integral_constant<int, -1>;
	using Bwd = std::integral_constant<int, 1>;

	if constexpr (PF_SPLIT == MODE) {

		float2 h[RA];
		load(h, col);
		pf_tables(a, tw, lin, nullptr);

		// fftmod of the other axes of this column
		float2 fo = make_float2(1.f, 0.f);
		const float2* fma = nullptr;

		if (nullptr != a.fm[0]) {
			int c[3];
			a.va.coords(in ? i : 0, o, 0, c);
#pragma unroll
			for (int d = 0; d < 3; d++) {
				if (d == a.va.axis)
					fma = a.fm[d];
				else
					fo = cmul(fo, a.fm[d][c[d]]);
			}
		}

		lds_barrier();

#pragma unroll 1
		for (int b = 0; b < 2; b++) {

			const float2* lb = lin + b * N + j;
			float2 x[RA];
#pragma unroll
			for (int r = 0; r < RA; r++)
				x[r] = cmul(h[r], lb[r * RB]);
			PfDft<RA, -1>::run(x);

			if (b > 0)
				lds_barrier();  // the first member's last pass has read LDS

			put(x);
			lds_barrier();

			float2* out = col + b * a.half;

			last(Fwd{}, [&](int r, float2 y) BAM_INLINE {
				if (nullptr != fma)
					y = cmul(y, cmul(fo, fma[j + r * RB]));
				if (in)
					out[r * step] = y;
			});
		}

	} else if constexpr (PF_MERGE == MODE) {

		// both members' loads in flight
		float2 x[RA], x1[RA];
		load(x, col);
		load(x1, col + a.half);
		pf_tables(a, tw, lin, nullptr);
		PfDft<RA, 1>::run(x);
		put(x);
		lds_barrier();

		const float2* lb = lin + j;
		float2 acc[RA];
		last(Bwd{}, [&](int r, float2 y) BAM_INLINE { acc[r] = cmulc(y, lb[r * RB]); });

		PfDft<RA, 1>::run(x1);
		lds_barrier();
		put(x1);
		lds_barrier();

		last(Bwd{}, [&](int r, float2 y) BAM_INLINE {
			if (in)
				col[r * step] = cadd(acc[r], cmulc(y, lb[N + r * RB]));
		});

	} else {

		float2 h[RA], acc[RA];
		load(h, col);
		pf_tables(a, tw, lin, nullptr);
#pragma unroll
		for (int r = 0; r < RA; r++)
			acc[r] = make_float2(0.f, 0.f);
		lds_barrier();

		const float2* psf = a.psf + (long)a.f_C.div(v) * a.va.N + vol0;

#pragma unroll 1
		for (int b = 0; b < 2; b++) {

			const float2* lb = lin + b * N + j;
			float2 x[RA];
#pragma unroll
			for (int r = 0; r < RA; r++)
				x[r] = cmul(h[r], lb[r * RB]);
			PfDft<RA, -1>::run(x);

			if (b > 0)
				lds_barrier();

			put(x);
			float2 ps[RA];
			load(ps, psf + b * a.psf_half);  // in flight across the exchange
			lds_barrier();
			last(Fwd{}, [&](int r, float2 y) BAM_INLINE { x[r] = cmul(y, ps[r]); });
			PfDft<RA, 1>::run(x);
			lds_barrier();
			put(x);
			lds_barrier();
			last(Bwd{}, [&](int r, float2 y) BAM_INLINE { acc[r] = cadd(acc[r], cmulc(y, lb[r * RB])); });
		}

#pragma unroll
		for (int r = 0; r < RA; r++)
			if (in)
				col[r * step] = acc[r];
	}
}

// ---------------------------------------------------------------------------
// First axis: P rows of the image per work-group.  Split: coil image c (or
// image x map c) x rolloff into volumes c and c + C; merge: the volumes of the
// coils of a group back to the coil image, or conj(map) x summed over the
// group into its partial image (no atomics, fixed order).
// ---------------------------------------------------------------------------

// rolloff and fftmod of the other axes of a row, fftmod table along it (null:
// no fftmod)
__device__ __forceinline__ void pf_row_factors(const PairArgs& a, uint32_t row, float& rr, float2& fo,
					       const float2*& fma)
{
	rr = 1.f;
	fo = make_float2(1.f, 0.f);
	fma = nullptr;

	if (nullptr == a.roll[0] && nullptr == a.fm[0])
		return;

	// along x: (y, z); along y: z (along z there is one row)
	uint32_t c1 = row, c2 = row;
	if (0 == a.va.axis)
		a.va.f_n1.divmod(row, c2, c1);
	const int c[3] = { 0, (int)c1, (int)c2 };
#pragma unroll
	for (int d = 0; d < 3; d++) {
		if (nullptr != a.roll[0] && d != a.va.axis)
			rr *= a.roll[d][c[d]];
		if (nullptr != a.fm[0]) {
			if (d == a.va.axis)
				fma = a.fm[d];
			else
				fo = cmul(fo, a.fm[d][c[d]]);
		}
	}
}

template <int MODE, bool MID>
__device__ __forceinline__ void pair_rows_block(const PairArgs& a, uint32_t w, float2* lds)
{
	const int n = a.pl.n;
	const int size = a.P * a.pitch;
	float2* tw = lds + 2 * size;
	float2* lin = tw + n;

	uint32_t rg, u, p, jj;
	a.f_ncg.divmod(w, u, rg);  // u: coil, or coil group
	const int b = __builtin_amdgcn_readfirstlane((int)threadIdx.x >= a.group ? 1 : 0);
	a.pl.fNJ.divmod(threadIdx.x - (uint32_t)(b * a.group), p, jj);

	const uint32_t row = rg * a.P + p;
	const long N = a.va.N;
	PfLane<true> t;
	t.ls = lds + b * size + p * a.pitch;
	t.tw = tw;
	t.n = n;
	t.logP = 0;
	t.j = (int)jj;
	t.in = (int)p < a.P && row < a.va.outer;
	const long ro = (long)row * n;
	const int r0 = a.pl.rad[0];
	const int nr = a.pl.nr;
	const int rl = a.pl.rad[nr - 1];
	const float2* lb = lin + b * n;
	float2 h[PF_MAXR];

	if constexpr (pf_is_split(MODE)) {

		const float2* im = (nullptr != a.sens) ? a.src + ro : a.src + (long)u * N + ro;
		const float2* mp = (nullptr != a.sens) ? a.sens + (long)u * N + ro : nullptr;

		BAM_PF_PASS(r0)
			if (act) {
#pragma unroll
				for (int r = 0; r < R; r++)
					h[r] = im[j + r * nR];
				if (nullptr != mp) {
					float2 m[R];
#pragma unroll
					for (int r = 0; r < R; r++)
						m[r] = mp[j + r * nR];
#pragma unroll
					for (int r = 0; r < R; r++)
						h[r] = cmul(h[r], m[r]);
				}
			}
		BAM_PF_END;

	}

	pf_tables(a, tw, lin, a.roll[a.va.axis]);

	float rr;
	float2 fo;
	const float2* fma;
	pf_row_factors(a, t.in ? row : 0, rr, fo, fma);

	lds_barrier();

	if constexpr (pf_is_split(MODE)) {

		float2* out = a.grid + (long)u * N + ro + b * a.half;
		const float2* psf = a.psf + ro + b * a.psf_half;

		auto store = [&](int k, float2 x) BAM_INLINE {
			if (nullptr != fma)
				x = cmul(x, cmul(fo, fma[k]));
			if constexpr (PF_SPLIT_PSF == MODE)
				x = cmul(x, psf[k]);
			out[k] = x;
		};

		BAM_PF_PASS(r0)
			if (act) {
				float2 x[R];
#pragma unroll
				for (int r = 0; r < R; r++)
					x[r] = cscale(cmul(h[r], lb[j + r * nR]), rr);
				PfDft<R, -1>::run(x);
				if (1 == nr) {
#pragma unroll
					for (int q = 0; q < R; q++)
						store(q, x[q]);
				} else {
					t.put(x);
				}
			}
		BAM_PF_END;

		if (1 == nr)
			return;

		lds_barrier();

		if constexpr (MID)
			t.template middle<-1>(a.pl.rad[1], r0, a.pl.fF, rl);

		BAM_PF_PASS(rl)
			if (act) {
				float2 x[R];
				t.template last<R, -1>(x);
#pragma unroll
				for (int q = 0; q < R; q++)
					store(j + q * nR, x[q]);
			}
		BAM_PF_END;

	} else {

		float2 acc[PF_MAXR];
#pragma unroll
		for (int q = 0; q < PF_MAXR; q++)
			acc[q] = make_float2(0.f, 0.f);

		// the coils of the group
#pragma unroll 1
		for (int m = 0; m < a.cc; m++) {

			const float2* mp = (nullptr != a.sens) ? a.sens + ((long)u * a.cc + m) * N + ro : nullptr;

			auto part = [&](float2 x, int k) BAM_INLINE {
				x = cmulc(x, lb[k]);
				return (nullptr != mp) ? cmulc(x, mp[k]) : x;
			};

			const float2* in = a.grid + ((long)u * a.cc + m) * N + b * a.half + ro;

			BAM_PF_PASS(r0)
				float2 x[R];
				if (act) {
#pragma unroll
					for (int r = 0; r < R; r++)
						x[r] = in[j + r * nR];
					PfDft<R, 1>::run(x);
				}
				if (nr > 1) {
					if (m > 0)
						lds_barrier();
					if (act)
						t.put(x);
				} else if (act) {
#pragma unroll
					for (int q = 0; q < R; q++)
						acc[q] = cadd(acc[q], part(x[q], q));
				}
			BAM_PF_END;

			if (1 == nr)
				continue;

			lds_barrier();

			if constexpr (MID)
				t.template middle<1>(a.pl.rad[1], r0, a.pl.fF, rl);

			BAM_PF_PASS(rl)
				if (act) {
					float2 x[R];
					t.template last<R, 1>(x);
#pragma unroll
					for (int q = 0; q < R; q++)
						acc[q] = cadd(acc[q], part(x[q], j + q * nR));
				}
			BAM_PF_END;
		}

		// sum of the members
		if (b > 0) {
			BAM_PF_PASS(rl)
				if (act)
#pragma unroll
					for (int q = 0; q < R; q++)
						t.ls[t.at(j + q * nR)] = acc[q];
			BAM_PF_END;
		}

		lds_barrier();

		if (0 == b) {

			float2* out = a.dst + (long)u * N + ro;

			BAM_PF_PASS(rl)
				if (act)
#pragma unroll
					for (int q = 0; q < R; q++) {
						const int k = j + q * nR;
						out[k] = cscale(cadd(acc[q], t.ls[size + t.at(k)]), rr);
					}
			BAM_PF_END;
		}
	}
}

// ---------------------------------------------------------------------------
// First axis of such a length: RB lanes per row and member, the two members of
// a row in the same wave.  A row never leaves its wave, so its exchange needs
// no barrier, and a merge's next coil is loaded while the present one is
// transformed (the coils of a group follow one another in the same lanes).
// 128^3, 16 coils with maps: merge 444 us in the general kernel, 180 here (0.8
// GB); split 235 -> 212.  CG of 256^2, 8 coils, 30 iterations: rows and columns
// together 1.96 -> 1.61 ms.
// ---------------------------------------------------------------------------

// LDS of a wave's own rows, written and read by its lanes
__device__ __forceinline__ void pf_wave_sync()
{
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
	__builtin_amdgcn_wave_barrier();
	__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int MODE, int RA, int RB>
__device__ __forceinline__ void pair_rows_fixed(const PairArgs& a, uint32_t w, float2* lds)
{
	constexpr int n = RA * RB, K = RA / RB;
	constexpr int PITCH = pf_row_pitch(n);
	const int P = a.P;  // of a batch's work-group maybe not all waves
	float2* tw = lds + 2 * P * PITCH;
	float2* lin = tw + n;

	uint32_t rg, u;
	a.f_ncg.divmod(w, u, rg);  // u: coil, or coil group
	const int tr = threadIdx.x / RB;  // transform of the work-group: row, member
	const int j = threadIdx.x % RB;
	const int b = tr & 1;
	const uint32_t row = rg * P + (tr >> 1);
	const bool in = tr < 2 * P && row < a.va.outer;
	const long N = a.va.N;
	const long ro = (long)(in ? row : 0) * n + j;
	float2* ls = lds + tr * PITCH;
	const float2* lb = lin + b * n + j;

	auto load = [&](float2 (&x)[RA], const float2* q) BAM_INLINE {
#pragma unroll
		for (int r = 0; r < RA; r++)
			x[r] = q[r * RB];
	};

	auto at = [](int k) BAM_INLINE { return k + (k >> 3); };

	// DFT of x, exchange, last pass: f(r, point j + r RB)
	auto transform = [&](auto sg, float2 (&x)[RA], auto&& f) BAM_INLINE {
		constexpr int SG = decltype(sg)::value;
		PfDft<RA, SG>::run(x);
		pf_wave_sync();
#pragma unroll
		for (int q = 0; q < RA; q++)
			ls[at(j * RA + q)] = x[q];
		pf_wave_sync();
#pragma unroll
		for (int m = 0; m < K; m++) {
			const int jb = j + m * RB;
			float2 y[RB];
#pragma unroll
			for (int r = 0; r < RB; r++) {
				y[r] = ls[at(jb + r * RA)];
				if (r > 0)
					y[r] = (SG > 0) ? cmulc(y[r], tw[r * jb]) : cmul(y[r], tw[r * jb]);
			}
			PfDft<RB, SG>::run(y);
#pragma unroll
			for (int q = 0; q < RB; q++)
				f(m + K * q, y[q]);
		}
	};

	float2 x[RA];

	if constexpr (pf_is_split(MODE)) {

		load(x, ((nullptr != a.sens) ? a.src : a.src + (long)u * N) + ro);

		if (nullptr != a.sens) {
			float2 m[RA];
			load(m, a.sens + (long)u * N + ro);
#pragma unroll
			for (int r = 0; r < RA; r++)
				x[r] = cmul(x[r], m[r]);
		}
	} else {
		load(x, a.grid + (long)u * a.cc * N + b * a.half + ro);
	}

	pf_tables(a, tw, lin, a.roll[a.va.axis]);

	float rr;
	float2 fo;
	const float2* fma;
	pf_row_factors(a, in ? row : 0, rr, fo, fma);
	lds_barrier();

	if (tr >= 2 * P)
		return;  // a whole wave

	if constexpr (pf_is_split(MODE)) {

#pragma unroll
		for (int r = 0; r < RA; r++)
			x[r] = cscale(cmul(x[r], lb[r * RB]), rr);

		float2* out = a.grid + (long)u * N + ro + b * a.half;
		const float2* psf = a.psf + ro + b * a.psf_half;

		transform(std::integral_constant<int, -1>{}, x, [&](int r, float2 y) BAM_INLINE {
			if (nullptr != fma)
				y = cmul(y, cmul(fo, fma[j + r * RB]));
			if constexpr (PF_SPLIT_PSF == MODE)
				y = cmul(y, psf[r * RB]);
			if (in)
				out[r * RB] = y;
		});

	} else {

		float2 acc[RA];
#pragma unroll
		for (int r = 0; r < RA; r++)
			acc[r] = make_float2(0.f, 0.f);

#pragma unroll 1
		for (int m = 0; m < a.cc; m++) {

			const long c = (long)u * a.cc + m;
			float2 xn[RA], mp[RA];

			if (nullptr != a.sens)
				load(mp, a.sens + c * N + ro);

			if (m + 1 < a.cc)
				load(xn, a.grid + (c + 1) * N + b * a.half + ro);

			transform(std::integral_constant<int, 1>{}, x, [&](int r, float2 y) BAM_INLINE {
				y = cmulc(y, lb[r * RB]);
				if (nullptr != a.sens)
					y = cmulc(y, mp[r]);
				acc[r] = cadd(acc[r], y);
			});

			if (m + 1 < a.cc)
#pragma unroll
				for (int r = 0; r < RA; r++)
					x[r] = xn[r];
		}

		// sum of the members: each takes half of the points
		float2* out = a.dst + (long)u * N + ro + b * (n / 2);

#pragma unroll
		for (int r = 0; r < RA / 2; r++) {
			const float2 own = (b > 0) ? acc[r + RA / 2] : acc[r];
			const float2 oth = (b > 0) ? acc[r] : acc[r + RA / 2];
			const float2 rec = make_float2(__shfl_xor(oth.x, RB), __shfl_xor(oth.y, RB));
			if (in)
				out[r * RB] = cscale(cadd(own, rec), rr);
		}
	}
}

#undef BAM_PF_PASS
#undef BAM_PF_END

// work-groups are dealt to the 8 XCDs in turn: each XCD takes a contiguous
// part of the work, so that neighbours share its L2
__device__ __forceinline__ uint32_t pf_xcd_order(uint32_t b, uint32_t nblk)
{
	const uint32_t q = nblk >> 3, r = nblk & 7, x = b & 7;
	return x * q + min(x, r) + (b >> 3);
}

template <int MODE, bool ROWS, bool MID>
__device__ __forceinline__ void pair_block(const PairArgs& a, uint32_t w, float2* lds)
{
	if (nullptr != a.skip && 0 != *a.skip)
		return;

	if constexpr (ROWS)
		pair_rows_block<MODE, MID>(a, w, lds);
	else
		pair_cols_block<MODE, MID>(a, w, lds);
}

template <int MODE, bool ROWS, bool MID>
__global__ __launch_bounds__(pf_threads(ROWS, MID)) void k_pair(PairArgs a)
{
	extern __shared__ float2 pf_lds[];
	pair_block<MODE, ROWS, MID>(a, pf_xcd_order(blockIdx.x, gridDim.x), pf_lds);
}

template <int MODE, bool ROWS, int RA, int RB>
__device__ __forceinline__ void pair_fixed_block(const PairArgs& a, uint32_t w, float2* lds)
{
	if (nullptr != a.skip && 0 != *a.skip)
		return;

	if constexpr (ROWS)
		pair_rows_fixed<MODE, RA, RB>(a, w, lds);
	else
		pair_cols_fixed<MODE, RA, RB>(a, w, lds);
}

template <int MODE, bool ROWS, int RA, int RB>
__global__ __launch_bounds__(ROWS ? 256 : PF_FP * RB) void k_pair_fixed(PairArgs a)
{
	extern __shared__ float2 pf_lds[];
	pair_fixed_block<MODE, ROWS, RA, RB>(a, pf_xcd_order(blockIdx.x, gridDim.x), pf_lds);
}

// one pass of many plans in one launch: btab[b] = (plan, its work-group)
template <int MODE, bool ROWS, bool MID>
__global__ __launch_bounds__(pf_threads(ROWS, MID)) void k_pair_batch(const PairArgs* __restrict__ items,
										const int2* __restrict__ btab)
{
	extern __shared__ float2 pf_lds[];
	const int2 e = btab[blockIdx.x];
	pair_block<MODE, ROWS, MID>(items[e.x], (uint32_t)e.y, pf_lds);
}

template <int MODE, bool ROWS, int RA, int RB>
__global__ __launch_bounds__(ROWS ? 256 : PF_FP * RB) void k_pair_fixed_batch(const PairArgs* __restrict__ items,
									     const int2* __restrict__ btab)
{
	extern __shared__ float2 pf_lds[];
	const int2 e = btab[blockIdx.x];
	pair_fixed_block<MODE, ROWS, RA, RB>(items[e.x], (uint32_t)e.y, pf_lds);
}

// launches (pair.hip)
void pair_launch(int mode, bool rows, const PairArgs& a, const char* name, hipStream_t st);
void pair_launch_batch(int mode, bool rows, int cl, const PairArgs* items, const int2* btab, int nblk,
		       unsigned threads, size_t lds, const char* name, hipStream_t st);

}  // namespace bam
