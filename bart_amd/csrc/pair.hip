// pair.hip -- host side of the pair passes: radices, work-group geometry,
// launches.
#include "pair.hpp"

#include <algorithm>

namespace bam {

// n as at most three radices of 2 .. 16, the smallest as large as possible
// (a transform takes n / (smallest radix) lanes), fewer radices first
PairPlan make_pair_plan(const AxisPlan& a)
{
	PairPlan p;
	const int n = a.n;
	p.n = n;
	p.tw = a.tw;

	if (n < 2 || n > PF_MAXN)
		return p;

	if (n <= PF_MAXR) {
		// 2 .. 16 are all radices
		p.nr = 1;
		p.rad[0] = n;
		p.rad[1] = p.rad[2] = 1;
	}

	// two: the larger one as small as possible
	for (int r = 2; r <= PF_MAXR && 0 == p.nr; r++)
		if (0 == n % r && n / r <= r) {
			p.nr = 2;
			p.rad[0] = n / r;
			p.rad[1] = r;
			p.rad[2] = 1;
		}

	int low = 1;

	for (int x = 2; x <= PF_MAXR && 2 != p.nr && 1 != p.nr; x++)
		for (int y = x; y <= PF_MAXR; y++) {
			if (0 != n % (x * y))
				continue;
			const int z = n / (x * y);
			if (z < y || z > PF_MAXR || x <= low)
				continue;
			low = x;
			p.nr = 3;
			p.rad[0] = x;
			p.rad[1] = y;
			p.rad[2] = z;
		}

	if (0 == p.nr)
		return p;

	for (int i = 0; i < p.nr; i++)
		p.NJ = std::max(p.NJ, n / p.rad[i]);

	if (p.NJ > 256) {
		p.nr = 0;
		return p;
	}

	p.fF = FastDiv((uint32_t)p.rad[0]);
	p.fB = FastDiv((uint32_t)p.rad[2]);
	p.fNJ = FastDiv((uint32_t)p.NJ);
	return p;
}

size_t pair_lds_bytes(const PairArgs& a, bool rows)
{
	return sizeof(float2) * ((size_t)a.P * (rows ? 2 * a.pitch : a.pl.n) + 3 * (size_t)a.pl.n);
}

unsigned pair_threads(const PairArgs& a, bool rows) { return (rows ? 2 : 1) * (unsigned)a.group; }

void pair_geometry(PairArgs& a, bool rows, uint32_t units, int ncu)
{
	const int n = a.pl.n;
	const int lim = pf_threads(rows, 3 == a.pl.nr) / (rows ? 2 : 1);  // lanes of a member
	const uint32_t count = rows ? a.va.outer : a.va.inner;
	int P = 1;

	a.cl = pf_class(n, a.pl.nr);

	if (a.cl >= PF_32) {
		const int RB = pf_fixed_lanes(a.cl);
		P = PF_FP;
		a.group = P * RB;

		if (rows) {
			// both members of a row in one wave; four waves per work-group,
			// one where that would leave compute units without a work-group
			// (Toeplitz normal, one and four: 64^2, 8 coils 31.1 and 31.9 us;
			// 128^2, 4 coils 36.5 and 37.7, 16 coils 39.5 and 39.8; from there
			// on four: 256^2, 8 coils 47.5 and 46.4, 32 coils 80.5 and 76.4;
			// 128^3, 4 coils 416 and 413)
			const int rw = 32 / RB;
			const int waves = ((long)units * count / (4 * rw) >= ncu) ? 4 : 1;
			P = rw * waves;
			a.group = 32 * waves;
		}
	} else if (rows) {
		// whole waves, twice as many once there are enough work-groups
		while (P * a.pl.NJ < 64 && 2 * P * a.pl.NJ <= lim)
			P *= 2;
		if ((long)units * (count / P) > 16l * ncu && 2 * P * a.pl.NJ <= lim)
			P *= 2;
	} else {
		// 16 columns (128-byte rows); 64 where a lane holds a whole transform
		const int want = (1 == a.pl.nr) ? 64 : 16;
		while (P < want && 2 * P * a.pl.NJ <= lim && 2l * P * n <= 8192)
			P *= 2;
	}

	a.P = P;
	a.logP = 0;
	while ((1 << a.logP) < P)
		a.logP++;
	if (a.cl < PF_32)
		a.group = (P * a.pl.NJ + 63) / 64 * 64;

	a.pitch = pf_row_pitch(n);
	a.ncg = (count + P - 1) / P;
	a.f_ncg = FastDiv(a.ncg);
	a.f_outer = FastDiv(a.va.outer);
	a.f_nvol = FastDiv((uint32_t)a.va.nvol);
	a.f_C = FastDiv((uint32_t)a.C);
	const long nblk = rows ? (long)a.ncg * units : (long)a.ncg * a.va.outer * a.va.nvol;
	BAM_CHECK(nblk < (1l << 31), "pair pass: too many work-groups");
	a.nblk = (uint32_t)nblk;
}

#define BAM_PF_CLASSES(cl, F)    \
	switch (cl) {            \
	case PF_32:              \
		F(8, 4);         \
		break;           \
	case PF_64:              \
		F(8, 8);         \
		break;           \
	case PF_128:             \
		F(16, 8);        \
		break;           \
	case PF_256:             \
		F(16, 16);       \
		break;           \
	default:                 \
		break;           \
	}

template <int MODE, bool ROWS>
static void launch_m(const PairArgs& a, hipStream_t st)
{
	const dim3 gb(a.nblk), tb(pair_threads(a, ROWS));
	const size_t lds = pair_lds_bytes(a, ROWS);

#define BAM_PF_FIXED(RA, RB) hipLaunchKernelGGL((k_pair_fixed<MODE, ROWS, RA, RB>), gb, tb, lds, st, a)
	if (a.cl >= PF_32)
		BAM_PF_CLASSES(a.cl, BAM_PF_FIXED)
	else if (PF_THREE == a.cl)
		hipLaunchKernelGGL((k_pair<MODE, ROWS, true>), gb, tb, lds, st, a);
	else
		hipLaunchKernelGGL((k_pair<MODE, ROWS, false>), gb, tb, lds, st, a);
#undef BAM_PF_FIXED
}

void pair_launch(int mode, bool rows, const PairArgs& a, const char* name, hipStream_t st)
{
	if (0 == a.nblk)
		return;

	BAM_CHECK(a.pl.nr >= 1 && a.pl.nr <= 3 && pair_lds_bytes(a, rows) <= 160 * 1024 &&
			  pair_threads(a, rows) <= (unsigned)pf_threads(rows, 3 == a.pl.nr),
		  "pair pass: no kernel for length %d", a.pl.n);
	ProfScope prof(name, st);

	if (rows) {
		if (PF_SPLIT == mode)
			launch_m<PF_SPLIT, true>(a, st);
		else if (PF_SPLIT_PSF == mode)
			launch_m<PF_SPLIT_PSF, true>(a, st);
		else
			launch_m<PF_MERGE, true>(a, st);
	} else {
		if (PF_SPLIT == mode)
			launch_m<PF_SPLIT, false>(a, st);
		else if (PF_MERGE == mode)
			launch_m<PF_MERGE, false>(a, st);
		else
			launch_m<PF_TURN, false>(a, st);
	}

	BAM_HIP(hipGetLastError());
}

template <int MODE, bool ROWS>
static void launch_b(int cl, const PairArgs* items, const int2* btab, dim3 gb, dim3 tb, size_t lds, hipStream_t st)
{
#define BAM_PF_FIXED(RA, RB) \
	hipLaunchKernelGGL((k_pair_fixed_batch<MODE, ROWS, RA, RB>), gb, tb, lds, st, items, btab)
	if (cl >= PF_32)
		BAM_PF_CLASSES(cl, BAM_PF_FIXED)
	else if (PF_THREE == cl)
		hipLaunchKernelGGL((k_pair_batch<MODE, ROWS, true>), gb, tb, lds, st, items, btab);
	else
		hipLaunchKernelGGL((k_pair_batch<MODE, ROWS, false>), gb, tb, lds, st, items, btab);
#undef BAM_PF_FIXED
}

void pair_launch_batch(int mode, bool rows, int cl, const PairArgs* items, const int2* btab, int nblk,
		       unsigned threads, size_t lds, const char* name, hipStream_t st)
{
	if (nblk <= 0)
		return;

	ProfScope prof(name, st);
	const dim3 gb((unsigned)nblk), tb(threads);

	if (rows && PF_SPLIT == mode)
		launch_b<PF_SPLIT, true>(cl, items, btab, gb, tb, lds, st);
	else if (rows)
		launch_b<PF_MERGE, true>(cl, items, btab, gb, tb, lds, st);
	else
		launch_b<PF_TURN, false>(cl, items, btab, gb, tb, lds, st);

	BAM_HIP(hipGetLastError());
}

}  // namespace bam
