// grid.hip -- Kaiser-Bessel gridding for gfx950.
//
// Maths of noncart/grid.c:153-253 and :403-512 (tap range, clamp or wrap,
// separable weights from the 1001-entry KB table with linear interpolation,
// weight product in the order z, y, x).  Execution differs from
// gpu_grid.cu:
//   * samples are sorted once per trajectory by the cell (2^d grid points)
//     that holds their position; the plan lives with the operator;
//   * adjoint (k-space -> grid) is output-stationary: a work-group owns a tile
//     of all sub-grids for a group of coils, each wave a block of every
//     sub-grid (in 3-d 2 x 2 x 2 points = a 4 x 4 x 4 block of the 2x grid),
//     accumulated on the matrix cores; a wave walks only the samples that
//     reach its block, four at a time.  There are no atomics and no zero-fill
//     of the grid;
//   * forward (grid -> k-space): a thread per sample gathers its taps in
//     cell-sorted order and stores k-space at the original positions.
#include "nufft_impl.hpp"
#include "prof.hpp"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include <sys/stat.h>

namespace bam {

// ---------------------------------------------------------------------------
// Kaiser-Bessel table (noncart/grid.c:38-97, 516-519)
// ---------------------------------------------------------------------------

static double bessel_i0(double x)
{
	double q = 0.25 * x * x;
	double term = 1., sum = 1.;

	for (int k = 1; k < 500; k++) {
		term *= q / ((double)k * (double)k);
		sum += term;
		if (term < 1.e-17 * sum)
			break;
	}

	return sum;
}

double calc_beta(float os, float width)
{
	return M_PI * sqrt(pow((double)(width / os) * (os - 0.5), 2.) - 0.8);
}

void kb_table_host(double beta, float* table)
{
	double i0b = bessel_i0(beta);

	for (int i = 0; i < KB_SIZE + 1; i++) {

		double x = (double)i / (double)(KB_SIZE - 1) / 2.;
		table[i] = (fabs(x) >= 0.5) ? 0.f : (float)(bessel_i0(beta * sqrt(1. - pow(2. * x, 2.))) / i0b);
	}
}


// conj(fftmod) of grid point (x, y, z) applied to an adjoint gridding result
__device__ inline float2 apply_conj_fm(const GridGeom& g, float2 v, int x, int y, int z)
{
	if (nullptr == g.fm[0])
		return v;

	float2 f = g.fm[0][x];
	f = cmul(f, g.fm[1][y]);
	f = cmul(f, g.fm[2][z]);
	return cmulc(v, f);
}

// ---------------------------------------------------------------------------
// Plan: cell sort and tilings
// ---------------------------------------------------------------------------

constexpr int MAX_RANGES = 256;

// visits (samples of a tile's cells and their ring) per adjoint work item at
// most, and at least where a tile is split.  Every part costs a partial tile
// written and read, but a longer item is a longer chain of 32-bit sums: the
// 128^3 kooshball with 16 coils takes 4.34 ms at 2048 visits and 4.20 ms at
// 8192, with an error against 64 bits of 1.8e-7 and 5.5e-7.
constexpr int ADJ_MAXV = 2048;
constexpr int ADJ_MINV = 512;

// sample position on the grid, pos = os (k + shift) + n / 2, rounded as
// noncart/grid.c:181-187 rounds it (the device twin is grid_pos)
static float host_pos(const GridGeom& g, int s, int d, float k)
{
	const float b = (float)((double)g.os * ((double)k + (double)g.shift[s][d]));
	return b + (float)(g.n[d] / 2);
}

// Adjoint tiling.  A wave owns a block of every sub-grid: 2 x 2 x 2 points
// in 3-d (a 4 x 4 x 4 block of the 2x oversampled grid), 4 x 4 in 2-d, 32 in
// 1-d, one lane per (sub-grid, point), up to 16 coils per lane in registers.
// Tiles are 8 x 4 x 4 (16 waves), 16 x 16 (16 waves), 32 (1 wave); a tile
// dim is cut to the grid rounded up to the block.
static GridTiling choose_tiling(const GridGeom& g)
{
	int nd = 0;
	for (int d = 0; d < 3; d++)
		nd += (g.n[d] > 1);

	const int Tdef3[3] = { 8, 4, 4 };
	const int Tdef2[3] = { 16, 16, 1 };
	const int bdim = (3 == nd) ? 2 : ((2 == nd) ? 4 : 32);

	GridTiling t = {};
	int k = 0;
	int e = 0;
	t.ntiles = 1;
	t.Wtot = 1;
	t.nw = 1;

	for (int d = 0; d < 3; d++) {

		t.eoff[d] = 0;

		if (1 == g.n[d]) {
			t.T[d] = 1;
			t.b[d] = 1;
		} else {
			int want = (3 == nd) ? Tdef3[k] : ((2 == nd) ? Tdef2[k] : 32);
			k++;
			t.b[d] = bdim;
			t.T[d] = std::min(want, ((g.n[d] + bdim - 1) / bdim) * bdim);
			t.act[t.nd++] = d;
			t.eoff[d] = e;
			e += 2 * ((t.T[d] + 3) / 4 * 4);
		}

		t.Tp[d] = (t.T[d] + 3) / 4 * 4;

		t.nt[d] = (g.n[d] + t.T[d] - 1) / t.T[d];
		t.ntiles *= t.nt[d];
		t.Wtot *= t.T[d];
		t.nb[d] = t.T[d] / t.b[d];
		t.nw *= t.nb[d];
	}

	BAM_CHECK(e <= 64 && t.nw <= 16 && 64 == g.S * t.b[0] * t.b[1] * t.b[2] &&
			  64 * t.nw == g.S * t.Wtot, "gridding: bad tiling");

	auto ilog2 = [](int v) {
		int l = 0;
		while ((1 << l) < v)
			l++;
		BAM_CHECK((1 << l) == v, "gridding: block dims must be powers of two");
		return l;
	};
	t.lb0 = ilog2(t.b[0]);
	t.lb01 = t.lb0 + ilog2(t.b[1]);
	t.lb = t.lb01 + ilog2(t.b[2]);
	t.cc = (g.C <= 4) ? 4 : ((g.C <= 8) ? 8 : 16);
	t.ntap = (int)ceilf(g.width);
	t.rwidth = 1.f / g.width;
	t.fW = FastDiv((uint32_t)t.Wtot);
	t.fT0 = FastDiv((uint32_t)t.T[0]);
	t.fT1 = FastDiv((uint32_t)t.T[1]);

	// cell rows visited by one work-group must fit the range list
	long rows = 2;
	for (int d = 1; d < 3; d++)
		if (g.n[d] > 1)
			rows *= (long)ceil((t.T[d] + g.reach_lo + g.reach_hi) / g.CS[d]) + 2;
	BAM_CHECK(rows <= MAX_RANGES, "gridding: tile too large for the cell range list");

	return t;
}

// cell that holds position x on the axis of dim d.  The cells of a periodic
// grid continue beyond both ends, where the last cell of an odd dim, which
// holds one point, takes the place of a whole one.
__host__ __device__ inline int cell_at(const GridGeom& g, int d, float x)
{
	int turns = 0;

	if (g.periodic)
		turns = (x < 0.f) ? -1 : ((x >= (float)g.n[d]) ? 1 : 0);

	return (int)floorf((x - (float)(turns * g.n[d])) / (float)g.CS[d]) + turns * g.ncell[d];
}

// cells [clo, chi] of one dim as up to two spans {a0, n0, a1, n1} (wrapped
// for periodic grids, clamped otherwise, every cell at most once); the
// device twin is cell_span()
static void host_cell_span(const GridGeom& g, int d, int clo, int chi, int sp[4])
{
	const int nc = g.ncell[d];
	sp[2] = 0;
	sp[3] = 0;

	if (chi - clo + 1 >= nc) {
		sp[0] = 0;
		sp[1] = nc;
		return;
	}

	if (!g.periodic) {
		clo = std::max(clo, 0);
		chi = std::min(chi, nc - 1);
		sp[0] = clo;
		sp[1] = std::max(0, chi - clo + 1);
		return;
	}

	int lo = ((clo % nc) + nc) % nc;
	int len = chi - clo + 1;
	sp[0] = lo;

	if (lo + len <= nc) {
		sp[1] = len;
	} else {
		sp[1] = nc - lo;
		sp[3] = len - sp[1];
	}
}

// Forward gather work list of 3-D grids (non-periodic, kernel width < 4):
// the samples in home-tile order (cell order within a tile) and work items of
// at most FW_MAXS samples of one tile.
constexpr int FW_T = 8;          // tile edge, grid points
constexpr int FW_SPT = 4;        // samples per thread
constexpr int FW_THREADS = 512;
constexpr int FW_MAXS = FW_SPT * FW_THREADS;
constexpr int FW_CC = 4;         // coils per staged region
constexpr int FW_E = 12;         // staged region edge: tile + halo of a kernel of width 3
constexpr int FW_NT = 3;         // taps of such a kernel (an edge of 12 means a width over 2, up to 3)

static int taps_bound(const GridGeom& g);

void GridPlan::build_forward_tiles(const GridGeom& gg, const std::vector<int>& hsm, const std::vector<float4>& hsk,
				   const std::vector<int>& cell)
{
	ft = FwdTiling();

	// BART_AMD_FWD_TILES=off keeps the per-sample gather (for comparisons)
	const char* env = getenv("BART_AMD_FWD_TILES");

	if (nullptr != env && 0 == strcmp(env, "off"))
		return;

	bool all3 = gg.n[0] > 1 && gg.n[1] > 1 && gg.n[2] > 1;

	if (!all3 || gg.periodic || 4 != taps_bound(gg) || 0 == gg.M || gg.N * FW_CC >= (1l << 31))
		return;

	ft.T = FW_T;
	long ntiles = 1;

	for (int d = 0; d < 3; d++) {
		BAM_CHECK(0 == FW_T % gg.CS[d], "gridding: tile is not a multiple of the cell");
		ft.nt[d] = (gg.n[d] + FW_T - 1) / FW_T;
		ft.HL[d] = (int)ceilf(gg.reach_lo);
		ft.E[d] = FW_T + ft.HL[d] + (int)ceilf(gg.reach_hi);
		ntiles *= ft.nt[d];
	}

	ft.Etot = ft.E[0] * ft.E[1] * ft.E[2];

	// the kernel is built for one region edge; the region rows are loaded in
	// 16-byte pairs of points starting at even x
	if (FW_E != ft.E[0] || FW_E != ft.E[1] || FW_E != ft.E[2] || 0 != gg.n[0] % 2 || 0 != ft.HL[0] % 2)
		return;

	// the staged region of FW_CC coils and the KB table fit into 64 KiB
	if (((size_t)ft.Etot + 2 * FW_E) * FW_CC * sizeof(float2) + (KB_SIZE + 4) * sizeof(float) > 64 * 1024)
		return;

	const int cpt = FW_T / gg.CS[0];  // cells per tile edge (CS is equal in every dim)
	std::vector<int> tile_of(gg.M);
	std::vector<long> cnt(ntiles + 1, 0);

	// hsm/hsk are in cell order; cell[] is indexed by the original sample
	for (long i = 0; i < gg.M; i++) {
		int c = cell[hsm[i]];
		int cx = c % gg.ncell[0];
		int cy = (c / gg.ncell[0]) % gg.ncell[1];
		int cz = c / (gg.ncell[0] * gg.ncell[1]);
		int t = cx / cpt + ft.nt[0] * (cy / cpt + ft.nt[1] * (cz / cpt));
		tile_of[i] = t;
		cnt[t + 1]++;
	}

	for (long t = 0; t < ntiles; t++)
		cnt[t + 1] += cnt[t];

	std::vector<int> osm(gg.M);
	std::vector<float4> osk(gg.M);
	std::vector<long> pos(cnt.begin(), cnt.end() - 1);

	for (long i = 0; i < gg.M; i++) {
		long j = pos[tile_of[i]]++;
		osm[j] = hsm[i];
		osk[j] = hsk[i];
	}

	std::vector<int4> items;

	for (long t = 0; t < ntiles; t++)
		for (long a = cnt[t]; a < cnt[t + 1]; a += FW_MAXS)
			items.push_back(make_int4((int)t, (int)a, (int)std::min(cnt[t + 1], a + FW_MAXS), 0));

	std::stable_sort(items.begin(), items.end(), [](const int4& a, const int4& b) { return (a.z - a.y) > (b.z - b.y); });

	ft.nitems = (int)items.size();
	fsm.alloc(gg.M);
	fsk.alloc(gg.M);
	fwork.alloc(std::max(ft.nitems, 1));
	BAM_HIP(hipMemcpy(fsm.ptr, osm.data(), sizeof(int) * gg.M, hipMemcpyHostToDevice));
	BAM_HIP(hipMemcpy(fsk.ptr, osk.data(), sizeof(float4) * gg.M, hipMemcpyHostToDevice));
	BAM_HIP(hipMemcpy(fwork.ptr, items.data(), sizeof(int4) * ft.nitems, hipMemcpyHostToDevice));
	ft.on = true;
}

void GridPlan::build(const GridGeom& geom, const float* traj)
{
	g = geom;

	float maxshift = 0.f;
	for (int s = 0; s < g.S; s++)
		for (int d = 0; d < 3; d++)
			maxshift = std::max(maxshift, fabsf(g.shift[s][d] - g.shift[0][d]));

	g.reach_lo = 0.5f * g.width + g.os * maxshift;
	g.reach_hi = 0.5f * g.width;

	// distinct shift values per dim (the decomposition uses two: 0 and -1/2,
	// plus the odd-size correction) and the variant of every sub-grid
	for (int d = 0; d < 3; d++) {

		g.shv[d][0] = g.shift[0][d];
		g.shv[d][1] = g.shift[0][d];
		g.nshv[d] = 1;

		for (int s = 0; s < g.S; s++) {

			if (g.shift[s][d] == g.shv[d][0]) {
				g.sbit[s][d] = 0;
			} else if (1 == g.nshv[d] || g.shift[s][d] == g.shv[d][1]) {
				g.shv[d][1] = g.shift[s][d];
				g.nshv[d] = 2;
				g.sbit[s][d] = 1;
			} else {
				BAM_CHECK(false, "gridding: more than two shifts per dim");
			}
		}
	}

	long ncells = 1;

	for (int d = 0; d < 3; d++) {
		g.CS[d] = (g.n[d] > 1) ? 2 : 1;
		g.ncell[d] = (g.n[d] + g.CS[d] - 1) / g.CS[d];
		ncells *= g.ncell[d];
	}

	std::vector<int> cell(g.M);
	std::vector<int> count(ncells + 1, 0);

	for (long m = 0; m < g.M; m++) {

		int cb[3];

		for (int d = 0; d < 3; d++) {

			if (1 == g.n[d]) {
				cb[d] = 0;
				continue;
			}

			float p = host_pos(g, 0, d, traj[3 * m + d]);

			if (!std::isfinite(p))
				p = 0.f;

			if (g.periodic)
				p = p - (float)g.n[d] * floorf(p / (float)g.n[d]);

			int b = (int)floorf(p / (float)g.CS[d]);
			cb[d] = std::min(std::max(b, 0), g.ncell[d] - 1);
		}

		cell[m] = cb[0] + g.ncell[0] * (cb[1] + g.ncell[1] * cb[2]);
		count[cell[m] + 1]++;
	}

	for (long c = 0; c < ncells; c++)
		count[c + 1] += count[c];

	std::vector<int> hsm(std::max<long>(g.M, 1));
	std::vector<float4> hsk(std::max<long>(g.M, 1));
	std::vector<int> pos(count.begin(), count.end() - 1);

	for (long m = 0; m < g.M; m++) {

		long i = pos[cell[m]]++;
		hsm[i] = (int)m;
		hsk[i] = make_float4(traj[3 * m + 0], traj[3 * m + 1], traj[3 * m + 2], 0.f);
	}

	BAM_CHECK(g.M < (1l << 31), "too many samples");

	build_forward_tiles(g, hsm, hsk, cell);

	ta = choose_tiling(g);

	sm.alloc(std::max<long>(g.M, 1));
	si.alloc(std::max<long>(g.M, 1));
	sk.alloc(std::max<long>(g.M, 1));
	cstart.alloc(ncells + 1);

	BAM_HIP(hipMemcpy(sm.ptr, hsm.data(), sizeof(int) * std::max<long>(g.M, 1), hipMemcpyHostToDevice));
	{
		std::vector<int> hsi(std::max<long>(g.M, 1), 0);
		for (long i = 0; i < g.M; i++)
			hsi[hsm[i]] = (int)i;
		BAM_HIP(hipMemcpy(si.ptr, hsi.data(), sizeof(int) * std::max<long>(g.M, 1), hipMemcpyHostToDevice));
	}
	BAM_HIP(hipMemcpy(sk.ptr, hsk.data(), sizeof(float4) * std::max<long>(g.M, 1), hipMemcpyHostToDevice));

	BAM_HIP(hipMemcpy(cstart.ptr, count.data(), sizeof(int) * (ncells + 1), hipMemcpyHostToDevice));

	// room for every coils-per-work-group value the autotuner may pick
	// (4 .. the default): the coils rounded up to each
	cc_max = ta.cc;
	long kch = 0;
	for (int c = 4; c <= ta.cc; c *= 2)
		kch = std::max<long>(kch, (long)((g.C + c - 1) / c) * c);
	kspS.alloc((size_t)kch * std::max<long>(g.M, 1));

	ncu = device_cus();

	// adjoint work list: the visits of a tile (its cells and their ring)
	const GridTiling& t = ta;
	std::vector<int> visits(t.ntiles);
	long total = 0;

	for (int tile = 0; tile < t.ntiles; tile++) {

		int tb[3] = { tile % t.nt[0], (tile / t.nt[0]) % t.nt[1], tile / (t.nt[0] * t.nt[1]) };
		int span[3][4];

		for (int d = 0; d < 3; d++) {

			int clo = 0, chi = 0;

			if (g.n[d] > 1) {
				int t0 = tb[d] * t.T[d];
				clo = cell_at(g, d, (float)t0 - g.reach_hi);
				chi = cell_at(g, d, (float)(t0 + t.T[d] - 1) + g.reach_lo);
			}

			host_cell_span(g, d, clo, chi, span[d]);
		}

		long F = 0;

		for (int zs = 0; zs < 2; zs++)
			for (int cz = span[2][2 * zs]; cz < span[2][2 * zs] + span[2][2 * zs + 1]; cz++)
				for (int ys = 0; ys < 2; ys++)
					for (int cy = span[1][2 * ys]; cy < span[1][2 * ys] + span[1][2 * ys + 1]; cy++)
						for (int xs = 0; xs < 2; xs++) {
							long row = (long)g.ncell[0] * (cy + (long)g.ncell[1] * cz);
							long a = row + span[0][2 * xs];
							F += count[a + span[0][2 * xs + 1]] - count[a];
						}

		visits[tile] = (int)F;
		total += F;
	}

	// Items of at most MAXV visits; tiles with more are split, at the cost of
	// a partial tile per item.  Two items per compute unit where the visits
	// of the whole plan make them (a 2-D problem's dense tiles would keep a
	// few compute units busy while the others wait), between ADJ_MINV and
	// ADJ_MAXV.
	const long share = total * ((g.C + ta.cc - 1) / ta.cc) / (2l * ncu);
	const long MAXV = std::min<long>(ADJ_MAXV, std::max<long>(ADJ_MINV, (share + 255) / 256 * 256));
	std::vector<int4> hw;
	std::vector<int4> hsplit;
	int slots = 0;

	for (int tile = 0; tile < t.ntiles; tile++) {

		const long F = visits[tile];

		if (F <= MAXV) {
			hw.push_back(make_int4(tile, 0, (int)F, 0));
		} else {
			const int first = slots;
			for (long b = 0; b < F; b += MAXV)
				hw.push_back(make_int4(tile, (int)b, (int)std::min(F, b + MAXV), 1 + slots++));
			hsplit.push_back(make_int4(tile, first, slots - first, 0));
		}
	}

	// largest items first: the persistent work-groups take them in this order
	std::stable_sort(hw.begin(), hw.end(), [](const int4& a, const int4& b) { return (a.z - a.y) > (b.z - b.y); });

	nwork = (int)hw.size();
	nsplit = (int)hsplit.size();
	ta.nwork = nwork;
	queue.alloc(1);
	nslot = slots;
	work.alloc(std::max(nwork, 1));
	split_tiles.alloc(std::max(nsplit, 1));
	BAM_HIP(hipMemcpy(work.ptr, hw.data(), sizeof(int4) * nwork, hipMemcpyHostToDevice));
	if (nsplit > 0)
		BAM_HIP(hipMemcpy(split_tiles.ptr, hsplit.data(), sizeof(int4) * nsplit, hipMemcpyHostToDevice));
	spart.alloc((size_t)std::max(nslot, 1) * g.S * g.C * t.Wtot);
}

// taps per dim: floor(p + w/2) - ceil(p - w/2) + 1 <= floor(w) + 1
static int taps_bound(const GridGeom& g)
{
	int tp = (int)floor(g.width) + 1;
	BAM_CHECK(tp <= MAX_TAPS, "gridding: kernel width %f too large", g.width);
	return (tp <= 4) ? 4 : 8;
}

// ---------------------------------------------------------------------------
// Adjoint input permutation: kspS[(ch M + i) cc + cl] = ksp[(ch cc + cl) M + m(i)] conj(w(m))
// (the weights of noncart/nufft.c:1474-1479 are applied here), written
// from the original sample order with si = the inverse of m(i)
// ---------------------------------------------------------------------------

// A work-group takes PERM_S samples of a coil chunk: the coil values are read
// along m (coalesced), exchanged through LDS, and CC lanes write a sample's
// values as one run at its sorted position si[m].  Bound by HBM; a thread
// that wrote a sample's 128-byte run by itself reached 0.87 TB/s (128^3
// kooshball, 16 coils: 615 us, now 108 us or 5 TB/s).  Also clears the work
// queue of the gridding that follows on the stream.
constexpr int PERM_S = 256;

template <int CC>
__global__ __launch_bounds__(256) void k_permute_ksp(long M, int C, const int* __restrict__ si,
						     const float2* __restrict__ ksp,
						     const float2* __restrict__ weights, float2* __restrict__ kspS,
						     int* __restrict__ queue)
{
	__shared__ float2 buf[CC * (PERM_S + 1)];
	__shared__ int pos[PERM_S];

	if (0 == blockIdx.x && 0 == blockIdx.y && 0 == threadIdx.x)
		queue[0] = 0;

	const long m0 = (long)blockIdx.x * PERM_S;
	const int c0 = blockIdx.y * CC;
	const long m = m0 + threadIdx.x;

	if (m < M) {

		const float2 w = (nullptr != weights) ? weights[m] : make_float2(1.f, 0.f);
		float2 v[CC];

#pragma unroll
		for (int cl = 0; cl < CC; cl++)
			v[cl] = (c0 + cl < C) ? ksp[(long)(c0 + cl) * M + m] : make_float2(0.f, 0.f);

#pragma unroll
		for (int cl = 0; cl < CC; cl++)
			buf[cl * (PERM_S + 1) + threadIdx.x] = (nullptr != weights) ? cmulc(v[cl], w) : v[cl];

		pos[threadIdx.x] = si[m];
	}

	__syncthreads();

	float2* out = kspS + (long)blockIdx.y * M * CC;
	const int ns = (int)min((long)PERM_S, M - m0);

#pragma unroll
	for (int e = threadIdx.x; e < CC * PERM_S; e += 256) {
		const int i = e / CC;
		const int cl = e % CC;
		if (i < ns)
			out[(long)pos[i] * CC + cl] = buf[cl * (PERM_S + 1) + i];
	}
}

// ---------------------------------------------------------------------------
// Cell ranges of a work-group: the sorted samples of the cells [clo, chi] per
// dim (wrapped for periodic grids, clamped otherwise; every cell at most
// once) as contiguous index ranges, one per row of cells along x (two when x
// wraps).
// ---------------------------------------------------------------------------

struct CellRanges {
	int start[MAX_RANGES];
	int pre[MAX_RANGES + 1];
	int n;
	int pad[2];
};

// dynamic LDS layout: KB table, cell ranges, then the float2 data (16-byte aligned)
constexpr size_t SMEM_TABLE = (KB_SIZE + 4) * sizeof(float);
constexpr size_t SMEM_DATA = ((SMEM_TABLE + sizeof(CellRanges) + 15) / 16) * 16;

__device__ inline void cell_span(const GridGeom& g, int d, int clo, int chi, int& a0, int& n0, int& a1, int& n1)
{
	const int nc = g.ncell[d];
	a1 = 0;
	n1 = 0;

	if (chi - clo + 1 >= nc) {
		a0 = 0;
		n0 = nc;
		return;
	}

	if (!g.periodic) {
		clo = max(clo, 0);
		chi = min(chi, nc - 1);
		a0 = clo;
		n0 = max(0, chi - clo + 1);
		return;
	}

	int lo = ((clo % nc) + nc) % nc;
	int len = chi - clo + 1;

	a0 = lo;

	if (lo + len <= nc) {
		n0 = len;
	} else {
		n0 = nc - lo;
		n1 = len - n0;
	}
}

// Builds the ranges in LDS, one per row of cells along x (and x span), in
// the order z, y, x; empty rows are kept (their prefix entries repeat).
// Returns the total sample count.
__device__ inline int build_ranges(const GridGeom& g, const int* __restrict__ cstart, const int clo[3],
				   const int chi[3], CellRanges& R)
{
	int xa[2], xn[2], ya[2], yn[2], za[2], zn[2];
	cell_span(g, 0, clo[0], chi[0], xa[0], xn[0], xa[1], xn[1]);
	cell_span(g, 1, clo[1], chi[1], ya[0], yn[0], ya[1], yn[1]);
	cell_span(g, 2, clo[2], chi[2], za[0], zn[0], za[1], zn[1]);

	const int nxs = (xn[0] > 0) + (xn[1] > 0);
	const int ny = yn[0] + yn[1];
	const int nrow = min(nxs * ny * (zn[0] + zn[1]), MAX_RANGES);  // the plan checks the bound

	for (int r = threadIdx.x; r < nrow; r += blockDim.x) {

		const int xs = (xn[0] > 0) ? (r % nxs) : 1;
		const int q = r / nxs;
		const int yi = q % ny;
		const int zi = q / ny;
		const int cy = (yi < yn[0]) ? (ya[0] + yi) : (ya[1] + yi - yn[0]);
		const int cz = (zi < zn[0]) ? (za[0] + zi) : (za[1] + zi - zn[0]);
		const long row = (long)g.ncell[0] * (cy + (long)g.ncell[1] * cz) + xa[xs];
		const int a = cstart[row];
		R.start[r] = a;
		R.pre[r + 1] = cstart[row + xn[xs]] - a;
	}

	__syncthreads();

	// prefix sums by the first wave, 64 rows at a time
	if (threadIdx.x < 64) {

		int tot = 0;

		for (int r0 = 0; r0 < nrow; r0 += 64) {

			const int r = r0 + (int)threadIdx.x;
			int v = (r < nrow) ? R.pre[r + 1] : 0;

#pragma unroll
			for (int o = 1; o < 64; o <<= 1) {
				const int u = __shfl_up(v, o, 64);
				v += ((int)threadIdx.x >= o) ? u : 0;
			}

			if (r < nrow)
				R.pre[r + 1] = tot + v;

			tot += __shfl(v, 63, 64);
		}

		if (0 == threadIdx.x) {
			R.pre[0] = 0;
			R.n = nrow;
		}
	}

	__syncthreads();
	return R.pre[R.n];
}

template <typename X>
__device__ inline X sel3(int d, X a, X b, X c)
{
	return (0 == d) ? a : ((1 == d) ? b : c);
}

// x / width, correctly rounded from the rounded reciprocal (one residual
// step, Markstein)
__device__ inline float div_width(float x, float width, float rwidth)
{
	const float q = x * rwidth;
	return __builtin_fmaf(__builtin_fmaf(-q, width, x), rwidth, q);
}

// ---------------------------------------------------------------------------
// Taps of one sample along one dim (noncart/grid.c:415-457): NT = ceil(width)
// of them -- of the width + 1 taps of a sample half way between grid points
// both ends weigh 0 -- with weight 0 for those the grid's edge cuts off.
// last: the last tap with a weight.  Returns whether there is one.
// ---------------------------------------------------------------------------

__device__ inline float sample_pos_v(const GridGeom& g, int d, int v, float k)
{
	return grid_pos(g.os, k, g.shv[d][v], (float)(g.n[d] / 2));
}

template <int NT>
__device__ inline bool taps_of(const GridGeom& g, int d, int v, float k, const float* table, float rwidth, int& start,
			       int& last, float (&w)[NT])
{
	if (1 == g.n[d]) {
		start = 0;
		last = 0;
#pragma unroll
		for (int j = 0; j < NT; j++)
			w[j] = (0 == j) ? 1.f : 0.f;
		return true;
	}

	const float pos = sample_pos_v(g, d, v, k);
	int sti = (int)ceil((double)pos - 0.5 * (double)g.width);
	int eni = (int)floor((double)pos + 0.5 * (double)g.width);

	if (!g.periodic) {
		sti = max(sti, 0);
		eni = min(eni, g.n[d] - 1);
	}

	// (positions beyond the range of int saturate: taps are counted first)
	const int cnt = max(eni - sti + 1, 0);
	last = max(min(cnt, NT), 1) - 1;
	// (of a sample without taps: some point of the grid)
	start = g.periodic ? sti : min(sti, g.n[d] - 1);

#pragma unroll
	for (int j = 0; j < NT; j++)
		w[j] = (j < cnt) ? kb_lookup(table, div_width(fabsf((float)(int)((unsigned)sti + j) - pos), g.width, rwidth)) : 0.f;

	return cnt > 0;
}

// The same in a staged region whose points off the grid are 0, so that no tap
// has to be cut off: start is tap 0 of an unbounded grid, and a tap beyond the
// kernel (width < NT) weighs 0 by its distance.
template <int NT>
__device__ inline bool taps_staged(const GridGeom& g, int d, int v, float k, const float* table, float rwidth,
				   int& start, int& last, float (&w)[NT])
{
	const float pos = sample_pos_v(g, d, v, k);
	start = (int)ceil((double)pos - 0.5 * (double)g.width);
	last = min(max((int)floor((double)pos + 0.5 * (double)g.width) - start, 0), NT - 1);

#pragma unroll
	for (int j = 0; j < NT; j++)
		w[j] = kb_lookup(table, div_width(fabsf((float)(int)((unsigned)start + j) - pos), g.width, rwidth));

	// a tap on the grid: start in (-NT, n)
	return (unsigned)start + (NT - 1) < (unsigned)(g.n[d] + NT - 1);
}

// acc += val where `in`, whatever val holds elsewhere.  The mask goes through an
// empty asm: given a select or a branch the compiler moves the loads behind val
// around (those of all samples of a thread come at once and spill 140 registers).
template <int CC>
__device__ inline void acc_where(float2 (&acc)[CC], const float2 (&val)[CC], bool in)
{
	unsigned m = in ? ~0u : 0u;
	asm("" : "+v"(m));

#pragma unroll
	for (int cl = 0; cl < CC; cl++) {
		acc[cl].x += __uint_as_float(__float_as_uint(val[cl].x) & m);
		acc[cl].y += __uint_as_float(__float_as_uint(val[cl].y) & m);
	}
}

// grid index of tap start + j, wrapped on a periodic grid
__device__ inline int tap_index(const GridGeom& g, int d, int start, int j)
{
	if (!g.periodic)
		return start + j;

	const int n = g.n[d];
	const int w = (int)((unsigned)start + j) % n;
	return w + ((w < 0) ? n : 0);
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
constexpr int ADJ_BATCH = 256;  // visits per batch (4 groups of 64)
constexpr int ADJ_WROW = 68;    // weight table row of a visit: 64 entries, 16-byte aligned, bank spread

// LDS of the adjoint after the KB table and the ranges
struct AdjLds {
	float2* vbuf;         // [ADJ_BATCH + 1][CC] coil values per visit
	float* wtab;          // [ADJ_BATCH + 1][ADJ_WROW] tap weights per visit
	unsigned* rows;       // [6][ADJ_BATCH] tile rows hit, per active dim and variant
	float* kc;            // [3][ADJ_BATCH] coordinates of the active dims
	int* sidx;            // [2][ADJ_BATCH] sorted sample of each visit, two batches
	unsigned short* list; // [16][ADJ_BATCH + 4] a wave's visits of the batch
};

template <int CC>
constexpr size_t adj_work_bytes()
{
	return sizeof(float2) * (ADJ_BATCH + 1) * CC + sizeof(float) * (ADJ_BATCH + 1) * ADJ_WROW +
	       sizeof(unsigned) * 6 * ADJ_BATCH + sizeof(float) * 3 * ADJ_BATCH + sizeof(int) * 2 * ADJ_BATCH +
	       sizeof(unsigned short) * 16 * (ADJ_BATCH + 4);
}

// Adjoint gridding (k-space -> grid), output-stationary and atomic-free.
// grid layout [S][C][N].  Persistent work-groups (a few per CU) take work
// items (tile, visit range, coil chunk) from a queue, largest first.
//
// A wave owns a block of b points per dim in every sub-grid (64 outputs:
// sub-grid s, point).  For each batch of visits (samples of the tile's cells
// and of the ring of neighbouring cells, in cell order):
//   1. a wave takes 64 visits, one dim and one shift variant (its parameters
//      are scalars): a lane evaluates the taps of its visit, clears its row
//      of tile weights and scatters the taps there, with a bit mask of the
//      rows hit; the coil values and coordinates of the batch, loaded during
//      the previous batch, go to LDS;
//   2. every wave lists the visits that reach its block (from the masks) and
//      walks them four at a time on the matrix cores: C[out][j] += sum_k
//      A[out][k] B[k][j], v_mfma_f32_16x16x4_f32 with A = tap weight of output
//      out for visit k and B = value j (coil j / 2, re / im) of visit k.  The
//      64 outputs are 4 groups of 16 rows; sub-grids that differ in the last
//      one (two) active dims are in the same lane, so that 4 to 5 weights
//      per lane and visit make the 4 rows' products.
// Each product is accumulated in visit order, as in the sequential gridding
// of noncart/grid.c:240-250.  Tiles whose visits are split over several
// work items store partial tiles, summed in order by k_sum_split.
//
// Bound by the vector instructions of both steps, the latencies at the start
// of an item and, for 2-D problems, by the largest item.  When a lane chose
// one of its taps for every tile row, two visits were multiplied per step
// (32x32x2 tiles, half empty with 8 coils) and the store formed an address
// and a factor per value: 128^3 kooshball, 16 coils 5040 -> 2755 us; 256^2
// radial, 8 coils 197 -> 45 us.
template <int TP, int CC, int ND>
__global__ __launch_bounds__(1024) void k_grid_adj(GridGeom g, GridTiling t, const float* __restrict__ kbt,
						   const float4* __restrict__ sk, const int* __restrict__ cstart,
						   const int4* __restrict__ work, int nitems, int* __restrict__ queue,
						   const float2* __restrict__ kspS, float2* __restrict__ grid,
						   float2* __restrict__ spart)
{
	constexpr int NCB = (CC + 7) / 8;  // blocks of 16 columns (8 coils)
	extern __shared__ float4 smem4[];
	char* smem = (char*)smem4;
	float* table = (float*)smem;
	CellRanges& R = *(CellRanges*)(smem + SMEM_TABLE);
	AdjLds L;
	L.vbuf = (float2*)(smem + SMEM_DATA);
	L.wtab = (float*)(L.vbuf + (ADJ_BATCH + 1) * CC);
	L.rows = (unsigned*)(L.wtab + (ADJ_BATCH + 1) * ADJ_WROW);
	L.kc = (float*)(L.rows + 6 * ADJ_BATCH);
	L.sidx = (int*)(L.kc + 3 * ADJ_BATCH);
	const size_t otile_bytes = sizeof(float2) * g.S * CC * (t.Wtot + 1);
	const size_t data_bytes = max(adj_work_bytes<CC>(), otile_bytes);
	int* qitem = (int*)(smem + SMEM_DATA + (data_bytes + 15) / 16 * 16);
	float2* fml = (float2*)(qitem + 4);                   // [n0 + n1 + n2] fftmod tables (when t.fmlds)

	const int nthr = blockDim.x;
	const int nwv = nthr >> 6;
	const int lane = threadIdx.x & 63;
	const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform
	const int nwork = t.nwork;
	L.list = (unsigned short*)(L.sidx + 2 * ADJ_BATCH) + wid * (ADJ_BATCH + 4);

	for (int i = threadIdx.x; i < KB_SIZE + 1; i += nthr)
		table[i] = kbt[i];

	if (0 == threadIdx.x)
		qitem[1] = 0;

	const bool fm = (nullptr != g.fm[0]);
	const bool fmlds = fm && (0 != t.fmlds);

	if (fmlds) {
		for (int i = threadIdx.x; i < g.n[0]; i += nthr)
			fml[i] = g.fm[0][i];
		for (int i = threadIdx.x; i < g.n[1]; i += nthr)
			fml[g.n[0] + i] = g.fm[1][i];
		for (int i = threadIdx.x; i < g.n[2]; i += nthr)
			fml[g.n[0] + g.n[1] + i] = g.fm[2][i];
	}

	// the wave's block, and the weight table entries of the lane's rows
	// 16 q + l16, q = 0 .. 3 (row = sub-grid x B + point): wo[d][bit], the
	// entry of active dim d for shift variant bit.  In 3-d the x bit follows
	// from l16, y and z bits from q; in 2-d both from q; in 1-d the bit and
	// the upper half of the points.
	constexpr int LB = (3 == ND) ? 3 : ((2 == ND) ? 4 : 5);  // points per block and sub-grid
	constexpr int B = 1 << LB;
	const int wb[3] = { wid % t.nb[0], (wid / t.nb[0]) % t.nb[1], wid / (t.nb[0] * t.nb[1]) };
	const int l16 = lane & 15;
	int wo[ND][2], wo1[4];

	// the lane's point and sub-grid of the output store
	uint32_t srs, spq, sx0, sx1, sx2;
	{
		uint32_t r;
		t.fW.divmod(threadIdx.x, srs, spq);
		t.fT0.divmod(spq, r, sx0);
		t.fT1.divmod(r, sx2, sx1);
	}

	{
		const int cb = l16 & (B - 1);
		int q[3];
		q[0] = wb[0] * t.b[0] + (cb & (t.b[0] - 1));
		q[1] = wb[1] * t.b[1] + ((cb >> t.lb0) & (t.b[1] - 1));
		q[2] = wb[2] * t.b[2] + (cb >> t.lb01);

#pragma unroll
		for (int a = 0; a < ND; a++) {
			const int d = t.act[a];
			const int e = t.eoff[d] + min(sel3(d, q[0], q[1], q[2]), t.T[d] - 1);
			wo[a][0] = e;
			wo[a][1] = e + t.Tp[d];
		}

		if (3 == ND && l16 >= 8)
			wo[0][0] = wo[0][1];

		if (1 == ND) {
			const int d = t.act[0];
#pragma unroll
			for (int r = 0; r < 4; r++)
				wo1[r] = t.eoff[d] + (r >> 1) * t.Tp[d] +
					 min(sel3(d, wb[0], wb[1], wb[2]) * t.b[d] + 16 * (r & 1) + l16, t.T[d] - 1);
		}
	}

	constexpr int VPT = (ADJ_BATCH * CC + 1023) / 1024;  // coil values carried per lane (1024 lanes)

	// the first work-groups' first items are their own; later ones come from
	// the queue, asked for one item ahead
	int next = (int)blockIdx.x;

	while (true) {

		// next work item (the barrier also ends every wave's use of the
		// previous item's LDS data)
		if (0 == threadIdx.x)
			qitem[0] = next;

		__syncthreads();

		const int item = qitem[0];

		if (item >= nitems)
			break;

		if (0 == threadIdx.x)
			next = (int)gridDim.x + atomicAdd(queue, 1);

		// the visit that fills up groups of four: no weight, no value (the
		// output store of the previous item reused this memory)
		for (int i = threadIdx.x; i < ADJ_WROW; i += nthr)
			L.wtab[ADJ_BATCH * ADJ_WROW + i] = 0.f;
		for (int i = threadIdx.x; i < CC; i += nthr)
			L.vbuf[ADJ_BATCH * CC + i] = make_float2(0.f, 0.f);

		const int ch = item / nwork;
		const int4 wk = work[item - ch * nwork];  // (tile, first visit, end visit, partial slot + 1 or 0)
		const int tile = wk.x;
		const int c0 = ch * CC;
		const int ncc = min(CC, g.C - c0);

		int tb[3], t0[3], clo[3], chi[3];
		tb[0] = tile % t.nt[0];
		tb[1] = (tile / t.nt[0]) % t.nt[1];
		tb[2] = tile / (t.nt[0] * t.nt[1]);

		for (int d = 0; d < 3; d++) {
			t0[d] = tb[d] * t.T[d];
			if (1 == g.n[d]) {
				clo[d] = 0;
				chi[d] = 0;
			} else {
				clo[d] = cell_at(g, d, (float)t0[d] - g.reach_hi);
				chi[d] = cell_at(g, d, (float)(t0[d] + t.T[d] - 1) + g.reach_lo);
			}
		}

		const int Ftile = build_ranges(g, cstart, clo, chi, R);
		const int fb = min(wk.y, Ftile);
		const int fe = min(wk.z, Ftile);
		const int F = fe - fb;

		// sorted sample of the visits of batch q into its half of sidx
		// (visits past the end: the last one)
		auto find = [&](int q) {
			for (int v = threadIdx.x; v < ADJ_BATCH; v += nthr) {
				const int f = fb + min(q * ADJ_BATCH + v, F - 1);
				int lo = 0, hi = R.n;
				while (hi - lo > 1) {
					const int mid = (lo + hi) >> 1;
					if (R.pre[mid] <= f)
						lo = mid;
					else
						hi = mid;
				}
				L.sidx[(q & 1) * ADJ_BATCH + v] = R.start[lo] + (f - R.pre[lo]);
			}
		};

		if (F > 0) {
			find(0);
			find(1);
		}

		__syncthreads();

		// coil values: lane carries VPT float2 of the next batch (entries
		// threadIdx.x + 1024 q: visit e / CC, coil e % CC) through the current
		// one; the first ADJ_BATCH lanes its coordinates
		const float2* kch = kspS + (long)ch * g.M * CC;
		float2 vnext[VPT];
		float4 knext = make_float4(0.f, 0.f, 0.f, 0.f);

#pragma unroll
		for (int q = 0; q < VPT; q++) {
			const int e = threadIdx.x + 1024 * q;
			vnext[q] = (e < ADJ_BATCH * CC && F > 0) ? kch[(long)L.sidx[e / CC] * CC + (e % CC)] : make_float2(0.f, 0.f);
		}

		if (threadIdx.x < ADJ_BATCH && F > 0)
			knext = sk[L.sidx[threadIdx.x]];

		f32x4 acc[NCB][4];
#pragma unroll
		for (int c = 0; c < NCB; c++)
#pragma unroll
			for (int q = 0; q < 4; q++)
				acc[c][q] = f32x4{ 0.f, 0.f, 0.f, 0.f };

		for (int base = 0; base < F; base += ADJ_BATCH) {

			const int nb = min(ADJ_BATCH, F - base);
			const int bi = base / ADJ_BATCH;
			const int* scur = L.sidx + (bi & 1) * ADJ_BATCH;
			const int* snext = L.sidx + (1 - (bi & 1)) * ADJ_BATCH;

			// the previous batch is done with the LDS buffers
			lds_barrier();

#pragma unroll
			for (int q = 0; q < VPT; q++) {
				const int e = threadIdx.x + 1024 * q;
				if (e < ADJ_BATCH * CC)
					L.vbuf[e] = vnext[q];
			}

			if (threadIdx.x < ADJ_BATCH) {
				const float kk[3] = { knext.x, knext.y, knext.z };
#pragma unroll
				for (int a = 0; a < ND; a++)
					L.kc[a * ADJ_BATCH + threadIdx.x] = sel3(t.act[a], kk[0], kk[1], kk[2]);
			}

			// work-groups of fewer than 1024 lanes load the rest now
			for (int e = threadIdx.x + nthr; e < ADJ_BATCH * CC; e += nthr)
				if (e % 1024 >= nthr)
					L.vbuf[e] = kch[(long)scur[e / CC] * CC + (e % CC)];

			for (int v = threadIdx.x + nthr; v < ADJ_BATCH; v += nthr) {
				const float4 k = sk[scur[v]];
#pragma unroll
				for (int a = 0; a < ND; a++)
					L.kc[a * ADJ_BATCH + v] = sel3(t.act[a], k.x, k.y, k.z);
			}

			// the next batch's values are loaded while this one is processed
			if (base + ADJ_BATCH < F) {
#pragma unroll
				for (int q = 0; q < VPT; q++) {
					const int e = threadIdx.x + 1024 * q;
					if (e < ADJ_BATCH * CC)
						vnext[q] = kch[(long)snext[e / CC] * CC + (e % CC)];
				}
				if (threadIdx.x < ADJ_BATCH)
					knext = sk[snext[threadIdx.x]];
			}

			lds_barrier();

			// the batch after the next (this one's half of sidx is free)
			if (base + 2 * ADJ_BATCH < F)
				find(bi + 2);

			// 1. taps of the batch: wave task (64 visits, dim, variant)
			for (int task = wid; task < 4 * 2 * ND; task += nwv) {

				const int vg = task / (2 * ND);
				const int k = task - vg * (2 * ND);
				const int var = k & 1;

				if (vg * 64 >= nb)
					break;

				const int v = vg * 64 + lane;
				const int d = t.act[k >> 1];
				const int n = g.n[d];
				const float sh = g.shv[d][(g.nshv[d] > 1) ? var : 0];
				const float kd = L.kc[(k >> 1) * ADJ_BATCH + v];
				const float pos = grid_pos(g.os, kd, sh, (float)(n / 2));
				int sti = (int)ceil((double)pos - 0.5 * (double)g.width);
				int eni = (int)floor((double)pos + 0.5 * (double)g.width);

				if (!g.periodic) {
					sti = max(sti, 0);
					eni = min(eni, n - 1);
				}

				const int cnt = min(max(eni - sti + 1, 0), TP);
				const int T = t.T[d], Tp = t.Tp[d];
				const int td = sel3(d, t0[0], t0[1], t0[2]);
				float* wr = L.wtab + v * ADJ_WROW + t.eoff[d] + var * Tp;
				unsigned bits = 0u;

				for (int l = 0; l < Tp; l += 4)
					*(f32x4*)(wr + l) = f32x4{ 0.f, 0.f, 0.f, 0.f };

				int l0 = sti - td;

				if (g.periodic) {
					l0 = sti % n;
					l0 += (l0 < 0) ? n : 0;
					l0 -= td;
				}

#pragma unroll
				for (int q = 0; q < TP; q++) {

					if (q >= t.ntap)
						break;

					int l = l0 + q;

					if (g.periodic && l + td >= n)
						l -= n;

					const float w = kb_lookup(table, div_width(fabsf((float)(sti + q) - pos), g.width, t.rwidth));

					if (q < min(cnt, n) && l >= 0 && l < T) {
						wr[l] = w;
						bits |= 1u << l;
					}
				}

				// more taps than points of the period: a point gets several, the
				// first ones are in
				if (g.periodic && n < t.ntap)
					for (int q = n; q < cnt; q++) {

						const int l = (l0 + td + q) % n - td;

						if (l >= 0 && l < T)
							wr[l] += kb_lookup(table, div_width(fabsf((float)(sti + q) - pos), g.width, t.rwidth));
					}

				L.rows[k * ADJ_BATCH + v] = bits;
			}

			lds_barrier();

			// 2. the visits that reach this wave's block (taps in its rows in
			// every active dim, either variant), in order
			int cnt = 0;

			for (int gb = 0; gb < nb; gb += 64) {

				bool reach = lane < nb - gb;

#pragma unroll
				for (int a = 0; a < ND; a++) {
					const int d = t.act[a];
					const unsigned m = L.rows[2 * a * ADJ_BATCH + gb + lane] |
							   L.rows[(2 * a + 1) * ADJ_BATCH + gb + lane];
					const unsigned sel = (32 == t.b[d]) ? ~0u : ((1u << t.b[d]) - 1u) << (sel3(d, wb[0], wb[1], wb[2]) * t.b[d]);
					reach = reach && 0u != (m & sel);
				}

				const unsigned long long mh = __ballot(reach);

				if (reach)
					L.list[cnt + __builtin_amdgcn_mbcnt_hi((unsigned)(mh >> 32),
									       __builtin_amdgcn_mbcnt_lo((unsigned)mh, 0u))] =
						(unsigned short)(gb + lane);

				cnt += (int)__popcll(mh);
			}

			if (lane < 4)
				L.list[cnt + lane] = (unsigned short)ADJ_BATCH;

			// the list is this wave's own
			__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
			__builtin_amdgcn_wave_barrier();
			__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");

			const unsigned short* lp = L.list + (lane >> 4);

#pragma unroll 2
			for (int i = 0; i < cnt; i += 4) {

				const int v = lp[i];
				const float* wv = L.wtab + v * ADJ_WROW;
				const float* bp = (const float*)L.vbuf + v * 2 * CC;
				float bv[NCB];

#pragma unroll
				for (int c = 0; c < NCB; c++)
					bv[c] = bp[16 * c + ((4 == CC) ? (l16 & 7) : l16)];

				float a[4];

				if constexpr (3 == ND) {
					const float x = wv[wo[0][0]];
					const float y0 = wv[wo[1][0]] * x, y1 = wv[wo[1][1]] * x;
					const float z0 = wv[wo[2][0]], z1 = wv[wo[2][1]];
					a[0] = z0 * y0;
					a[1] = z0 * y1;
					a[2] = z1 * y0;
					a[3] = z1 * y1;
				} else if constexpr (2 == ND) {
					const float x0 = wv[wo[0][0]], x1 = wv[wo[0][1]];
					const float y0 = wv[wo[1][0]], y1 = wv[wo[1][1]];
					a[0] = y0 * x0;
					a[1] = y0 * x1;
					a[2] = y1 * x0;
					a[3] = y1 * x1;
				} else {
#pragma unroll
					for (int q = 0; q < 4; q++)
						a[q] = wv[wo1[q]];
				}

#pragma unroll
				for (int c = 0; c < NCB; c++)
#pragma unroll
					for (int q = 0; q < 4; q++)
						acc[c][q] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q], bv[c], acc[c][q], 0, 0, 0);
			}
		}

		// Store through LDS: the waves put their outputs into the tile
		// buffer otile[s][c][point] (plane pitch Wtot + 1, spread over the
		// banks; it reuses the batch buffers), then a lane writes one point of
		// one sub-grid for all coils (S Wtot lanes: the whole work-group), so
		// that its address and fftmod factor are formed once.  Column j = l16
		// of block c is coil 8 c + j / 2 (re, im); register r of group q holds
		// row 16 q + 4 (lane / 16) + r.
		const int OP = t.Wtot + 1;
		float* otile = (float*)L.vbuf;

		lds_barrier();

		{
			// (zero is 0, read from LDS here so that the row decoding is
			// not hoisted out of the item loop, where its copies would stay
			// live)
			const int zero = qitem[1];
			const int kg = (lane + zero) >> 4;

#pragma unroll
			for (int h = 0; h < ((LB > 4) ? 2 : 1); h++)
#pragma unroll
				for (int r = 0; r < 4; r++) {

					// rows 16 q + i: sub-grid (16 q + i) / B, point of the block
					// i % B (+ 16 h where a block spans two groups)
					const int i = 4 * kg + r;
					const int rc = (LB > 4) ? i + 16 * h : (i & (B - 1));
					const int q0 = wb[0] * t.b[0] + (rc & (t.b[0] - 1));
					const int q1 = wb[1] * t.b[1] + ((rc >> t.lb0) & (t.b[1] - 1));
					const int q2 = wb[2] * t.b[2] + (rc >> t.lb01);
					const int pt = q0 + t.T[0] * (q1 + t.T[1] * q2);
					float* op = otile + (((i >> LB) * CC + (l16 >> 1)) * OP + pt) * 2 + (l16 & 1);

#pragma unroll
					for (int q = h; q < 4; q += ((LB > 4) ? 2 : 1)) {
						const int rs = (16 * q) >> LB;
#pragma unroll
						for (int c = 0; c < NCB; c++)
							if (4 != CC || l16 < 8)
								op[((rs * CC + 8 * c) * OP) * 2] = acc[c][q][r];
					}
				}
		}

		lds_barrier();

		{
			const int x0 = t0[0] + (int)sx0, x1 = t0[1] + (int)sx1, x2 = t0[2] + (int)sx2;

			if ((int)srs < g.S && x0 < g.n[0] && x1 < g.n[1] && x2 < g.n[2]) {

				const float2* op = (const float2*)otile + (long)srs * CC * OP + spq;

				if (0 == wk.w) {

					float2 f = make_float2(1.f, 0.f);

					if (fmlds) {
						f = fml[x0];
						f = cmul(f, fml[g.n[0] + x1]);
						f = cmul(f, fml[g.n[0] + g.n[1] + x2]);
					} else if (fm) {
						f = cmul(cmul(g.fm[0][x0], g.fm[1][x1]), g.fm[2][x2]);
					}

					float2* out = grid + ((long)srs * g.C + c0) * g.N + x0 + (long)g.n[0] * (x1 + (long)g.n[1] * x2);

					for (int c = 0; c < ncc; c++)
						out[(long)c * g.N] = cmulc(op[c * OP], f);

				} else {

					// tile split over several work items (dense region): the
					// partial tile goes to its own slot, summed by k_sum_split
					float2* out = spart + (((long)(wk.w - 1) * g.S + srs) * g.C + c0) * t.Wtot + spq;

					for (int c = 0; c < ncc; c++)
						out[(long)c * t.Wtot] = op[c * OP];
				}
			}
		}
	}
}

// tiles split over several work items: sum of their partial tiles in slot
// order (deterministic, no atomics); work-group (split tile, sub-grid, group
// of nc coils), thread per (coil, point)

__global__ __launch_bounds__(256) void k_sum_split(GridGeom g, GridTiling t, const int4* __restrict__ tiles,
						   const float2* __restrict__ spart, float2* __restrict__ grid, int nc)
{
	const int4 st = tiles[blockIdx.x];
	const int tile = st.x;
	const int tb0 = tile % t.nt[0], tb1 = (tile / t.nt[0]) % t.nt[1], tb2 = tile / (t.nt[0] * t.nt[1]);
	const int c0 = blockIdx.z * nc;
	const int ncc = min(nc, g.C - c0);
	const long slot = (long)g.S * g.C * t.Wtot;

	for (uint32_t e = threadIdx.x; e < (uint32_t)(ncc * t.Wtot); e += 256) {

		uint32_t cl, pnt, r, x0, x1, x2;
		t.fW.divmod(e, cl, pnt);
		t.fT0.divmod(pnt, r, x0);
		t.fT1.divmod(r, x2, x1);
		const int gx = tb0 * t.T[0] + (int)x0;
		const int gy = tb1 * t.T[1] + (int)x1;
		const int gz = tb2 * t.T[2] + (int)x2;

		if (gx >= g.n[0] || gy >= g.n[1] || gz >= g.n[2])
			continue;

		const long sc = (long)blockIdx.y * g.C + c0 + cl;
		const float2* p = spart + (long)st.y * slot + sc * t.Wtot + pnt;
		float2 a = make_float2(0.f, 0.f);

#pragma unroll 4
		for (int k = 0; k < st.z; k++)
			a = cadd(a, p[k * slot]);

		grid[sc * g.N + gx + (long)g.n[0] * (gy + (long)g.n[1] * gz)] = apply_conj_fm(g, a, gx, gy, gz);
	}
}

void grid_adjoint(const GridPlan& gp, const float* kb, float2* grid, const float2* ksp, const float2* weights,
		  hipStream_t st)
{
	const GridGeom& g = gp.g;
	const GridTiling& t = gp.ta;

	if (0 == g.C)
		return;

	BAM_CHECK(t.cc <= 16, "gridding: at most 16 coils per work-group");

	{
		ProfScope prof("permute_ksp", st);
		const int nch = (g.C + t.cc - 1) / t.cc;
		const dim3 blocks(std::max(1u, ceil_div(g.M, PERM_S)), nch);
#define BAM_PERM(CC) \
	hipLaunchKernelGGL(k_permute_ksp<CC>, blocks, dim3(256), 0, st, g.M, g.C, gp.si.ptr, ksp, weights, \
			   gp.kspS.ptr, gp.queue.ptr)
		if (t.cc <= 4)
			BAM_PERM(4);
		else if (t.cc <= 8)
			BAM_PERM(8);
		else
			BAM_PERM(16);
#undef BAM_PERM
		BAM_HIP(hipGetLastError());
	}

	ProfScope prof("grid_adjoint", st);

	const int tp = taps_bound(g);
	const int nthr = 64 * t.nw;
	const int nch = (g.C + t.cc - 1) / t.cc;
	const int nitems = gp.nwork * nch;
	const unsigned nwg = (unsigned)std::max(1, std::min(nitems, gp.wpc * gp.ncu));
	const size_t workb = (t.cc <= 4) ? adj_work_bytes<4>() : ((t.cc <= 8) ? adj_work_bytes<8>() : adj_work_bytes<16>());
	// the output tile (plane pitch Wtot + 1) reuses the batch buffers
	const size_t otile = (size_t)g.S * t.cc * (t.Wtot + 1) * sizeof(float2);
	size_t lds = SMEM_DATA + (std::max(workb, otile) + 15) / 16 * 16 + sizeof(int) * 4;

	// fftmod tables in LDS when they fit (160 KiB per work-group)
	GridTiling tl = t;
	const size_t fmb = sizeof(float2) * ((size_t)g.n[0] + g.n[1] + g.n[2]);
	tl.fmlds = (nullptr != g.fm[0] && lds + fmb <= 160 * 1024) ? 1 : 0;
	if (tl.fmlds)
		lds += fmb;

#define BAM_ADJ(TP, CC, ND)                                                                                     \
	hipLaunchKernelGGL((k_grid_adj<TP, CC, ND>), dim3(nwg), dim3(nthr), lds, st, g, tl, kb, gp.sk.ptr, gp.cstart.ptr, \
			   gp.work.ptr, nitems, gp.queue.ptr, gp.kspS.ptr, grid, gp.spart.ptr)
#define BAM_ADJ_ND(TP, CC)             \
	do {                           \
		if (3 == t.nd)         \
			BAM_ADJ(TP, CC, 3); \
		else if (2 == t.nd)    \
			BAM_ADJ(TP, CC, 2); \
		else                   \
			BAM_ADJ(TP, CC, 1); \
	} while (0)

	if (4 == tp) {
		if (t.cc <= 4) BAM_ADJ_ND(4, 4);
		else if (t.cc <= 8) BAM_ADJ_ND(4, 8);
		else BAM_ADJ_ND(4, 16);
	} else {
		if (t.cc <= 4) BAM_ADJ_ND(8, 4);
		else if (t.cc <= 8) BAM_ADJ_ND(8, 8);
		else BAM_ADJ_ND(8, 16);
	}
#undef BAM_ADJ_ND
#undef BAM_ADJ

	BAM_HIP(hipGetLastError());

	if (gp.nsplit > 0) {
		ProfScope prof2("grid_adjoint_sum_split", st);
		const int nc = std::max(1, 256 / t.Wtot);
		hipLaunchKernelGGL(k_sum_split, dim3((unsigned)gp.nsplit, (unsigned)g.S, ceil_div(g.C, nc)), dim3(256), 0, st, g,
				   t, gp.split_tiles.ptr, gp.spart.ptr, grid, nc);
		BAM_HIP(hipGetLastError());
	}
}

// ---------------------------------------------------------------------------
// Forward gridding (grid -> k-space), per-sample form for the grids the
// tiled kernel below does not take: one thread per sample and coil chunk
// gathers the taps of all sub-grids from the grid; sub-grids are summed in
// order s = 0 .. S-1 (noncart/nufft.c:1444-1445) and the result is
// multiplied by the weights (:1456-1457).  Samples are taken in cell-sorted
// order, so that the lanes of a wave read neighbouring grid lines (in the
// original order a 3-d readout crosses many lines: measured 8x slower on a
// 128^3 kooshball); the k-space stores go to the original positions.  Small
// problems are bound by a thread's chain of loads, so the dims and taps are
// constants and every load of a sample (sub-grids x taps) is in flight before
// the first is used, without branches around taps cut off at the edge; with
// run-time dims and taps the loads went one by one (64^2, 4 coils: 38 us; now
// 6.2.  320^2 spiral, 32 coils: 155; now 112).
// Launch (ceil(M / 256), ceil(C / CC)).
// ---------------------------------------------------------------------------

template <int NT, int CC, int ND>
__global__ __launch_bounds__(256) void k_grid_fwd(GridGeom g, const float* __restrict__ kbt,
						  const int* __restrict__ sm, const float4* __restrict__ sk,
						  const float2* __restrict__ grid, const float2* __restrict__ weights,
						  float2* __restrict__ ksp, int a0, int a1, int a2, float rwidth)
{
	__shared__ float table[KB_SIZE + 1];

	for (int i = threadIdx.x; i < KB_SIZE + 1; i += 256)
		table[i] = kbt[i];

	__syncthreads();

	const long i = (long)blockIdx.x * 256 + threadIdx.x;

	if (i >= g.M)
		return;

	const int c0 = blockIdx.y * CC;
	const int ncc = min(CC, g.C - c0);
	const float4 kc = sk[i];
	const int act[3] = { a0, a1, a2 };  // active dims, x first

	// taps of the active dims and shift variants: weights, and offsets of the
	// grid points in a coil plane (unsigned: a plane of 2^31 points and more
	// fits the memory).  A tap without a weight takes the last one's point, and
	// a sub-grid where the sample has no taps adds nothing, so that a non-finite
	// grid point reaches only the samples next to it.
	float w[ND][2][NT];
	unsigned off[ND][2][NT];
	bool any[ND][2];

#pragma unroll
	for (int a = 0; a < ND; a++) {

		const int d = act[a];
		const unsigned str = (0 == d) ? 1u : ((1 == d) ? (unsigned)g.n[0] : (unsigned)g.n[0] * (unsigned)g.n[1]);
		const float k = sel3(d, kc.x, kc.y, kc.z);

#pragma unroll
		for (int v = 0; v < 2; v++) {

			if (v > 0 && g.nshv[d] < 2) {
#pragma unroll
				for (int j = 0; j < NT; j++) {
					w[a][1][j] = w[a][0][j];
					off[a][1][j] = off[a][0][j];
				}
				any[a][1] = any[a][0];
				continue;
			}

			int start, last;
			any[a][v] = taps_of<NT>(g, d, v, k, table, rwidth, start, last, w[a][v]);

#pragma unroll
			for (int j = 0; j < NT; j++)
				off[a][v][j] = str * (unsigned)tap_index(g, d, start, min(j, last));
		}
	}

	float2 acc[CC];
#pragma unroll
	for (int cl = 0; cl < CC; cl++)
		acc[cl] = make_float2(0.f, 0.f);

	auto subgrid = [&](int s, auto checked) {

		float ws[ND][NT];
		unsigned os[ND][NT];
		bool in = true;

#pragma unroll
		for (int a = 0; a < ND; a++) {
#pragma unroll
			for (int j = 0; j < NT; j++) {
				ws[a][j] = ((s >> a) & 1) ? w[a][1][j] : w[a][0][j];
				os[a][j] = ((s >> a) & 1) ? off[a][1][j] : off[a][0][j];
			}
			in = in && (((s >> a) & 1) ? any[a][1] : any[a][0]);
		}

		float2 val[CC];
#pragma unroll
		for (int cl = 0; cl < CC; cl++)
			val[cl] = make_float2(0.f, 0.f);

		const float2* gs = grid + ((long)s * g.C + c0) * g.N;
		constexpr int NZ = (ND > 2) ? NT : 1, NY = (ND > 1) ? NT : 1;

#pragma unroll
		for (int iz = 0; iz < NZ; iz++) {

			const float dz = (ND > 2) ? ws[ND - 1][iz] : 1.f;
			const unsigned oz = (ND > 2) ? os[ND - 1][iz] : 0u;

#pragma unroll
			for (int iy = 0; iy < NY; iy++) {

				const float dy = (ND > 1) ? dz * ws[(ND > 1) ? 1 : 0][iy] : dz;
				const unsigned oy = oz + ((ND > 1) ? os[(ND > 1) ? 1 : 0][iy] : 0u);

#pragma unroll
				for (int ix = 0; ix < NT; ix++) {

					const float dd = dy * ws[0][ix];
					const float2* p = gs + (oy + os[0][ix]);

#pragma unroll
					for (int cl = 0; cl < CC; cl++) {
						if (CC == 1 || cl < ncc) {
							float2 x = p[(long)cl * g.N];
							val[cl].x += x.x * dd;
							val[cl].y += x.y * dd;
						}
					}
				}
			}
		}

		if (!decltype(checked)::value || in)
#pragma unroll
			for (int cl = 0; cl < CC; cl++)
				acc[cl] = cadd(acc[cl], val[cl]);
	};

	// sub-grids: one bit per active dim (unrolled, with all their loads in
	// flight, while the registers last; a check per sub-grid would keep the
	// loads apart)
	bool all = true;

#pragma unroll
	for (int a = 0; a < ND; a++)
		all = all && any[a][0] && any[a][1];

	if (__all(all)) {

		constexpr int UNROLL = (ND <= 2 && NT <= 4) ? (1 << ND) : 1;

#pragma unroll UNROLL
		for (int s = 0; s < (1 << ND); s++)
			subgrid(s, std::false_type{});

	} else {

#pragma unroll 1
		for (int s = 0; s < (1 << ND); s++)
			subgrid(s, std::true_type{});
	}

	const int m = sm[i];
	const float2 wm = (nullptr != weights) ? weights[m] : make_float2(1.f, 0.f);

#pragma unroll
	for (int cl = 0; cl < CC; cl++)
		if (cl < ncc)
			ksp[(long)(c0 + cl) * g.M + m] = (nullptr != weights) ? cmul(acc[cl], wm) : acc[cl];
}

// ---------------------------------------------------------------------------
// Tiled forward gather (3-D grids): one work-group per work item, i.e. up to
// FW_MAXS samples of one home tile.  For every coil chunk and sub-grid the
// work-group stages the tile with its halo -- E^3 points of FW_CC coils, zero
// outside the grid -- in LDS with row-wise coalesced loads, and each thread
// gathers the taps of its samples from there.  The arithmetic is that of
// k_grid_fwd, term by term in the same order, so both give the same bits.
// A wave's samples come from the same or neighbouring cells, so that its
// lanes read points up to one apart in every dim: a point is 8 banks, a row
// 12 points and a plane 2 points more than its rows, which puts the 8 points
// of such a cube into 8 different bank groups.  All taps are taken (weight 0
// beyond an edge) instead of branching around the ones that are cut off.  Plans
// with such tiles have kernels of more than 2 and at most 3 points.
// Bound by LDS reads (27 float2 per sample, coil and sub-grid) and the waits of
// the staging: 128^3 kooshball, 16 coils, 3.31 -> 2.85 ms with constant taps
// and the padded planes (39.6 thousand vector instructions per wave, 47.6
// before).
// ---------------------------------------------------------------------------

constexpr size_t FW_TABLE_BYTES = ((KB_SIZE + 4) * sizeof(float) + 15) / 16 * 16;
constexpr int FW_ZPAD = 2;

// points of the staged region: planes with their padding
constexpr int fw_region(int E) { return E * (E * E + FW_ZPAD); }

// E: staged region edge (tile + halo); LDS region layout [z][y][x][coil].
// FULL: the kernel width is NT, so that only a grid's edge takes taps away and
// the taps off the grid are points of the halo, which is 0 there; otherwise a
// tap without a weight takes the last one's point.
template <int CCH, int E, int NT, bool FULL>
__global__ __launch_bounds__(FW_THREADS) void k_grid_fwd_tile(GridGeom g, FwdTiling ft, const float* __restrict__ kbt,
							      const int4* __restrict__ work,
							      const int* __restrict__ fsm,
							      const float4* __restrict__ fsk,
							      const float2* __restrict__ grid,
							      const float2* __restrict__ weights,
							      float2* __restrict__ ksp, float rwidth)
{
	constexpr int ZS = E * E + FW_ZPAD;
	static_assert(CCH == 4 && E <= 16 && 0 == E % 2, "region rows are loaded by 8 lanes, 4 coils per point");

	extern __shared__ __align__(16) unsigned char fw_smem[];
	float* table = (float*)fw_smem;
	float2* reg = (float2*)(fw_smem + FW_TABLE_BYTES);

	for (int i = threadIdx.x; i < KB_SIZE + 1; i += FW_THREADS)
		table[i] = kbt[i];

	const int4 it = work[blockIdx.x];
	const int tile = it.x;
	const int o0 = (tile % ft.nt[0]) * ft.T - ft.HL[0];
	const int o1 = ((tile / ft.nt[0]) % ft.nt[1]) * ft.T - ft.HL[1];
	const int o2 = (tile / (ft.nt[0] * ft.nt[1])) * ft.T - ft.HL[2];
	const int n0 = g.n[0], n1 = g.n[1], n2 = g.n[2];
	const int Ni = (int)g.N;

	// region loads: 8 lanes per row of E points (two points per lane),
	// rows (coil, z, y)
	const int lx2 = 2 * (threadIdx.x & 7);
	const int gx = o0 + lx2;
	const bool xin = lx2 < E && gx >= 0 && gx < n0;
	constexpr int NROW = CCH * E * E;
	constexpr int RSTEP = FW_THREADS / 8;

	float4 kc[FW_SPT];
	bool valid[FW_SPT];

#pragma unroll
	for (int q = 0; q < FW_SPT; q++) {
		const int j = it.y + threadIdx.x + FW_THREADS * q;
		valid[q] = j < it.z;
		kc[q] = valid[q] ? fsk[j] : make_float4(0.f, 0.f, 0.f, 0.f);
	}

	for (int c0 = 0; c0 < g.C; c0 += CCH) {

		const int ncc = min(CCH, g.C - c0);
		float2 acc[FW_SPT][CCH];

#pragma unroll
		for (int q = 0; q < FW_SPT; q++)
#pragma unroll
			for (int cl = 0; cl < CCH; cl++)
				acc[q][cl] = make_float2(0.f, 0.f);

		for (int s = 0; s < g.S; s++) {

			const float2* gs = grid + ((long)s * g.C + c0) * g.N;

			// the previous region has been consumed (and the table is in)
			__syncthreads();

			for (int r = threadIdx.x >> 3; r < NROW; r += RSTEP) {

				const int cl = r / (E * E);
				const int zy = r - cl * (E * E);
				const int z = zy / E;
				const int gy = o1 + zy - z * E;
				const int gz = o2 + z;
				float4 v = make_float4(0.f, 0.f, 0.f, 0.f);

				// 32-bit offsets within the chunk (the plan bounds CCH N);
				// x pairs start at even points (even origin and row length)
				if (xin && cl < ncc && gy >= 0 && gy < n1 && gz >= 0 && gz < n2)
					v = *(const float4*)(gs + cl * Ni + gx + n0 * (gy + n1 * gz));

				if (lx2 < E) {
					float2* d = reg + (z * ZS + (zy - z * E) * E + lx2) * CCH + cl;
					d[0] = make_float2(v.x, v.y);
					d[CCH] = make_float2(v.z, v.w);
				}
			}

			__syncthreads();

			const int v0 = g.sbit[s][0], v1 = g.sbit[s][1], v2 = g.sbit[s][2];

#pragma unroll
			for (int q = 0; q < FW_SPT; q++) {

				if (!valid[q])
					continue;

				int b0, b1, b2, e0, e1, e2;
				float w0[NT], w1[NT], w2[NT];
				const bool a0 = taps_staged<NT>(g, 0, v0, kc[q].x, table, rwidth, b0, e0, w0);
				const bool a1 = taps_staged<NT>(g, 1, v1, kc[q].y, table, rwidth, b1, e1, w1);
				const bool a2 = taps_staged<NT>(g, 2, v2, kc[q].z, table, rwidth, b2, e2, w2);

				// in the staged region (outside it: a sample without taps)
				b0 = min(max(b0, o0) - o0, E - NT);
				b1 = min(max(b1, o1) - o1, E - NT);
				b2 = min(max(b2, o2) - o2, E - NT);
				const float2* pt = reg + (b0 + E * b1 + ZS * b2) * CCH;

				float2 val[CCH];
#pragma unroll
				for (int cl = 0; cl < CCH; cl++)
					val[cl] = make_float2(0.f, 0.f);

#pragma unroll
				for (int iz = 0; iz < NT; iz++) {

					const float dz = w2[iz];
					const int lz = (FULL ? iz : min(iz, e2)) * ZS;

#pragma unroll
					for (int iy = 0; iy < NT; iy++) {

						const float dy = dz * w1[iy];
						const int ly = lz + (FULL ? iy : min(iy, e1)) * E;

#pragma unroll
						for (int ix = 0; ix < NT; ix++) {

							const float dd = dy * w0[ix];
							const float4* p = (const float4*)(pt + (ly + (FULL ? ix : min(ix, e0))) * CCH);
							const float4 x01 = p[0];
							const float4 x23 = p[1];
							val[0].x += x01.x * dd;
							val[0].y += x01.y * dd;
							val[1].x += x01.z * dd;
							val[1].y += x01.w * dd;
							val[2].x += x23.x * dd;
							val[2].y += x23.y * dd;
							val[3].x += x23.z * dd;
							val[3].y += x23.w * dd;
						}
					}
				}

				acc_where<CCH>(acc[q], val, a0 && a1 && a2);
			}
		}

#pragma unroll
		for (int q = 0; q < FW_SPT; q++) {

			if (!valid[q])
				continue;

			const int m = fsm[it.y + threadIdx.x + FW_THREADS * q];
			const float2 w = (nullptr != weights) ? weights[m] : make_float2(1.f, 0.f);

#pragma unroll
			for (int cl = 0; cl < CCH; cl++)
				if (cl < ncc)
					ksp[(long)(c0 + cl) * g.M + m] = (nullptr != weights) ? cmul(acc[q][cl], w) : acc[q][cl];
		}
	}
}

void grid_forward(const GridPlan& gp, const float* kb, float2* ksp, const float2* grid, const float2* weights,
		  hipStream_t st)
{
	const GridGeom& g = gp.g;

	if (0 == g.M || 0 == g.C)
		return;

	ProfScope prof("grid_forward", st);

	if (gp.ft.on) {

		const FwdTiling& ft = gp.ft;
		const size_t lds = FW_TABLE_BYTES + (size_t)FW_CC * fw_region(FW_E) * sizeof(float2);
		BAM_CHECK(FW_NT == gp.ta.ntap && !g.periodic && lds <= 64 * 1024 && FW_E == ft.E[0] &&
			  FW_E == ft.E[1] && FW_E == ft.E[2], "grid_forward: bad tiling");
#define BAM_FWT(FULL)                                                                                               \
	hipLaunchKernelGGL((k_grid_fwd_tile<FW_CC, FW_E, FW_NT, FULL>), dim3(ft.nitems), dim3(FW_THREADS), lds, st, g, ft, \
			   kb, gp.fwork.ptr, gp.fsm.ptr, gp.fsk.ptr, grid, weights, ksp, gp.ta.rwidth)
		if ((float)FW_NT == g.width)
			BAM_FWT(true);
		else
			BAM_FWT(false);
#undef BAM_FWT
		BAM_HIP(hipGetLastError());
		return;
	}

	const int tp = taps_bound(g);
	const GridTiling& t = gp.ta;

	// 4 coils per thread: the launch walks the samples chunk by chunk, so the
	// grid planes in use at a time are those of 4 coils (measured on a 128^3,
	// 16-coil kooshball: 7.7 ms at 4 coils, 12.4 ms at 16; 1 or 2 coils gain
	// nothing more).  One coil per thread in 2-D, where the taps cost little
	// beside the loads and all of a sample's loads fit in flight (320^2 spiral,
	// 32 coils: 112 us against 121; forward of 256^2, 98304 samples: 8 coils 82
	// against 97, 16 coils 113 against 115, 32 coils 179 against 187), and where 4 would leave less than 8 waves
	// per compute unit: a thread's chain of loads is then what the launch waits
	// for (64^2, 4 coils, 3968 samples: 38 -> 6 us).
	const bool one = t.ntap <= 3 && (t.nd < 3 || (long)g.M * ceil_div(g.C, 4) < 8l * 64 * gp.ncu);
	const dim3 blocks(ceil_div(g.M, 256), one ? (unsigned)g.C : ceil_div(g.C, 4));

#define BAM_FWD(NT, CC, ND)                                                                                      \
	hipLaunchKernelGGL((k_grid_fwd<NT, CC, ND>), blocks, dim3(256), 0, st, g, kb, gp.sm.ptr, gp.sk.ptr, grid, \
			   weights, ksp, t.act[0], t.act[1], t.act[2], t.rwidth)
#define BAM_FWD_CC(NT, ND)               \
	do {                             \
		if (one)                 \
			BAM_FWD(3, 1, ND); \
		else                     \
			BAM_FWD(NT, 4, ND); \
	} while (0)
#define BAM_FWD_ND(NT)                \
	do {                          \
		if (3 == t.nd)        \
			BAM_FWD_CC(NT, 3); \
		else if (2 == t.nd)   \
			BAM_FWD_CC(NT, 2); \
		else                  \
			BAM_FWD_CC(NT, 1); \
	} while (0)

	if (t.ntap <= 3)
		BAM_FWD_ND(3);
	else if (4 == tp)
		BAM_FWD_ND(4);
	else
		BAM_FWD_ND(8);
#undef BAM_FWD_ND
#undef BAM_FWD_CC
#undef BAM_FWD

	BAM_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Autotuner of the adjoint gridding launch
// ---------------------------------------------------------------------------

struct TuneEntry {
	std::string key;
	int cc, wpc;
	float ms;
	int tried;
};

static std::mutex tune_mtx;
static std::vector<TuneEntry> tune_table;  // this process's choices (and the file's)
static bool tune_loaded = false;

static std::string tune_file()
{
	const char* f = getenv("BART_AMD_TUNE_FILE");
	if (nullptr != f)
		return f;
	const char* h = getenv("HOME");
	return std::string(nullptr != h ? h : "/tmp") + "/.cache/bart_amd_tune.txt";
}

static void tune_load()
{
	if (tune_loaded)
		return;
	tune_loaded = true;
	FILE* fp = fopen(tune_file().c_str(), "r");
	if (nullptr == fp)
		return;
	char key[256];
	int cc, wpc;
	float ms;
	while (4 == fscanf(fp, "%255s %d %d %f", key, &cc, &wpc, &ms))
		tune_table.push_back(TuneEntry{ key, cc, wpc, ms, 0 });
	fclose(fp);
}

static void tune_store(const TuneEntry& e)
{
	std::string f = tune_file();
	std::string dir = f.substr(0, f.find_last_of('/'));
	if (!dir.empty())
		(void)mkdir(dir.c_str(), 0755);
	FILE* fp = fopen(f.c_str(), "a");
	if (nullptr == fp)
		return;  // not writable: the choice holds for this process only
	fprintf(fp, "%s %d %d %.4f\n", e.key.c_str(), e.cc, e.wpc, e.ms);
	fclose(fp);
}

void tune_grid_adjoint(GridPlan& gp, const float* kb, float2* grid, hipStream_t st)
{
	const GridGeom& g = gp.g;

	static const bool on = [] {
		const char* e = getenv("BART_AMD_AUTOTUNE");
		return !(nullptr != e && 0 == strcmp(e, "off"));
	}();

	if (!on || 0 == g.C || 0 == g.M || 0 == gp.nwork)
		return;

	char kbuf[256];
	snprintf(kbuf, sizeof(kbuf), "adj:%dx%dx%d:S%d:C%d:M%ld:ccmax%d:quads", g.n[0], g.n[1], g.n[2], g.S, g.C, g.M,
		 gp.cc_max);
	const std::string key = kbuf;

	{
		std::lock_guard<std::mutex> lock(tune_mtx);
		tune_load();
		for (const TuneEntry& e : tune_table)
			if (e.key == key && e.cc >= 4 && e.cc <= gp.cc_max && e.wpc >= 1 && e.wpc <= 4) {
				gp.ta.cc = e.cc;
				gp.wpc = e.wpc;
				return;
			}
	}

	// time every candidate on the plan with a zero k-space (two launches,
	// the second timed; the output is the same for all of them)
	DevBuf<float2> ksp((size_t)g.C * g.M);
	BAM_HIP(hipMemsetAsync(ksp.ptr, 0, sizeof(float2) * g.C * g.M, st));
	hipEvent_t e0, e1;
	BAM_HIP(hipEventCreate(&e0));
	BAM_HIP(hipEventCreate(&e1));
	const int cc0 = gp.ta.cc, wpc0 = gp.wpc;
	TuneEntry best{ key, cc0, wpc0, 1e30f, 0 };

	for (int cc = 4; cc <= gp.cc_max; cc *= 2) {
		for (int wpc = 1; wpc <= 4; wpc *= 2) {
			gp.ta.cc = cc;
			gp.wpc = wpc;
			grid_adjoint(gp, kb, grid, ksp.ptr, nullptr, st);
			BAM_HIP(hipEventRecord(e0, st));
			grid_adjoint(gp, kb, grid, ksp.ptr, nullptr, st);
			BAM_HIP(hipEventRecord(e1, st));
			BAM_HIP(hipEventSynchronize(e1));
			float ms = 0.f;
			BAM_HIP(hipEventElapsedTime(&ms, e0, e1));
			best.tried++;
			if (ms < best.ms) {
				best.ms = ms;
				best.cc = cc;
				best.wpc = wpc;
			}
		}
	}

	(void)hipEventDestroy(e0);
	(void)hipEventDestroy(e1);
	gp.ta.cc = best.cc;
	gp.wpc = best.wpc;

	std::lock_guard<std::mutex> lock(tune_mtx);
	tune_table.push_back(best);
	tune_store(best);
}

std::string tuning_report()
{
	std::lock_guard<std::mutex> lock(tune_mtx);
	std::string out = "[";
	for (size_t i = 0; i < tune_table.size(); i++) {
		const TuneEntry& e = tune_table[i];
		char b[512];
		snprintf(b, sizeof(b), "%s{\"shape\": \"%s\", \"coils_per_workgroup\": %d, \"workgroups_per_cu\": %d, "
			 "\"ms\": %.4f, \"candidates_timed\": %d}", i ? ", " : "", e.key.c_str(), e.cc, e.wpc, e.ms,
			 e.tried);
		out += b;
	}
	return out + "]";
}

}  // namespace bam
