// nufft.hip -- the decomposed 2x-oversampled NUFFT, its Toeplitz normal
// operator and PSF on gfx950.
//
// Algorithm of noncart/nufft.c (decomp = true, os = 2):
//   forward  (:1388-1458): roll -> x linphase_s -> FFT -> x fftmod -> sum_s gridH_s -> x weights
//   adjoint  (:1462-1540): x conj(weights) -> grid_s -> x conj(fftmod) -> IFFT -> sum_s conj(linphase_s) -> roll
//   normal   (:1546-1625): sum_s conj(linphase_s) IFFT(psf_s FFT(linphase_s x))
//   psf      (:727-776):   decompose(fftuc_2n(NUFFT^H_2n(|w|^2; 2 traj), periodic))
// Every element-wise factor is fused into the first or last FFT pass; the
// product with the coil maps (sense/modelnc.c, linops/fmac.c) and the sum
// over coils of S^H are fused there as well.
#include "cg.hpp"
#include "nufft_impl.hpp"
#include "prof.hpp"

#include <algorithm>
#include <cmath>
#include <complex>
#include <cstdlib>
#include <cstring>

namespace bam {

// ---------------------------------------------------------------------------
// Separable tables (host, FP64 maths)
// ---------------------------------------------------------------------------

// num/fft.c:64-90
double fftmod_phase(long length, long j)
{
	long center1 = length / 2;
	double shift = (double)center1 / (double)length;
	return ((double)j - (double)center1 / 2.) * shift;
}

std::complex<double> fftmod_value(double phase)
{
	double rem = phase - floor(phase);

	if (rem == 0.)
		return 1.;
	if (rem == 0.5)
		return -1.;
	if (rem == 0.25)
		return std::complex<double>(0., 1.);
	if (rem == 0.75)
		return std::complex<double>(0., -1.);

	return std::polar(1., 2. * M_PI * rem);
}

static double bessel_i0_d(double x)
{
	double q = 0.25 * x * x, term = 1., sum = 1.;

	for (int k = 1; k < 500; k++) {
		term *= q / ((double)k * (double)k);
		sum += term;
		if (term < 1.e-17 * sum)
			break;
	}

	return sum;
}

// noncart/grid.c:100-117, 522-531
double rolloff_1d(int d, int i, float os, double beta, double width)
{
	if (1 == d)
		return 1.;

	int od = os * d;
	int oi = i + (od / 2 - d / 2);
	float x = ((float)oi - (float)(od / 2)) / (float)od;

	double i0b = bessel_i0_d(beta);
	double a = beta * beta - pow(M_PI * x * width, 2.);
	double ft;

	if (0. == a)
		ft = 1. / i0b;
	else if (a > 0)
		ft = (sinh(sqrt(a)) / sqrt(a)) / i0b;
	else
		ft = (sin(sqrt(-a)) / sqrt(-a)) / i0b;

	return 1. / ft / width;
}

static void build_tables(Nufft& p)
{
	long tot = 0;
	long totr = 0;

	for (int d = 0; d < 3; d++) {
		tot += 3 * p.n[d];
		totr += p.n[d];
	}

	std::vector<float2> h2(tot);
	std::vector<float> hr(totr);
	long o2[3], orr[3];
	long a2 = 0, ar = 0;

	int bit = 0;

	for (int d = 0; d < 3; d++) {

		int n = p.n[d];
		o2[d] = a2;
		orr[d] = ar;
		a2 += 3 * n;
		ar += n;

		p.tabs.n[d] = n;
		p.tabs.bitpos[d] = (n > 1) ? bit++ : -1;

		for (int j = 0; j < n; j++) {

			hr[orr[d] + j] = (float)rolloff_1d(n, j, p.os, p.beta, p.width);

			std::complex<double> fm = (n > 1) ? fftmod_value(fftmod_phase(n, j)) : 1.;
			h2[o2[d] + 2 * n + j] = make_float2((float)fm.real(), (float)fm.imag());

			for (int b = 0; b < 2; b++) {

				std::complex<double> v = 1.;

				if (n > 1) {

					// compute_linphases (nufft.c:196-248) with linear_phase
					// (num/filter.c:241-265), one dim at a time
					double shift = -0.5 * b + (n / 2. - n / 2);
					double grad = 2. * M_PI * shift / (double)n;
					double ph = grad * (double)j - grad * (double)n / 2.;
					v = std::polar(1., ph) * fm / sqrt((double)n);
				}

				h2[o2[d] + b * n + j] = make_float2((float)v.real(), (float)v.imag());
			}
		}
	}

	p.tab2.alloc(tot);
	p.tabr.alloc(totr);
	BAM_HIP(hipMemcpy(p.tab2.ptr, h2.data(), sizeof(float2) * tot, hipMemcpyHostToDevice));
	BAM_HIP(hipMemcpy(p.tabr.ptr, hr.data(), sizeof(float) * totr, hipMemcpyHostToDevice));

	for (int d = 0; d < 3; d++) {
		p.tabs.lin[d][0] = p.tab2.ptr + o2[d];
		p.tabs.lin[d][1] = p.tab2.ptr + o2[d] + p.n[d];
		p.tabs.fm[d] = p.tab2.ptr + o2[d] + 2 * p.n[d];
		p.tabs.roll[d] = p.tabr.ptr + orr[d];
	}
}

__device__ inline float2 fm_val(const SepTables& T, const int c[3])
{
	float2 v = make_float2(1.f, 0.f);

#pragma unroll
	for (int d = 0; d < 3; d++)
		if (T.bitpos[d] >= 0)
			v = cmul(v, T.fm[d][c[d]]);

	return v;
}

// ---------------------------------------------------------------------------
// Pass functors
// ---------------------------------------------------------------------------

// Passes of the run-time FFT kernel over the members of sub-grid pairs (see
// pair.hpp): a block holds nm members of Q = P / nm columns, transform p of it
// member b0 + p / Q of the block's column p % Q.  Both members (nm = 2) share
// the loads of a split and the stores of a merge; where two do not fit (over
// FFT_MAX_ELEMS / 2 points) a launch takes one.
struct MemberGeom {

	VolAxis va;       // nvol: volumes split or merged
	int nm, b0;
	int logP, logQ;
	uint32_t nblk;
	long ncol;        // columns in all
	int cc;           // rows: coils per group, neighbours in a block
	FastDiv f_cc;

	// column of transform t: false beyond the last one
	__device__ bool column(long t, uint32_t& i, uint32_t& o, uint32_t& v, int& b) const
	{
		const uint32_t p = (uint32_t)t & ((1u << logP) - 1u);
		uint32_t blk = (uint32_t)(t >> logP);

		// neighbouring columns share cache lines
		if (1 != va.inner)
			blk = pf_xcd_order(blk, nblk);

		const long q = ((long)blk << logQ) + (p & ((1u << logQ) - 1u));
		b = b0 + (int)(p >> logQ);

		if (q >= ncol)
			return false;

		if (1 == cc) {
			va.split(q, i, o, v);
		} else {
			uint32_t r, cl, g;
			f_cc.divmod((uint32_t)q, r, cl);
			i = 0;
			va.f_outer.divmod(r, g, o);
			v = g * cc + cl;
		}

		return true;
	}
};

// split: the image side (src, with maps sens; x rolloff) or the grid, x the
// linear phases l; merge (no l): the members
struct LdMember {

	MemberGeom m;
	SepTables T;
	const float2* src;
	const float2* sens;
	bool roll;
	const float2* l[2];
	const float2* grid;
	long half;

	__device__ float2 operator()(long t, int k) const
	{
		uint32_t i, o, v;
		int b;

		if (!m.column(t, i, o, v, b))
			return make_float2(0.f, 0.f);

		const long at = m.va.offset_iov(i, o, v, k);

		if (nullptr == l[0])
			return grid[at + b * half];

		float2 x;

		if (nullptr == src)
			x = grid[at];
		else if (nullptr != sens)
			x = cmul(src[at - (long)v * m.va.N], sens[at]);
		else
			x = src[at];

		if (roll) {
			int c[3];
			m.va.coords(i, o, k, c);
			x = cscale(x, T.roll[0][c[0]] * T.roll[1][c[1]] * T.roll[2][c[2]]);
		}

		return cmul(x, l[b][k]);
	}
};

// PSFs of the members
struct MdMember {
	static constexpr bool active = true;
	MemberGeom m;
	FastDiv f_C;
	const float2* psf;
	long half;

	__device__ float2 operator()(long t, int k, float2 x) const
	{
		uint32_t i, o, v;
		int b;

		if (!m.column(t, i, o, v, b))
			return x;

		return cmul(x, psf[m.va.offset_iov(i, o, f_C.div(v), k) + b * half]);
	}
};

struct StSplit {

	MemberGeom m;
	SepTables T;
	float2* grid;
	long half;
	bool fm;

	__device__ void store(const float2* lds, const FftLaunch& L, long t0) const
	{
		store_each(lds, L, t0, [&](long t, int k, float2 x) {
			uint32_t i, o, v;
			int b;

			if (!m.column(t, i, o, v, b))
				return;

			if (fm) {
				int px[3];
				m.va.coords(i, o, k, px);
				x = cmul(x, fm_val(T, px));
			}

			grid[m.va.offset_iov(i, o, v, k) + b * half] = x;
		});
	}
};

// Sum over the members (and with maps over the coils of a group, into its
// partial image) into dst, without dst into the grid in place; the second
// launch of single members adds to what the first has left there.
struct StMerge {

	MemberGeom m;
	SepTables T;
	float2* dst;
	const float2* sens;
	bool roll;
	const float2* l[2];
	float2* grid;

	__device__ void store(const float2* lds, const FftLaunch& L, long t0) const
	{
		const int n = L.plan.n;
		const int Q = 1 << m.logQ;
		const int ng = Q / m.cc;  // sums per block and point

		for (int e = threadIdx.x; e < ng * n; e += FFT_THREADS) {

			// rows: points next to each other; columns: columns
			const int g = L.contig ? e / n : e & (Q - 1);
			const int k = L.contig ? e - g * n : e >> m.logQ;
			float2 a = make_float2(0.f, 0.f);
			uint32_t i, o, v = 0;
			int b;

			if (!m.column(t0 + g * m.cc, i, o, v, b))
				continue;

			const long at = m.va.offset_iov(i, o, v, k);

			for (int c = 0; c < m.cc; c++) {

				const float2* x = lds + (g * m.cc + c) * L.pitch + k;
				float2 s = cmulc(x[0], l[m.b0][k]);

				if (2 == m.nm)
					s = cadd(s, cmulc(x[Q * L.pitch], l[1][k]));

				if (nullptr != sens)
					s = cmulc(s, sens[at + c * m.va.N]);

				a = cadd(a, s);
			}

			if (roll) {
				int px[3];
				m.va.coords(i, o, k, px);
				a = cscale(a, T.roll[0][px[0]] * T.roll[1][px[1]] * T.roll[2][px[2]]);
			}

			if (nullptr == dst)
				grid[at] = (m.b0 > 0) ? cadd(grid[at], a) : a;
			else
				dst[m.va.offset_iov(i, o, v / (uint32_t)m.cc, k)] = a;
		}
	}
};

// ---------------------------------------------------------------------------
// Small element-wise kernels
// ---------------------------------------------------------------------------

__global__ void k_fill(float2* p, long n, float2 v, const int* skip)
{
	if (nullptr != skip && 0 != *skip)
		return;

	for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
		p[i] = v;
}

// dst[i] = sum_g part[g N + i], g = 0 .. G-1 in order
__global__ void k_sum_groups(float2* __restrict__ dst, const float2* __restrict__ part, long N, int G,
			     const int* skip)
{
	if (nullptr != skip && 0 != *skip)
		return;

	for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += (long)gridDim.x * blockDim.x) {

		float2 a = part[i];

		// (loads of several groups in flight)
#pragma unroll 8
		for (int g = 1; g < G; g++)
			a = cadd(a, part[(long)g * N + i]);

		dst[i] = a;
	}
}

static void sum_groups(float2* dst, const float2* part, long N, int G, hipStream_t st, const int* skip)
{
	ProfScope prof("sum_coil_groups", st);
	unsigned blocks = (unsigned)std::min<long>((N + 255) / 256, 4096);
	hipLaunchKernelGGL(k_sum_groups, dim3(blocks), dim3(256), 0, st, dst, part, N, G, skip);
	BAM_HIP(hipGetLastError());
}

__global__ void k_axpy(float2* __restrict__ d, const float2* __restrict__ x, float a, long n, const int* skip)
{
	if (nullptr != skip && 0 != *skip)
		return;

	for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
		const float2 v = x[i];
		d[i] = make_float2(d[i].x + a * v.x, d[i].y + a * v.y);
	}
}

void axpy(float2* d, const float2* x, float a, long n, hipStream_t st, const int* skip)
{
	const unsigned blocks = (unsigned)std::min<long>((n + 255) / 256, 8192);
	hipLaunchKernelGGL(k_axpy, dim3(blocks), dim3(256), 0, st, d, x, a, n, skip);
	BAM_HIP(hipGetLastError());
}

void sum_images(float2* dst, const float2* part, long N, int G, hipStream_t st, const int* skip)
{
	sum_groups(dst, part, N, G, st, skip);
}

void fill(float2* p, long n, float2 v, hipStream_t st, const int* skip)
{
	if (n <= 0)
		return;
	ProfScope prof("fill", st);
	unsigned blocks = (unsigned)std::min<long>((n + 255) / 256, 8192);
	hipLaunchKernelGGL(k_fill, dim3(blocks), dim3(256), 0, st, p, n, v, skip);
	BAM_HIP(hipGetLastError());
}

// ---------------------------------------------------------------------------
// Plan creation
// ---------------------------------------------------------------------------

void Nufft::create(const int dims[3], int C_, long M_, const float* traj, const float2* weights_host,
		   bool toeplitz_, bool periodic_, float width_, float os_, bool compute_psf)
{
	create_geometry(dims, C_, toeplitz_, periodic_, width_, os_);
	set_traj(M_, traj, weights_host, compute_psf);
}

static int merge_group(const Nufft& p);

void Nufft::create_geometry(const int dims[3], int C_, bool toeplitz_, bool periodic_, float width_, float os_)
{
	BAM_CHECK(2.f == os_, "only oversampling 2 is supported (got %f)", os_);
	BAM_CHECK(width_ > 0.f && width_ / 2.f <= (float)(MAX_TAPS - 1), "kernel width %f not supported", width_);

	ncu = device_cus();
	N = 1;
	nact = 0;
	S = 1;

	for (int d = 0; d < 3; d++) {

		n[d] = dims[d];
		BAM_CHECK(n[d] >= 1, "bad image dims");
		N *= n[d];

		if (n[d] > 1) {
			BAM_CHECK(fft_size_supported(n[d]), "image dim %d not supported by the FFT", n[d]);
			act[nact++] = d;
			S *= 2;
		}
	}

	BAM_CHECK(nact >= 1, "NUFFT needs at least one non-trivial image dim");

	C = C_;
	M = 0;
	width = width_;
	os = os_;
	// BART's KB table is built by the first kb_init call, which
	// rolloff_correction makes with beta passed as float (noncart/nufft.c:898,
	// noncart/grid.c:537-540); the table, I0(beta) and the rolloff all use
	// the float-rounded beta
	beta = (double)(float)calc_beta(os, width);
	periodic = periodic_;
	toeplitz = toeplitz_;

	std::vector<float> kbh(KB_SIZE + 1);
	kb_table_host(beta, kbh.data());
	kb.alloc(KB_SIZE + 1);
	BAM_HIP(hipMemcpy(kb.ptr, kbh.data(), sizeof(float) * (KB_SIZE + 1), hipMemcpyHostToDevice));

	build_tables(*this);

	for (int j = 0; j < nact; j++) {
		axis[j] = make_axis_plan(n[act[j]]);
		pair[j] = make_pair_plan(axis[j]);
	}

	grid.alloc((size_t)S * C * N);

	// partial images of the coil groups of S^H (allocated here so that no
	// allocation happens inside a captured CG iteration)
	const int G = C / merge_group(*this);

	if (G > 1)
		part.alloc((size_t)G * N);
}

// Trajectory, weights, gridding plan and (Toeplitz) PSF -- nufft_set_traj
// (noncart/nufft.c:1002-1159).  Called again by nufft_update_traj: the
// sample count stays that of the k-space dims.
void Nufft::set_traj(long M_, const float* traj, const float2* weights_host, bool compute_psf)
{
	M = M_;
	has_traj = false;
	has_psf = false;
	has_weights = (nullptr != weights_host);

	if (has_weights) {
		weights.alloc(std::max<long>(M, 1));
		if (M > 0)
			BAM_HIP(hipMemcpy(weights.ptr, weights_host, sizeof(float2) * M, hipMemcpyHostToDevice));
	}

	// gridding geometry of the decomposition (nufft.c:147-188)
	GridGeom g = {};

	for (int d = 0; d < 3; d++)
		g.n[d] = n[d];

	g.N = N;
	g.C = C;
	g.M = M;
	g.S = S;
	g.os = 1.f;
	g.width = width / 2.f;
	g.periodic = periodic;

	for (int d = 0; d < 3; d++)
		g.fm[d] = tabs.fm[d];

	for (int s = 0; s < S; s++) {

		int idx = s;

		for (int d = 0; d < 3; d++) {

			int f = (n[d] > 1) ? 2 : 1;
			float sh = -(float)(idx % f) / f;
			idx /= f;

			if (f > 1)
				sh += (n[d] / 2.0 - n[d] / 2) / g.os;

			g.shift[s][d] = sh;
		}
	}

	gp.build(g, traj);
	has_traj = true;
	if (tune)
		tune_grid_adjoint(gp, kb.ptr, grid.ptr, stream);

	if (toeplitz && compute_psf)
		compute_psf_from_traj(traj, weights_host, true);
}

// ---------------------------------------------------------------------------
// Forward / adjoint / normal
// ---------------------------------------------------------------------------

// ---------------------------------------------------------------------------
// Axis passes of the decomposition (see pair.hpp).  Axis j (of the active
// ones) doubles the volumes: split takes the C 2^j volumes c + C s of the
// grid (axis 0: the image side) to C 2^(j + 1), merge back.  Lengths beyond
// the pair kernels (over PF_MAXN, or no three radices) run on the run-time FFT
// kernel (LdMember, ...).
// ---------------------------------------------------------------------------

// its coils per partial image: a block of at most 4096 points
static int member_group(const Nufft& p)
{
	int cc = 1;

	while (0 == p.C % (2 * cc) && 4l * cc * p.n[p.act[0]] <= FFT_MAX_ELEMS / 2)
		cc *= 2;

	return cc;
}

// coils per partial image of the last merge: the most that leave 16 waves per
// compute unit to share the work (the partial images cost a pass over G N
// values in all), but not more than MERGE_IMAGES partial images, each of which
// a point of the sum waits for (256 points, 1024 coils, normal with maps: 260 us
// with 1024 of them, 64 with 64)
constexpr int MERGE_IMAGES = 64;

static int merge_group(const Nufft& p)
{
	const PairPlan& pl = p.pair[0];
	const long lanes = (p.N / p.n[p.act[0]]) * std::max(1, pl.NJ);
	int cc = 1;

	if (0 == pl.nr)
		return member_group(p);

	for (int c = 2; c <= p.C; c++)
		if (0 == p.C % c && (lanes * (p.C / c) >= 16l * 64 * p.ncu || p.C / cc > MERGE_IMAGES))
			cc = c;

	return cc;
}

static PairArgs pair_args(const Nufft& p, int j, const int* skip)
{
	PairArgs a = {};
	a.pl = p.pair[j];
	a.va = VolAxis::make(p.n, p.act[j], (0 == j) ? 1 : ((long)p.C << j));
	a.skip = skip;
	a.l[0] = p.tabs.lin[p.act[j]][0];
	a.l[1] = p.tabs.lin[p.act[j]][1];
	a.grid = p.grid.ptr;
	a.half = ((long)p.C << j) * p.N;
	a.C = p.C;
	a.cc = 1;
	return a;
}

static PairArgs rows_split_args(const Nufft& p, const float2* src, const float2* sens, bool roll, bool fm,
				const int* skip)
{
	PairArgs a = pair_args(p, 0, skip);
	a.src = src;
	a.sens = sens;
	for (int d = 0; d < 3; d++) {
		a.roll[d] = roll ? p.tabs.roll[d] : nullptr;
		a.fm[d] = fm ? p.tabs.fm[d] : nullptr;
	}
	pair_geometry(a, true, (uint32_t)p.C, p.ncu);
	return a;
}

static PairArgs rows_merge_args(const Nufft& p, float2* dst, const float2* sens, bool roll, const int* skip)
{
	PairArgs a = pair_args(p, 0, skip);
	a.dst = dst;
	a.sens = sens;
	a.cc = (nullptr != sens) ? merge_group(p) : 1;
	for (int d = 0; d < 3; d++)
		a.roll[d] = roll ? p.tabs.roll[d] : nullptr;
	pair_geometry(a, true, (uint32_t)(p.C / a.cc), p.ncu);
	return a;
}

static PairArgs turn_args(const Nufft& p, const int* skip)
{
	const int j = p.nact - 1;
	PairArgs a = pair_args(p, j, skip);
	a.psf = p.psf.ptr;
	a.psf_half = (1l << j) * p.N;
	pair_geometry(a, false, 0, p.ncu);
	return a;
}

// Members of axis j on the run-time kernel: geometry.  Rows: blocks of 2048 points
// and more; columns: 16 next to each other (128 bytes), as far as 128 KB of LDS
// hold them and no compute unit is left without a block (12 x 1040, 2 coils,
// normal: 98 us with four columns per block, 62 with one).
static FftLaunchCfg member_config(const Nufft& p, int j, int nm, int b0, int cc, float sign, MemberGeom& m)
{
	const int n = p.n[p.act[j]];
	m.va = VolAxis::make(p.n, p.act[j], (long)p.C << j);
	m.nm = nm;
	m.b0 = b0;
	m.cc = cc;
	m.f_cc = FastDiv((uint32_t)cc);
	m.ncol = m.va.transforms();

	const bool contig = m.va.contig();
	int Q = contig ? cc : 1;

	if (contig)
		while (nm * Q * n < 2048)
			Q *= 2;
	else
		while (Q < 16 && 2l * nm * Q * n <= 2 * FFT_MAX_ELEMS && m.ncol >= 2l * Q * p.ncu)
			Q *= 2;

	BAM_CHECK((long)nm * Q * n <= 2 * FFT_MAX_ELEMS, "FFT block of %d x %d exceeds LDS budget", nm * Q, n);

	m.logQ = 0;
	while ((1 << m.logQ) < Q)
		m.logQ++;
	m.logP = m.logQ + (nm - 1);
	m.nblk = (uint32_t)((m.ncol + Q - 1) / Q);

	FftLaunchCfg c;
	c.L.plan = p.axis[j];
	c.L.P = nm * Q;
	c.L.logP = m.logP;
	c.L.contig = contig;
	c.L.total = (long)m.nblk * c.L.P;
	c.L.sign = sign;
	c.L.pitch = n;
	c.blocks = m.nblk;
	c.lds_bytes = (size_t)nm * Q * n * sizeof(float2);
	c.ept = (nm * Q * n <= 4096) ? 8 : ((nm * Q * n <= 8192) ? 16 : 32);
	return c;
}

// members per block: both, as far as they fit
static int members(const Nufft& p, int j) { return (2 * p.n[p.act[j]] <= FFT_MAX_ELEMS) ? 2 : 1; }

static LdMember member_load(const Nufft& p, int j, const MemberGeom& m, const float2* src, const float2* sens, bool roll,
			    bool phase)
{
	const int d = p.act[j];
	return LdMember{ m, p.tabs, src, sens, roll, { phase ? p.tabs.lin[d][0] : nullptr, phase ? p.tabs.lin[d][1] : nullptr },
			 p.grid.ptr, m.va.nvol * p.N };
}

static StMerge member_sum(const Nufft& p, int j, const MemberGeom& m, float2* dst, const float2* sens, bool roll)
{
	const int d = p.act[j];
	return StMerge{ m, p.tabs, dst, sens, roll, { p.tabs.lin[d][0], p.tabs.lin[d][1] }, p.grid.ptr };
}

static void member_split(const Nufft& p, int j, const float2* src, const float2* sens, bool roll, bool fm,
			 const int* skip, const char* name)
{
	const int nm = members(p, j);

	// single members: the second first, as the first takes the source's place
	for (int b0 = 2 - nm; b0 >= 0; b0--) {
		MemberGeom m;
		FftLaunchCfg cfg = member_config(p, j, nm, b0, 1, -1.f, m);
		cfg.L.skip = skip;
		cfg.name = name;
		launch_fft_any(cfg, p.stream, member_load(p, j, m, src, sens, roll, true), NoMid{},
			       StSplit{ m, p.tabs, p.grid.ptr, m.va.nvol * p.N, fm });
	}
}

static void member_merge(const Nufft& p, int j, float2* dst, const float2* sens, bool roll, int cc, const int* skip,
			 const char* name)
{
	const int nm = members(p, j);

	for (int b0 = 0; b0 <= 2 - nm; b0++) {
		MemberGeom m;
		FftLaunchCfg cfg = member_config(p, j, nm, b0, cc, +1.f, m);
		cfg.L.skip = skip;
		cfg.name = name;
		launch_fft_any(cfg, p.stream, member_load(p, j, m, nullptr, nullptr, false, false), NoMid{},
			       member_sum(p, j, m, dst, sens, roll));
	}
}

// split, PSFs and merge of the last axis
static void member_turn(const Nufft& p, int j, float2* dst, const float2* src, const float2* sens, int cc,
			const int* skip, const char* name)
{
	MemberGeom m;
	FftLaunchCfg cfg = member_config(p, j, 2, 0, cc, -1.f, m);
	cfg.L.skip = skip;
	cfg.name = name;
	launch_fft_any(cfg, p.stream, member_load(p, j, m, src, sens, false, true),
		       MdMember{ m, FastDiv((uint32_t)p.C), p.psf.ptr, (1l << j) * p.N },
		       member_sum(p, j, m, dst, sens, false));
}

// the image side's forms: src / dst non-null on axis 0 only
static void axis_split(const Nufft& p, int j, const float2* src, const float2* sens, bool roll, bool fm,
		       const int* skip, const char* name)
{
	if (0 == p.pair[j].nr) {
		member_split(p, j, src, sens, roll, fm, skip, name);
		return;
	}

	if (0 == j) {
		pair_launch(PF_SPLIT, true, rows_split_args(p, src, sens, roll, fm, skip), name, p.stream);
		return;
	}

	PairArgs a = pair_args(p, j, skip);
	for (int d = 0; d < 3; d++)
		a.fm[d] = fm ? p.tabs.fm[d] : nullptr;
	pair_geometry(a, false, 0, p.ncu);
	pair_launch(PF_SPLIT, false, a, name, p.stream);
}

static void axis_merge(const Nufft& p, int j, float2* dst, const float2* sens, bool roll, const int* skip,
		       const char* name)
{
	if (0 == p.pair[j].nr) {
		member_merge(p, j, dst, sens, roll, (nullptr != sens) ? member_group(p) : 1, skip, name);
		return;
	}

	if (0 == j) {
		pair_launch(PF_MERGE, true, rows_merge_args(p, dst, sens, roll, skip), name, p.stream);
		return;
	}

	PairArgs a = pair_args(p, j, skip);
	pair_geometry(a, false, 0, p.ncu);
	pair_launch(PF_MERGE, false, a, name, p.stream);
}

// The range of the entry points: the S transforms of a row of the first axis in
// one LDS block of the FFT.  (No pass needs it any more; a plan beyond it stays
// refused.)
static void check_first_axis(const Nufft& p)
{
	BAM_CHECK((long)p.S * p.n[p.act[0]] <= FFT_MAX_ELEMS, "FFT block of %d x %d exceeds LDS budget", p.S,
		  p.n[p.act[0]]);
}

// partial images of S^H of cc coils each: their number, and where the last merge
// writes
static float2* merge_target(Nufft& p, float2* dst, const float2* sens, int cc, int& G)
{
	G = (nullptr != sens) ? p.C / cc : 1;

	if (G <= 1)
		return dst;

	if ((long)p.part.n < (long)G * p.N)
		p.part.alloc((size_t)G * p.N);

	return p.part.ptr;
}

void Nufft::forward(float2* ksp, const float2* src, const float2* sens)
{
	check_first_axis(*this);
	axis_split(*this, 0, src, sens, true, 1 == nact, nullptr, "fft_fwd_first");

	for (int j = 1; j < nact; j++)
		axis_split(*this, j, nullptr, nullptr, false, j == nact - 1, nullptr, "fft_fwd_axis");

	grid_forward(gp, kb.ptr, ksp, grid.ptr, has_weights ? weights.ptr : nullptr, stream);
}

void Nufft::adjoint(float2* dst, const float2* ksp, const float2* sens)
{
	// the output-stationary adjoint gridding writes every grid point
	grid_adjoint(gp, kb.ptr, grid.ptr, ksp, has_weights ? weights.ptr : nullptr, stream);

	check_first_axis(*this);

	for (int j = nact - 1; j >= 1; j--)
		axis_merge(*this, j, nullptr, nullptr, false, nullptr, "fft_adj_axis");

	int G;
	float2* out = merge_target(*this, dst, sens, merge_group(*this), G);
	axis_merge(*this, 0, out, sens, true, nullptr, "fft_adj_last");

	if (out != dst)
		sum_groups(dst, part.ptr, N, G, stream, nullptr);
}

// the coil-group sum that ends a normal operator, or with fuse the CG step
// fused into it
static bool sum_groups_or_fuse(float2* dst, const float2* part, long N, int G, hipStream_t st, const int* skip,
			       const CgApFuse* fuse)
{
	if (nullptr != fuse) {
		BAM_CHECK((const float*)dst == fuse->Ap && fuse->len == 2 * N, "normal: fused CG step mismatch");
		cg_apdot_groups(*fuse, part, N, G, st);
		return true;
	}

	sum_groups(dst, part, N, G, st, skip);
	return false;
}

bool Nufft::normal(float2* dst, const float2* src, const float2* sens, const int* skip, const CgApFuse* fuse)
{
	BAM_CHECK(has_psf, "Toeplitz normal operator without PSF");
	BAM_CHECK(0 == nbasis, "normal: a plan with a subspace basis takes normal_basis");

	check_first_axis(*this);
	const int last = nact - 1;
	const int cc = merge_group(*this);
	int G;
	float2* out = merge_target(*this, dst, sens, cc, G);

	if (0 == last) {

		// one axis: the PSFs are multiplied where the split stores, or the
		// run-time kernel takes both directions
		if (pair[0].nr > 0) {
			PairArgs a = rows_split_args(*this, src, sens, false, false, skip);
			a.psf = psf.ptr;
			a.psf_half = N;
			pair_launch(PF_SPLIT_PSF, true, a, "fft_toeplitz_fwd", stream);
			axis_merge(*this, 0, out, sens, false, skip, "fft_toeplitz_inv");
		} else {
			member_turn(*this, 0, out, src, sens, (nullptr != sens) ? cc : 1, skip, "fft_toeplitz");
		}

	} else {

		axis_split(*this, 0, src, sens, false, false, skip, "fft_toeplitz_fwd");

		for (int j = 1; j < last; j++)
			axis_split(*this, j, nullptr, nullptr, false, false, skip, "fft_toeplitz_fwd");

		if (pair[last].nr > 0) {
			pair_launch(PF_TURN, false, turn_args(*this, skip), "fft_toeplitz", stream);
		} else if (2 == members(*this, last)) {
			member_turn(*this, last, nullptr, nullptr, nullptr, 1, skip, "fft_toeplitz");
		} else {
			axis_split(*this, last, nullptr, nullptr, false, false, skip, "fft_toeplitz_fwd");
			basis_psf_apply(grid.ptr, psf.ptr, S, C, 1, N, stream, skip);
			axis_merge(*this, last, nullptr, nullptr, false, skip, "fft_toeplitz_inv");
		}

		for (int j = last - 1; j >= 1; j--)
			axis_merge(*this, j, nullptr, nullptr, false, skip, "fft_toeplitz_inv");

		axis_merge(*this, 0, out, sens, false, skip, "fft_toeplitz_inv");
	}

	if (out != dst)
		return sum_groups_or_fuse(dst, part.ptr, N, G, stream, skip, fuse);

	return false;
}

void Nufft::set_basis(int K, int T, long Mf, const float2* B_host)
{
	BAM_CHECK(K >= 1 && K <= BASIS_MAX, "basis: %d coefficients (at most %d)", K, BASIS_MAX);
	BAM_CHECK(T >= 1 && Mf >= 0, "basis: bad frame dims");
	nbasis = K;
	bT = T;
	bMf = Mf;
	bas.alloc((size_t)K * T);
	BAM_HIP(hipMemcpy(bas.ptr, B_host, sizeof(float2) * K * T, hipMemcpyHostToDevice));
}

// Toeplitz normal operator with a subspace basis (noncart/nufft.c:1546-1625
// with the K x K PSF of nufft_set_traj): per sub-grid s, FFT(linphase_s x_k)
// for every coil and coefficient, the PSF product over the coefficients,
// IFFT, conj(linphase_s), sum over s.  The last axis is transformed forward,
// multiplied (basis_psf_apply) and transformed back in three launches.
void Nufft::normal_basis(float2* dst, const float2* src, const int* skip)
{
	BAM_CHECK(has_psf && nbasis > 0, "normal_basis: no subspace PSF");
	BAM_CHECK(0 == C % nbasis, "normal_basis: channels %d not a multiple of %d coefficients", C, nbasis);
	const int Cc = C / nbasis;

	check_first_axis(*this);
	axis_split(*this, 0, src, nullptr, false, false, skip, "fft_toeplitz_basis_first");

	for (int j = 1; j < nact; j++)
		axis_split(*this, j, nullptr, nullptr, false, false, skip, "fft_toeplitz_basis_fwd");

	basis_psf_apply(grid.ptr, psf.ptr, S, Cc, nbasis, N, stream, skip);

	for (int j = nact - 1; j >= 1; j--)
		axis_merge(*this, j, nullptr, nullptr, false, skip, "fft_toeplitz_basis_inv");

	axis_merge(*this, 0, dst, nullptr, false, skip, "fft_toeplitz_basis_last");
}

// ---------------------------------------------------------------------------
// Strang's circulant preconditioner (noncart/precond.c:46-71, 92-106)
// ---------------------------------------------------------------------------

__device__ inline float2 sep_fm(const SepTables& T, long i, const int n[3])
{
	const int x = (int)(i % n[0]);
	const int y = (int)((i / n[0]) % n[1]);
	const int z = (int)(i / ((long)n[0] * n[1]));
	return cmul(cmul(T.fm[0][x], T.fm[1][y]), T.fm[2][z]);
}

__device__ inline float2 sep_lin(const SepTables& T, int s, long i, const int n[3])
{
	const int c[3] = { (int)(i % n[0]), (int)((i / n[0]) % n[1]), (int)(i / ((long)n[0] * n[1])) };
	float2 v = make_float2(1.f, 0.f);
	for (int d = 0; d < 3; d++)
		if (T.bitpos[d] >= 0)
			v = cmul(v, T.lin[d][(s >> T.bitpos[d]) & 1][c[d]]);
	return v;
}

struct Int3 {
	int v[3];
};

// tmp[s][i] = psf[s][i] conj(fm(i)) (ifftmod before the inverse FFT)
__global__ void k_pre_load(SepTables T, Int3 n, long N, int S, const float2* __restrict__ psf, float2* __restrict__ tmp)
{
	for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < (long)S * N; e += (long)gridDim.x * blockDim.x)
		tmp[e] = cmulc(psf[e], sep_fm(T, e % N, n.v));
}

// acc(i) = sum_s conj(fm(i)) tmp[s](i) conj(lin_s(i)) (ifftmod after the
// inverse FFT, the cropped PSF of md_zfmacc2), then x fm(i) (fftmod before
// the forward FFT)
__global__ void k_pre_sum(SepTables T, Int3 n, long N, int S, const float2* __restrict__ tmp, float2* __restrict__ acc)
{
	for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += (long)gridDim.x * blockDim.x) {
		const float2 fm = sep_fm(T, i, n.v);
		float2 a = make_float2(0.f, 0.f);
		for (int s = 0; s < S; s++)
			a = cadd(a, cmulc(cmulc(tmp[(long)s * N + i], fm), sep_lin(T, s, i, n.v)));
		acc[i] = cmul(a, fm);
	}
}

// pre(i) = |fm(i) acc(i)| + 1e-3 (fftmod after the forward FFT, md_zabs,
// md_zsadd)
__global__ void k_pre_abs(SepTables T, Int3 n, long N, float2* __restrict__ acc)
{
	for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < N; i += (long)gridDim.x * blockDim.x) {
		const float2 v = cmul(acc[i], sep_fm(T, i, n.v));
		acc[i] = make_float2(sqrtf(v.x * v.x + v.y * v.y) + 1e-3f, 0.f);
	}
}

// dst[c][i] = src[c][i] / pre[i]
__global__ void k_pre_div(float2* __restrict__ dst, const float2* __restrict__ pre, long N, long total)
{
	for (long e = (long)blockIdx.x * blockDim.x + threadIdx.x; e < total; e += (long)gridDim.x * blockDim.x) {
		const float2 v = dst[e];
		const float p = pre[e % N].x;
		dst[e] = make_float2(v.x / p, v.y / p);
	}
}

void Nufft::compute_precond(DevBuf<float2>& pre) const
{
	BAM_CHECK(toeplitz && has_psf, "nufft_precond_create: needs a Toeplitz operator with its PSF");
	DevBuf<float2> tmp((size_t)S * N);
	pre.alloc(N);
	const Int3 nn{ { n[0], n[1], n[2] } };
	const unsigned blk = (unsigned)std::min<long>(((long)S * N + 255) / 256, 8192);
	const float sc = 1.f / sqrtf((float)N);

	hipLaunchKernelGGL(k_pre_load, dim3(blk), dim3(256), 0, stream, tabs, nn, N, S, psf.ptr, tmp.ptr);
	fft_nd(n, S, 7, +1.f, tmp.ptr, tmp.ptr, sc, stream);
	hipLaunchKernelGGL(k_pre_sum, dim3(blk), dim3(256), 0, stream, tabs, nn, N, S, tmp.ptr, pre.ptr);
	fft_nd(n, 1, 7, -1.f, pre.ptr, pre.ptr, sc, stream);
	hipLaunchKernelGGL(k_pre_abs, dim3(blk), dim3(256), 0, stream, tabs, nn, N, pre.ptr);
	BAM_HIP(hipGetLastError());
	BAM_HIP(hipStreamSynchronize(stream));
}

// dst = IFFT(FFT(src) / pre) per coil, unnormalised FFTs over the image
// dims (linop_fft_create, linops/someops.c:1732-1776): BART's
// nufft_precond_apply (noncart/precond.c:92-106)
void Nufft::apply_precond(const float2* pre, float2* dst, const float2* src, int ncoil) const
{
	fft_nd(n, ncoil, 7, -1.f, dst, src, 1.f, stream);
	const long total = (long)ncoil * N;
	const unsigned blk = (unsigned)std::min<long>((total + 255) / 256, 8192);
	hipLaunchKernelGGL(k_pre_div, dim3(blk), dim3(256), 0, stream, dst, pre, N, total);
	BAM_HIP(hipGetLastError());
	fft_nd(n, ncoil, 7, +1.f, dst, dst, 1.f, stream);
}

// ---------------------------------------------------------------------------
// Normal operators of many 2-D plans in one launch per pass (batched CG)
// ---------------------------------------------------------------------------

// The three passes of Nufft::normal's 2-D path (split of the first axis with
// maps, turn of the second, merge of the first with the sums over coil
// groups) for every plan, each pass one launch per kernel that its lengths
// take: the same work-groups and arithmetic as the plans' own launches, so the
// results are the same bits.
struct NormalGroupSet {

	struct Pass {
		int nb = 0;
		unsigned threads = 0;
		size_t lds = 0;
		DevBuf<PairArgs> items;
		DevBuf<int2> bt;
	};

	Pass pass[3][PF_CLASSES];
};

bool normal_groupable(const Nufft& p, const float2* sens)
{
	if (2 != p.nact || !p.toeplitz || !p.has_psf || nullptr == sens || p.nbasis > 0)
		return false;

	if (0 == p.pair[0].nr || 0 == p.pair[1].nr || (long)p.S * p.n[p.act[0]] > FFT_MAX_ELEMS)
		return false;

	const int G = p.C / merge_group(p);
	return G <= 1 || (long)p.part.n >= (long)G * p.N;
}

std::shared_ptr<NormalGroupSet> normal_groups_build(const std::vector<const Nufft*>& plans,
						    const std::vector<const float2*>& sens,
						    const std::vector<const float2*>& src, const std::vector<float2*>& dst,
						    const std::vector<const int*>& skip)
{
	auto set = std::make_shared<NormalGroupSet>();
	std::vector<PairArgs> items[3][PF_CLASSES];

	for (size_t q = 0; q < plans.size(); q++) {

		const Nufft& p = *plans[q];
		float2* out = (p.C / merge_group(p) > 1) ? p.part.ptr : dst[q];
		const PairArgs a[3] = { rows_split_args(p, src[q], sens[q], false, false, skip[q]), turn_args(p, skip[q]),
					rows_merge_args(p, out, sens[q], false, skip[q]) };

		for (int ph = 0; ph < 3; ph++) {
			const int cl = a[ph].cl;
			NormalGroupSet::Pass& P = set->pass[ph][cl];
			P.threads = std::max(P.threads, pair_threads(a[ph], 1 != ph));
			P.lds = std::max(P.lds, pair_lds_bytes(a[ph], 1 != ph));
			items[ph][cl].push_back(a[ph]);
		}
	}

	for (int ph = 0; ph < 3; ph++)
		for (int cl = 0; cl < PF_CLASSES; cl++) {

			NormalGroupSet::Pass& P = set->pass[ph][cl];
			const std::vector<PairArgs>& it = items[ph][cl];
			std::vector<int2> bt;

			for (size_t i = 0; i < it.size(); i++)
				for (uint32_t b = 0; b < it[i].nblk; b++)
					bt.push_back(make_int2((int)i, (int)b));

			P.nb = (int)bt.size();

			if (0 == P.nb)
				continue;

			P.items.alloc(it.size());
			P.bt.alloc(bt.size());
			BAM_HIP(hipMemcpy(P.items.ptr, it.data(), sizeof(PairArgs) * it.size(), hipMemcpyHostToDevice));
			BAM_HIP(hipMemcpy(P.bt.ptr, bt.data(), sizeof(int2) * bt.size(), hipMemcpyHostToDevice));
		}

	return set;
}

void normal_groups_launch(const NormalGroupSet& set, hipStream_t st)
{
	static const char* name[3] = { "fft_toeplitz_fwd", "fft_toeplitz", "fft_toeplitz_inv" };
	static const int mode[3] = { PF_SPLIT, PF_TURN, PF_MERGE };

	for (int ph = 0; ph < 3; ph++)
		for (int cl = 0; cl < PF_CLASSES; cl++) {
			const NormalGroupSet::Pass& P = set.pass[ph][cl];
			pair_launch_batch(mode[ph], 1 != ph, cl, P.items.ptr, P.bt.ptr, P.nb, P.threads, P.lds, name[ph],
					  st);
		}
}

// the partial images of a plan's grouped normal operator: (pointer, groups)
std::pair<const float2*, int> normal_group_partials(const Nufft& p, float2* dst)
{
	const int G = p.C / merge_group(p);
	return (G > 1) ? std::make_pair((const float2*)p.part.ptr, G) : std::make_pair((const float2*)dst, 1);
}

// ---------------------------------------------------------------------------
// PSF (noncart/nufft.c:727-776 compute_psf2, :535-586 compute_psf_int)
// ---------------------------------------------------------------------------

// fftuc over the 2x grid: first pass loads x fftmod; the last pass stores
// x fftmod x 1/sqrt(N2) into the decomposed layout psf[s][n] (md_decompose,
// num/shuffle.c:84-130)
struct LdFm2 {
	VolAxis g;
	SepTables T2;
	const float2* src;
	bool fm;

	__device__ float2 operator()(long t, int k) const
	{
		uint32_t i, o, v;
		g.split(t, i, o, v);
		float2 x = src[g.offset_iov(i, o, v, k)];

		if (fm) {
			int px[3];
			g.coords(i, o, k, px);
			x = cmul(x, fm_val(T2, px));
		}

		return x;
	}
};

struct StDecomp {
	VolAxis g;
	SepTables T2;
	float2* dst;      // 2x grid (intermediate passes) or decomposed psf (last)
	bool last;
	bool fm_first;    // single-axis case: the load already applied the first fftmod
	float scale;
	int n1[3];        // sub-grid dims
	long N1;
	long vstride = 0; // output stride of the volumes (K x K basis PSFs)

	__device__ void store(const float2* lds, const FftLaunch& L, long t0) const
	{
		store_each(lds, L, t0, [&](long t, int k, float2 x) {
			uint32_t i, o, v;
			g.split(t, i, o, v);

			if (!last) {
				dst[g.offset_iov(i, o, v, k)] = x;
				return;
			}

			int px[3];
			g.coords(i, o, k, px);
			x = cmul(x, fm_val(T2, px));
			x = cscale(x, scale);

			int s = 0;
			int q[3];

			for (int d = 0; d < 3; d++) {
				if (T2.bitpos[d] >= 0) {
					s |= (px[d] & 1) << T2.bitpos[d];
					q[d] = px[d] >> 1;
				} else {
					q[d] = px[d];
				}
			}

			dst[(long)v * vstride + (long)s * N1 + q[0] + (long)n1[0] * (q[1] + (long)n1[1] * q[2])] = x;
		});
	}
};

void Nufft::compute_psf_from_traj(const float* traj, const float2* weights_host, bool periodic_psf)
{
	int n2[3];

	for (int d = 0; d < 3; d++)
		n2[d] = (1 == n[d]) ? 1 : 2 * n[d];

	std::vector<float> traj2(3 * M);

	for (long i = 0; i < 3 * M; i++)
		traj2[i] = traj[i] * 2.f;

	std::vector<float2> sqw;

	if (nullptr != weights_host) {

		sqw.resize(M);

		for (long m = 0; m < M; m++) {
			float2 w = weights_host[m];
			sqw[m] = make_float2(w.x * w.x + w.y * w.y, w.y * w.x - w.x * w.y);
		}
	}

	// with a basis, J = K^2 channels whose k-space is conj(B_k) B_k' in
	// place of the ones (compute_psf_int, noncart/nufft.c:535-586)
	const int J = (nbasis > 0) ? nbasis * nbasis : 1;
	BAM_CHECK(0 == nbasis || bMf * bT == M, "psf: basis frames (%d x %ld) do not match the samples (%ld)", bT, bMf,
		  M);

	Nufft p2;
	p2.stream = stream;
	p2.tune = false;  // one adjoint only
	p2.create(n2, J, M, traj2.data(), sqw.empty() ? nullptr : sqw.data(), false, periodic_psf, width, os, false);

	long N2 = p2.N;
	DevBuf<float2> ones(std::max<long>((long)J * M, 1));
	DevBuf<float2> psft((size_t)J * N2);

	if (nbasis > 0)
		basis_psf_vals(ones.ptr, bas.ptr, nbasis, bT, bMf, stream);
	else
		fill(ones.ptr, M, make_float2(1.f, 0.f), stream);

	p2.adjoint(psft.ptr, ones.ptr, nullptr);

	psf.alloc((size_t)J * S * N);

	const float scale = 1.f / sqrtf((float)N2);
	int last = p2.act[p2.nact - 1];

	for (int j = 0; j < p2.nact; j++) {

		int a = p2.act[j];
		VolAxis va = VolAxis::make(n2, a, J);
		FftLaunchCfg cfg = fft_config(p2.axis[j], va.transforms(), va.contig(), 1, -1.f);
		cfg.name = "fft_psf";
		LdFm2 ld{ va, p2.tabs, psft.ptr, 0 == j };
		StDecomp st{ va, p2.tabs, (a == last) ? psf.ptr : psft.ptr, a == last, false, scale,
			     { n[0], n[1], n[2] }, N, (long)S * N };
		launch_fft_axis(cfg, stream, ld, st);
	}

	apply_real_psf();
	BAM_HIP(hipStreamSynchronize(stream));
	has_psf = true;
}

__global__ void k_real_part(float2* p, long n)
{
	for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
		p[i].y = 0.f;
}

void Nufft::apply_real_psf()
{
	if (!real_psf)
		return;

	const long n = (long)psf.n;
	const unsigned blocks = (unsigned)std::min<long>((n + 255) / 256, 4096);
	hipLaunchKernelGGL(k_real_part, dim3(blocks), dim3(256), 0, stream, psf.ptr, n);
	BAM_HIP(hipGetLastError());
}

}  // namespace bam
