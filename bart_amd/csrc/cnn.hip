// cnn.hip -- 3x3 convolutions of the CG warm-start network on the matrix
// cores (gfx950): BF16 operands, FP32 accumulation.
//
// No counterpart in BART: the network that supplies a CG initial guess (the
// x0 of pics -W, iter/itop.c:54-66) is new.  Layout: activations
// [B][C][H][W] float, weights [Cout][Cin][3][3] float (k = ci 9 + 3 u + v),
// zero padding, cross-correlation:
//   y[b][co][i][j] = bias[co] + sum_{ci,u,v} w[co][ci][u][v] x[b][ci][i+u-1][j+v-1]
// Every layer is a GEMM of M = output channels, N = pixels, K = Cin 9 taps
// (forward), or M = output channels, N = Cin 9 taps, K = pixels (weight
// gradient), on v_mfma_f32_16x16x32_bf16: lane l supplies A[l % 16][8 (l / 16)
// + t] and B[8 (l / 16) + t][l % 16], t < 8; accumulator register r of lane
// l holds D[4 (l / 16) + r][l % 16].  Operands are rounded to bfloat16
// (nearest, ties to even) when they are staged into LDS.
#include "cnn.hpp"

#include <algorithm>
#include <cmath>
#include <mutex>
#include <random>
#include <vector>

namespace bam {

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int CV_MAXC = 64;     // channels (in and out) per layer at most
constexpr int CV_THREADS = 512; // 8 waves
constexpr int CV_STRIP = 256;   // forward: pixels (row segment) per work-group at most
constexpr int CV_MAXROWS = 16;  // image rows per work-group at most
constexpr int CV_WG_MAXW = 256;

// two floats rounded to bfloat16 (nearest, ties to even), the first in the
// low half
__device__ inline unsigned bf_pack(float a, float b)
{
	const f32x2 v = { a, b };
	return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
}

// image rows per work-group: nwg work-groups where there are rows enough (each
// one reads two rows of halo), down to one row
static int conv_rows(long total_rows, int nwg)
{
	return (int)std::min<long>(CV_MAXROWS, std::max<long>(1, (total_rows + nwg - 1) / nwg));
}

// ---------------------------------------------------------------------------
// Forward.  Bound by HBM: 48 channels of 256^2 are 2 x 100 MB per batch of 8
// against 22 GFLOP.  A work-group takes a strip of CV_STRIP pixels and walks
// down its image rows, so that a row is read once (and two halo rows per
// work-group) and stays in LDS, channel-fastest, for the three output rows
// that need it; the next row's loads are in flight while the matrix cores
// work on the present one.  K is ordered (tap, channel) with the channels
// padded to 8 G, in steps of 32 (four groups of 8 channels, each of one
// tap): the B fragment of a lane is one 16-byte LDS read at its pixel and
// tap (pixel pitch 4 x odd dwords: no bank conflicts), and the weights of
// all steps stay in registers (A fragments, k_conv_wprep's order).  Waves
// share the 16-pixel tiles of the row; with many channels also the output
// channel tiles (TPW per wave, ncog groups: three tiles of 48 channels per
// wave spill 120 registers, 124 us; two groups 81 us).  48 -> 48 channels,
// batch 8 of 256^2: 187 -> 81 us (2.5 TB/s) against 64-pixel, 4-row blocks
// that staged 2-byte elements.
// ---------------------------------------------------------------------------

__host__ __device__ constexpr int conv_steps(int G) { return (9 * G + 3) / 4; }
__host__ __device__ constexpr int conv_pitch(int G) { return 8 * (G | 1); }

// A fragments wb[tile][step][lane][8]: w[co = 16 tile + lane % 16][k = 32 step
// + 8 (lane / 16) + i], zero for padded channels and taps.  flip: the
// weights of the transposed convolution (the data gradient), w'[o][i][t] =
// w[i][o][8 - t].
__global__ void k_conv_wprep(const float* __restrict__ w, int Cin, int Cout, int G, int ntiles, int flip,
			     unsigned short* __restrict__ wb)
{
	const int steps = conv_steps(G);
	const int n = ntiles * steps * 512;

	for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < n; e += gridDim.x * blockDim.x) {
		const int lane = (e >> 3) & 63;
		const int ts = e >> 9;
		const int tile = ts / steps;
		const int k8 = 4 * (ts - tile * steps) + (lane >> 4);
		const int t = k8 / G;
		const int ci = (k8 - t * G) * 8 + (e & 7);
		const int co = 16 * tile + (lane & 15);
		float v = 0.f;
		if (co < Cout && ci < Cin && t < 9)
			v = flip ? w[(ci * Cout + co) * 9 + (8 - t)] : w[(co * Cin + ci) * 9 + t];
		wb[e] = (unsigned short)(bf_pack(v, 0.f) & 0xFFFFu);
	}
}

template <int G, int TPW>
__global__ __launch_bounds__(CV_THREADS) void k_conv3x3_fwd(const float* __restrict__ x, int Cin, int H, int W,
							    const unsigned short* __restrict__ wb,
							    const float* __restrict__ bias,
							    const float* __restrict__ res, int Cout, int relu,
							    float* __restrict__ y, int strip, int rows, int ncog)
{
	constexpr int STEPS = conv_steps(G);
	constexpr int PITCH = conv_pitch(G);
	constexpr int ROWSZ = (CV_STRIP + 2) * PITCH;
	constexpr int NT = (G * CV_STRIP + CV_THREADS - 1) / CV_THREADS;
	extern __shared__ __align__(16) unsigned char cv_smem[];
	unsigned short* xl = (unsigned short*)cv_smem;  // [3][CV_STRIP + 2][PITCH]

	const int x0 = blockIdx.x * strip;
	const int y0 = blockIdx.y * rows;
	const int b = blockIdx.z;
	const int nrow = min(rows, H - y0);
	const long HW = (long)H * W;
	const float* xb = x + (long)b * Cin * HW;

	const int lane = threadIdx.x & 63;
	const int wv = threadIdx.x >> 6;
	const int l16 = lane & 15;
	const int kg = lane >> 4;
	const int cog = wv % ncog;
	const int pg = wv / ncog;
	const int npg = 8 / ncog;

	bf16x8 A[TPW][STEPS];

#pragma unroll
	for (int q = 0; q < TPW; q++)
#pragma unroll
		for (int s = 0; s < STEPS; s++)
			A[q][s] = *(const bf16x8*)(wb + (((long)(cog * TPW + q) * STEPS + s) * 64 + lane) * 8);

	// one image row in registers: 8 channels of a pixel per task, NT tasks
	// of the strip and one of the two halo pixels (the first 2 G threads)
	float v[NT + 1][8];

	// (a strip's right halo pixel included; it is the extra task's where the
	// strip takes all of CV_STRIP)
	const int xe = min(W, x0 + strip + 1);

	auto load8 = [&](float (&d)[8], int g, int gy, int gx) {
		const bool ok = gy >= 0 && gy < H && gx >= 0 && gx < xe;
		const float* p = xb + (long)(8 * g) * HW + (long)gy * W;
#pragma unroll
		for (int i = 0; i < 8; i++)
			d[i] = (ok && 8 * g + i < Cin) ? (p + i * HW)[gx] : 0.f;
	};

	// the strip's channel groups are wave-uniform (scalar row addresses)
	const int g0 = __builtin_amdgcn_readfirstlane(threadIdx.x / CV_STRIP);

	auto load_row = [&](int gy) {
#pragma unroll
		for (int i = 0; i < NT; i++)
			load8(v[i], g0 + i * (CV_THREADS / CV_STRIP), gy, x0 + (int)threadIdx.x % CV_STRIP);
		if (threadIdx.x < 2 * G)
			load8(v[NT], threadIdx.x >> 1, gy, (threadIdx.x & 1) ? x0 + CV_STRIP : x0 - 1);
	};

	auto put8 = [&](const float (&d)[8], unsigned short* p) {
		*(uint4*)p = make_uint4(bf_pack(d[0], d[1]), bf_pack(d[2], d[3]), bf_pack(d[4], d[5]),
					bf_pack(d[6], d[7]));
	};

	auto store_row = [&](int slot) {
		unsigned short* r = xl + slot * ROWSZ;
#pragma unroll
		for (int i = 0; i < NT; i++) {
			const int e = threadIdx.x + i * CV_THREADS;
			if (0 == (G * CV_STRIP) % CV_THREADS || e < G * CV_STRIP)
				put8(v[i], r + (1 + e % CV_STRIP) * PITCH + 8 * (e / CV_STRIP));
		}
		if (threadIdx.x < 2 * G)
			put8(v[NT], r + ((threadIdx.x & 1) ? CV_STRIP + 1 : 0) * PITCH + 8 * (threadIdx.x >> 1));
	};

	load_row(y0 - 1);
	store_row(0);
	load_row(y0);
	store_row(1);
	load_row(y0 + 1);

	const int ntile = (min(strip, W - x0) + 15) / 16;

	for (int r = 0; r < nrow; r++) {

		// image row y0 + r + 1; rows y0 + r - 1 + u are in slots (r + u) % 3
		store_row((r + 2) % 3);
		lds_barrier();

		if (r + 1 < nrow)
			load_row(y0 + r + 2);

		// LDS offsets of this lane's 8 channels of every step, pixel 0
		int off[STEPS];
#pragma unroll
		for (int s = 0; s < STEPS; s++) {
			const int k8 = min(4 * s + kg, 9 * G - 1);
			const int t = k8 / G;
			const int u = t / 3;
			off[s] = ((r + u) % 3) * ROWSZ + (l16 + t - 3 * u) * PITCH + (k8 - t * G) * 8;
		}

		for (int pt = pg; pt < ntile; pt += npg) {

			f32x4 acc[TPW];
#pragma unroll
			for (int q = 0; q < TPW; q++)
				acc[q] = f32x4{ 0.f, 0.f, 0.f, 0.f };

			const unsigned short* xp = xl + pt * 16 * PITCH;

#pragma unroll
			for (int s = 0; s < STEPS; s++) {
				uint4 raw = *(const uint4*)(xp + off[s]);
				// the last step's groups beyond the nine taps: zero
				if (STEPS * 4 > 9 * G && STEPS - 1 == s && 4 * s + kg >= 9 * G)
					raw = make_uint4(0u, 0u, 0u, 0u);
				const bf16x8 bv = __builtin_bit_cast(bf16x8, raw);
#pragma unroll
				for (int q = 0; q < TPW; q++)
					acc[q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[q][s], bv, acc[q], 0, 0, 0);
			}

			const int gx = x0 + pt * 16 + l16;

			if (gx < W) {

				const long at0 = ((long)b * Cout + 16 * (cog * TPW) + 4 * kg) * HW + (long)(y0 + r) * W + gx;

#pragma unroll
				for (int q = 0; q < TPW; q++)
#pragma unroll
					for (int i = 0; i < 4; i++) {
						const int co = 16 * (cog * TPW + q) + 4 * kg + i;
						if (co < Cout) {
							float o = acc[q][i] + ((nullptr != bias) ? bias[co] : 0.f);
							if (relu)
								o = fmaxf(o, 0.f);
							const long at = at0 + (16 * q + i) * HW;
							if (nullptr != res)
								o += res[at];
							y[at] = o;
						}
					}
			}
		}

		lds_barrier();  // the oldest slot is rewritten next
	}
}

// ---------------------------------------------------------------------------
// Weight gradient.  Bound by HBM (x and dy once).  A work-group walks down
// its image rows: the input rows y - 1, y, y + 1 and the output-gradient row
// y are in LDS pixel-fastest, so that a lane's 8 consecutive pixels of one
// channel (K = pixels) are one 16-byte read; the three horizontal taps of
// an input row come from that read and the two neighbouring pixels by
// funnel shifts in registers.  Wave (it, ks) owns input-channel tile it and
// every output-channel tile and tap (9 NCO accumulator tiles), for the
// pixel chunks ks, ks + KS, ...; the KS parts are summed through LDS in
// order, and each work-group writes one partial gradient [9][16 NCO][16 NCI]
// (k_conv_wgrad_sum adds them in order).  The bias gradient's sums of the
// unrounded dy are taken while its rows are staged.  48 x 48 channels, batch
// 8 of 256^2: 600 + 508 (bias) + 72 (sum) -> 52 + 7 us (3.8 TB/s) against
// 2-byte LDS reads of the input patch, one work-group per bias channel and a
// thread per entry of the sum.
// ---------------------------------------------------------------------------

__host__ __device__ constexpr int wg_pitch(int n) { return ((n + 7) / 8 | 1) * 8; }
__host__ __device__ constexpr int wg_pitch_x(int W) { return wg_pitch(8 + (W + 31) / 32 * 32 + 8); }
__host__ __device__ constexpr int wg_pitch_dy(int W) { return wg_pitch((W + 31) / 32 * 32); }

template <int NCO, int NCI>
__global__ __launch_bounds__(CV_THREADS) void k_conv3x3_wgrad(const float* __restrict__ x,
							      const float* __restrict__ dy, int Cin, int Cout, int H,
							      int W, int rows, int aligned, float* __restrict__ part,
							      float* __restrict__ bpart)
{
	constexpr int NW = CV_THREADS / 64;
	constexpr int KS = NW / NCI;
	constexpr int XI = 2 * NCI;  // float4 of x (of dy) per thread and row at most
	constexpr int DI = 2 * NCO;
	extern __shared__ __align__(16) unsigned char cv_smem[];
	const int PX = wg_pitch_x(W), PD = wg_pitch_dy(W);
	unsigned short* xl = (unsigned short*)cv_smem;     // [3][16 NCI][PX], pixel p at 8 + p
	unsigned short* dl = xl + 3 * 16 * NCI * PX;       // [16 NCO][PD]

	const int nrg = (H + rows - 1) / rows;
	const int b = blockIdx.x / nrg;
	const int y0 = (blockIdx.x - b * nrg) * rows;
	const int nrow = min(rows, H - y0);
	const long HW = (long)H * W;
	const float* xb = x + (long)b * Cin * HW;
	const float* db = dy + (long)b * Cout * HW;

	const int lane = threadIdx.x & 63;
	const int wv = threadIdx.x >> 6;

	// staging: LG lanes per channel row (four pixels each), 64 / LG channels
	// per wave and step
	int lgl = 1;
	while ((4 << lgl) < W)
		lgl++;
	const int cstep = NW << (6 - lgl);
	const int c0 = (wv << (6 - lgl)) + (lane >> lgl);
	const int px = 4 * (lane & ((1 << lgl) - 1));
	const bool pin = px < W;

	// zero once: padded channels, the halo pixels and the pixels beyond W
	for (int e = threadIdx.x; e < (3 * 16 * NCI * PX + 16 * NCO * PD) / 8; e += CV_THREADS)
		((uint4*)cv_smem)[e] = make_uint4(0u, 0u, 0u, 0u);

	f32x4 xv[XI], dv[DI];
	float bs[DI];
#pragma unroll
	for (int i = 0; i < DI; i++)
		bs[i] = 0.f;

	auto ld4 = [&](const float* p) {
		if (aligned)
			return *(const f32x4*)p;
		return f32x4{ p[0], p[1], p[2], p[3] };
	};

	auto load_x = [&](int gy) {
#pragma unroll
		for (int i = 0; i < XI; i++) {
			const int c = c0 + i * cstep;
			xv[i] = f32x4{ 0.f, 0.f, 0.f, 0.f };
			if (pin && c < Cin && gy >= 0 && gy < H)
				xv[i] = ld4(xb + c * HW + (long)gy * W + px);
		}
	};

	auto load_dy = [&](int gy) {
#pragma unroll
		for (int i = 0; i < DI; i++) {
			const int c = c0 + i * cstep;
			dv[i] = f32x4{ 0.f, 0.f, 0.f, 0.f };
			if (pin && c < Cout)
				dv[i] = ld4(db + c * HW + (long)gy * W + px);
		}
	};

	auto put4 = [&](const f32x4& f, unsigned short* p) {
		*(uint2*)p = make_uint2(bf_pack(f[0], f[1]), bf_pack(f[2], f[3]));
	};

	auto store_x = [&](int slot) {
#pragma unroll
		for (int i = 0; i < XI; i++) {
			const int c = c0 + i * cstep;
			if (pin && c < Cin)
				put4(xv[i], xl + (slot * 16 * NCI + c) * PX + 8 + px);
		}
	};

	auto store_dy = [&]() {
#pragma unroll
		for (int i = 0; i < DI; i++) {
			const int c = c0 + i * cstep;
			if (pin && c < Cout) {
				bs[i] += (dv[i][0] + dv[i][1]) + (dv[i][2] + dv[i][3]);
				put4(dv[i], dl + c * PD + px);
			}
		}
	};

	const int it = wv % NCI;
	const int ks = wv / NCI;
	const int l16 = lane & 15;
	const int kg = lane >> 4;

	f32x4 acc[9][NCO];
#pragma unroll
	for (int t = 0; t < 9; t++)
#pragma unroll
		for (int q = 0; q < NCO; q++)
			acc[t][q] = f32x4{ 0.f, 0.f, 0.f, 0.f };

	load_x(y0 - 1);
	__syncthreads();  // the zeroes are in
	store_x(0);
	load_x(y0);
	store_x(1);
	load_x(y0 + 1);
	load_dy(y0);

	for (int r = 0; r < nrow; r++) {

		store_x((r + 2) % 3);
		store_dy();
		lds_barrier();

		if (r + 1 < nrow) {
			load_x(y0 + r + 2);
			load_dy(y0 + r + 1);
		}

		if (ks < KS) {

			for (int p0 = 32 * ks; p0 < W; p0 += 32 * KS) {

				const int p = p0 + 8 * kg;
				// beyond the row dy is 0, and a 0 of dy must not meet the
				// row's last pixel, which may be infinite
				const unsigned pm = (p < W) ? ~0u : 0u;
				bf16x8 a[NCO];
#pragma unroll
				for (int q = 0; q < NCO; q++)
					a[q] = *(const bf16x8*)(dl + (16 * q + l16) * PD + p);

#pragma unroll
				for (int u = 0; u < 3; u++) {

					const unsigned short* xr = xl + ((((r + u) % 3) * NCI + it) * 16 + l16) * PX + 8 + p;
					const uint4 d = *(const uint4*)xr;
					const unsigned pv = *(const unsigned*)(xr - 2) & pm;
					const unsigned nx = *(const unsigned*)(xr + 8);
					// 8 pixels from p - 1 and from p + 1
					const unsigned m0 = __builtin_amdgcn_alignbyte(d.x, pv, 2);
					const unsigned m1 = __builtin_amdgcn_alignbyte(d.y, d.x, 2);
					const unsigned m2 = __builtin_amdgcn_alignbyte(d.z, d.y, 2);
					const unsigned m3 = __builtin_amdgcn_alignbyte(d.w, d.z, 2);
					const unsigned m4 = __builtin_amdgcn_alignbyte(nx, d.w, 2);
					const bf16x8 bv[3] = { __builtin_bit_cast(bf16x8, make_uint4(m0, m1, m2, m3)),
							       __builtin_bit_cast(bf16x8, d),
							       __builtin_bit_cast(bf16x8, make_uint4(m1, m2, m3, m4)) };
#pragma unroll
					for (int h = 0; h < 3; h++)
#pragma unroll
						for (int q = 0; q < NCO; q++)
							acc[3 * u + h][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
								a[q], bv[h], acc[3 * u + h][q], 0, 0, 0);
				}
			}
		}

		lds_barrier();
	}

	// sum of the KS parts in order, through LDS (the rows are done with)
	f32x4* sh = (f32x4*)cv_smem;  // [NCI][9 NCO][64]

	for (int k = 1; k < KS; k++) {

		if (k == ks) {
#pragma unroll
			for (int t = 0; t < 9; t++)
#pragma unroll
				for (int q = 0; q < NCO; q++)
					sh[((it * 9 + t) * NCO + q) * 64 + lane] = acc[t][q];
		}

		lds_barrier();

		if (0 == ks) {
#pragma unroll
			for (int t = 0; t < 9; t++)
#pragma unroll
				for (int q = 0; q < NCO; q++)
					acc[t][q] += sh[((it * 9 + t) * NCO + q) * 64 + lane];
		}

		lds_barrier();
	}

	if (0 == ks) {

		float* pp = part + (long)blockIdx.x * 9 * 16 * NCO * 16 * NCI;

#pragma unroll
		for (int t = 0; t < 9; t++)
#pragma unroll
			for (int q = 0; q < NCO; q++)
#pragma unroll
				for (int i = 0; i < 4; i++)
					pp[((t * 16 * NCO) + 16 * q + 4 * kg + i) * 16 * NCI + 16 * it + l16] = acc[t][q][i];
	}

	if (nullptr != bpart) {
#pragma unroll
		for (int i = 0; i < DI; i++) {
			float s = bs[i];
			for (int o = (1 << lgl) >> 1; o > 0; o >>= 1)
				s += __shfl_xor(s, o, 64);
			const int c = c0 + i * cstep;
			if (0 == px && c < Cout)
				bpart[(long)blockIdx.x * CV_MAXC + c] = s;
		}
	}
}

// Sums of the partials: dw[co][ci][t] (work-groups below nblk, 64 entries of a
// partial each) and db[co] (the work-group after them): four threads per
// entry take every fourth partial in order, their sums are added in order.
__global__ __launch_bounds__(256) void k_conv_wgrad_sum(const float* __restrict__ part, const float* __restrict__ bpart,
							int nparts, int Cin, int Cout, int PO, int PI, int nblk,
							float* __restrict__ dw, float* __restrict__ db)
{
	__shared__ float sh[256];
	const int j = threadIdx.x & 63;
	const int g = threadIdx.x >> 6;
	const bool wsum = (int)blockIdx.x < nblk;
	const long stride = wsum ? 9l * PO * PI : CV_MAXC;
	const int e = wsum ? (int)blockIdx.x * 64 + j : j;
	const float* p = (wsum ? part : bpart) + e;
	float s = 0.f;

	if (wsum || e < Cout) {
#pragma unroll 8
		for (int k = g; k < nparts; k += 4)
			s += p[k * stride];
	}

	sh[threadIdx.x] = s;
	__syncthreads();

	if (0 != g)
		return;

	s = ((sh[j] + sh[64 + j]) + sh[128 + j]) + sh[192 + j];

	if (wsum) {
		const int t = e / (PO * PI);
		const int r = e - t * (PO * PI);
		const int co = r / PI;
		const int ci = r - co * PI;
		if (co < Cout && ci < Cin)
			dw[(co * Cin + ci) * 9 + t] = s;
	} else if (e < Cout) {
		db[e] = s;
	}
}

// work buffers: the weights as matrix-core fragments, the partial gradients
struct CnnWork {
	std::mutex mtx;
	DevBuf<float> part;
	DevBuf<unsigned short> wb;
};

static CnnWork& cnn_work()
{
	static CnnWork w;
	return w;
}

static void check_shape(int B, int Cin, int Cout, int H, int W)
{
	BAM_CHECK(B >= 1 && H >= 1 && W >= 1, "conv3x3: bad shape");
	BAM_CHECK(Cin >= 1 && Cin <= CV_MAXC && Cout >= 1 && Cout <= CV_MAXC,
		  "conv3x3: 1 to %d channels in and out (got %d, %d)", CV_MAXC, Cin, Cout);
}

template <int G>
static void fwd_launch_g(dim3 grid, int tpw, const float* x, int Cin, int H, int W, const unsigned short* wb,
			 const float* bias, const float* res, int Cout, bool relu, float* y, int strip, int rows,
			 int ncog, hipStream_t st)
{
	const size_t lds = sizeof(unsigned short) * 3 * (CV_STRIP + 2) * conv_pitch(G);

#define BAM_CONV(T)                                                                                               \
	hipLaunchKernelGGL((k_conv3x3_fwd<G, T>), grid, dim3(CV_THREADS), lds, st, x, Cin, H, W, wb, bias, res, Cout, \
			   relu ? 1 : 0, y, strip, rows, ncog)
	if (1 == tpw)
		BAM_CONV(1);
	else if (2 == tpw)
		BAM_CONV(2);
	else if constexpr (G <= 4)
		BAM_CONV(3);
	else
		fail("conv3x3: no kernel for %d channel tiles", tpw);
#undef BAM_CONV
}

// the weights as bfloat16 fragments (prepared per call), then the layer;
// flip: w holds the forward weights of the transposed convolution
static void fwd_launch(const float* x, int B, int Cin, int H, int W, const float* w, const float* bias,
		       const float* res, int Cout, bool relu, float* y, hipStream_t st, DevBuf<unsigned short>& wb,
		       bool flip)
{
	check_shape(B, Cin, Cout, H, W);
	BAM_CHECK(H <= 65535 && B <= 65535, "conv3x3: too many rows or images");

	// a wave keeps the weights of its output-channel tiles in registers (4
	// per tile and step of 32): three tiles up to 32 input channels, two above
	// (208 to 244 registers in all at 48 to 64 channels, none spilled; three
	// tiles of 48 channels spill 120)
	const int G = (Cin + 7) / 8;
	const int nco = (Cout + 15) / 16;
	const int ncog = (4 == nco || (3 == nco && G > 4)) ? 2 : 1;
	const int tpw = (nco + ncog - 1) / ncog;
	const int ntiles = ncog * tpw;
	const long nw = (long)ntiles * conv_steps(G) * 512;
	if ((long)wb.n < nw)
		wb.alloc(nw);
	hipLaunchKernelGGL(k_conv_wprep, dim3((unsigned)((nw + 255) / 256)), dim3(256), 0, st, w, Cin, Cout, G, ntiles,
			   flip ? 1 : 0, wb.ptr);
	// Strips of equal width (320 as 256 + 64: 286 us for 48 channels, batch 8 of
	// 320^2, as 160 + 160: 225).  A work-group per compute unit, or two where the
	// weights of a lane and the rows in LDS are few (2 -> 48 channels, batch 8 of
	// 320^2: 88 -> 59 us; four: 61), in halves of a strip where these would walk
	// down less than two rows (one image of 320^2: 17.9 -> 14.4; 512^2, 16
	// channels, with two rows: 14.8 and 15.2).
	int nx = (W + CV_STRIP - 1) / CV_STRIP;
	const int nwg = device_cus() * ((G <= 2) ? 2 : 1);
	if (G <= 2 && (long)nx * H * B < 2l * nwg)
		nx = (W + CV_STRIP / 2 - 1) / (CV_STRIP / 2);
	const int strip = ((W + nx - 1) / nx + 15) / 16 * 16;
	const int rows = conv_rows((long)nx * H * B, nwg);
	dim3 grid(nx, (H + rows - 1) / rows, B);

#define BAM_CONV_G(NG) \
	case NG: fwd_launch_g<NG>(grid, tpw, x, Cin, H, W, wb.ptr, bias, res, Cout, relu, y, strip, rows, ncog, st); break
	switch (G) {
		BAM_CONV_G(1);
		BAM_CONV_G(2);
		BAM_CONV_G(3);
		BAM_CONV_G(4);
		BAM_CONV_G(5);
		BAM_CONV_G(6);
		BAM_CONV_G(7);
		BAM_CONV_G(8);
	default:
		fail("conv3x3: no kernel for %d channels", Cin);
	}
#undef BAM_CONV_G

	BAM_HIP(hipGetLastError());
}

void conv3x3_fwd(const float* x, int B, int Cin, int H, int W, const float* w, const float* bias, const float* res,
		 int Cout, bool relu, float* y, hipStream_t st)
{
	// the prepared weights are rewritten by the next call: calls are ordered
	// on the one stream every layer call uses
	CnnWork& cw = cnn_work();
	std::lock_guard<std::mutex> lock(cw.mtx);
	fwd_launch(x, B, Cin, H, W, w, bias, res, Cout, relu, y, st, cw.wb, false);
}

void conv3x3_bwd_data(const float* dy, int B, int Cout, int H, int W, const float* w, int Cin, float* dx,
		      hipStream_t st)
{
	check_shape(B, Cin, Cout, H, W);
	CnnWork& cw = cnn_work();
	std::lock_guard<std::mutex> lock(cw.mtx);
	fwd_launch(dy, B, Cout, H, W, w, nullptr, nullptr, Cin, false, dx, st, cw.wb, true);
	BAM_HIP(hipStreamSynchronize(st));
}

template <int NCO>
static void wgrad_launch(int nci, int nparts, const float* x, const float* dy, int Cin, int Cout, int H, int W,
			 int rows, int aligned, float* part, float* bpart, hipStream_t st)
{
	// the rows, later the accumulator tiles of the in-order sum
	const size_t lds = std::max(sizeof(unsigned short) * (3 * 16 * (size_t)nci * wg_pitch_x(W) +
							      16 * (size_t)NCO * wg_pitch_dy(W)),
				    sizeof(f32x4) * 64 * 9 * (size_t)nci * NCO);

#define BAM_WGRAD(NI)                                                                                              \
	case NI: hipLaunchKernelGGL((k_conv3x3_wgrad<NCO, NI>), dim3(nparts), dim3(CV_THREADS), lds, st, x, dy, Cin, Cout, \
				    H, W, rows, aligned, part, bpart); break
	switch (nci) {
		BAM_WGRAD(1);
		BAM_WGRAD(2);
		BAM_WGRAD(3);
		BAM_WGRAD(4);
	default:
		fail("conv3x3 weight gradient: no kernel for %d channels", Cin);
	}
#undef BAM_WGRAD
}

void conv3x3_bwd_weights(const float* x, const float* dy, int B, int Cin, int Cout, int H, int W, float* dw,
			 float* db, hipStream_t st)
{
	check_shape(B, Cin, Cout, H, W);
	BAM_CHECK(W <= CV_WG_MAXW && 0 == W % 8, "conv3x3 weight gradient: width a multiple of 8, at most %d",
		  CV_WG_MAXW);
	// the entry point's range (57 to 64 channels in with more than 32 out stay
	// outside of it), not a limit of the kernel
	BAM_CHECK(((Cout + 31) / 32) * ((Cin * 9 + 31) / 32) <= 32, "conv3x3 weight gradient: too many tiles");
	CnnWork& cw = cnn_work();
	std::lock_guard<std::mutex> lock(cw.mtx);
	const int nco = (Cout + 15) / 16, nci = (Cin + 15) / 16;
	const int PO = 16 * nco, PI = 16 * nci;
	const int rows = conv_rows((long)B * H, device_cus());
	const int nparts = B * ((H + rows - 1) / rows);
	const long np = (long)nparts * (9 * PO * PI + CV_MAXC);
	if ((long)cw.part.n < np)
		cw.part.alloc(np);
	float* bpart = (nullptr != db) ? cw.part.ptr + (long)nparts * 9 * PO * PI : nullptr;
	const int aligned = (0 == ((uintptr_t)x | (uintptr_t)dy) % 16) ? 1 : 0;

	switch (nco) {
	case 1: wgrad_launch<1>(nci, nparts, x, dy, Cin, Cout, H, W, rows, aligned, cw.part.ptr, bpart, st); break;
	case 2: wgrad_launch<2>(nci, nparts, x, dy, Cin, Cout, H, W, rows, aligned, cw.part.ptr, bpart, st); break;
	case 3: wgrad_launch<3>(nci, nparts, x, dy, Cin, Cout, H, W, rows, aligned, cw.part.ptr, bpart, st); break;
	default: wgrad_launch<4>(nci, nparts, x, dy, Cin, Cout, H, W, rows, aligned, cw.part.ptr, bpart, st); break;
	}

	const int nblk = 9 * PO * PI / 64;
	hipLaunchKernelGGL(k_conv_wgrad_sum, dim3(nblk + (nullptr != db ? 1 : 0)), dim3(256), 0, st, cw.part.ptr, bpart,
			   nparts, Cin, Cout, PO, PI, nblk, dw, db);
	BAM_HIP(hipGetLastError());
	BAM_HIP(hipStreamSynchronize(st));
}

}  // namespace bam

// ---------------------------------------------------------------------------
// The warm-start network: 6 convolution layers 2 -> C -> C -> C -> C -> C -> 2
// with ReLU after the first five and the input added to the output
// (residual), trained on mean squared error with Adam.
// ---------------------------------------------------------------------------

namespace bam {

// g[i] = 0 where the layer's output a[i] was clipped by the ReLU
__global__ void k_relu_bwd(float* __restrict__ g, const float* __restrict__ a, long n)
{
	for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
		if (!(a[i] > 0.f))
			g[i] = 0.f;
}

// d = 2 (out - t) / n; per-work-group partial sums of (out - t)^2
__global__ __launch_bounds__(256) void k_mse(const float* __restrict__ out, const float* __restrict__ t, long n,
					      float* __restrict__ d, double* __restrict__ part)
{
	__shared__ double sh[256];
	double s = 0.;

	for (long i = (long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long)gridDim.x * 256) {
		const float e = out[i] - t[i];
		d[i] = 2.f * e / (float)n;
		s += (double)e * (double)e;
	}

	sh[threadIdx.x] = s;
	__syncthreads();

	for (int h = 128; h > 0; h >>= 1) {
		if (threadIdx.x < h)
			sh[threadIdx.x] += sh[threadIdx.x + h];
		__syncthreads();
	}

	if (0 == threadIdx.x)
		part[blockIdx.x] = sh[0];
}

// Adam (Kingma & Ba, ICLR 2015) with bias correction
__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
		       float* __restrict__ v, long n, float lr, float b1, float b2, float eps, float c1, float c2)
{
	for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
		const float gi = g[i];
		const float mi = b1 * m[i] + (1.f - b1) * gi;
		const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
		m[i] = mi;
		v[i] = vi;
		p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
	}
}

constexpr int WN_LAYERS = 6;
constexpr int WN_MSE_BLOCKS = 256;

WarmNet::WarmNet(int channels, unsigned long seed)
{
	BAM_CHECK(channels >= 1 && channels <= CV_MAXC, "warm-start network: 1 to %d channels", CV_MAXC);
	ch[0] = 2;
	for (int l = 1; l < WN_LAYERS; l++)
		ch[l] = channels;
	ch[WN_LAYERS] = 2;

	long n = 0;
	for (int l = 0; l < WN_LAYERS; l++) {
		woff[l] = n;
		n += (long)ch[l + 1] * ch[l] * 9;
		boff[l] = n;
		n += ch[l + 1];
	}
	nparams = n;

	// He-normal weights (std sqrt(2 / fan-in)); the last layer x 0.1 so that
	// the untrained network is close to the identity; zero biases
	std::vector<float> h(n, 0.f);
	std::mt19937_64 rng(seed);
	std::normal_distribution<double> nd(0., 1.);
	for (int l = 0; l < WN_LAYERS; l++) {
		const double sd = sqrt(2. / (9. * ch[l])) * ((WN_LAYERS - 1 == l) ? 0.1 : 1.);
		for (long i = 0; i < (long)ch[l + 1] * ch[l] * 9; i++)
			h[woff[l] + i] = (float)(sd * nd(rng));
	}

	params.alloc(n);
	grads.alloc(n);
	m.alloc(n);
	v.alloc(n);
	BAM_HIP(hipMemcpy(params.ptr, h.data(), sizeof(float) * n, hipMemcpyHostToDevice));
	BAM_HIP(hipMemset(m.ptr, 0, sizeof(float) * n));
	BAM_HIP(hipMemset(v.ptr, 0, sizeof(float) * n));
	lpart.alloc(WN_MSE_BLOCKS);
}

void WarmNet::ensure(int B, int H, int W)
{
	const long hid = (long)B * ch[1] * H * W;
	if ((long)act.n < (WN_LAYERS - 1) * hid)
		act.alloc((WN_LAYERS - 1) * hid);
	if ((long)g0.n < hid) {
		g0.alloc(hid);
		g1.alloc(hid);
	}
	const long io = (long)B * 2 * H * W;
	if ((long)out.n < io)
		out.alloc(io);
}

// a_l: input of layer l (a_0 = x)
const float* WarmNet::a(int l, const float* x, int B, int H, int W) const
{
	return (0 == l) ? x : act.ptr + (long)(l - 1) * B * ch[1] * H * W;
}

void WarmNet::forward(const float* x, int B, int H, int W, float* y, hipStream_t st)
{
	ensure(B, H, W);

	for (int l = 0; l < WN_LAYERS; l++) {
		const bool last = WN_LAYERS - 1 == l;
		float* dst = last ? y : (float*)a(l + 1, x, B, H, W);
		conv3x3_fwd(a(l, x, B, H, W), B, ch[l], H, W, params.ptr + woff[l], params.ptr + boff[l],
			    last ? x : nullptr, ch[l + 1], !last, dst, st);
	}
}

// Backpropagation of the output gradient in g0 through the layer outputs of
// the last forward (input x), then one Adam step.
void WarmNet::backward_update(const float* x, int B, int H, int W, float lr, hipStream_t st)
{
	float* g = g0.ptr;      // gradient at the output of layer l
	float* gn = g1.ptr;

	for (int l = WN_LAYERS - 1; l >= 0; l--) {

		const float* al = a(l, x, B, H, W);
		conv3x3_bwd_weights(al, g, B, ch[l], ch[l + 1], H, W, grads.ptr + woff[l], grads.ptr + boff[l], st);

		if (l > 0) {
			conv3x3_bwd_data(g, B, ch[l + 1], H, W, params.ptr + woff[l], ch[l], gn, st);
			const long na = (long)B * ch[l] * H * W;
			hipLaunchKernelGGL(k_relu_bwd, dim3(1024), dim3(256), 0, st, gn, al, na);
			BAM_HIP(hipGetLastError());
			std::swap(g, gn);
		}
	}

	step++;
	const float b1 = 0.9f, b2 = 0.999f;
	const float c1 = 1.f - (float)pow(b1, step), c2 = 1.f - (float)pow(b2, step);
	hipLaunchKernelGGL(k_adam, dim3(256), dim3(256), 0, st, params.ptr, grads.ptr, m.ptr, v.ptr, nparams, lr, b1, b2,
			   1e-8f, c1, c2);
	BAM_HIP(hipGetLastError());
}

double WarmNet::train_step(const float* x, const float* t, int B, int H, int W, float lr, hipStream_t st)
{
	ensure(B, H, W);
	forward(x, B, H, W, out.ptr, st);

	const long n = (long)B * 2 * H * W;
	hipLaunchKernelGGL(k_mse, dim3(WN_MSE_BLOCKS), dim3(256), 0, st, out.ptr, t, n, g0.ptr, lpart.ptr);
	BAM_HIP(hipGetLastError());

	backward_update(x, B, H, W, lr, st);

	std::vector<double> hp(WN_MSE_BLOCKS);
	BAM_HIP(hipMemcpyAsync(hp.data(), lpart.ptr, sizeof(double) * WN_MSE_BLOCKS, hipMemcpyDeviceToHost, st));
	BAM_HIP(hipStreamSynchronize(st));
	double s = 0.;
	for (double v : hp)
		s += v;
	return s / (double)n;
}

void WarmNet::train_step_grad(const float* x, const float* dout, int B, int H, int W, float lr, hipStream_t st)
{
	ensure(B, H, W);
	const long n = (long)B * 2 * H * W;
	BAM_HIP(hipMemcpyAsync(g0.ptr, dout, sizeof(float) * n, hipMemcpyDeviceToDevice, st));
	backward_update(x, B, H, W, lr, st);
	BAM_HIP(hipStreamSynchronize(st));
}

// ---------------------------------------------------------------------------
// The network's input and the guess it gives (first CG iterate from zero,
// scale, channels)
// ---------------------------------------------------------------------------

constexpr int GS_BLOCKS = 256;
constexpr int GS_THREADS = 256;

// partial sums of the first step along a direction d for the right-hand
// side b: d^H b (re, im), d^H (A^H A d + lambda d) and max |d|^2, per block
// (FP64; d = b gives CG's first step from zero)
__global__ __launch_bounds__(GS_THREADS) void k_guess_partials(const float* __restrict__ d, const float* __restrict__ b,
							       const float* __restrict__ Ad, float lambda, long n,
							       double* __restrict__ part)
{
	__shared__ double sh[4][GS_THREADS / 64];
	double db = 0., dbi = 0., dad = 0., mx = 0.;

	for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
		const float2 dv = ((const float2*)d)[i];
		const float2 bv = ((const float2*)b)[i];
		const float2 av = ((const float2*)Ad)[i];
		const float a0 = av.x + lambda * dv.x;
		const float a1 = av.y + lambda * dv.y;
		db += (double)(dv.x * bv.x) + (double)(dv.y * bv.y);
		dbi += (double)(dv.x * bv.y) - (double)(dv.y * bv.x);
		dad += (double)(dv.x * a0) + (double)(dv.y * a1);
		mx = fmax(mx, (double)dv.x * dv.x + (double)dv.y * dv.y);
	}

	for (int off = 32; off > 0; off >>= 1) {
		db += __shfl_down(db, off, 64);
		dbi += __shfl_down(dbi, off, 64);
		dad += __shfl_down(dad, off, 64);
		mx = fmax(mx, __shfl_down(mx, off, 64));
	}

	const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;

	if (0 == lane) {
		sh[0][wid] = db;
		sh[1][wid] = dad;
		sh[2][wid] = mx;
		sh[3][wid] = dbi;
	}

	__syncthreads();

	if (0 == threadIdx.x) {
		double a = 0., c = 0., m = 0., ai = 0.;
		for (int w = 0; w < GS_THREADS / 64; w++) {
			a += sh[0][w];
			c += sh[1][w];
			m = fmax(m, sh[2][w]);
			ai += sh[3][w];
		}
		part[blockIdx.x] = a;
		part[GS_BLOCKS + blockIdx.x] = c;
		part[2 * GS_BLOCKS + blockIdx.x] = m;
		part[3 * GS_BLOCKS + blockIdx.x] = ai;
	}
}

// sc = { re alpha, s, 1 / s, im alpha }: x1 = alpha d with alpha =
// d^H b / d^H (A^H A + lambda I) d, s = max |x1| (1 when x1 = 0)
__global__ void k_guess_scalars(const double* __restrict__ part, float* __restrict__ sc)
{
	if (0 != threadIdx.x)
		return;

	double a = 0., c = 0., m = 0., ai = 0.;
	for (int i = 0; i < GS_BLOCKS; i++) {
		a += part[i];
		c += part[GS_BLOCKS + i];
		m = fmax(m, part[2 * GS_BLOCKS + i]);
		ai += part[3 * GS_BLOCKS + i];
	}

	const float rs = (float)a;
	const float rsi = (float)ai;
	const float pAp = (float)c;
	const float alpha = (0.f != pAp) ? rs / pAp : 0.f;
	const float alpha_i = (0.f != pAp) ? rsi / pAp : 0.f;
	float s = sqrtf(alpha * alpha + alpha_i * alpha_i) * (float)sqrt(m);
	if (!(s > 0.f))
		s = 1.f;
	sc[0] = alpha;
	sc[1] = s;
	sc[2] = 1.f / s;
	sc[3] = alpha_i;
}

// ch[0][i] = re(v_i) f, ch[1][i] = im(v_i) f with v = alpha d (mode 0) or
// v = img (mode 1; f = 1 / scale given)
__global__ void k_guess_pack(const float2* __restrict__ v, const float* __restrict__ sc, float f, long npix,
			     int mode, float* __restrict__ ch)
{
	for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < npix; i += (long)gridDim.x * blockDim.x) {
		float2 x = v[i];
		float g = f;
		if (0 == mode) {
			x = make_float2(sc[0] * x.x - sc[3] * x.y, sc[0] * x.y + sc[3] * x.x);
			g = sc[2];
		}
		ch[i] = x.x * g;
		ch[npix + i] = x.y * g;
	}
}

// x0 = s (ch[0] + i ch[1])
__global__ void k_guess_unpack(const float* __restrict__ ch, const float* __restrict__ sc, long npix,
			       float2* __restrict__ x0)
{
	for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < npix; i += (long)gridDim.x * blockDim.x)
		x0[i] = make_float2(sc[1] * ch[i], sc[1] * ch[npix + i]);
}

void guess_scalars(const float2* d, const float2* b, const float2* Ad, float lambda, long npix, double* part,
		   float* sc, hipStream_t st)
{
	hipLaunchKernelGGL(k_guess_partials, dim3(GS_BLOCKS), dim3(GS_THREADS), 0, st, (const float*)d,
			   (const float*)b, (const float*)Ad, lambda, npix, part);
	hipLaunchKernelGGL(k_guess_scalars, dim3(1), dim3(64), 0, st, part, sc);
	BAM_HIP(hipGetLastError());
}

void guess_pack(const float2* v, const float* sc, float f, long npix, bool scaled_first_iterate, float* ch,
		hipStream_t st)
{
	const unsigned blocks = (unsigned)std::min<long>((npix + 255) / 256, 2048);
	hipLaunchKernelGGL(k_guess_pack, dim3(blocks), dim3(256), 0, st, v, sc, f, npix, scaled_first_iterate ? 0 : 1,
			   ch);
	BAM_HIP(hipGetLastError());
}

void guess_unpack(const float* ch, const float* sc, long npix, float2* x0, hipStream_t st)
{
	const unsigned blocks = (unsigned)std::min<long>((npix + 255) / 256, 2048);
	hipLaunchKernelGGL(k_guess_unpack, dim3(blocks), dim3(256), 0, st, ch, sc, npix, x0);
	BAM_HIP(hipGetLastError());
}

}  // namespace bam
