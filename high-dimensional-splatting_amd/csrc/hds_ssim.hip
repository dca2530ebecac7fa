// SSIM loss kernels: forward (map + the three per-pixel partials the backward needs) and backward.
//
// Zero-padded separable 11-tap Gaussian window, sigma 1.5, C1 = 0.01^2, C2 = 0.03^2, on interleaved
// [H, W, 3] images (ssim.cu:6-113, utils/loss.py:8-9, 39-54). Both directions are one walk: a wave is a
// work-group of its own and owns a strip of 64 channel elements, one per lane, and some rows of it. It brings
// each input row and its halo into LDS (the next row's loads in flight during this one, no barrier between
// waves), blurs it horizontally, keeps the last 11 blurred rows in a ring of registers and blurs those
// vertically; the row loop is unrolled by the ring's length, so that its slots are registers. Out-of-image taps
// read zeros, which add +0 exactly where the reference skips them.
//
// Bound by VALU issue: the forward's differences of moments cancel, so its sums keep the order and the separate
// rounding of every product and sum (20 operations per tap of both blurs together); the backward is linear
// and takes fused multiply-adds. At 1920x1080: forward 107 -> 61 us, backward 150 -> 41 us against strips
// staged whole in LDS before the first row (forward) and tiles blurred by way of LDS twice (backward).
#include "hds_internal.h"
#include "hds_rasterizer.h"

namespace {

constexpr int kR = 5;                     // window radius
constexpr int kTaps = 2 * kR + 1;
constexpr int kE = 64;                    // output elements per row of a strip: a wave
constexpr int kHalo = 3 * kR;             // input elements on either side
constexpr int kEin = kE + 2 * kHalo;
constexpr float kC1 = 0.01f * 0.01f, kC2 = 0.03f * 0.03f;

// exp(-x^2 / (2 * 1.5^2)) / sum over x = -5..5, evaluated in double and rounded to float.
__device__ constexpr float kWin[kTaps] = {0x1.0d956cp-10f, 0x1.f1fe02p-8f, 0x1.26eb18p-5f, 0x1.bff0fep-4f,
										  0x1.b43c40p-3f,  0x1.106560p-2f, 0x1.b43c40p-3f, 0x1.bff0fep-4f,
										  0x1.26eb18p-5f,  0x1.f1fe02p-8f, 0x1.0d956cp-10f};

// The element `bytes` past p[offset]: a uniform pointer and a 32-bit offset per lane.
template <typename T>
__device__ inline T& at(T* p, int64_t offset, uint32_t bytes) {
	asm volatile("" : "+v"(bytes));  // widened here, where the address mode takes it as it is
	return *(T*)((const char*)(p + offset) + bytes);
}

// Keeps the compiler from moving the loads of v into a branch on what selects them.
__device__ inline void pin(float2& v) { asm volatile("" : "+v"(v.x), "+v"(v.y)); }
__device__ inline void pin(float3& v) { asm volatile("" : "+v"(v.x), "+v"(v.y), "+v"(v.z)); }

// Walks the strip of work-group blockIdx.x (strips vary fastest), `rows` rows of it. load(row offset, lane's bytes)
// gives an input element and centre(...) what an output element needs besides (row offsets are uniform); tap(weight,
// element, sums, first) adds one horizontal tap to the kQ sums, column(ring, first slot, sums) blurs the ring's
// rows vertically and out(row offset, lane's bytes, sums, centre) takes this lane's result.
template <int kQ, typename Row, typename Centre, typename Load, typename LoadCentre, typename Tap, typename Column,
		  typename Out>
__device__ inline void walk_strip(int height, int width, int rows, Load&& load, LoadCentre&& centre, Tap&& tap,
								  Column&& column, Out&& out) {
	__shared__ Row s_line[2][2 * kE];
	const int lane = threadIdx.x;
	const int64_t stride = (int64_t)width * 3;  // elements per row
	const int strips = (int)((stride + kE - 1) / kE);
	const int64_t e0 = (int64_t)(blockIdx.x % strips) * kE;
	const int y0 = blockIdx.x / strips * rows, y1 = min(y0 + rows, height);
	// This lane's elements of the row with its halo, lane and 64 + lane, counted from the strip's first one
	// inside the image. What lies outside reads the nearest element inside and becomes zero, and the lanes past
	// the image's edge repeat its last element: no load or store hangs on a branch, so a wait for the next row's
	// loads need not wait for this row's stores.
	const int64_t first = max(e0 - kHalo, (int64_t)0);
	const int last = (int)min(stride - first, (int64_t)kEin) - 1;
	const int off = lane - (int)(first - (e0 - kHalo));
	const uint32_t bytes_a = 4u * (uint32_t)min(max(off, 0), last), bytes_b = 4u * (uint32_t)min(off + kE, last);
	const bool in_a = off >= 0 && off <= last, in_b = off + kE <= last;
	const int lane_out = (int)min((int64_t)lane, stride - 1 - e0);
	const uint32_t bytes_out = 4u * (uint32_t)lane_out;
	Row next_a, next_b;
	auto fetch = [&](int y) {
		const int64_t g = min(max(y, 0), height - 1) * stride + first;
		next_a = load(g, bytes_a);
		next_b = load(g, bytes_b);
	};
	int buffer = 0;
	fetch(y0 - kR);
	// Horizontal blur of input row y, whose elements were fetched one row ahead.
	auto blur_row = [&](int y, float (&sums)[kQ]) {
		Row* const line = s_line[buffer];
		buffer ^= 1;
		const bool in = y >= 0 && y < height;
		pin(next_a);
		pin(next_b);
		line[lane] = in && in_a ? next_a : Row{};
		line[kE + lane] = in && in_b ? next_b : Row{};
		fetch(y + 1);
		__syncthreads();  // one wave: orders its own LDS accesses
#pragma unroll
		for (int k = 0; k < kTaps; k++) tap(kWin[k], line[lane_out + 3 * k], sums, k == 0);
#pragma unroll
		for (int q = 0; q < kQ; q++) asm volatile("" : "+v"(sums[q]));  // blurred here, not where the ring is read
	};
	float ring[kTaps][kQ];
#pragma unroll
	for (int r = 0; r < 2 * kR; r++) blur_row(y0 - kR + r, ring[r]);
	Centre next_centre = centre(y0 * stride + e0, bytes_out);
#pragma unroll 1
	for (int y = y0; y < y1; y += kTaps) {
#pragma unroll
		for (int j = 0; j < kTaps; j++) {
			if (y + j >= y1) break;  // uniform
			const Centre c = next_centre;
			next_centre = centre(min(y + j + 1, height - 1) * stride + e0, bytes_out);
			blur_row(y + j + kR, ring[(j + 2 * kR) % kTaps]);
			float sums[kQ];
			column(ring, j, sums);
			out((y + j) * stride + e0, bytes_out, sums, c);
			// The ring's values are new to the compiler: it would keep products of one row for a later one.
#pragma unroll
			for (int k = 0; k < kTaps; k++) {
#pragma unroll
				for (int q = 0; q < kQ; q++) asm volatile("" : "+v"(ring[k][q]));
			}
		}
	}
}

// Forward: moments a, b, aa, bb, ab blurred -> ssim, d_mu, d_aa, d_ab (ssim.cu:39-72).
__global__ __launch_bounds__(kE, 4) void ssim_forward_kernel(int height, int width, int rows,
															 const float* __restrict__ img_a,
															 const float* __restrict__ img_b, float* __restrict__ ssim_map,
															 float* __restrict__ d_mu, float* __restrict__ d_aa,
															 float* __restrict__ d_ab) {
	struct None {};
	walk_strip<5, float2, None>(
		height, width, rows, [&](int64_t g, uint32_t i) { return make_float2(at(img_a, g, i), at(img_b, g, i)); },
		[](int64_t, uint32_t) { return None{}; },
		[](float w, float2 p, float (&s)[5], bool first) {
			const float wa = w * p.x, wb = w * p.y;
			const float m[5] = {wa, wb, wa * p.x, wb * p.y, wa * p.y};
#pragma unroll
			for (int q = 0; q < 5; q++) s[q] = first ? m[q] : s[q] + m[q];
		},
		[](const float (&ring)[kTaps][5], int slot, float (&s)[5]) {
#pragma unroll
			for (int k = 0; k < kTaps; k++) {
#pragma unroll
				for (int q = 0; q < 5; q++) {
					const float m = kWin[k] * ring[(slot + k) % kTaps][q];
					s[q] = k == 0 ? m : s[q] + m;
				}
			}
		},
		[&](int64_t g, uint32_t i, const float (&e)[5], None) {
			const float mu_a = e[0], mu_b = e[1], e_aa = e[2], e_bb = e[3], e_ab = e[4];
			const float a1 = 2.0f * mu_a * mu_b + kC1;
			const float a2 = 2.0f * (e_ab - mu_a * mu_b) + kC2;
			const float b1 = mu_a * mu_a + mu_b * mu_b + kC1;
			const float b2 = (e_aa - mu_a * mu_a) + (e_bb - mu_b * mu_b) + kC2;
			const float inv_b = 1.0f / (b1 * b2);
			const float sv = a1 * a2 * inv_b;
			at(ssim_map, g, i) = sv;
			at(d_mu, g, i) = (2.0f * mu_b * (a2 - a1) - 2.0f * mu_a * sv * (b2 - b1)) * inv_b;
			at(d_aa, g, i) = -sv / b2;
			at(d_ab, g, i) = 2.0f * a1 * inv_b;
		});
}

// Backward: grad = dL/dmean / n * (blur(d_mu) + 2 a blur(d_aa) + b blur(d_ab)) (ssim.cu:74-113); the window's
// transpose is itself.
__global__ __launch_bounds__(kE, 4) void ssim_backward_kernel(int height, int width, int rows,
															  const float* __restrict__ grad_mean,
															  const float* __restrict__ img_a, const float* __restrict__ img_b,
															  const float* __restrict__ p_mu, const float* __restrict__ p_aa,
															  const float* __restrict__ p_ab, float* __restrict__ grad) {
	const float scale = grad_mean[0] / (float)((int64_t)height * width * 3);
	walk_strip<3, float3, float2>(
		height, width, rows,
		[&](int64_t g, uint32_t i) { return make_float3(at(p_mu, g, i), at(p_aa, g, i), at(p_ab, g, i)); },
		[&](int64_t g, uint32_t i) { return make_float2(at(img_a, g, i), at(img_b, g, i)); },
		[](float w, float3 p, float (&s)[3], bool first) {
			s[0] = first ? w * p.x : fmaf(w, p.x, s[0]);
			s[1] = first ? w * p.y : fmaf(w, p.y, s[1]);
			s[2] = first ? w * p.z : fmaf(w, p.z, s[2]);
		},
		[](const float (&ring)[kTaps][3], int slot, float (&s)[3]) {
#pragma unroll
			for (int k = 0; k < kTaps; k++) {
#pragma unroll
				for (int q = 0; q < 3; q++) {
					const float v = ring[(slot + k) % kTaps][q];
					s[q] = k == 0 ? kWin[k] * v : fmaf(kWin[k], v, s[q]);
				}
			}
		},
		[&](int64_t g, uint32_t i, const float (&e)[3], float2 c) {
			at(grad, g, i) = scale * (e[0] + 2.0f * c.x * e[1] + c.y * e[2]);
		});
}

// Rows per strip: a strip blurs 10 rows more than it writes, so long strips save work, but the waves have to fill
// the chip's 1,024 SIMDs evenly. Takes the fewest row steps of the busiest SIMD.
int strip_rows(int height, int strips) {
	constexpr int64_t kSimds = 1024;
	int best = 0;
	int64_t least = INT64_MAX;
	for (int rows = 4; rows <= 64; rows += 4) {
		const int64_t waves = (int64_t)strips * ((height + rows - 1) / rows);
		const int64_t steps = ((waves + kSimds - 1) / kSimds) * (rows + 2 * kR);
		if (steps < least) best = rows, least = steps;
	}
	return best;
}

}  // namespace

extern "C" int hds_ssim_forward(int height, int width, const float* rendered, const float* gt, float* ssim_map,
								float* d_mu, float* d_aa, float* d_ab, hds_stream_t stream) {
	HDS_REQUIRE(height > 0 && width > 0, "ssim inputs must both be [H, W, 3] with H, W > 0");
	HDS_REQUIRE(rendered && gt && ssim_map && d_mu && d_aa && d_ab, "ssim_forward: null pointer argument");
	hipStream_t s = (hipStream_t)stream;
	const int strips = (int)(((int64_t)width * 3 + kE - 1) / kE), rows = strip_rows(height, strips);
	const dim3 grid((unsigned)(strips * (int64_t)((height + rows - 1) / rows)));
	HdsKernelTimer timer1("ssim_forward_kernel", s);
	ssim_forward_kernel<<<grid, kE, 0, s>>>(height, width, rows, rendered, gt, ssim_map, d_mu, d_aa, d_ab);
	timer1.stop();
	HDS_LAUNCH_CHECK("ssim_forward", s);
	return HDS_OK;
}

extern "C" int hds_ssim_backward(int height, int width, const float* grad_mean, const float* rendered, const float* gt,
								 const float* d_mu, const float* d_aa, const float* d_ab, float* grad_rendered,
								 hds_stream_t stream) {
	HDS_REQUIRE(height > 0 && width > 0, "ssim inputs must both be [H, W, 3] with H, W > 0");
	HDS_REQUIRE(grad_mean && rendered && gt && d_mu && d_aa && d_ab && grad_rendered, "ssim_backward: null pointer argument");
	hipStream_t s = (hipStream_t)stream;
	const int strips = (int)(((int64_t)width * 3 + kE - 1) / kE), rows = strip_rows(height, strips);
	const dim3 grid((unsigned)(strips * (int64_t)((height + rows - 1) / rows)));
	HdsKernelTimer timer2("ssim_backward_kernel", s);
	ssim_backward_kernel<<<grid, kE, 0, s>>>(height, width, rows, grad_mean, rendered, gt, d_mu, d_aa, d_ab, grad_rendered);
	timer2.stop();
	HDS_LAUNCH_CHECK("ssim_backward", s);
	return HDS_OK;
}
