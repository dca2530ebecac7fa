// Blend backward through per-block gaussian lists and stored gradient rows (hds_render_backward_rows).
//
// 1. backward_lists_kernel: per tile, the gaussians that blend into each of its four 8x8 pixel blocks (from the
//    render's marks; without marks, those that can reach the block, up to its deepest contributor), deepest first,
//    as one list per block; every (gaussian, block) hit
//    gets the next row number of its gaussian.
// 2. backward_base_kernel: one contiguous range of rows per gaussian.
// 3. backward_geometry_kernel: the replay. Work-group = one block x slice of S channels, two waves; it walks
//    the block's list from every pixel's final T and n_contrib (backward.cu:53-163, features.cu:419-541) in
//    groups of 16 gaussians. Inside a group a lane is a (gaussian, pixel quarter) pair: lane 16 h + q
//    holds gaussian q of the group (q = 0 deepest) and the 16 pixels 16 n + 4 h + i (n, i < 4), so that
//    - alpha, T, the weights and dL/dalpha of a group are 16 independent chains per lane: nothing waits
//      for the previous gaussian, the recurrences over the gaussians are prefix scans over q (DPP);
//    - the gaussian's record sits in the lane's registers, and its geometry gradients are plain fp32 sums
//      over the lane's pixels, reduced over the four h lanes once per group;
//    - dot[px][q] = sum_c dL/dF[px][c] F[q][c] comes out of the 16x16x32 MFMA in exactly this layout
//      (rows = pixels, column = gaussian), with F read as the gaussian's own row;
//    - the weights w[q][px] are the A operand of dF[q][c] += sum_px w[q][px] dL/dF[px][c] as they stand: the
//      order of the pixels along K is free as long as both operands agree.
//    dL/dF of the block stays in LDS as split-bf16 planes for the whole walk; the dot products read it by
//    rows, the contraction by columns (ds_read_b64_tr_b16). The gradients of each (gaussian, block) are
//    stored as one row.
// 4. backward_features_kernel: sums every gaussian's rows.
//
// With R_q = prod_{j <= q} (1 - alpha_j) over the group (from its deepest gaussian) and T_out, U the
// transmittance and sum_{behind} w d (plus T_final bg . g) behind the group:
//   T_q = T_out / R_q,  w_q = alpha_q T_q,  U_q = U + T_out sum_{j < q} alpha_j d_j / R_j,
//   dL/dalpha_q = T_q d_q - U_q / (1 - alpha_q),  d = f . dL/dF + c . dL/dRGB
// (the reference's RGB term (c - rec) . g T and its feature term T (dot - behind_dot) are this one
// expression; geometry gradients only where the raw alpha <= 0.99, backward.cu:126-135). Only (T_out, U)
// chain from group to group, so the two waves evaluate consecutive groups at once and exchange 1 / R and
// the sum of each whole group through LDS, one barrier per pair of groups.
//
// Rows instead of atomics: the L2s perform about 20 G atomic requests (of up to 64 bytes) per second,
// whatever their scope or locality: 2.32M feature rows of 512 B took 0.91 ms as atomics, and 0.20 ms as
// stores plus 0.17 ms as loads.
//
// Measured at 1.18M gaussians, 979x546, against the two kernels of hds_render_backward (lane = pixel, a
// serial chain per gaussian, atomics; side by side): C = 128 lists 0.08 + replay 0.71 + sums 0.39 ms for 1.68,
// RGB alone 0.08 + 0.27 + 0.06 for 0.66, C = 512 4.5 for 6.4; 4M gaussians at 1920x1080, C = 256: 2.6 for 4.2. The
// replay issues 1,290 VALU instructions per group (0.36 ms), 106 MFMAs (0.11 ms), and moves 1.3 GB of feature
// rows in and 1.5 GB of gradient rows out; it runs two waves per SIMD (250 VGPRs, 40 KB of LDS per block).
#include <algorithm>

#include "hds_internal.h"
#include "hds_rasterizer.h"
#include "hds_stage.h"

namespace {

constexpr int kGroup = 16;                // gaussians per group
constexpr int kWaves = 2;                 // groups in flight per block
constexpr int kThreads = 64 * kWaves;
constexpr int kRound = kWaves * kGroup;   // gaussians per round
constexpr int kGeo = 16;                  // floats of a row's geometry part, one part per slice:
constexpr int kGeoGid = 9;                //   dopacity, dmean2D, dconic, dcolour, the gaussian's index
constexpr int kWaitVmem = 0x0f70;         // s_waitcnt vmcnt(0)
constexpr int kLong = 64;                 // gaussians with more rows are summed in pieces of this many
constexpr int kSpareRows = 1024;          // rows past the capacity that take what no gaussian's row needs
constexpr int64_t kMaxRows = 1 << 30;     // row numbers stay below 2^31: base <= 2^30, ordinals < blocks of an image

// The gaussians that reach each block: entries [4 range.x + b (range.y - range.x), + hits[4 tile + b]) of the
// three arrays belong to block b of a tile.
struct BlockLists {
	int* gid;
	int* idx;      // position in the tile's list
	int* ordinal;  // row number within the gaussian's rows
	int* hits;
};

// Row storage: gaussian g's rows are [base[g], base[g] + count[g]): a feature part of one float per channel and
// one geometry part per slice each, in arrays of their own so that both start on cache lines. Rows from
// `capacity` on do not exist: their gradients are added atomically.
struct Rows {
	float* features;
	float* geo;
	int* count;
	int* base;
	unsigned long long* total;  // allocation cursor of backward_base_kernel
	int64_t capacity;
	int slices;
};

struct BackwardArgs {
	int width, height, tiles_x, channels, num_tiles;
	int64_t n;
	const int2* ranges;
	const int* values;
	const float2* means2D;
	const float4* conic4;
	const float4* color_op4;
	const float* background;
	const float* final_T;
	const int* n_contrib;
	const uint8_t* contributes;  // the render's marks (hds_render_contributes), or null
	const float* grad_image;
	const float* features;
	const float* grad_feature_image;
	float* grad_means2D;
	float* grad_conics;
	float* grad_colors;
	float* grad_opacities;
	float* grad_features;
	BlockLists lists;
	Rows rows;
};

// One work-group per tile, a list entry per thread and step, what the next step needs in flight meanwhile. With the
// render's marks (kMarked) a block's list holds exactly what blends into it; without them, what can reach it: a
// thread tests its entry against the tile's four blocks (their tests share most of the arithmetic, and every
// record is gathered once). Bound by latency and the one returning atomic per (gaussian, tile). At 1.18M
// gaussians, 979x546, C = 128 marks take 0.020 ms of the render and save 0.026 here (0.108 -> 0.082), 0.065 of the
// geometry and 0.036 of the sums, which have a tenth fewer rows.
constexpr int kListThreads = 256;
template <bool kMarked>
__global__ __launch_bounds__(kListThreads) void backward_lists_kernel(const BackwardArgs a) {
	__shared__ int s_last[4];
	__shared__ int s_count[2][4][4];  // per step parity: [wave][block]
	const int tile = blockIdx.x, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
	const int tx0 = (tile % a.tiles_x) * HDS_TILE, ty0 = (tile / a.tiles_x) * HDS_TILE;
	const int2 range = a.ranges[tile];
	const int len = range.y - range.x;
	{
		// Wave = block, lane = pixel: the block's deepest contributor.
		const int x = tx0 + (wave & 1) * 8 + (lane & 7), y = ty0 + (wave >> 1) * 8 + (lane >> 3);
		const int last = x < a.width && y < a.height ? a.n_contrib[(int64_t)y * a.width + x] : 0;
		const int deepest = hds_wave_max(last);
		if (lane == 0) s_last[wave] = min(deepest, len);
	}
	__syncthreads();
	int last[4], found[4] = {0, 0, 0, 0};
#pragma unroll
	for (int b = 0; b < 4; b++) last[b] = __builtin_amdgcn_readfirstlane(s_last[b]);
	const int num = max(max(last[0], last[1]), max(last[2], last[3]));
	const int* const list = a.values + range.x;
	const int64_t out = 4 * (int64_t)range.x;
	int gid = 0, later = 0;
	float2 mean = make_float2(0.0f, 0.0f);
	float4 conic = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
	uint8_t mark[4] = {0, 0, 0, 0};
	// The records or marks of entry e (gaussian gid).
	auto fetch = [&](int e) {
		if constexpr (kMarked) {
#pragma unroll
			for (int b = 0; b < 4; b++) mark[b] = a.contributes[out + (int64_t)b * len + max(e, 0)];
		} else {
			mean = a.means2D[gid];
			conic = a.conic4[gid];
		}
	};
	if (num > 0) {
		gid = list[max(num - 1 - tid, 0)];
		later = list[max(num - 1 - kListThreads - tid, 0)];
		fetch(num - 1 - tid);
	}
	for (int step = 0; step * kListThreads < num; step++) {
		const int e = num - 1 - step * kListThreads - tid, g = gid;
		const float2 m = mean;
		const float4 c = conic;
		const uint8_t marked[4] = {mark[0], mark[1], mark[2], mark[3]};
		gid = later;
		fetch(e - kListThreads);
		later = list[max(e - 2 * kListThreads, 0)];
		uint64_t hits[4];
		int mask = 0;
#pragma unroll
		for (int b = 0; b < 4; b++) {
			const float x0 = (float)(tx0 + (b & 1) * 8) + 0.5f, y0 = (float)(ty0 + (b >> 1) * 8) + 0.5f;
			const bool hit = e >= 0 && e < last[b] && (kMarked ? marked[b] != 0 : hds_block_reach(m, c, x0, x0 + 7.0f, y0, y0 + 7.0f));
			hits[b] = hds_ballot(hit);
			mask |= (int)hit << b;
		}
		int ordinal = 0;
		if (mask) ordinal = atomicAdd(a.rows.count + g, __popc(mask));
		int(*const count)[4] = s_count[step & 1];
		if (lane < 4) count[wave][lane] = __popcll(lane == 0 ? hits[0] : lane == 1 ? hits[1] : lane == 2 ? hits[2] : hits[3]);
		__syncthreads();
#pragma unroll
		for (int b = 0; b < 4; b++) {
			int before = 0, all = 0;
#pragma unroll
			for (int w = 0; w < 4; w++) {
				const int k = count[w][b];
				before += w < wave ? k : 0;
				all += k;
			}
			if ((mask >> b) & 1) {
				const int64_t to = out + (int64_t)b * len + found[b] + before + hds_rank_below(hits[b]);
				a.lists.gid[to] = g;
				a.lists.idx[to] = e;
				a.lists.ordinal[to] = ordinal++;
			}
			found[b] += all;
		}
	}
	if (tid == 0) {
#pragma unroll
		for (int b = 0; b < 4; b++) a.lists.hits[4 * tile + b] = found[b];
	}
}

// Whether a gaussian with these rows is summed by plain stores; the others' gradients are added atomically.
__device__ inline bool summed_whole(const Rows& rows, int base, int count) {
	return count <= kLong && (int64_t)base + count <= rows.capacity;
}

// Row ranges: a work-group places the rows of 4096 gaussians in one run, taken from the cursor (fewer, larger
// runs: the cursor's atomics queue up, 1024 per run took 0.020 ms for 1.18M gaussians).
constexpr int kBaseThreads = 1024, kBaseItems = 4;
__global__ __launch_bounds__(kBaseThreads) void backward_base_kernel(const BackwardArgs a) {
	__shared__ uint32_t s_wave[kBaseThreads / 64];
	__shared__ unsigned long long s_base;
	const int64_t g0 = ((int64_t)blockIdx.x * kBaseThreads + threadIdx.x) * kBaseItems;
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	uint32_t count[kBaseItems], sum = 0;
#pragma unroll
	for (int k = 0; k < kBaseItems; k++) {
		count[k] = g0 + k < a.n ? (uint32_t)a.rows.count[g0 + k] : 0u;
		sum += count[k];
	}
	const uint32_t upto = hds_wave_inclusive_scan(sum);
	if (lane == 63) s_wave[wave] = upto;
	__syncthreads();
	unsigned long long before = 0, all = 0;
#pragma unroll
	for (int w = 0; w < kBaseThreads / 64; w++) {
		before += w < wave ? s_wave[w] : 0u;
		all += s_wave[w];
	}
	if (threadIdx.x == 0) s_base = atomicAdd(a.rows.total, all);
	__syncthreads();
	unsigned long long at = s_base + before + (upto - sum);
#pragma unroll
	for (int k = 0; k < kBaseItems; k++) {
		const int64_t g = g0 + k;
		if (g >= a.n) break;
		const int base = (int)min(at, (unsigned long long)kMaxRows);
		a.rows.base[g] = base;
		at += count[k];
	}
}

// x[k] <- x[k] OP x[k] of the lanes below in the 16-lane row (inclusive prefix), for 8 independent chains.
// A lane whose source lies outside the row keeps its value (bound_ctrl off). s_nop: the two wait states
// between a VALU write and its DPP read; inside the block the same register comes round after eight.
#define HDS_SCAN_STEP(OP, SHIFT)                                        \
	OP " %0, %0, %0 row_shr:" SHIFT " row_mask:0xf bank_mask:0xf\n"     \
	OP " %1, %1, %1 row_shr:" SHIFT " row_mask:0xf bank_mask:0xf\n"     \
	OP " %2, %2, %2 row_shr:" SHIFT " row_mask:0xf bank_mask:0xf\n"     \
	OP " %3, %3, %3 row_shr:" SHIFT " row_mask:0xf bank_mask:0xf\n"     \
	OP " %4, %4, %4 row_shr:" SHIFT " row_mask:0xf bank_mask:0xf\n"     \
	OP " %5, %5, %5 row_shr:" SHIFT " row_mask:0xf bank_mask:0xf\n"     \
	OP " %6, %6, %6 row_shr:" SHIFT " row_mask:0xf bank_mask:0xf\n"     \
	OP " %7, %7, %7 row_shr:" SHIFT " row_mask:0xf bank_mask:0xf\n"
#define HDS_SCAN8(OP, x, b)                                                                               \
	asm("s_nop 1\n" HDS_SCAN_STEP(OP, "1") HDS_SCAN_STEP(OP, "2") HDS_SCAN_STEP(OP, "4") HDS_SCAN_STEP(OP, "8") \
		: "+v"(x[b]), "+v"(x[b + 1]), "+v"(x[b + 2]), "+v"(x[b + 3]), "+v"(x[b + 4]), "+v"(x[b + 5]),       \
		  "+v"(x[b + 6]), "+v"(x[b + 7]))

__device__ inline void scan_products(float (&x)[16]) {
	HDS_SCAN8("v_mul_f32_dpp", x, 0);
	HDS_SCAN8("v_mul_f32_dpp", x, 8);
}
__device__ inline void scan_sums(float (&x)[16]) {
	HDS_SCAN8("v_add_f32_dpp", x, 0);
	HDS_SCAN8("v_add_f32_dpp", x, 8);
}

// x times the r of the lane below in the 16-lane row; x in the row's lane 0. The s_nop covers a write of r
// right before.
__device__ inline float scale_by_row_below(float x, float r) {
	float v = x;
	asm("s_nop 1\n\tv_mul_f32_dpp %0, %1, %2 row_shr:1 row_mask:0xf bank_mask:0xf" : "+v"(v) : "v"(r), "v"(x));
	return v;
}
// v -= b * (s of the lane below in the row; 0 for the row's lane 0).
__device__ inline void subtract_row_below(float& v, float s, float b) {
	asm("s_nop 1\n\tv_fmac_f32_dpp %0, -%1, %2 row_shr:1 row_mask:0xf bank_mask:0xf" : "+v"(v) : "v"(s), "v"(b));
}

// min(0.99, raw alpha), 0.99 for NaN, without the canonicalising move of fminf.
__device__ inline float min_alpha(float raw) {
	float r;
	asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(raw), "v"(HDS_MAX_ALPHA));
	return r;
}

// a * b, with 0 * anything = 0.
__device__ inline float mul_legacy(float a, float b) {
	float r;
	asm("v_mul_legacy_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
	return r;
}

// dL/dF planes: pixel row px holds its S channels as bf16 in S / 8 chunks of 16 bytes. Chunk 4 kk + h has
// the K slots of lane group h in step kk of the dot products: slot 4 j2 + e is channel
// (S / 2) j2 + (S / 8) h + (S / 32) e + kk. A gaussian's F row is then read as two contiguous runs per lane,
// and a lane's results of the contraction are S / 32 consecutive channels (one store). The chunk index is
// XORed with plane_swizzle(px): both reads (16 pixels at one chunk; 8 consecutive pixels at an aligned
// pair of chunks) touch every bank once.
template <int S>
__device__ inline int plane_swizzle(int px) {
	constexpr int kBits = S >= 128 ? 4 : S == 64 ? 3 : 2;
	const int t = (px & 15) >> (4 - kBits);
	return ((t << 1) & ((1 << kBits) - 1)) | (t >> (kBits - 1));
}

typedef short hds_i16x4 __attribute__((ext_vector_type(4)));
typedef short hds_i16x8 __attribute__((ext_vector_type(8)));

// ds_read_b64_tr_b16: within 16 lanes, lane L supplies the address of four values of row L / 4, and lane l
// receives value l % 4 of the lanes l / 4, 4 + l / 4, 8 + l / 4, 12 + l / 4 (checked on hardware).
__device__ inline hds_i16x4 read_transposed(const char* p) {
	return __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) hds_i16x4*)p);
}
__device__ inline hds_bf16x8 join8(hds_i16x4 a, hds_i16x4 b) {
	return __builtin_bit_cast(hds_bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// One fp32 value as three bf16 terms (24 bits).
__device__ inline void split3(float x, __bf16& hi, __bf16& mid, __bf16& lo) {
	hi = (__bf16)x;
	const float r = x - (float)hi;
	mid = (__bf16)r;
	lo = (__bf16)(r - (float)mid);
}

__device__ inline float element(const float4& v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// Sums of two values over the lane pairs (l, l + 32): lanes 0-31 get a's, lanes 32-63 b's.
__device__ inline float fold32(float a, float b) {
	const auto r = __builtin_amdgcn_permlane32_swap(hds_swap_operand(a), hds_swap_operand(b), false, false);
	return hds_u2f(r[0]) + hds_u2f(r[1]);
}
// Sums over the row pairs (0, 1) and (2, 3): the even row gets a's, the odd row b's.
__device__ inline float fold16(float a, float b) {
	const auto r = __builtin_amdgcn_permlane16_swap(hds_swap_operand(a), hds_swap_operand(b), false, false);
	return hds_u2f(r[0]) + hds_u2f(r[1]);
}

// REST: the second launch where the rows might not fit: it returns at once when they did, and otherwise adds the
// gradients of the rows past the capacity atomically.
// RGB alone fits three waves per SIMD (167 VGPRs; 0.317 -> 0.270 ms at 1.18M gaussians, 979x546); a slice of 32 channels
// would spill 16 registers for it and gains nothing.
template <int S, bool RGB, bool WANT, bool REST>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(S == 0 ? 3 : 2))) void backward_geometry_kernel(
	const BackwardArgs a) {
	constexpr int kKc = S > 0 ? S / 32 : 1;    // K steps of the dot products
	constexpr int kRun = S > 0 ? S / 8 : 4;    // channels per run of an F row
	constexpr int kRowBytes = 2 * S;           // one pixel's channels in a plane
	constexpr int kPlane = 64 * kRowBytes;

	__shared__ __attribute__((aligned(16))) char s_df[S > 0 ? 2 * kPlane : 16];  // hi plane, lo plane
	// Per round parity and wave: 1 / R and the sum of its group, by pixel.
	__shared__ __attribute__((aligned(16))) float s_x[2][kWaves][2][64];
	// Per wave: T_out and U of its group, by pixel.
	__shared__ __attribute__((aligned(16))) float s_in[kWaves][2][64];
	__shared__ __attribute__((aligned(16))) int s_last[64];
	// dL/dRGB of pixel 16 n + q, channel h, as the dot products' A operand (below).
	__shared__ __attribute__((aligned(16))) hds_bf16x8 s_g[RGB ? 4 : 1][RGB ? 64 : 1];

	const int block = hds_xcd_block(blockIdx.x, a.tiles_x, a.num_tiles);
	if (block < 0) return;
	const int tile = block >> 2;
	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int q = lane & 15, h = lane >> 4;
	const int slice = blockIdx.y, c0 = slice * S;
	const bool do_rgb = RGB && slice == 0;
	const int wx0 = (tile % a.tiles_x) * HDS_TILE + (block & 1) * 8;
	const int wy0 = (tile / a.tiles_x) * HDS_TILE + ((block >> 1) & 1) * 8;
	const int hits = a.lists.hits[block];
	if (hits == 0) return;
	if (REST && *a.rows.total <= (unsigned long long)a.rows.capacity) return;
	const int2 range = a.ranges[tile];
	const int64_t list = 4 * (int64_t)range.x + (int64_t)(block & 3) * (range.y - range.x);

	// T and U behind the current round, pixel = lane (both waves keep both).
	float T = 1.0f, U = 0.0f;
	{
		const int x = wx0 + (lane & 7), y = wy0 + (lane >> 3);
		const bool in = x < a.width && y < a.height;
		const int64_t pix = (int64_t)y * a.width + x;
		if (in) {
			T = a.final_T[pix];
			if (do_rgb)
				U = T * (a.background[0] * a.grad_image[pix * 3 + 0] + a.background[1] * a.grad_image[pix * 3 + 1] +
						 a.background[2] * a.grad_image[pix * 3 + 2]);
		}
		if (wave == 0) s_last[lane] = in ? a.n_contrib[pix] : 0;
	}

	// dL/dF of the block -> split-bf16 planes (zeros outside the image); a unit is one run of one pixel.
	if constexpr (S > 0) {
#pragma unroll
		for (int k = 0; k < 64 * 8 / kThreads; k++) {
			const int u = k * kThreads + tid, p = u >> 3, seg = u & 7;
			const int x = wx0 + (p & 7), y = wy0 + (p >> 3);
			float v[kRun];
			const bool in = x < a.width && y < a.height;
			const float* src = a.grad_feature_image + ((int64_t)y * a.width + x) * a.channels + c0 + kRun * seg;
#pragma unroll
			for (int j = 0; j < kRun; j += 4) {
				const float4 t = in ? *reinterpret_cast<const float4*>(src + j) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
				v[j] = t.x, v[j + 1] = t.y, v[j + 2] = t.z, v[j + 3] = t.w;
			}
			const int swizzle = plane_swizzle<S>(p);
#pragma unroll
			for (int kk = 0; kk < kKc; kk++) {
				uint2 hi, lo;
				hds_split_pair(v[kk], v[kKc + kk], hi.x, lo.x);
				hds_split_pair(v[2 * kKc + kk], v[3 * kKc + kk], hi.y, lo.y);
				char* dst = s_df + p * kRowBytes + (((4 * kk + (seg & 3)) ^ swizzle) << 4) + ((seg >> 2) << 3);
				*reinterpret_cast<uint2*>(dst) = hi;
				*reinterpret_cast<uint2*>(dst + kPlane) = lo;
			}
		}
	}

	// dL/dRGB as MFMA operands. For the dot c . g (kept at fp32 accuracy: three bf16 terms per factor, the
	// six products above 2^-24) lane group h carries channel h in its eight K slots; for the colour
	// gradient sum_px w g, columns 0-2 hold g's hi terms and 4-6 its lo terms.
	hds_bf16x8 g_col[2];
	if (do_rgb) {
#pragma unroll
		for (int k = 0; k < 4 / kWaves; k++) {
			const int n = wave + kWaves * k, p = 16 * n + q, x = wx0 + (p & 7), y = wy0 + (p >> 3);
			const bool in = h < 3 && x < a.width && y < a.height;
			const float v = in ? a.grad_image[((int64_t)y * a.width + x) * 3 + h] : 0.0f;
			__bf16 hi, mid, lo;
			split3(v, hi, mid, lo);
			s_g[n][lane] = hds_bf16x8{hi, hi, mid, hi, mid, lo, (__bf16)0.0f, (__bf16)0.0f};
		}
#pragma unroll
		for (int kp = 0; kp < 2; kp++)
#pragma unroll
			for (int j = 0; j < 8; j++) {
				const int p = 16 * (2 * kp + (j >> 2)) + 4 * h + (j & 3), x = wx0 + (p & 7), y = wy0 + (p >> 3);
				const bool in = q < 8 && (q & 3) < 3 && x < a.width && y < a.height;
				const float v = in ? a.grad_image[((int64_t)y * a.width + x) * 3 + (q & 3)] : 0.0f;
				const __bf16 hi = (__bf16)v;
				g_col[kp][j] = q < 4 ? hi : (__bf16)(v - (float)hi);
			}
	}

	// The lane's pixel centres: columns x0 + i, rows y0 + 2 n.
	const float x0 = (float)(wx0 + 4 * (h & 1)) + 0.5f, y0 = (float)(wy0 + (h >> 1)) + 0.5f;
	// Dot products read pixel 16 n + q at chunk 4 kk + h; the contraction reads pixel 16 n + 4 h + q / 4 at
	// chunk 4 kk + 2 u + (q / 2) % 2, half q % 2.
	const char* const dot_row = s_df + q * kRowBytes;
	const char* const tr_row = s_df + (4 * h + (q >> 2)) * kRowBytes + ((q & 1) << 3);
	const int dot_chunk = S > 0 ? h ^ plane_swizzle<S>(q) : 0;
	const int tr_chunk = S > 0 ? ((q >> 1) & 1) ^ plane_swizzle<S>(4 * h + (q >> 2)) : 0;

	// What a group needs from memory is loaded in the middle of the round before (its list entries one round
	// earlier still), and always before that round's stores: the waits then count past the stores, which are in
	// flight for the whole next round (1.18M gaussians, 979x546: RGB 0.41 -> 0.36 ms, C = 128 0.83 -> 0.81 ms). The
	// compiler can count them because every round issues the same loads and stores whatever its lanes do:
	// positions past the list's end repeat its last hit, never contribute and store to a spare row.
	struct Entry {
		int gid, idx, ordinal;
	};
	struct Group {
		int gid, idx, base, ordinal;
		float2 mean;
		float4 conic;
		float color;              // colour channel h
		float4 f[2][kRun / 4];    // the lane's two runs of the F row
	};
	auto load_entry = [&](int first) {
		const int at = first + wave * kGroup + q;
		const int64_t e = list + min(at, hits - 1);
		Entry r;
		r.gid = a.lists.gid[e];
		r.idx = a.lists.idx[e];
		r.ordinal = a.lists.ordinal[e];
		return r;
	};
	auto keep = [](auto v) { return __builtin_bit_cast(decltype(v), hds_opaque(__builtin_bit_cast(uint32_t, v))); };
	auto load_group = [&](Group& r, const Entry& e) {
		r.gid = keep(e.gid);
		r.idx = keep(e.idx);
		r.ordinal = keep(e.ordinal);
		r.base = a.rows.base[r.gid];
		r.mean = a.means2D[r.gid];
		r.conic = a.conic4[r.gid];
		r.color = reinterpret_cast<const float*>((RGB ? a.color_op4 : a.conic4) + r.gid)[hds_opaque(h)];
		if constexpr (S > 0) {
			const float* src = a.features + (size_t)r.gid * a.channels + c0 + kRun * h;
#pragma unroll
			for (int j2 = 0; j2 < 2; j2++)
#pragma unroll
				for (int j = 0; j < kRun / 4; j++) r.f[j2][j] = *reinterpret_cast<const float4*>(src + (S / 2) * j2 + 4 * j);
		}
	};
	Group g;
	load_group(g, load_entry(0));
	Entry later = load_entry(kRound);
	// vmcnt(0) in the form that the compiler reads: with nothing in flight on entry, the loop's waits count the
	// loads and stores of one round and the next alone.
	__builtin_amdgcn_s_waitcnt(kWaitVmem);
	__syncthreads();

	for (int round = 0, first = 0; first < hits; round++, first += kRound) {
		const bool work = first + wave * kGroup < hits;  // wave-uniform
		float raw[16];  // raw alpha where the gaussian contributes to the pixel, else 0
		float A[16], B[16], W[16], S_q[16], rc[16];
		uint32_t active = 0;  // positions that contribute to at least one pixel
		hds_f32x4 X[4];
#pragma unroll
		for (int k = 0; k < 16; k++) {
			rc[k] = 1.0f;
			S_q[k] = 0.0f;
		}
		if (work) {
			const int idx = first + wave * kGroup + q < hits ? g.idx : 0x7fffffff;
			uint32_t any = 0;
#pragma unroll
			for (int n = 0; n < 4; n++) {
				const int4 last = *reinterpret_cast<const int4*>(&s_last[16 * n + 4 * h]);
				const int last_of[4] = {last.x, last.y, last.z, last.w};
#pragma unroll
				for (int i = 0; i < 4; i++) {
					float G, dx, dy;
					const float v = hds_raw_alpha(x0 + (float)i, y0 + (float)(2 * n), g.mean, g.conic, G, dx, dy);
					const bool on = idx < last_of[i] && !(v < HDS_MIN_ALPHA);
					raw[4 * n + i] = on ? v : 0.0f;
					any |= hds_f2u(raw[4 * n + i]);
				}
			}
			uint64_t lanes = hds_ballot(any != 0);
			lanes |= lanes >> 32;
			active = (uint32_t)(lanes | (lanes >> 16)) & 0xffffu;
		}
		if (active != 0) {
#pragma unroll
			for (int k = 0; k < 16; k++) {
				W[k] = min_alpha(raw[k]);
				B[k] = 1.0f - W[k];
			}
			scan_products(B);
#pragma unroll
			for (int k = 0; k < 16; k++) {
				rc[k] = __builtin_amdgcn_rcpf(B[k]);     // 1 / R_q
				B[k] = scale_by_row_below(rc[k], B[k]);  // R_{q-1} / R_q = 1 / (1 - alpha)
				W[k] *= rc[k];                           // w / T_out
			}
#pragma unroll
			for (int n = 0; n < 4; n++) X[n] = hds_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
			if (do_rgb) {
				__bf16 hi, mid, lo;
				split3(h < 3 ? g.color : 0.0f, hi, mid, lo);
				const hds_bf16x8 c_dot = {hi, mid, hi, lo, mid, hi, (__bf16)0.0f, (__bf16)0.0f};
#pragma unroll
				for (int n = 0; n < 4; n++) X[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(s_g[n][lane], c_dot, X[n], 0, 0, 0);
			}
			if constexpr (S > 0) {
#pragma unroll
				for (int kk = 0; kk < kKc; kk++) {
					float v[8];
#pragma unroll
					for (int j = 0; j < 8; j++) {
						const int r = kKc * (j & 3) + kk;
						v[j] = element(g.f[j >> 2][r >> 2], r & 3);
					}
					hds_bf16x8 f_hi, f_lo;
					hds_split8(v, f_hi, f_lo);
					const char* src = dot_row + ((dot_chunk ^ (4 * kk)) << 4);
#pragma unroll
					for (int n = 0; n < 4; n++) {
						const hds_bf16x8 p_hi = *reinterpret_cast<const hds_bf16x8*>(src + 16 * n * kRowBytes);
						const hds_bf16x8 p_lo = *reinterpret_cast<const hds_bf16x8*>(src + 16 * n * kRowBytes + kPlane);
						X[n] = hds_mfma_split(p_hi, p_lo, f_hi, f_lo, X[n]);
					}
				}
			}
		}
		// What the rest of the round needs of this group moves out of the way of the next one.
		const int gid = keep(g.gid), row = keep(g.base + g.ordinal);
		const float2 mean = make_float2(keep(g.mean.x), keep(g.mean.y));
		const float4 conic = make_float4(keep(g.conic.x), keep(g.conic.y), keep(g.conic.z), keep(g.conic.w));
		load_group(g, later);
		later = load_entry(first + 2 * kRound);
		if (active != 0) {
#pragma unroll
			for (int k = 0; k < 16; k++) {
				const float d = X[k >> 2][k & 3];
				A[k] = rc[k] * d;
				// 0 * anything is 0: a pixel's infinite or NaN d reaches only the gaussians it sees.
				S_q[k] = mul_legacy(W[k], d);
			}
			scan_sums(S_q);
#pragma unroll
			for (int k = 0; k < 16; k++) subtract_row_below(A[k], S_q[k], B[k]);
		}
		float(*const x)[2][64] = s_x[round & 1];
		if (q == 15) {
#pragma unroll
			for (int n = 0; n < 4; n++) {
				*reinterpret_cast<float4*>(&x[wave][0][16 * n + 4 * h]) =
					make_float4(rc[4 * n], rc[4 * n + 1], rc[4 * n + 2], rc[4 * n + 3]);
				*reinterpret_cast<float4*>(&x[wave][1][16 * n + 4 * h]) =
					make_float4(S_q[4 * n], S_q[4 * n + 1], S_q[4 * n + 2], S_q[4 * n + 3]);
			}
		}
		__syncthreads();
		{
			// (T_out, U) of this wave's group, and behind the next round, pixel = lane.
			const float T1 = T * x[0][0][lane], U1 = fmaf(T, x[0][1][lane], U);
			s_in[wave][0][lane] = wave ? T1 : T;
			s_in[wave][1][lane] = wave ? U1 : U;
			U = fmaf(T1, x[1][1][lane], U1);
			T = T1 * x[1][0][lane];
			hds_wave_fence();
		}
		// Geometry gradients in terms of s = raw dL/dalpha = op G dL/dalpha and d = pixel - mean: dopacity = sum s / op,
		// dmean = Q sum s d, dconic = -(sum s dx^2 / 2, sum s dx dy, sum s dy^2 / 2) (backward.cu:136-160).
		float m0 = 0.0f, mx = 0.0f, my = 0.0f, mxx = 0.0f, mxy = 0.0f, myy = 0.0f;
		uint32_t w_hi[8], w_lo[8];
		if (active != 0) {
#pragma unroll
			for (int n = 0; n < 4; n++) {
				const float4 tg = *reinterpret_cast<const float4*>(&s_in[wave][0][16 * n + 4 * h]);
				const float4 ug = *reinterpret_cast<const float4*>(&s_in[wave][1][16 * n + 4 * h]);
				const float dy = y0 + (float)(2 * n) - mean.y;
				float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f;
#pragma unroll
				for (int i = 0; i < 4; i++) {
					const int k = 4 * n + i;
					const float dL = element(tg, i) * A[k] - element(ug, i) * B[k];
					// A clamped alpha no longer depends on the gaussian (backward.cu:126-135).
					const float s = mul_legacy(raw[k] <= HDS_MAX_ALPHA ? raw[k] : 0.0f, dL);
					W[k] *= element(tg, i);
					const float dx = x0 + (float)i - mean.x, t = s * dx;
					s0 += s;
					s1 += t;
					s2 = fmaf(t, dx, s2);
				}
				const float t = s0 * dy;
				m0 += s0;
				mx += s1;
				my += t;
				mxx += s2;
				mxy = fmaf(s1, dy, mxy);
				myy = fmaf(t, dy, myy);
				hds_split_pair(W[4 * n], W[4 * n + 1], w_hi[2 * n], w_lo[2 * n]);
				hds_split_pair(W[4 * n + 2], W[4 * n + 3], w_hi[2 * n + 1], w_lo[2 * n + 1]);
			}
		} else {
#pragma unroll
			for (int k = 0; k < 8; k++) w_hi[k] = w_lo[k] = 0u;
		}
		// Contractions of the weights over the pixels.
		hds_bf16x8 a_hi[2], a_lo[2];
#pragma unroll
		for (int kp = 0; kp < 2; kp++) {
			a_hi[kp] = __builtin_bit_cast(hds_bf16x8, hds_u32x4{w_hi[4 * kp], w_hi[4 * kp + 1], w_hi[4 * kp + 2], w_hi[4 * kp + 3]});
			a_lo[kp] = __builtin_bit_cast(hds_bf16x8, hds_u32x4{w_lo[4 * kp], w_lo[4 * kp + 1], w_lo[4 * kp + 2], w_lo[4 * kp + 3]});
		}
		// The geometry part as three floats of lane (h, q) for gaussian q, elements h, 4 + h and 8 + h of the part: the
		// sums over the h lanes (and of the colour gradient's hi and lo rows) by swaps of lane halves and rows.
		float geo0, geo1, geo2;
		{
			hds_f32x4 C = {0.0f, 0.0f, 0.0f, 0.0f};  // rows 0-2: colour gradient from g's hi terms, 4-6: from its lo terms
			if (do_rgb) {
#pragma unroll
				for (int kp = 0; kp < 2; kp++) {
					C = __builtin_amdgcn_mfma_f32_16x16x32_bf16(g_col[kp], a_lo[kp], C, 0, 0, 0);
					C = __builtin_amdgcn_mfma_f32_16x16x32_bf16(g_col[kp], a_hi[kp], C, 0, 0, 0);
				}
			}
			const float g1 = conic.x * mx + conic.y * my, g2 = conic.y * mx + conic.z * my;
			geo0 = fold16(fold32(m0 / conic.w, g2), fold32(g1, -0.5f * mxx));
			geo1 = fold16(fold32(-mxy, C[0]), fold32(-0.5f * myy, C[1]));
			const float blue = fold16(C[2], 0.0f);
			const bool live = (active >> q) & 1u;
			geo0 = live ? geo0 : 0.0f;
			geo1 = live ? geo1 : 0.0f;
			geo2 = h == 1 ? hds_u2f((uint32_t)gid) : live ? blue : 0.0f;
		}
		hds_f32x4 D[2][kKc];  // rows: gaussian 4 h + i; columns: channel + (S / 4) u + kk
		if constexpr (WANT) {
#pragma unroll
			for (int u = 0; u < 2; u++)
#pragma unroll
				for (int kk = 0; kk < kKc; kk++) {
					D[u][kk] = hds_f32x4{0.0f, 0.0f, 0.0f, 0.0f};
					const char* src = tr_row + ((tr_chunk ^ (4 * kk + 2 * u)) << 4);
#pragma unroll
					for (int kp = 0; kp < 2; kp++) {
						const char* p = src + 32 * kp * kRowBytes;
						const hds_bf16x8 p_hi = join8(read_transposed(p), read_transposed(p + 16 * kRowBytes));
						const hds_bf16x8 p_lo = join8(read_transposed(p + kPlane), read_transposed(p + kPlane + 16 * kRowBytes));
						D[u][kk] = hds_mfma_split(a_hi[kp], a_lo[kp], p_hi, p_lo, D[u][kk]);
					}
				}
		}
		const int qq = (int)hds_opaque((uint32_t)q), hh = (int)hds_opaque((uint32_t)h);
		const int channel = c0 + (S / 2) * ((qq >> 2) & 1) + (S / 8) * (qq >> 3) + (S / 32) * (qq & 3);
		const bool valid = first + wave * kGroup + q < hits;
		if constexpr (REST) {
			const bool mine = valid && row >= a.rows.capacity;
			if (mine) {
				float* const out[4] = {a.grad_opacities + gid, a.grad_means2D + 2 * (int64_t)gid, a.grad_means2D + 2 * (int64_t)gid + 1,
									   a.grad_conics + 3 * (int64_t)gid};
				atomicAdd(hh == 0 ? out[0] : hh == 1 ? out[1] : hh == 2 ? out[2] : out[3], geo0);
				if (hh < 2) atomicAdd(a.grad_conics + 3 * (int64_t)gid + 1 + hh, geo1);
				if (do_rgb && hh >= 2) atomicAdd(a.grad_colors + 3 * (int64_t)gid + hh - 2, geo1);
				if (do_rgb && hh == 0) atomicAdd(a.grad_colors + 3 * (int64_t)gid + 2, geo2);
			}
			if constexpr (WANT) {
#pragma unroll
				for (int i = 0; i < 4; i++) {
					const int gid_of = __builtin_amdgcn_ds_bpermute(4 * (4 * h + i), mine ? gid : -1);
					if (gid_of < 0) continue;
					float* const to = a.grad_features + (int64_t)gid_of * a.channels + channel;
#pragma unroll
					for (int u = 0; u < 2; u++)
#pragma unroll
						for (int kk = 0; kk < kKc; kk++) atomicAdd(to + (S / 4) * u + kk, D[u][kk][i]);
				}
			}
		} else {
			const int slot = valid && row < a.rows.capacity ? row : (int)a.rows.capacity + (block & (kSpareRows - 1));
			float* const geo = a.rows.geo + ((int64_t)slot * a.rows.slices + slice) * kGeo + hh;
			geo[0] = geo0;
			geo[4] = geo1;
			geo[8] = geo2;
			if constexpr (WANT) {
#pragma unroll
				for (int i = 0; i < 4; i++) {
					const int slot_of = __builtin_amdgcn_ds_bpermute(4 * (4 * h + i), slot);
					float* const to = a.rows.features + (int64_t)slot_of * a.channels + channel;
#pragma unroll
					for (int u = 0; u < 2; u++) {
						float* p = to + (S / 4) * u;
						// Whole lines, read again only after the launch: past the caches, which keep the feature rows
						// (1.18M, C = 128: replay 0.734 -> 0.708 ms, sums 0.414 -> 0.393; non-temporal reads of the rows save
						// 0.010 more there and cost 0.003 of 0.037 at 200k, C = 32).
						if constexpr (kKc == 4)
							__builtin_nontemporal_store(hds_f32x4{D[u][0][i], D[u][1][i], D[u][2][i], D[u][3][i]}, reinterpret_cast<hds_f32x4*>(p));
						else if constexpr (kKc == 2)
							*reinterpret_cast<float2*>(p) = make_float2(D[u][0][i], D[u][1][i]);
						else
							*p = D[u][0][i];
					}
				}
			}
		}
	}
}

// Sums every gaussian's rows into its gradients, which hold zeros. A wave lists, in LDS, which of 64 consecutive
// gaussians have rows, and sums those, a row per group of C / 4 lanes (4 lanes for the geometry) and two
// gaussians' rows in flight per group; the work-groups past `gaussian_blocks` sum the gaussians of more
// than kLong rows in pieces of kLong rows, which hold the end of one such gaussian and the start of another
// at most. Bound by HBM: every row is read once.
struct SumGrid {
	int gaussian_blocks, piece_blocks;
	int feature_parts, quads_log2;                   // parts of a feature row of at most 64 float4s (a wave); the geometry last
	int64_t gaussians_per_pass;                      // by all waves of gaussian_blocks
};

__device__ inline float4 add4(float4 a, float4 b) { return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); }

struct RowBatch {
	float4 v[4];
};
// Rows [from, to), at most four, of an array of rows of `stride` float4s.
__device__ inline RowBatch load_rows(const float4* src, int stride, int64_t from, int64_t to) {
	RowBatch r;
#pragma unroll
	for (int k = 0; k < 4; k++) {
		r.v[k] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		if (from + k < to) r.v[k] = src[(from + k) * stride];
	}
	return r;
}
__device__ inline float4 sum_rows(const RowBatch& r) { return add4(add4(r.v[0], r.v[1]), add4(r.v[2], r.v[3])); }
// The whole sum, its first batch given.
__device__ inline float4 finish_rows(const RowBatch& first, const float4* src, int stride, int64_t from, int64_t to) {
	float4 sum = sum_rows(first);
	for (int64_t r = from + 4; r < to; r += 4) sum = add4(sum, sum_rows(load_rows(src, stride, r, to)));
	return sum;
}

// The same over the geometry parts of all slices (colours, floats 6-8, come from slice 0 alone).
__device__ inline float4 sum_geometry(const Rows& rows, int quad, int64_t from, int64_t to) {
	const int stride = rows.slices * kGeo / 4;
	float4 sum = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
	for (int s = 0; s < rows.slices; s++) {
		const float4* const src = reinterpret_cast<const float4*>(rows.geo + s * kGeo) + quad;
		const float4 v = finish_rows(load_rows(src, stride, from, to), src, stride, from, to);
		sum.x += s == 0 || quad < 2 ? v.x : 0.0f;
		sum.y += s == 0 || quad < 2 ? v.y : 0.0f;
		sum.z += s == 0 || quad < 1 ? v.z : 0.0f;
		sum.w += s == 0 || quad < 1 ? v.w : 0.0f;
	}
	return sum;
}

// put(output, value) for each float of quad `quad` of gaussian gid's geometry part.
template <typename Put>
__device__ inline void put_geometry(const BackwardArgs& a, int64_t gid, int quad, float4 v, Put put) {
	if (quad == 0) {
		put(a.grad_opacities + gid, v.x);
		put(a.grad_means2D + 2 * gid, v.y);
		put(a.grad_means2D + 2 * gid + 1, v.z);
		put(a.grad_conics + 3 * gid, v.w);
	} else if (quad == 1) {
		put(a.grad_conics + 3 * gid + 1, v.x);
		put(a.grad_conics + 3 * gid + 2, v.y);
		if (a.grad_image) {
			put(a.grad_colors + 3 * gid, v.z);
			put(a.grad_colors + 3 * gid + 1, v.w);
		}
	} else if (quad == 2 && a.grad_image) {
		put(a.grad_colors + 3 * gid + 2, v.x);
	}
}

__global__ __launch_bounds__(256) void backward_features_kernel(const BackwardArgs a, const SumGrid grid) {
	__shared__ int s_gid[4][64], s_base[4][64], s_count[4][64];
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const bool geometry = (int)blockIdx.y == grid.feature_parts;
	const int quads = 1 << grid.quads_log2;       // float4s of a row this wave covers, from quad0
	const int quad0 = (int)blockIdx.y << 6;
	const int quad = lane & (quads - 1), sub = lane >> grid.quads_log2, subs = 64 >> grid.quads_log2;
	const int stride = a.channels / 4;
	const float4* const features = reinterpret_cast<const float4*>(a.rows.features) + quad0 + quad;
	if ((int)blockIdx.x < grid.gaussian_blocks) {
		int* const gids = s_gid[wave];
		int* const bases = s_base[wave];
		int* const counts = s_count[wave];
		for (int64_t g0 = ((int64_t)blockIdx.x * 4 + wave) * 64; g0 < a.n; g0 += grid.gaussians_per_pass) {
			const int64_t g = g0 + lane;
			const int count = g < a.n ? a.rows.count[g] : 0, base = g < a.n ? a.rows.base[g] : 0;
			const bool some = count > 0 && summed_whole(a.rows, base, count);
			const uint64_t mask = hds_ballot(some);
			const int listed = __popcll(mask);
			hds_wave_fence();
			if (some) {
				const int to = hds_rank_below(mask);
				gids[to] = (int)g;
				bases[to] = base;
				counts[to] = count;
			}
			hds_wave_fence();
			if (!geometry) {
				for (int i = sub; i < listed; i += 2 * subs) {
					const int j = i + subs < listed ? i + subs : i;
					const int64_t from0 = bases[i], to0 = from0 + counts[i], from1 = bases[j], to1 = i == j ? from1 : from1 + counts[j];
					const RowBatch batch0 = load_rows(features, stride, from0, to0);
					const RowBatch batch1 = load_rows(features, stride, from1, to1);
					float4* const out = reinterpret_cast<float4*>(a.grad_features) + quad0 + quad;
					out[(int64_t)gids[i] * stride] = finish_rows(batch0, features, stride, from0, to0);
					if (i != j) out[(int64_t)gids[j] * stride] = finish_rows(batch1, features, stride, from1, to1);
				}
			} else if ((lane & 3) < 3) {
				for (int i = lane >> 2; i < listed; i += 16)
					put_geometry(a, gids[i], lane & 3, sum_geometry(a.rows, lane & 3, bases[i], (int64_t)bases[i] + counts[i]),
								 [](float* p, float v) { *p = v; });
			}
		}
		return;
	}
	const int64_t rows = (int64_t)min(*a.rows.total, (unsigned long long)a.rows.capacity);
	const int64_t pieces = (rows + kLong - 1) / kLong;
	for (int64_t piece = (int64_t)((int)blockIdx.x - grid.gaussian_blocks) * 4 + wave; piece < pieces;
		 piece += 4 * (int64_t)grid.piece_blocks) {
		const int64_t first = piece * kLong, last = min(first + kLong, rows);
		int64_t done = -1;
#pragma unroll
		for (int side = 0; side < 2; side++) {
			const int64_t row = side ? last - 1 : first;
			const int64_t gid = (int64_t)(int)hds_f2u(a.rows.geo[row * a.rows.slices * kGeo + kGeoGid]);
			const int count = a.rows.count[gid], base = a.rows.base[gid];
			if (gid == done || summed_whole(a.rows, base, count)) continue;
			done = gid;
			const int64_t from = max((int64_t)base, first), to = min((int64_t)base + count, last);
			if (!geometry) {
				// The lane groups take equal shares of the rows.
				const int64_t share = (to - from + subs - 1) / subs, f = from + sub * share, e = min(f + share, to);
				if (f < e) {
					const float4 v = finish_rows(load_rows(features, stride, f, e), features, stride, f, e);
					float* const out = a.grad_features + (gid * stride + quad0 + quad) * 4;
					atomicAdd(out + 0, v.x);
					atomicAdd(out + 1, v.y);
					atomicAdd(out + 2, v.z);
					atomicAdd(out + 3, v.w);
				}
			}
			if (geometry && lane < 3)
				put_geometry(a, gid, lane, sum_geometry(a.rows, lane, from, to), [](float* p, float v) { atomicAdd(p, v); });
		}
	}
}

// Zeroes up to five ranges of 4-byte words in one launch.
struct ZeroList {
	uint32_t* p[5];
	int64_t end[5];  // running sums of the range lengths
};

__global__ __launch_bounds__(256) void zero_words_kernel(const ZeroList z) {
	const int64_t stride = (int64_t)gridDim.x * 256;
	for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < z.end[4]; i += stride) {
		int64_t begin = 0;
#pragma unroll
		for (int k = 0; k < 5; k++) {
			if (i >= begin && i < z.end[k]) z.p[k][i - begin] = 0u;
			begin = z.end[k];
		}
	}
}

template <int S, bool RGB, bool WANT>
int launch_geometry(const BackwardArgs& a, int slices, bool rest, hipStream_t s) {
	const dim3 grid(hds_xcd_block_grid(a.tiles_x, a.num_tiles), (unsigned)slices);
	HdsKernelTimer timer("backward_geometry_kernel", s);
	backward_geometry_kernel<S, RGB, WANT, false><<<grid, kThreads, 0, s>>>(a);
	if (rest) backward_geometry_kernel<S, RGB, WANT, true><<<grid, kThreads, 0, s>>>(a);
	timer.stop();
	return hds_check_launch("backward_geometry", s);
}

template <int S>
int launch_geometry(const BackwardArgs& a, int slices, bool rgb, bool rest, hipStream_t s) {
	if (a.grad_features)
		return rgb ? launch_geometry<S, true, true>(a, slices, rest, s) : launch_geometry<S, false, true>(a, slices, rest, s);
	return rgb ? launch_geometry<S, true, false>(a, slices, rest, s) : launch_geometry<S, false, false>(a, slices, rest, s);
}

// Layout of the workspace; every part starts on a 256-byte boundary.
struct Layout {
	size_t gid, idx, ordinal, hits, count, base, total, features, geo, bytes;
};

Layout layout_of(int64_t n, int width, int height, int64_t num_pairs, int64_t row_capacity, int row_channels, int slices) {
	Layout l{};
	size_t at = 0;
	auto take = [&](int64_t words) {
		const size_t here = at;
		at += ((size_t)words * 4 + 255) & ~(size_t)255;
		return here;
	};
	const int64_t tiles = (int64_t)((width + HDS_TILE - 1) / HDS_TILE) * ((height + HDS_TILE - 1) / HDS_TILE);
	l.gid = take(4 * num_pairs);
	l.idx = take(4 * num_pairs);
	l.ordinal = take(4 * num_pairs);
	l.hits = take(4 * tiles);
	l.count = take(n);
	l.total = take(2);  // right after count: both are cleared together
	l.base = take(n);
	l.features = take((row_capacity + kSpareRows) * row_channels);
	l.geo = take((row_capacity + kSpareRows) * slices * kGeo);
	l.bytes = at;
	return l;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
int log2_of(int v) { return 31 - __builtin_clz((unsigned)v); }

}  // namespace

#define HDS_BACKWARD_ARGS                                                                                     \
	int64_t n, int width, int height, int channels, int slice_width, const int32_t *tile_ranges,               \
		const int32_t *values_sorted, int64_t num_pairs, const float *means2D, const float *conic4,             \
		const float *color_opacity4, const float *background, const float *final_T, const int32_t *n_contrib,   \
		const float *grad_image, const float *features, const float *grad_feature_image, float *grad_means2D,   \
		float *grad_conics, float *grad_colors, float *grad_opacities, float *grad_features

extern "C" size_t hds_render_backward_workspace_bytes(int64_t n, int width, int height, int channels, int slice_width,
													  int want_features, int64_t num_pairs, int64_t row_capacity) {
	if (n < 0 || width <= 0 || height <= 0 || channels < 0 || (channels > 0 && slice_width <= 0) || num_pairs < 0 ||
		row_capacity < 0)
		return 0;
	return layout_of(n, width, height, num_pairs, row_capacity, want_features ? channels : 0,
					 channels > 0 ? channels / slice_width : 1).bytes;
}

extern "C" int hds_render_backward_rows(HDS_BACKWARD_ARGS, int zeroed, const uint8_t* contributes, int64_t row_capacity,
										void* workspace, size_t workspace_bytes, hds_stream_t stream) {
	HDS_REQUIRE(width > 0 && height > 0, "render_backward: image size %dx%d must be positive", width, height);
	HDS_REQUIRE(n >= 0, "render_backward: negative gaussian count");
	HDS_REQUIRE(tile_ranges && final_T && n_contrib && (n == 0 || (grad_means2D && grad_conics && grad_opacities)),
				"render_backward: null pointer argument");
	const bool rgb = grad_image != nullptr;
	const bool feats = features != nullptr;
	HDS_REQUIRE(rgb || feats, "render_backward: neither grad_image nor features given");
	HDS_REQUIRE(!rgb || n == 0 || (grad_colors && background && color_opacity4), "render_backward: RGB term needs colors / background");
	if (feats) {
		HDS_REQUIRE(channels == 32 || channels == 64 || channels == 128 || channels == 256 || channels == 512,
					"features must have 32, 64, 128, 256 or 512 channels, got %d", channels);
		HDS_REQUIRE(grad_feature_image, "render_backward: features given without grad_feature_image");
		HDS_REQUIRE((slice_width == 32 || slice_width == 64 || slice_width == 128) && slice_width <= channels &&
						channels % slice_width == 0,
					"no feature backward for %d channels in slices of %d", channels, slice_width);
		HDS_REQUIRE(aligned16(features) && aligned16(grad_feature_image) && aligned16(grad_features),
					"render_backward: features must be 16-byte aligned");
	}
	HDS_REQUIRE(aligned16(conic4) && (!color_opacity4 || aligned16(color_opacity4)), "render_backward: misaligned conic4");
	HDS_REQUIRE(row_capacity >= 0 && row_capacity <= kMaxRows - kSpareRows, "render_backward: row capacity outside 0..2^30");
	const bool want = feats && grad_features;
	const int c = feats ? channels : 0;
	hipStream_t s = (hipStream_t)stream;
	const bool run = n > 0 && num_pairs > 0;
	const int slices = feats ? channels / slice_width : 1;
	const Layout l = layout_of(n, width, height, num_pairs, row_capacity, want ? c : 0, slices);
	HDS_REQUIRE(!run || (workspace && aligned16(workspace) && workspace_bytes >= l.bytes),
				"render_backward: workspace missing, misaligned or too small");
	char* const ws = reinterpret_cast<char*>(workspace);

	ZeroList z{};
	int64_t words = 0;
	auto zero = [&](int k, void* p, int64_t count) {
		z.p[k] = reinterpret_cast<uint32_t*>(p);
		words += p ? count : 0;
		z.end[k] = words;
	};
	zero(0, zeroed ? nullptr : grad_means2D, 2 * n);
	zero(1, zeroed ? nullptr : grad_conics, 3 * n);
	zero(2, zeroed ? nullptr : grad_opacities, n);
	zero(3, zeroed || !rgb ? nullptr : grad_colors, 3 * n);
	zero(4, run ? ws + l.count : nullptr, (int64_t)(l.total - l.count) / 4 + 2);
	if (words > 0) {
		HdsKernelTimer timer("zero_kernel", s);
		zero_words_kernel<<<(unsigned)std::min<int64_t>(hds_blocks(words, 256), 4096), 256, 0, s>>>(z);
		timer.stop();
		HDS_LAUNCH_CHECK("zero_gradients", s);
	}
	if (want && !zeroed && n > 0) {
		const int st = hds_zero_async(grad_features, (int64_t)channels * n, 0, stream);
		if (st != HDS_OK) return st;
	}
	if (!run) return HDS_OK;

	const int tiles_x = (width + HDS_TILE - 1) / HDS_TILE, tiles_y = (height + HDS_TILE - 1) / HDS_TILE;
	const int num_tiles = tiles_x * tiles_y;
	auto ints = [&](size_t at) { return reinterpret_cast<int*>(ws + at); };
	BackwardArgs a{};
	a.width = width;
	a.height = height;
	a.tiles_x = tiles_x;
	a.channels = c;
	a.num_tiles = num_tiles;
	a.n = n;
	a.ranges = reinterpret_cast<const int2*>(tile_ranges);
	a.values = values_sorted;
	a.means2D = reinterpret_cast<const float2*>(means2D);
	a.conic4 = reinterpret_cast<const float4*>(conic4);
	a.color_op4 = reinterpret_cast<const float4*>(color_opacity4);
	a.background = background;
	a.final_T = final_T;
	a.n_contrib = n_contrib;
	a.contributes = contributes;
	a.grad_image = grad_image;
	a.features = features;
	a.grad_feature_image = grad_feature_image;
	a.grad_means2D = grad_means2D;
	a.grad_conics = grad_conics;
	a.grad_colors = grad_colors;
	a.grad_opacities = grad_opacities;
	a.grad_features = want ? grad_features : nullptr;
	a.lists = BlockLists{ints(l.gid), ints(l.idx), ints(l.ordinal), ints(l.hits)};
	a.rows = Rows{reinterpret_cast<float*>(ws + l.features),
				  reinterpret_cast<float*>(ws + l.geo),
				  ints(l.count),
				  ints(l.base),
				  reinterpret_cast<unsigned long long*>(ws + l.total),
				  row_capacity,
				  slices};
	{
		HdsKernelTimer timer("backward_lists_kernel", s);
		if (contributes)
			backward_lists_kernel<true><<<(unsigned)num_tiles, kListThreads, 0, s>>>(a);
		else
			backward_lists_kernel<false><<<(unsigned)num_tiles, kListThreads, 0, s>>>(a);
		timer.stop();
		HDS_LAUNCH_CHECK("backward_lists", s);
	}
	{
		HdsKernelTimer timer("backward_base_kernel", s);
		backward_base_kernel<<<hds_blocks(n, kBaseThreads * kBaseItems), kBaseThreads, 0, s>>>(a);
		timer.stop();
		HDS_LAUNCH_CHECK("backward_base", s);
	}
	// A pair has at most four rows, one per block of its tile.
	const bool rest = row_capacity < 4 * num_pairs;
	int st;
	if (!feats) {
		st = launch_geometry<0, true, false>(a, 1, rest, s);
	} else {
		switch (slice_width) {
			case 32: st = launch_geometry<32>(a, slices, rgb, rest, s); break;
			case 64: st = launch_geometry<64>(a, slices, rgb, rest, s); break;
			default: st = launch_geometry<128>(a, slices, rgb, rest, s); break;
		}
	}
	if (st != HDS_OK) return st;
	// 64 gaussians per wave; the pieces of rows by enough work-groups to fill the chip, each looping.
	SumGrid grid{};
	grid.quads_log2 = want ? std::min(log2_of(channels / 4), 6) : 0;
	grid.gaussian_blocks = (int)std::min<int64_t>(hds_blocks(n, 256), 1 << 20);
	grid.gaussians_per_pass = (int64_t)grid.gaussian_blocks * 256;
	grid.piece_blocks = (int)std::min<int64_t>(hds_blocks(row_capacity, 4 * kLong), 1024);
	grid.feature_parts = want ? (channels / 4 + 63) / 64 : 0;
	const dim3 blocks((unsigned)(grid.gaussian_blocks + grid.piece_blocks), (unsigned)grid.feature_parts + 1u);
	HdsKernelTimer timer("backward_features_kernel", s);
	backward_features_kernel<<<blocks, 256, 0, s>>>(a, grid);
	timer.stop();
	return hds_check_launch("backward_features", s);
}
