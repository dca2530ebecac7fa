// Front-to-back blend of RGB and C feature channels in one walk.
//
// Work-group = one wave = one 8x8 block of a tile (and one slice of S <= 128 channels), lane l the pixel (l & 7,
// l >> 3) of it. The wave tests 64 entries of the tile's sorted list at a time against its block, keeps those that
// can reach it, in order, and takes them 16 at a time, updating T, RGB and n_contrib per lane exactly as
// render_gaussians does (forward.cu:181-225): alpha = min(0.99, op * exp(-m/2)), skip below 1/255, stop before T
// would drop below 1e-4, n_contrib = 1-based list index of the last blended gaussian.
//
// Features: the 16 hits are, in list order, the K dimension of
//   out[c][px] += sum_k F[k][c] * W[k][px],
// one v_mfma_f32_32x32x16_bf16 per 32 channels x 32 pixels, both operands in split-bf16 (3 MFMAs
// per tile, ~2^-16 relative error; CDNA4 has no TF32). Each lane keeps its own pixel's 16 weights
// w = alpha * T (0 where it did not blend) in registers as packed bf16 pairs; one
// v_permlane32_swap per register pair then forms the B operands of the two 32-pixel halves, so the
// weights never touch LDS. The 16-hit groups depend on geometry only, so each output channel sees the same
// operation sequence whatever C or the slicing is: channels are bitwise independent and RGB is bitwise equal with or
// without features (the properties the reference's tests/test_properties.py pins). The accumulators take S registers
// per lane (ordinary VGPRs: the compiler assigns no AGPRs here), so the 128-channel slice runs two waves per
// SIMD, the 64-channel slice three, the 32-channel slice four.
//
// Bound by VALU issue (about 35 operations per hit and 230 per group of 16 for the split operands) and, where the
// feature image or the cleared range is large, by stores. Against one work-group per tile, whose four waves shared a
// staged batch and met at a barrier after each: no wave waits for another, groups run on over batches
// (145k full ones instead of 226k at 1.18M gaussians, 979x546), rows no block can see are not copied, and a wave's
// slot is free when its block is done. Alphas are evaluated four at a time before the chain through T, which has
// no branch but one per four hits for pixels that stop there. The image leaves in whole lines, non-temporal.
// At 979x546: C = 32, 200k gaussians, 0.100 -> 0.070 ms; 1.18M: RGB 0.230 -> 0.187, C = 128 0.62 -> 0.49; at 4M,
// 1920x1080, C = 256: 1.61 -> 1.37.
#include <cstdlib>

#include "hds_internal.h"
#include "hds_rasterizer.h"
#include "hds_stage.h"

namespace {

constexpr int kBatch = 64;  // entries of the tile's list tested together, one per lane
constexpr int kGroup = 16;  // K of one MFMA: hits per group
constexpr int kHits = kGroup + kBatch;  // most hits pending, and more than a group reads past the last
constexpr int kIlp = 4;     // hits whose alpha is evaluated together
constexpr float kDone = 2.0f;  // alpha that none reaches

// Waits for this wave's outstanding vector-memory operations, LDS copies included.
__device__ inline void wait_vmem() {
	__builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0), which the compiler's own count knows of
	asm volatile("" ::: "memory");
}

struct RenderArgs {
	int width, height, tiles_x, channels, num_tiles;
	const int2* ranges;
	const int* values;
	const float2* means2D;
	const float4* conic4;
	const float4* color_op4;
	const float* background;
	const float* features;
	float* image;
	float* final_T;
	int* n_contrib;
	float* feature_image;
	float4* clear;   // hds_render_clear's range (clear4 16-byte words), or null
	int64_t clear4;
	uint8_t* contributes;  // hds_render_contributes' marks, or null
};

// Feature rows of a group in LDS, S floats each, in the order of their copy: wave instruction i brings 1 KB, in its
// lower half rows i * kRowsPerHalf .. of hits 0-7 and in its upper half the same rows of hits 8-15.
template <int S>
struct RowLayout {
	static constexpr int kLanes = S / 4;                   // lanes (16 bytes each) per row
	static constexpr int kRowsPerHalf = 32 / kLanes;       // rows per half instruction
	static constexpr int kOps = (kGroup / 2) / kRowsPerHalf;
	// Float offset of row 8 h + j.
	static __device__ constexpr int at(int h, int j) { return (j / kRowsPerHalf) * 256 + h * 128 + (j % kRowsPerHalf) * S; }
};

// acc[m][cb] += F^T W for one group. w_hi / w_lo hold this lane's pixel's packed weights for
// positions (2i, 2i+1); after the swaps, words 0-3 are the B operand of pixels 0-31 and words 4-7
// that of pixels 32-63. A = features: lane = (channel lane % 32, positions 8 (lane / 32) + 0..7),
// read as raw fp32 from the staged rows and split here.
template <int S>
__device__ inline void flush_group(hds_f32x16 (&acc)[2][S / 32], uint32_t (&w_hi)[8], uint32_t (&w_lo)[8],
								   const float* feat, int lane) {
#pragma unroll
	for (int i = 0; i < 4; i++) {
		const auto h = __builtin_amdgcn_permlane32_swap(w_hi[i], w_hi[4 + i], false, false);
		w_hi[i] = h[0];
		w_hi[4 + i] = h[1];
		const auto l = __builtin_amdgcn_permlane32_swap(w_lo[i], w_lo[4 + i], false, false);
		w_lo[i] = l[0];
		w_lo[4 + i] = l[1];
	}
	hds_bf16x8 b_hi[2], b_lo[2];
#pragma unroll
	for (int m = 0; m < 2; m++) {
		b_hi[m] = __builtin_bit_cast(hds_bf16x8, hds_u32x4{w_hi[4 * m], w_hi[4 * m + 1], w_hi[4 * m + 2], w_hi[4 * m + 3]});
		b_lo[m] = __builtin_bit_cast(hds_bf16x8, hds_u32x4{w_lo[4 * m], w_lo[4 * m + 1], w_lo[4 * m + 2], w_lo[4 * m + 3]});
	}
	const float* const mine = feat + RowLayout<S>::at(lane >> 5, 0) + (lane & 31);
#pragma unroll
	for (int cb = 0; cb < S / 32; cb++) {
		float v[8];
#pragma unroll
		for (int j = 0; j < 8; j++) v[j] = mine[RowLayout<S>::at(0, j) + 32 * cb];
		hds_bf16x8 a_hi, a_lo;
		hds_split8(v, a_hi, a_lo);
#pragma unroll
		for (int m = 0; m < 2; m++) acc[m][cb] = hds_mfma32_split(a_hi, a_lo, b_hi[m], b_lo[m], acc[m][cb]);
		asm volatile("" : "+v"(acc[0][cb]), "+v"(acc[1][cb]));  // summed here, not on either side of the loop's exit
	}
}

// Stages group hits first .. first + rows - 1 of the list: feature rows into feat, colours into rgb. Rows past the
// last hit (only a walk's last group has any) become zeros.
template <int S, bool RGB>
__device__ inline void stage_group(float* feat, float* rgb, const RenderArgs& a, const int* gids, int first, int rows, int c0) {
	const int lane = (int)hds_opaque(threadIdx.x);  // what follows from it is worked out here, not held through the walk
	if (rows < kGroup) {
		// The buffer is idle: zeros first, then what there is.
		if constexpr (S > 0)
			for (int i = lane; i < kGroup * S / 4; i += 64) reinterpret_cast<hds_f32x4*>(feat)[i] = hds_f32x4{};
		if constexpr (RGB)
			if (lane < 3 * kGroup) rgb[lane] = 0.0f;
		__builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
		asm volatile("" ::: "memory");
	}
	if constexpr (S > 0) {
		using L = RowLayout<S>;
		const int row0 = 8 * (lane >> 5) + (lane & 31) / L::kLanes;
		const float* const src = a.features + c0 + 4 * (lane % L::kLanes);
#pragma unroll
		for (int i = 0; i < L::kOps; i++) {
			const int row = row0 + i * L::kRowsPerHalf;
			if (row < rows)
				__builtin_amdgcn_global_load_lds(src + (size_t)gids[first + row] * a.channels, (hds_lds_void*)(feat + 256 * i), 16, 0, 0);
		}
	}
	if constexpr (RGB) {
		if (lane < rows) {
			const float4* const color = a.color_op4 + gids[first + lane];
			__builtin_amdgcn_global_load_lds(&color->x, (hds_lds_void*)(rgb), 4, 0, 0);
			__builtin_amdgcn_global_load_lds(&color->y, (hds_lds_void*)(rgb + kGroup), 4, 0, 0);
			__builtin_amdgcn_global_load_lds(&color->z, (hds_lds_void*)(rgb + 2 * kGroup), 4, 0, 0);
		}
	}
}

// Per-lane state of the walk. A gaussian blends where its alpha reaches `reach`: 1/255 until the pixel is done (or
// from the start outside the image), 2 afterwards.
struct Pixel {
	float T;
	float reach;
	int n_contrib;
	float r, g, b;
};

// hds_render_clear: every work-group zeroes a share of the caller's range before its walk. The walks leave most of the
// HBM bandwidth unused, so the stores drain beside those of other waves instead of in a fill launch of their own;
// non-temporal, so that the zeros do not push feature rows out of L2. (After the walk: 1.43 ms instead of 1.37 at 4M
// gaussians, C = 256; a piece per group: 1.72 instead of 1.65 before the image's stores became whole lines.)
__device__ inline void clear_share(const RenderArgs& a, int lane) {
	constexpr int kPiece = 256;  // 4 KB dealt out in turn
	const int64_t stride = (int64_t)gridDim.x * gridDim.y * kPiece;
	hds_f32x4* const clear = reinterpret_cast<hds_f32x4*>(a.clear);
	for (int64_t e = ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * kPiece + lane; e < a.clear4; e += stride) {
#pragma unroll
		for (int k = 0; k < kPiece; k += 64)
			if (e + k < a.clear4) __builtin_nontemporal_store(hds_f32x4{}, clear + e + k);
	}
}

// A wave is a work-group of its own: nothing in it waits for another. Per group of 16 hits it tests batches of entries
// until so many are pending (a batch's records are read while the one before is worked on), issues the copies
// of the group's feature rows and colours, evaluates the alphas and the chain through T while those are on their way,
// and then adds the colours and features.
template <int S, bool RGB>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(S >= 128 ? 2 : S == 64 ? 3 : 4))) void render_forward_kernel(
	const RenderArgs a) {
	constexpr int kNcb = S > 0 ? S / 32 : 1;

	// Hits in list order: mean and conic, and the gaussian and its place in the tile's list.
	__shared__ hds_f32x4 s_mean_ab[kHits];
	__shared__ hds_f32x2 s_c_op[kHits];
	__shared__ int s_gid[kHits], s_idx[kHits];
	// Feature rows and colours (16 reds, greens, blues) of the group; at the end, 32 channels of 32 pixels of the image.
	constexpr int kChunk = 32 * 32;
	constexpr int kFeat = S == 0 ? 4 : kGroup * S < kChunk ? kChunk : kGroup * S;
	__shared__ __attribute__((aligned(16))) float s_feat[kFeat];
	__shared__ __attribute__((aligned(16))) float s_rgb[RGB ? 3 * kGroup : 4];

	const int block = hds_xcd_block(blockIdx.x, a.tiles_x, a.num_tiles);
	const int lane = threadIdx.x;
	clear_share(a, lane);
	if (block < 0) return;
	const int slice = blockIdx.y;
	const int tile = block >> 2;
	const int wx0 = (tile % a.tiles_x) * HDS_TILE + (block & 1) * 8, wy0 = (tile / a.tiles_x) * HDS_TILE + (block >> 1 & 1) * 8;
	const int px = wx0 + (lane & 7), py = wy0 + (lane >> 3);
	const bool inside = px < a.width && py < a.height;
	const float fx = (float)px + 0.5f, fy = (float)py + 0.5f;
	const float rx0 = (float)wx0 + 0.5f, rx1 = (float)wx0 + 7.5f;
	const float ry0 = (float)wy0 + 0.5f, ry1 = (float)wy0 + 7.5f;
	const int2 range = a.ranges[tile];
	const int c0 = slice * S;

	Pixel st{1.0f, inside ? HDS_MIN_ALPHA : kDone, 0, 0.0f, 0.0f, 0.0f};
	hds_f32x16 acc[2][kNcb];
#pragma unroll
	for (int m = 0; m < 2; m++)
#pragma unroll
		for (int c = 0; c < kNcb; c++) acc[m][c] = hds_f32x16{};

	const int num = hds_ballot(inside) != 0 ? range.y - range.x : 0;
	// This block's marks, one byte per list entry: 0 from the test of an entry that cannot reach the block, the others
	// from the group they are blended in.
	uint8_t* const marks = a.contributes && slice == 0 ? a.contributes + 4 * (int64_t)range.x + (int64_t)(block & 3) * num : nullptr;
	if (num > 0) {
		const int* const values = a.values + range.x;
		// The next batch (entries pos .. pos + 63, its records in registers) and the gids of the one after.
		int pos = 0, gid = 0, gid_after = 0;
		float2 mean = make_float2(0.0f, 0.0f);
		float4 conic = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
		auto read_records = [&]() {
			if (pos + lane < num) {
				mean = a.means2D[gid];
				conic = a.conic4[gid];
			}
			if (pos + kBatch + lane < num) gid_after = values[pos + kBatch + lane];
		};
		if (lane < num) gid = values[lane];
		read_records();

		int head = 0, count = 0;  // pending hits: list positions head .. head + count - 1
		// Tests batches until `want` hits are pending or the list ends.
		auto top_up = [&](int want) {
			const int lane = (int)hds_opaque(threadIdx.x);
			while (count < want && pos < num) {
				const bool hit = pos + lane < num && hds_block_reach(mean, conic, rx0, rx1, ry0, ry1);
				const uint64_t hits = hds_ballot(hit);
				if (marks && !hit && pos + lane < num) marks[pos + lane] = 0;
				if (hits != 0) {
					if (head > 0) {
						// At most 31 hits are left: to the front.
						if (lane < count) {
							const hds_f32x4 m = s_mean_ab[head + lane];
							const hds_f32x2 c = s_c_op[head + lane];
							const int g = s_gid[head + lane], i = s_idx[head + lane];
							s_mean_ab[lane] = m;
							s_c_op[lane] = c;
							s_gid[lane] = g;
							s_idx[lane] = i;
						}
						hds_wave_fence();
						head = 0;
					}
					if (hit) {
						const int at = count + hds_rank_below(hits);
						s_mean_ab[at] = hds_f32x4{mean.x, mean.y, conic.x, conic.y};
						s_c_op[at] = hds_f32x2{conic.z, conic.w};
						s_gid[at] = gid;
						s_idx[at] = pos + lane;
					}
					count += __builtin_popcountll(hits);
				}
				pos += kBatch;
				gid = gid_after;
				read_records();
			}
			hds_wave_fence();
		};
		for (;;) {
			top_up(kGroup);
			const int n = min(count, kGroup), first = head;
			if (n == 0) break;
			head += n;
			count -= n;
			stage_group<S, RGB>(s_feat, s_rgb, a, s_gid, first, n, c0);
			float w[kGroup];
			int last = -1;
			uint32_t contribute = 0;  // bit q: hit q blends into some pixel
#pragma unroll
			for (int q0 = 0; q0 < kGroup; q0 += kIlp) {
				// The records of four hits, then their four alphas, then the chain through T: left alone, the
				// compiler takes the hits one by one, each behind its own LDS read and the alpha before it.
				hds_f32x4 ma[kIlp];
				hds_f32x2 co[kIlp];
				float alpha[kIlp];
#pragma unroll
				for (int u = 0; u < kIlp; u++) {
					ma[u] = s_mean_ab[first + q0 + u];
					co[u] = s_c_op[first + q0 + u];
				}
				asm volatile("" : "+v"(ma[0]), "+v"(ma[1]), "+v"(ma[2]), "+v"(ma[3]), "+v"(co[0]), "+v"(co[1]), "+v"(co[2]),
							 "+v"(co[3]));
#pragma unroll
				for (int u = 0; u < kIlp; u++) {
					float G, dx, dy;
					alpha[u] = fminf(HDS_MAX_ALPHA, hds_raw_alpha(fx, fy, make_float2(ma[u].x, ma[u].y),
																  make_float4(ma[u].z, ma[u].w, co[u].x, co[u].y), G, dx, dy));
				}
				asm volatile("" : "+v"(alpha[0]), "+v"(alpha[1]), "+v"(alpha[2]), "+v"(alpha[3]));
				bool blends[kIlp];
				float T[kIlp + 1];
				T[0] = st.T;
#pragma unroll
				for (int u = 0; u < kIlp; u++) {
					blends[u] = q0 + u < n && alpha[u] >= st.reach;
					alpha[u] = blends[u] ? alpha[u] : 0.0f;
					w[q0 + u] = alpha[u] * T[u];
					T[u + 1] = T[u] * (1.0f - alpha[u]);
				}
				if (hds_ballot(T[kIlp] < HDS_MIN_TRANSMITTANCE) != 0) {
					// Some pixel stops here, before the gaussian that takes its T below the limit.
					st.reach = T[kIlp] < HDS_MIN_TRANSMITTANCE ? kDone : st.reach;
					float kept = T[0];
#pragma unroll
					for (int u = 0; u < kIlp; u++) {
						const bool below = T[u + 1] < HDS_MIN_TRANSMITTANCE;
						blends[u] = blends[u] && !below;
						w[q0 + u] = below ? 0.0f : w[q0 + u];
						kept = below ? kept : T[u + 1];
					}
					T[kIlp] = kept;
				}
				st.T = T[kIlp];
#pragma unroll
				for (int u = 0; u < kIlp; u++) {
					last = blends[u] ? q0 + u : last;
					contribute |= hds_ballot(blends[u]) != 0 ? 1u << (q0 + u) : 0u;
				}
			}
			if (last >= 0) st.n_contrib = s_idx[first + last] + 1;
			wait_vmem();
			if (marks && lane < n) marks[s_idx[first + lane]] = (uint8_t)(contribute >> lane & 1u);
			if constexpr (RGB) {
				// fmaf as the oracle does: the RGB image is bit-exact. A colour that is not finite would turn the 0 of
				// a gaussian that does not blend into NaN.
				const float c = s_rgb[min(lane, 3 * kGroup - 1)];
				const bool any_odd = hds_ballot(!(c - c == 0.0f)) != 0;
#pragma unroll
				for (int q0 = 0; q0 < kGroup; q0 += 4) {
					hds_f32x4 color[3];
#pragma unroll
					for (int k = 0; k < 3; k++) color[k] = *reinterpret_cast<const hds_f32x4*>(s_rgb + k * kGroup + q0);
					if (__builtin_expect(any_odd, 0)) {
#pragma unroll
						for (int u = 0; u < 4; u++) {
							if (!(w[q0 + u] > 0.0f)) continue;
							st.r = fmaf(w[q0 + u], color[0][u], st.r);
							st.g = fmaf(w[q0 + u], color[1][u], st.g);
							st.b = fmaf(w[q0 + u], color[2][u], st.b);
						}
						asm volatile("" : "+v"(st.r));  // a branch, not three selects per hit
					} else {
#pragma unroll
						for (int u = 0; u < 4; u++) {
							st.r = fmaf(w[q0 + u], color[0][u], st.r);
							st.g = fmaf(w[q0 + u], color[1][u], st.g);
							st.b = fmaf(w[q0 + u], color[2][u], st.b);
						}
					}
				}
			}
			if constexpr (S > 0) {
				uint32_t w_hi[8], w_lo[8];
#pragma unroll
				for (int i = 0; i < 8; i++) hds_split_pair(w[2 * i], w[2 * i + 1], w_hi[i], w_lo[i]);
				flush_group<S>(acc, w_hi, w_lo, s_feat, lane);
			}
			if (hds_ballot(st.reach < kDone) == 0) break;
		}
	}

	if (inside && slice == 0) {
		const int64_t pix = (int64_t)py * a.width + px;
		if constexpr (RGB) {
			a.image[pix * 3 + 0] = fmaf(st.T, a.background[0], st.r);
			a.image[pix * 3 + 1] = fmaf(st.T, a.background[1], st.g);
			a.image[pix * 3 + 2] = fmaf(st.T, a.background[2], st.b);
		}
		a.final_T[pix] = st.T;
		a.n_contrib[pix] = st.n_contrib;
	}
	if constexpr (S > 0) {
		// D of a 32x32 tile: lane holds pixel 32m + lane % 32 and, for each group g of four accumulators, channels
		// 8g + 4 (lane / 32) + 0..3. By way of LDS, 32 channels of 32 pixels at a time, to whole lines: eight lanes
		// store a pixel's 128 bytes. The 16-byte pieces of a pixel are permuted by its number, against bank conflicts.
		hds_f32x4* const piece = reinterpret_cast<hds_f32x4*>(s_feat);
#pragma unroll
		for (int c = 0; c < kNcb; c++)
#pragma unroll
			for (int m = 0; m < 2; m++) {
				const hds_f32x16 v = acc[m][c];
				hds_f32x4* const half = piece + (kFeat >= 2 * kChunk ? kChunk / 4 * m : 0);
				hds_wave_fence();
#pragma unroll
				for (int g = 0; g < 4; g++)
					half[8 * (lane & 31) + ((2 * g + (lane >> 5)) ^ (lane & 7))] = hds_f32x4{v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]};
				hds_wave_fence();
#pragma unroll
				for (int i = 0; i < 4; i++) {
					const int p = 8 * i + (lane >> 3);
					const int x = wx0 + (p & 7), y = wy0 + 4 * m + (p >> 3);
					const hds_f32x4 out = half[8 * p + ((lane & 7) ^ (p & 7))];
					if (x < a.width && y < a.height)
						__builtin_nontemporal_store(out, reinterpret_cast<hds_f32x4*>(a.feature_image + ((int64_t)y * a.width + x) * a.channels +
																					  c0 + 32 * c) + (lane & 7));
				}
			}
	}
}

template <int S, bool RGB>
int launch(const RenderArgs& a, int num_tiles, int slices, hipStream_t s) {
	HdsKernelTimer timer1("render_forward_kernel", s);
	render_forward_kernel<S, RGB><<<dim3(hds_xcd_block_grid(a.tiles_x, num_tiles), (unsigned)slices), 64, 0, s>>>(a);
	timer1.stop();
	return hds_check_launch(RGB ? (S > 0 ? "render_rgb_features" : "render_rgb") : "render_features", s);
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

int render(int width, int height, int channels, const int32_t* tile_ranges, const int32_t* values_sorted,
		   int64_t num_pairs, const float* means2D, const float* conic4, const float* color_opacity4,
		   const float* background, const float* features, float* image, float* final_T, int32_t* n_contrib,
		   float* feature_image, float* clear, int64_t clear_count, uint8_t* contributes, hds_stream_t stream) {
	HDS_REQUIRE(clear_count >= 0, "render_clear: negative clear count");
	HDS_REQUIRE(clear_count == 0 || (clear && aligned16(clear) && clear_count % 4 == 0),
				"render_clear: needs a 16-byte aligned range of a multiple of 4 floats");
	HDS_REQUIRE(width > 0 && height > 0, "render: image size %dx%d must be positive", width, height);
	HDS_REQUIRE(tile_ranges && final_T && n_contrib, "render: null tile_ranges / final_T / n_contrib");
	const bool rgb = image != nullptr;
	const bool feats = features != nullptr;
	if (feats)
		HDS_REQUIRE(channels == 32 || channels == 64 || channels == 128 || channels == 256 || channels == 512,
					"features must have 32, 64, 128, 256 or 512 channels, got %d", channels);
	HDS_REQUIRE(!feats || feature_image, "render: features given without feature_image");
	HDS_REQUIRE(!rgb || (background && (color_opacity4 || num_pairs == 0)), "render: image requested without background / colors");
	HDS_REQUIRE(num_pairs == 0 || (values_sorted && means2D && conic4), "render: null gaussian arguments");
	HDS_REQUIRE(aligned16(conic4) && (!color_opacity4 || aligned16(color_opacity4)) && (!features || aligned16(features)) &&
					(!feature_image || aligned16(feature_image)) && (reinterpret_cast<uintptr_t>(means2D) & 7u) == 0 &&
					(reinterpret_cast<uintptr_t>(tile_ranges) & 7u) == 0,
				"render: misaligned buffer (conic4, color_opacity4, features, feature_image need 16 bytes)");
	const int tiles_x = (width + HDS_TILE - 1) / HDS_TILE, tiles_y = (height + HDS_TILE - 1) / HDS_TILE;
	const int num_tiles = tiles_x * tiles_y;
	RenderArgs a{width,
				 height,
				 tiles_x,
				 feats ? channels : 0,
				 num_tiles,
				 reinterpret_cast<const int2*>(tile_ranges),
				 values_sorted,
				 reinterpret_cast<const float2*>(means2D),
				 reinterpret_cast<const float4*>(conic4),
				 reinterpret_cast<const float4*>(color_opacity4),
				 background,
				 features,
				 image,
				 final_T,
				 n_contrib,
				 feature_image,
				 reinterpret_cast<float4*>(clear),
				 clear_count / 4,
				 contributes};
	hipStream_t s = (hipStream_t)stream;
	if (!feats) {
		HDS_REQUIRE(rgb, "render: nothing to render (no image and no features)");
		return launch<0, true>(a, num_tiles, 1, s);
	}
	// Channels per work-group: 128 unless HDS_FORWARD_SLICE_WIDTH (32, 64 or 128) asks for less. The
	// result does not depend on it: every channel runs the same operation sequence.
	int width_slice = channels < 128 ? channels : 128;
	if (const char* env = std::getenv("HDS_FORWARD_SLICE_WIDTH")) {
		const int w = std::atoi(env);
		if ((w == 32 || w == 64 || w == 128) && w <= channels) width_slice = w;
	}
	const int slices = channels / width_slice;
	switch (width_slice) {
		case 32: return rgb ? launch<32, true>(a, num_tiles, slices, s) : launch<32, false>(a, num_tiles, slices, s);
		case 64: return rgb ? launch<64, true>(a, num_tiles, slices, s) : launch<64, false>(a, num_tiles, slices, s);
		default: return rgb ? launch<128, true>(a, num_tiles, slices, s) : launch<128, false>(a, num_tiles, slices, s);
	}
}

}  // namespace

extern "C" int hds_render(int64_t n, int width, int height, int channels, const int32_t* tile_ranges,
						  const int32_t* values_sorted, int64_t num_pairs, const float* means2D, const float* conic4,
						  const float* color_opacity4, const float* background, const float* features, float* image,
						  float* final_T, int32_t* n_contrib, float* feature_image, hds_stream_t stream) {
	(void)n;
	return render(width, height, channels, tile_ranges, values_sorted, num_pairs, means2D, conic4, color_opacity4,
				  background, features, image, final_T, n_contrib, feature_image, nullptr, 0, nullptr, stream);
}

extern "C" int hds_render_clear(int64_t n, int width, int height, int channels, const int32_t* tile_ranges,
								const int32_t* values_sorted, int64_t num_pairs, const float* means2D,
								const float* conic4, const float* color_opacity4, const float* background,
								const float* features, float* image, float* final_T, int32_t* n_contrib,
								float* feature_image, float* clear, int64_t clear_count, hds_stream_t stream) {
	(void)n;
	return render(width, height, channels, tile_ranges, values_sorted, num_pairs, means2D, conic4, color_opacity4,
				  background, features, image, final_T, n_contrib, feature_image, clear, clear_count, nullptr, stream);
}

extern "C" int hds_render_contributes(int64_t n, int width, int height, int channels, const int32_t* tile_ranges,
									  const int32_t* values_sorted, int64_t num_pairs, const float* means2D,
									  const float* conic4, const float* color_opacity4, const float* background,
									  const float* features, float* image, float* final_T, int32_t* n_contrib,
									  float* feature_image, float* clear, int64_t clear_count, uint8_t* contributes,
									  hds_stream_t stream) {
	(void)n;
	HDS_REQUIRE(contributes || num_pairs == 0, "render_contributes: null marks");
	return render(width, height, channels, tile_ranges, values_sorted, num_pairs, means2D, conic4, color_opacity4,
				  background, features, image, final_T, n_contrib, feature_image, clear, clear_count, contributes, stream);
}
