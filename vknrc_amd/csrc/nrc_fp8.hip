// nrc_fp8.hip -- the inference forward on FP8 (OCP e4m3) MFMA, v_mfma_f32_32x32x16_fp8_fp8.
//
// Scales are powers of two folded into the weights, so the kernel carries the
// activations pre-scaled and multiplies only at the output:
//   a_l is stored as C_l a_l (C_0 = 1: the encoded features lie in [-1, 1]),
//   layer l's weights as c_l W_l, so relu(c_l W_l C_l a_l) = C_{l+1} a_{l+1}
//   with C_{l+1} = c_l C_l, and the output as c_H W_H, unscaled by 1/(c_H C_H).
// c_l targets a largest scaled activation of 224 (half the e4m3 maximum 448)
// from the largest |a_{l+1}| of the cache's last 16 FP8 inferences (delayed
// scaling), and never scales c_l W_l past 448.  Values are converted with
// v_cvt_pk_fp8_f32 after one v_med3 that applies the ReLU and saturates at 448
// (the conversion itself turns values past the e4m3 range into NaN).
#include "nrc_mfma.hpp"

namespace nrc {

namespace {

constexpr float kFp8Max = 448.0f;
constexpr float kFp8Target = 224.0f;
constexpr uint32_t kFp8SampleStride = 8; // tiles whose activation maxima feed the scales

typedef float float16_t __attribute__((ext_vector_type(16)));
typedef unsigned int uint3_t __attribute__((ext_vector_type(3)));

__device__ __forceinline__ float16_t mfma8(long a, long b, float16_t c) {
	return __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float relu_sat(float x) { return __builtin_amdgcn_fmed3f(x, 0.0f, kFp8Max); }

__device__ __forceinline__ uint32_t pack4_relu(float a, float b, float c, float d) {
	return pack4_fp8(relu_sat(a), relu_sat(b), relu_sat(c), relu_sat(d));
}

// D elements 4 k .. 4 k + 3 and 8 + 4 k .. of M-tile m -> the next layer's B operand for K-chunk 2 m + k
template <int k> __device__ __forceinline__ long pack_relu_fp8(float16_t d) {
	const uint32_t lo = pack4_relu(d[4 * k], d[4 * k + 1], d[4 * k + 2], d[4 * k + 3]);
	const uint32_t hi = pack4_relu(d[8 + 4 * k], d[8 + 4 * k + 1], d[8 + 4 * k + 2], d[8 + 4 * k + 3]);
	return (long)((uint64_t)lo | ((uint64_t)hi << 32));
}

// Writes feature quads of lane (n, r)'s record into a wave's LDS slot: quad p holds features
// 4p..4p+3, K-chunk 2 (p >> 3) + ((p >> 1) & 1), lane group p & 1, half (p >> 2) & 1 of the
// lane's 8 bytes; the two halves lie 256 bytes apart, so a wave's 4-byte stores are contiguous.
struct Fp8SlotEmit {
	uint32_t *s;
	int n, r;
	const uint32_t *sel; // the one-blob selector table
	__device__ __forceinline__ int at(int p) const { return (((n * 4 + 2 * (p >> 3) + ((p >> 1) & 1)) * 2 + ((p >> 2) & 1)) * 2 + (p & 1)) * 32 + r; }
	__device__ __forceinline__ void operator()(int p, float f0, float f1, float f2, float f3) const { s[at(p)] = pack4_fp8(f0, f1, f2, f3); }
	__device__ __forceinline__ void oneblob(int p, float x) const { s[at(p)] = oneblob4_fp8(x, sel); }
};

// Grouped and persistent, software-pipelined.  The 64-record tiles of the group's caches
// lie end to end; a workgroup takes a contiguous range and its four waves take the tiles of
// a cache in turn.  The cache's e4m3 weights (22 KB) are copied to LDS once a workgroup and
// cache.  A wave runs a tile as two N-tiles of 32 records through v_mfma_f32_32x32x16_fp8_fp8:
// lane 32h + r holds column r, K index group h; D element i of M-tile m is unit 32m +
// 8 (i >> 2) + 4h + (i & 3), so with K-chunk 2m + s taking features 32m + 8s + 4h + j (j < 4)
// and + 16 a layer's packed outputs are the next layer's operands in the same lanes.  Two
// such MFMAs add the products of one 16x16x32 over the same 32 features in the same order,
// bit for bit.  The A fragments of a layer are read in two groups of four, one group ahead;
// the encoding of the wave's next tile goes into its LDS slot, spread between the layers,
// once this tile's operands are read; nothing in a tile branches (records past the count
// encode the last record, the range-checked stores drop them).
// Bound by VALU and MFMA issue: 88 MFMAs of 32 cycles and about 830 VALU instructions a
// tile (1.5 an activation to clamp and pack).  2,073,600 queries: 100 us with the 16x16x32
// kernel that encoded between tiles from five knots, 81 us.
//
// Every kFp8SampleStride-th tile of a cache also records the largest pre-saturation
// activation of each layer (a sample that does not depend on how the tiles are split among
// waves, so a cache gets the same scales alone and in a group); the wave's maxima go to its
// block's slot of the cache's FP8 state.
template <int H, int ENC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void fp8_infer_kernel(const InferGroup grp) {
	__shared__ __attribute__((aligned(16))) long sW[(H * 8 + 4) * 64];
	__shared__ __attribute__((aligned(16))) uint32_t sX[4][16 * 64];
	__shared__ uint32_t sSel[4][8]; // each wave's one-blob selector table

	const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	oneblob_sel8_init(sSel[wave], lane);
	const int h = lane >> 5, r = lane & 31;
	const uint32_t tiles = infer_tiles(grp);
	const uint32_t t0 = (uint32_t)((uint64_t)tiles * blockIdx.x / gridDim.x);
	const uint32_t t1 = (uint32_t)((uint64_t)tiles * (blockIdx.x + 1) / gridDim.x);
	uint32_t *const slot = sX[wave];
	const Fp8SlotEmit emit{slot, h, r, sSel[wave]}; // this lane encodes record r of N-tile h

	for (uint32_t i = 0; i < grp.n_items; ++i) {
		const InferItem &it = grp.item[i];
		const uint32_t b0 = it.tile_begin, b1 = b0 + (it.max_count + 63) / 64;
		if (b1 <= t0) continue;
		if (b0 >= t1) break;
		const uint32_t count = __builtin_amdgcn_readfirstlane(effective_count(it.d_count, it.max_count, it.max_count));
		const uint32_t lt0 = (t0 > b0 ? t0 : b0) - b0;
		uint32_t lt1 = (t1 < b1 ? t1 : b1) - b0;
		const uint32_t ntiles = (count + 63) / 64;
		lt1 = lt1 < ntiles ? lt1 : ntiles;
		if (lt0 >= lt1) continue; // uniform over the workgroup

		const float out_scale = it.f8->out_scale;
		const float *queries = it.queries;
		float *out = it.out;
		const uint32_t last = count - 1, tlast = lt1 - 1;
		auto load_query = [&](uint32_t t, float *dst) __attribute__((always_inline)) {
			t = t < tlast ? t : tlast;
			uint32_t m = t * 64 + lane;
			m = m < last ? m : last;
			const float2 *qp = reinterpret_cast<const float2 *>(queries + (size_t)m * kQueryFloats);
#pragma unroll
			for (int k = 0; k < 7; ++k) {
				const float2 v = qp[k];
				dst[2 * k] = v.x;
				dst[2 * k + 1] = v.y;
			}
		};
		// wave w takes tiles lt0 + w, lt0 + w + 4, ..; two record buffers in ping-pong
		float ra[kQueryFloats], rb[kQueryFloats];
		const uint32_t tw = lt0 + wave;
		load_query(tw, ra);
		load_query(tw + 4, rb);
		block_lds_sync(); // the previous cache's weights are read
		for (int k = wave; k < (H * 8 + 4) / 2; k += 4)
			__builtin_amdgcn_global_load_lds(reinterpret_cast<const void *>(it.w8 + (k * 64 + lane) * 16),
			                                 (__attribute__((address_space(3))) void *)(sW + k * 128), 16, 0, 0);
		__builtin_amdgcn_s_waitcnt(0); // this wave's copies have landed
		block_lds_sync();
		if (tw >= lt1) continue;

		constexpr int NP = encode_pieces<ENC>();
		// piece k of the next tile's encoding goes into phase k * phases / NP
		constexpr int phases = 3 * H;
		auto pieces_at = [&](auto phase_c, const float *rec) __attribute__((always_inline)) {
			constexpr int phase = decltype(phase_c)::value;
			static_for<NP>([&](auto k_c) __attribute__((always_inline)) {
				constexpr int k = decltype(k_c)::value;
				if constexpr (k * phases / NP == phase) encode_piece<ENC, k>(rec, emit);
			});
		};
		// The A fragments of a layer in two groups of four, (M-tile, K-chunk) = (0, 0) (0, 1)
		// (1, 0) (1, 1), then chunks 2 and 3; the output layer's four are the last group.  The
		// groups of a tile are odd in number, so the buffer of group k of a tile with parity P
		// is (k + P) & 1.
		constexpr int NG = 2 * H + 1;
		long A[2][4];
		auto load_group = [&](auto k_c, long *dst) __attribute__((always_inline)) {
			constexpr int k = decltype(k_c)::value % NG;
#pragma unroll
			for (int j = 0; j < 4; ++j)
				dst[j] = k == NG - 1 ? sW[(H * 8 + j) * 64 + lane]
				                     : sW[((k >> 1) * 8 + (j >> 1) * 4 + 2 * (k & 1) + (j & 1)) * 64 + lane];
			// the reads stay above what follows: everything but LDS reads may cross
			__builtin_amdgcn_sched_barrier(0x27F);
		};
		float amax[H]; // largest pre-saturation a_1 .. a_H of the recorded tiles (scaled)
#pragma unroll
		for (int l = 0; l < H; ++l) amax[l] = 0.0f;
		auto run_tile = [&](auto par_c, auto track_c, uint32_t tile, const float *rec) __attribute__((always_inline)) {
			constexpr int P = decltype(par_c)::value;
			constexpr bool TRACK = decltype(track_c)::value;
			const uint32_t left = count - tile * 64;
			const uint32_t nrec = left < 64u ? left : 64u;
			const __amdgpu_buffer_rsrc_t rs =
			    __builtin_amdgcn_make_buffer_rsrc(out + (size_t)tile * 64 * kOut, (short)0, (int)(nrec * kOut * 4), 0x00020000);
			long B[2][4];
#pragma unroll
			for (int n = 0; n < 2; ++n)
#pragma unroll
				for (int c = 0; c < 4; ++c) {
					const uint32_t lo = slot[((n * 4 + c) * 2) * 64 + lane], hi = slot[((n * 4 + c) * 2 + 1) * 64 + lane];
					B[n][c] = (long)((uint64_t)lo | ((uint64_t)hi << 32));
				}
			static_for<H>([&](auto l_c) __attribute__((always_inline)) {
				constexpr int l = decltype(l_c)::value;
				float16_t acc[2][2]; // [M-tile][N-tile]
#pragma unroll
				for (int m = 0; m < 2; ++m)
#pragma unroll
					for (int n = 0; n < 2; ++n) acc[m][n] = (float16_t)0.0f;
				auto step = [&](long a, int m, int c) __attribute__((always_inline)) {
#pragma unroll
					for (int n = 0; n < 2; ++n) acc[m][n] = mfma8(a, B[n][c], acc[m][n]);
				};
				const long *A0 = A[(2 * l + P) & 1], *A1 = A[(2 * l + 1 + P) & 1];
				// the K-chunks of M-tile 0's features first, for both M-tiles: M-tile 1 of the
				// previous layer is still being packed
				load_group(std::integral_constant<int, 2 * l + 1>{}, A[(2 * l + 1 + P) & 1]);
				step(A0[0], 0, 0); step(A0[1], 0, 1); step(A0[2], 1, 0); step(A0[3], 1, 1);
				pieces_at(std::integral_constant<int, 3 * l>{}, rec);
				load_group(std::integral_constant<int, 2 * l + 2>{}, A[(2 * l + 2 + P) & 1]);
				step(A1[0], 0, 2); step(A1[1], 0, 3);
				pieces_at(std::integral_constant<int, 3 * l + 1>{}, rec);
				step(A1[2], 1, 2); step(A1[3], 1, 3);
				pieces_at(std::integral_constant<int, 3 * l + 2>{}, rec);
				if constexpr (TRACK) {
#pragma unroll
					for (int m = 0; m < 2; ++m)
#pragma unroll
						for (int n = 0; n < 2; ++n)
#pragma unroll
							for (int e = 0; e < 16; ++e) {
								const float x = acc[m][n][e];
								amax[l] = fmaxf(amax[l], x);
							}
				}
#pragma unroll
				for (int m = 0; m < 2; ++m)
#pragma unroll
					for (int n = 0; n < 2; ++n) {
						B[n][2 * m] = pack_relu_fp8<0>(acc[m][n]);
						B[n][2 * m + 1] = pack_relu_fp8<1>(acc[m][n]);
					}
			});
			load_group(std::integral_constant<int, 0>{}, A[(NG + P) & 1]); // of the next tile
			float16_t o[2] = {(float16_t)0.0f, (float16_t)0.0f};
#pragma unroll
			for (int c = 0; c < 4; ++c)
#pragma unroll
				for (int n = 0; n < 2; ++n) o[n] = mfma8(A[(NG - 1 + P) & 1][c], B[n][c], o[n]);
#pragma unroll
			for (int n = 0; n < 2; ++n) {
				uint3_t v;
#pragma unroll
				for (int e = 0; e < 3; ++e) {
					const float y = o[n][e] * out_scale;
					v[e] = __float_as_uint(grp.clamp0 ? fmaxf(y, 0.0f) : y);
				}
				const uint32_t off = h == 0 ? (uint32_t)((n * 32 + r) * kOut * 4) : 0x7ffffff0u;
				__builtin_amdgcn_raw_buffer_store_b96(v, rs, off, 0, 0);
			}
		};
		auto tile = [&](auto par_c, uint32_t t, const float *rec) __attribute__((always_inline)) {
			if (t % kFp8SampleStride == 0) // uniform
				run_tile(par_c, std::true_type{}, t, rec);
			else
				run_tile(par_c, std::false_type{}, t, rec);
			wave_lds_sync();
		};

		load_group(std::integral_constant<int, 0>{}, A[0]);
		encode_quads<ENC>(ra, emit);
		wave_lds_sync();
		for (uint32_t t = tw; t < lt1; t += 8) {
			load_query(t + 8, ra);
			tile(std::integral_constant<int, 0>{}, t, rb); // encodes tile t + 4 (a repeat of the last tile past the range)
			if (t + 4 >= lt1) break;
			load_query(t + 12, rb);
			tile(std::integral_constant<int, 1>{}, t + 4, ra); // encodes tile t + 8
		}
		// the wave's maxima into its block's slot (non-negative floats order as their bits)
#pragma unroll
		for (int l = 0; l < H; ++l) {
			float m = amax[l];
#pragma unroll
			for (int off = 32; off >= 1; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
			if (lane == 0 && m > 0.0f)
				atomicMax(reinterpret_cast<unsigned int *>(&it.f8->block_amax[blockIdx.x][l + 1]), __float_as_uint(m));
		}
	}
}

__device__ __forceinline__ float pow2_floor(float x) { return ldexpf(1.0f, ilogbf(x)); }

// The maximum over the 16 lanes of a row, in each of them (rotations by 8, 4, 2 and 1)
__device__ __forceinline__ float row_max(float x) {
	auto with = [](float v, auto ctrl) __attribute__((always_inline)) {
		const int o = __builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), decltype(ctrl)::value, 0xF, 0xF, false);
		return fmaxf(v, __uint_as_float((uint32_t)o));
	};
	x = with(x, std::integral_constant<int, 0x128>{}); // row_ror:8
	x = with(x, std::integral_constant<int, 0x124>{});
	x = with(x, std::integral_constant<int, 0x122>{});
	return with(x, std::integral_constant<int, 0x121>{});
}

// One block per cache: folds the last FP8 inference's per-block maxima into the history,
// chooses the layer scales and writes the e4m3 copy of c_l W_l.  Bound by latency: the
// maxima, the history, the scales and the weights (held in registers, five float4 a thread)
// are all loaded before anything waits, the barriers do not wait for the stores (nothing in
// this kernel reads them), and the maxima go over rows of lanes and then a wave each.
// 6.3 us; 8.2 with full barriers, shuffles over whole waves and one thread a maximum; a
// scale kernel of 256 threads and a quantize kernel took 8.5 + 4.8 us and a launch.
template <int H> __global__ __launch_bounds__(1024) void fp8_prep_kernel(const Fp8PrepGroup grp) {
	static_assert(kFp8MaxBlocks == 1024, "one slot of the last inference's maxima a thread");
	const Fp8PrepItem &it = grp.item[blockIdx.x];
	Fp8State *st = it.f8;
	const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
	__shared__ float red[2 * kFp8Layers][64]; // maxima of 16 threads: activations, then |W_l|
	__shared__ float largest[2 * kFp8Layers], hist_old[kFp8History][kFp8Layers], cscale[kFp8Layers];
	static_assert(kFp8History == 16 && 2 * kFp8Layers <= 16, "a row of lanes for the history, a wave for each maximum");

	// 1. every load: the last inference's activation maxima (scaled by its C_l), the history, the weights
	float m[2 * kFp8Layers];
#pragma unroll
	for (int l = 0; l < kFp8Layers; ++l) m[l] = st->block_amax[t][l];
	const uint32_t frames0 = st->frames;
	const bool recorded = st->scale[0] > 0.0f; // a previous call set the scales that inference used
	const float scale_old = st->scale[wave < kFp8Layers ? wave : 0];
	const float hv = t < kFp8History * kFp8Layers ? (&st->hist[0][0])[t] : 0.0f;
	const float4_t *w4 = reinterpret_cast<const float4_t *>(it.use32);
	float4_t w[H + 1];
#pragma unroll
	for (int l = 0; l < H; ++l) w[l] = w4[l * 1024 + t];
	w[H] = t < kOut * kWidth / 4 ? w4[H * 1024 + t] : (float4_t)0.0f;

	// 2. the maxima over the block, cleared in memory for the next inference
#pragma unroll
	for (int l = 0; l < kFp8Layers; ++l) st->block_amax[t][l] = 0.0f;
#pragma unroll
	for (int l = 0; l < kFp8Layers; ++l)
		m[kFp8Layers + l] = l <= H ? fmaxf(fmaxf(fabsf(w[l <= H ? l : 0][0]), fabsf(w[l <= H ? l : 0][1])),
		                                   fmaxf(fabsf(w[l <= H ? l : 0][2]), fabsf(w[l <= H ? l : 0][3])))
		                           : 0.0f;
#pragma unroll
	for (int k = 0; k < 2 * kFp8Layers; ++k) {
		m[k] = row_max(m[k]);
		if ((lane & 15) == 0) red[k][t >> 4] = m[k];
	}
	if (t < kFp8History * kFp8Layers) (&hist_old[0][0])[t] = hv;
	block_lds_sync();

	// 3. wave l <= H: the history maximum of layer l's input; waves kFp8Layers + l: |W_l|
	if (wave < 2 * kFp8Layers) {
		float mx = row_max(red[wave][lane]);
		mx = fmaxf(mx, __shfl_xor(mx, 16));
		mx = fmaxf(mx, __shfl_xor(mx, 32));
		if (wave < kFp8Layers) {
			uint32_t frames = frames0;
			float past = hist_old[lane & 15][wave];
			if (recorded && wave <= H) {
				const uint32_t slot = frames % kFp8History;
				const float v = wave == 0 ? 1.0f : mx / scale_old;
				if (lane == 0) st->hist[slot][wave] = v;
				if ((uint32_t)(lane & 15) == slot) past = v;
				++frames;
			}
			const uint32_t nh = frames < (uint32_t)kFp8History ? frames : (uint32_t)kFp8History;
			mx = fmaxf(row_max((uint32_t)(lane & 15) < nh ? past : 0.0f), 0.0f);
			if (nh == 0) mx = 4.0f; // no history yet: a first guess, corrected after one inference
		}
		if (lane == 0) largest[wave] = mx;
	}
	block_lds_sync();
	// the scales: c_l for l < H from the history, c_H from the weights (every wave has its
	// copy of what this overwrites)
	if (t == 0) {
		if (recorded) st->frames = frames0 + 1u;
		float C = 1.0f;
		st->scale[0] = 1.0f;
#pragma unroll
		for (int l = 0; l < H; ++l) {
			const float hmax = largest[l + 1], wmax = largest[kFp8Layers + l];
			float c = (hmax > 0.0f) ? pow2_floor(kFp8Target / (hmax * C)) : 1.0f;
			if (wmax > 0.0f && wmax * c > kFp8Max) c = pow2_floor(kFp8Max / wmax);
			st->wscale[l] = cscale[l] = c;
			C *= c;
			st->scale[l + 1] = C;
		}
		const float wmax = largest[kFp8Layers + H];
		const float cH = wmax > 0.0f ? pow2_floor(kFp8Max / wmax) : 1.0f;
		st->wscale[H] = cscale[H] = cH;
		st->out_scale = 1.0f / (cH * C);
	}
	block_lds_sync();

	// 4. the e4m3 copy: four weights of a row are four consecutive bytes of a fragment
#pragma unroll
	for (int l = 0; l <= H; ++l) {
		if (l == H && t >= kOut * kWidth / 4) break;
		const float c = cscale[l];
		float q[4];
#pragma unroll
		for (int e = 0; e < 4; ++e) q[e] = __builtin_amdgcn_fmed3f(w[l][e] * c, -kFp8Max, kFp8Max);
		*reinterpret_cast<uint32_t *>(it.w8 + fp8_frag_pos((uint32_t)l, (uint32_t)t >> 4, 4u * ((uint32_t)t & 15u))) =
		    pack4_fp8(q[0], q[1], q[2], q[3]);
	}
}

template <int H, int ENC> hipError_t fp8_launch(InferGroup &grp, const Fp8PrepGroup &prep, hipStream_t s) {
	fp8_prep_kernel<H><<<dim3(prep.n_items), dim3(1024), 0, s>>>(prep);
	hipError_t e = hipGetLastError();
	if (e != hipSuccess) return e;
	uint32_t blocks = (grp.total_tiles + 3) / 4;
	uint32_t cap = (uint32_t)device_cu_count() * infer_wg_per_cu();
	if (cap > (uint32_t)kFp8MaxBlocks) cap = kFp8MaxBlocks;
	if (blocks > cap) blocks = cap;
	if (blocks == 0) blocks = 1;
	// Every count: a workgroup copies the weights to LDS once whatever it runs, so an even deal
	// costs little and saves most (of 131 sizes and counts 0.88 of the time of the maximum's deal
	// in the mean: 524,288 queries of which 131,072, 15.4 -> 10.7 us; 196,608 of 393,216, 14.0 -> 15.1,
	// is the worst).
	grp.deal = deals_by_count(grp, blocks) ? kDealByCount : kDealByMaximum;
	fp8_infer_kernel<H, ENC><<<dim3(blocks), dim3(256), 0, s>>>(grp);
	return hipGetLastError();
}

template <int H> hipError_t fp8_h(int enc, InferGroup &grp, const Fp8PrepGroup &prep, hipStream_t s) {
	switch (enc) {
	case NRC_ENCODING_TRI12: return fp8_launch<H, NRC_ENCODING_TRI12>(grp, prep, s);
	case NRC_ENCODING_SINCOS6: return fp8_launch<H, NRC_ENCODING_SINCOS6>(grp, prep, s);
	default: return fp8_launch<H, NRC_ENCODING_UV_SINCOS16>(grp, prep, s);
	}
}

} // namespace

hipError_t launch_fp8_infer_group(int hidden, int encoding, InferGroup &grp, const float *const *use32,
                                  uint8_t *const *w8, hipStream_t stream) {
	uint32_t tiles = 0;
	Fp8PrepGroup prep{};
	prep.n_items = grp.n_items;
	for (uint32_t i = 0; i < grp.n_items; ++i) {
		grp.item[i].tile_begin = tiles;
		tiles += (grp.item[i].max_count + 63) / 64;
		prep.item[i] = Fp8PrepItem{grp.item[i].f8, use32[i], w8[i]};
	}
	grp.total_tiles = tiles;
	if (tiles == 0) return hipSuccess;
	if (hidden == 5) return fp8_h<5>(encoding, grp, prep, stream);
	return fp8_h<4>(encoding, grp, prep, stream);
}

} // namespace nrc
