// nrc_plain.hip -- the plain method: FP32 encoding, weights, products and sums.
//
// The layers run on v_mfma_f32_16x16x4_f32, whose products and sums are FP32: twice the
// rate of FP32 FMAs without packed instructions.  Lane l = 16 g + r holds A row r, B
// column r at K index g, and D column r, rows 4 g .. 4 g + 3.  A wave runs 16 records
// (the columns).  The rows of an A tile are permuted so that D element i of tile Mt in
// lane group g is unit 16 Mt + 4 i + g: K step s = 4 mt + i of the next layer takes
// features 4 s .. 4 s + 3 from lane groups 0 .. 3, which is exactly where they are.  So a
// layer's ReLU'd D registers are the next layer's B operands with no data movement at
// all, and every sum runs over k = 0 .. 63 in order, one fused multiply-add after the
// other, as one thread a record would compute it (the MFMA adds its K products in order,
// each rounded: the results equal the FMA loop's bit for bit).
//
// All weights of the network lie in LDS as A fragments: float4 (l, Mt, mt, g, r) holds
// W_l[16 Mt + 4 (r & 3) + (r >> 2)][16 mt + 4 i + g], i = 0..3, at slot 16 g + ((r + g) & 15)
// of its 1 KB block.  The rotation by g lets the backward read single floats of W_l^T from
// the same copy without bank conflicts (for one i, the 16 values (4 g + i + g') mod 16 of
// g, g' in 0..3 differ).
//
// The weight gradient is reduced over fixed kPlainChunk-record chunks in a fixed order,
// so the result is deterministic.  This path is the FP32 reference the fused FP16-MFMA
// path is measured against.
#include <type_traits>

#include "nrc_internal.hpp"

namespace nrc {

namespace {

typedef float float4_t __attribute__((ext_vector_type(4)));

// waves of a workgroup; one workgroup a CU (its LDS holds the FP32 weights)
constexpr int kPlainWaves = 8, kPlainInferWaves = 16;

__device__ __forceinline__ float4_t mfma4(float a, float b, float4_t c) {
	return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

template <int H> struct PlainSmem {
	float4_t frag[H * 16 * 64];
	float4_t frag_out[4 * 64]; // the output layer's A fragments: row c < 3 is output c, the rest zero
};

// All weights into LDS, every load in flight before the first store.
template <int H, int WAVES> __device__ __forceinline__ void stage_weights(PlainSmem<H> &S, const float *__restrict__ w32) {
	constexpr int kPer = H * 1024 / (64 * WAVES);
	const int t = threadIdx.x;
	const float4_t *src = reinterpret_cast<const float4_t *>(w32);
	float4_t v[kPer];
#pragma unroll
	for (int k = 0; k < kPer; ++k) v[k] = src[t + k * 64 * WAVES];
	if (t < 4 * 64) {
		const int mt = t >> 6, g = (t >> 4) & 3, r = t & 15;
		const float *wo = w32 + H * kWidth * kWidth + (r < kOut ? r : 0) * kWidth + 16 * mt + g;
		const float4_t o = {wo[0], wo[4], wo[8], wo[12]};
		S.frag_out[t] = r < kOut ? o : (float4_t)0.0f;
	}
	float *f = reinterpret_cast<float *>(S.frag);
#pragma unroll
	for (int k = 0; k < kPer; ++k) {
		// layer j >> 10, row (j >> 4) & 63, columns 16 mt + 4 i + 0..3
		const int j = t + k * 64 * WAVES, row = (j >> 4) & 63, mt = (j >> 2) & 3, i = j & 3;
		const int r = 4 * (row & 3) + ((row >> 2) & 3), blk = ((j >> 10) * 4 + (row >> 4)) * 4 + mt;
#pragma unroll
		for (int g = 0; g < 4; ++g) f[(blk * 64 + 16 * g + ((r + g) & 15)) * 4 + i] = v[k][g];
	}
	__syncthreads();
}

__device__ __forceinline__ float4_t relu4(float4_t v) {
#pragma unroll
	for (int i = 0; i < 4; ++i) v[i] = fmaxf(v[i], 0.0f);
	return v;
}

// The features 4 s + g, s = 0..15, of one record for lane group g (element g of every
// quad), by the arithmetic of encode_all.
template <int ENC> __device__ __forceinline__ void encode_lane(const float *rec, int g, float4_t *x) {
	auto pick = [g](float a, float b, float c, float d) __attribute__((always_inline)) {
		return g == 0 ? a : g == 1 ? b : g == 2 ? c : d;
	};
	if constexpr (ENC == NRC_ENCODING_UV_SINCOS16) {
#pragma unroll
		for (int a = 0; a < 2; ++a)
#pragma unroll
			for (int q = 0; q < 4; ++q) {
				float s[4], c[4];
				sincospi_poly(rec[a] * (float)(1 << (4 * q)), &s[0], &c[0]);
#pragma unroll
				for (int k = 1; k < 4; ++k) {
					s[k] = 2.0f * s[k - 1] * c[k - 1];
					c[k] = 1.0f - 2.0f * s[k - 1] * s[k - 1];
				}
				x[2 * a][q] = pick(s[0], s[1], s[2], s[3]);
				x[2 * a + 1][q] = pick(c[0], c[1], c[2], c[3]);
			}
	} else {
#pragma unroll
		for (int a = 0; a < 3; ++a) {
			if constexpr (ENC == NRC_ENCODING_TRI12) {
				const float p = rec[a] * (float)(1 << g);
#pragma unroll
				for (int q = 0; q < 3; ++q) x[(3 * a + q) >> 2][(3 * a + q) & 3] = tri(p * (float)(1 << (4 * q)));
			} else {
				float s[6], c[6];
				sincos_octaves<6>(rec[a], s, c);
				x[(3 * a) >> 2][(3 * a) & 3] = pick(s[0], s[1], s[2], s[3]);
				x[(3 * a + 1) >> 2][(3 * a + 1) & 3] = pick(s[4], s[5], c[0], c[1]);
				x[(3 * a + 2) >> 2][(3 * a + 2) & 3] = pick(c[2], c[3], c[4], c[5]);
			}
		}
		const float k0 = 0.25f * (float)g, k1 = k0 + 0.25f; // the knots of bin g
#pragma unroll
		for (int b = 0; b < 5; ++b) {
			const float u = b == 4 ? 1.0f - expf(-rec[7]) : rec[3 + b];
			x[(9 + b) >> 2][(9 + b) & 3] = quartic_cdf(k1 - u) - quartic_cdf(k0 - u);
		}
		x[3][2] = pick(rec[8], rec[9], rec[10], rec[11]);
		x[3][3] = pick(rec[12], rec[13], 1.0f, 1.0f);
	}
}

// The A fragments of layer l that the K steps 4 mt .. 4 mt + 3 take
template <int H> __device__ __forceinline__ void layer_fragments(const PlainSmem<H> &S, int l, int mt, int slot, float4_t *a) {
#pragma unroll
	for (int m = 0; m < 4; ++m) a[m] = S.frag[((l * 4 + m) * 4 + mt) * 64 + slot];
}

// x = relu(W_l x) of this wave's 16 records (NN_nv.glsl:99-127); four independent
// accumulator chains, one 16-byte LDS read per four MFMAs.  `next` holds the layer's first
// fragments and receives those of the layer after it (the first layer's after the last): a
// wave that has its SIMD to itself would otherwise wait for each read.
template <int H> __device__ __forceinline__ void layer_forward(const PlainSmem<H> &S, int l, int slot, float4_t *x, float4_t *next) {
	float4_t acc[4];
#pragma unroll
	for (int m = 0; m < 4; ++m) acc[m] = (float4_t)0.0f;
	const int after = l + 1 < H ? l + 1 : 0;
#pragma unroll
	for (int mt = 0; mt < 4; ++mt) {
		float4_t a[4];
#pragma unroll
		for (int m = 0; m < 4; ++m) a[m] = next[m];
		layer_fragments<H>(S, mt < 3 ? l : after, (mt + 1) & 3, slot, next);
		__builtin_amdgcn_sched_barrier(0);
#pragma unroll
		for (int i = 0; i < 4; ++i)
#pragma unroll
			for (int m = 0; m < 4; ++m) acc[m] = mfma4(a[m][i], x[mt][i], acc[m]);
		__builtin_amdgcn_sched_barrier(0);
	}
#pragma unroll
	for (int m = 0; m < 4; ++m) x[m] = relu4(acc[m]);
}

// o = W_H x (NN_nv.glsl:129-158), padded to 16 rows: lane group 0 holds the outputs
template <int H> __device__ __forceinline__ float4_t output_forward(const PlainSmem<H> &S, int lane, const float4_t *x) {
	float4_t acc = (float4_t)0.0f;
#pragma unroll
	for (int mt = 0; mt < 4; ++mt) {
		const float4_t a = S.frag_out[mt * 64 + lane];
#pragma unroll
		for (int i = 0; i < 4; ++i) acc = mfma4(a[i], x[mt][i], acc);
	}
	return acc;
}

__device__ __forceinline__ void load_query(const float *__restrict__ q, float *rec) {
	const float2 *p = reinterpret_cast<const float2 *>(q);
#pragma unroll
	for (int i = 0; i < 7; ++i) {
		const float2 v = p[i];
		rec[2 * i] = v.x;
		rec[2 * i + 1] = v.y;
	}
}

// nrc_inference.comp:30-48 (without the scene unpack and the epilogue).  Persistent, one
// workgroup a CU, 16-record tiles dealt to the waves in turn.  Bound by the FP32 MFMA
// rate, 336 MFMAs of 32 cycles a tile, plus the 270 (TRI12) vector instructions of a tile:
// FP32 MFMAs and vector instructions never overlap (no co-issued cycle counted), 4.9 us of a
// SIMD together.  Four waves a SIMD fill the waits that two left (87.3 -> 84.3 us for
// 230,400 queries back to back, 681 -> 660 us for 2,073,600; 655 with the fragments read
// ahead).  230,400 queries: 203 -> 80.3 us against one thread a query on the vector unit.
template <int H, int ENC>
__global__ __launch_bounds__(64 * kPlainInferWaves) void plain_infer_kernel(const float *__restrict__ queries,
                                                                       const uint32_t *__restrict__ d_count,
                                                                       uint32_t max_count,
                                                                       const float *__restrict__ w32,
                                                                       float *__restrict__ rgb) {
	__shared__ PlainSmem<H> S;
	const uint32_t count = effective_count(d_count, max_count, max_count);
	const int lane = threadIdx.x & 63, g = lane >> 4, r = lane & 15, slot = 16 * g + ((r + g) & 15);
	const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const uint32_t tiles = (count + 15) / 16, last = count - 1, stride = kPlainInferWaves * gridDim.x;
	uint32_t t = wave * gridDim.x + blockIdx.x;
	float rec[kQueryFloats];
	// the first records are on their way while the weights are staged, the next ones while
	// a tile runs (a tile past the last re-reads the last record)
	auto load_tile = [&](uint32_t tile) __attribute__((always_inline)) {
		const uint32_t n = tile < tiles ? tile * 16 + r : last;
		load_query(queries + (size_t)(n < last ? n : last) * kQueryFloats, rec);
	};
	if (blockIdx.x >= tiles) return; // no tile for any wave: nothing to stage the weights for (uniform)
	load_tile(t);
	stage_weights<H, kPlainInferWaves>(S, w32);
	float4_t next[4];
	layer_fragments<H>(S, 0, 0, slot, next);
	for (; t < tiles; t += stride) {
		const uint32_t n = t * 16 + r;
		float4_t x[4];
		encode_lane<ENC>(rec, g, x);
		load_tile(t + stride);
#pragma unroll 1
		for (int l = 0; l < H; ++l) layer_forward<H>(S, l, slot, x, next);
		const float4_t o = output_forward<H>(S, lane, x);
		if (g == 0 && n < count)
#pragma unroll
			for (int c = 0; c < kOut; ++c) rgb[(size_t)n * kOut + c] = fmaxf(o[c], 0.0f); // nrc_inference.comp:48
	}
}

// Per record: encode, forward keeping a_0..a_H, loss gradient, then the
// backward recurrence delta_{l-1} = (W_l^T delta_l) . 1[a_l > 0]
// (nrc_gradient.comp:26-58, NN_nv.glsl:162-278).  Writes the activations and deltas of a
// tile as one 4 KB block [64 features][16 records] a layer, so that every store here and
// every load of the reduction is a contiguous 256 or 1024 bytes a wave (rows of a whole
// batch put each load on 16 lines 64 KB apart: the reduction took 25.7 us instead of 17.7,
// before it went through LDS).  The records that pad the last tile are written as zeros, and
// the records of a tile are stored in the order 4 (r & 3) + (r >> 2) that the reduction
// reads.  Bound by the FP32 MFMA rate (592 of 32 cycles a tile for H = 5, 7.9 us of a SIMD;
// 16,384 records are one tile a SIMD), the 46 MB of activations and deltas written and the
// staging of the weights before the first tile.  16,384 records: 397 -> 25.8 us against one
// thread a record (64 workgroups on 256 CUs, a broadcast LDS read a product), 23.2 with the
// layers as loops and the weights read ahead; 4.4 of that are the launch and the staging,
// 2 to 3 the stores (non-temporal stores move as much to the reduction).
template <int H, int ENC, int LOSS>
__global__ __launch_bounds__(64 * kPlainWaves) void plain_fwdbwd_kernel(const float *__restrict__ records,
                                                           const uint32_t *__restrict__ d_count, uint32_t max_count,
                                                           uint32_t clamp, const float *__restrict__ w32,
                                                           const DeviceState *__restrict__ st, int parity,
                                                           float *__restrict__ acts, float *__restrict__ deltas,
                                                           float *__restrict__ sample_loss, uint32_t ldn) {
	__shared__ PlainSmem<H> S;
	const uint32_t count = effective_count(d_count, max_count, clamp);
	const int lane = threadIdx.x & 63, g = lane >> 4, r = lane & 15, slot = 16 * g + ((r + g) & 15);
	const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const uint32_t tiles = (count + 15) / 16;
	const size_t slab = (size_t)kWidth * ldn;
	const float s = st->pub[parity].loss_scale;
	// floats of W_l^T: row 16 mt + 4 i + g, column 16 Mt + 4 (r & 3) + (r >> 2) of W_l lies
	// in block (mt, Mt) at slot tslot(i), component r & 3
	const int gp = r >> 2;
	int tslot[4];
#pragma unroll
	for (int i = 0; i < 4; ++i) tslot[i] = (16 * gp + ((4 * g + i + gp) & 15)) * 4 + (r & 3);
	const float *sf = reinterpret_cast<const float *>(S.frag);
	const uint32_t last = count - 1, stride = kPlainWaves * gridDim.x;
	uint32_t t = wave * gridDim.x + blockIdx.x;
	float rec[kTrainFloats];
	auto load_tile = [&](uint32_t tile) __attribute__((always_inline)) {
		const uint32_t n = tile < tiles ? tile * 16 + r : last;
		const float *rp = records + (size_t)(n < last ? n : last) * kTrainFloats;
#pragma unroll
		for (int i = 0; i < kTrainFloats; ++i) rec[i] = rp[i];
	};
	if (blockIdx.x >= tiles) return; // no tile for any wave: nothing to stage the weights for (uniform)
	load_tile(t); // on their way while the weights are staged
	stage_weights<H, kPlainWaves>(S, w32);
	float4_t next[4];
	layer_fragments<H>(S, 0, 0, slot, next);
	for (; t < tiles; t += stride) {
		const uint32_t n = t * 16 + r;
		const bool valid = n < count;
		// features 16 mt + 4 i + g of this lane's record in the tile's block of a slab
		const size_t blk = (size_t)t * (16 * kWidth) + 4 * (r & 3) + (r >> 2);
		auto store = [&](float *dst, const float4_t *v) __attribute__((always_inline)) {
#pragma unroll
			for (int mt = 0; mt < 4; ++mt)
#pragma unroll
				for (int i = 0; i < 4; ++i) dst[blk + 16 * (16 * mt + 4 * i + g)] = v[mt][i];
		};
		float4_t x[4];
		encode_lane<ENC>(rec, g, x);
#pragma unroll
		for (int mt = 0; mt < 4; ++mt)
#pragma unroll
			for (int i = 0; i < 4; ++i) x[mt][i] = valid ? x[mt][i] : 0.0f;
		store(acts, x);
		// 1[a_l > 0] of this lane's units, 16 bits a layer, the latest layer lowest.  With the
		// bits instead of the activations in registers the layers are loops, whose code is
		// fetched once: a launch is one tile a wave, and its first pass over 25 KB of unrolled
		// layers waited for the instructions.
		uint32_t active[3] = {0u, 0u, 0u};
		static_assert(H <= 6, "16 H bits in three words");
#pragma unroll 1
		for (int l = 0; l < H; ++l) {
			layer_forward<H>(S, l, slot, x, next);
			store(acts + (size_t)(l + 1) * slab, x);
			active[2] = __builtin_amdgcn_alignbit(active[2], active[1], 16);
			active[1] = __builtin_amdgcn_alignbit(active[1], active[0], 16);
			active[0] <<= 16;
#pragma unroll
			for (int mt = 0; mt < 4; ++mt)
#pragma unroll
				for (int i = 0; i < 4; ++i) active[0] |= (x[mt][i] > 0.0f ? 1u : 0u) << (4 * mt + i);
		}
		auto relu_mask = [&active](float v, int unit) __attribute__((always_inline)) {
			return relu_bwd(v, (active[0] >> unit) & 1u ? 1.0f : 0.0f);
		};
		const float4_t ov = output_forward<H>(S, lane, x);
		const float o[kOut] = {__shfl(ov[0], r), __shfl(ov[1], r), __shfl(ov[2], r)}; // from lane group 0
		float go[kOut];
		const float v = loss_grad<LOSS>(o, rec + kQueryFloats, s, go);
#pragma unroll
		for (int c = 0; c < kOut; ++c) go[c] = valid ? go[c] : 0.0f;
		if (g == 0) {
			sample_loss[n] = valid ? v : 0.0f;
			float *dH = deltas + (size_t)H * slab;
#pragma unroll
			for (int c = 0; c < kOut; ++c) dH[blk + 16 * c] = go[c];
		}

		// delta_{H-1} = (W_H^T g_o) . 1[a_H > 0]   (NNBackwardDA3_ReLU, NN_nv.glsl:222-246)
		float4_t d[4];
#pragma unroll
		for (int mt = 0; mt < 4; ++mt) {
			const float4_t *w = S.frag_out + mt * 64 + 16 * g; // W_H[c][16 mt + 4 i + g] at lane row c
			const float4_t w0 = w[0], w1 = w[1], w2 = w[2];
#pragma unroll
			for (int i = 0; i < 4; ++i) {
				float y = w0[i] * go[0];
				y = fmaf(w1[i], go[1], y);
				y = fmaf(w2[i], go[2], y);
				d[mt][i] = relu_mask(y, 4 * mt + i);
			}
		}
		store(deltas + (size_t)(H - 1) * slab, d);
		// delta_{l-1} = (W_l^T delta_l) . 1[a_l > 0], l = H-1..1  (NNBackwardDA64_ReLU, NN_nv.glsl:248-278)
#pragma unroll 1
		for (int l = H - 1; l >= 1; --l) {
			active[0] = __builtin_amdgcn_alignbit(active[1], active[0], 16);
			active[1] = __builtin_amdgcn_alignbit(active[2], active[1], 16);
			active[2] >>= 16;
			float4_t acc[4];
			float w[2][4][4]; // the weights of four K steps, read while the four before them run
			auto read = [&](int mt) __attribute__((always_inline)) {
#pragma unroll
				for (int i = 0; i < 4; ++i)
#pragma unroll
					for (int m = 0; m < 4; ++m) w[mt & 1][i][m] = sf[((l * 4 + mt) * 4 + m) * 256 + tslot[i]];
			};
#pragma unroll
			for (int m = 0; m < 4; ++m) acc[m] = (float4_t)0.0f;
			read(0);
#pragma unroll
			for (int mt = 0; mt < 4; ++mt) {
				if (mt < 3) read(mt + 1);
				__builtin_amdgcn_sched_barrier(0);
#pragma unroll
				for (int i = 0; i < 4; ++i)
#pragma unroll
					for (int m = 0; m < 4; ++m) acc[m] = mfma4(w[mt & 1][i][m], d[mt][i], acc[m]);
				__builtin_amdgcn_sched_barrier(0);
			}
#pragma unroll
			for (int m = 0; m < 4; ++m)
#pragma unroll
				for (int i = 0; i < 4; ++i) d[m][i] = relu_mask(acc[m][i], 4 * m + i);
			store(deltas + (size_t)(l - 1) * slab, d);
		}
		if (t + stride < tiles) load_tile(t + stride); // uniform
	}
}

// Partial dW over one chunk of records: dW_l[m][k] = sum_n delta_l[m][n] a_l[k][n]
// (NNUpdateDW64 / NNUpdateDW3, NN_nv.glsl:280-367), the records in order.  Grid: x over
// the layers, y over chunks; wave w computes two of a layer's sixteen 16x16 tiles as dW^T (A =
// activations, B = deltas, K = records, so a lane stores four consecutive inputs): in the
// stored order a lane group's float4 holds records 4 j + g, the K index g of step j.  The 4 KB
// blocks pass through LDS, two groups of 64 records ahead, so each is read once a layer and
// chunk.  Also writes the chunk's loss sum after the weights and flags
// non-finite partials.  Bound by the FP32 MFMA rate on the CUs that hold a workgroup (160
// for 16,384 records: 512 MFMAs a SIMD, 6.8 us) and by the reads of what the kernel before
// wrote (46 MB, past the L2s).  16,384 records: 65 us with FMAs from LDS tiles, 17.7 with
// operands loaded by each wave for itself, 15.7 now.
constexpr int kTiles = 4; // 16-record tiles a step
template <int H>
__global__ __launch_bounds__(512) void plain_dw_kernel(const uint32_t *__restrict__ d_count, uint32_t max_count,
                                                       uint32_t clamp, const float *__restrict__ acts,
                                                       const float *__restrict__ deltas,
                                                       const float *__restrict__ sample_loss, uint32_t ldn,
                                                       float *__restrict__ partials, uint32_t pstride,
                                                       uint32_t *__restrict__ overflow) {
	constexpr int WC = weight_count(H);
	const uint32_t count = effective_count(d_count, max_count, clamp);
	const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const int g = lane >> 4, r = lane & 15;
	const int l = (int)blockIdx.x; // H: the output layer
	const size_t slab = (size_t)kWidth * ldn;
	const uint32_t nb0 = blockIdx.y * kPlainChunk;
	uint32_t nend = nb0 + kPlainChunk;
	if (nend > count) nend = count;
	float *pp = partials + (size_t)blockIdx.y * pstride;
	bool bad = false;
	auto put = [&](float *dst, float4_t v) __attribute__((always_inline)) {
		*reinterpret_cast<float4_t *>(dst) = v;
#pragma unroll
		for (int i = 0; i < 4; ++i) bad |= !isfinite(v[i]);
	};
	const uint32_t steps = nb0 < nend ? (nend - nb0 + 15) / 16 : 0; // 16-record tiles of this chunk
	if (l < H) {
		// kTiles tiles of a_l and delta_l are in LDS at a time, as they lie in memory; the next
		// two groups are on their way through registers (direct copies to LDS would be waited
		// for, all of them, before every read)
		constexpr int kFloats = kTiles * 16 * kWidth, kPer = kFloats / 4 / 512, kGroups = (int)kPlainChunk / (16 * kTiles);
		__shared__ __attribute__((aligned(16))) float buf[2][2][kFloats];
		const float *src[2] = {acts + (size_t)l * slab + (size_t)nb0 * kWidth, deltas + (size_t)l * slab + (size_t)nb0 * kWidth};
		const uint32_t words = steps * (16 * kWidth), tid = threadIdx.x;
		float4_t next[2][2][kPer];
		auto load = [&](int grp) __attribute__((always_inline)) {
#pragma unroll
			for (int op = 0; op < 2; ++op)
#pragma unroll
				for (int k = 0; k < kPer; ++k) {
					// past the chunk the loads repeat its last piece, which no step reads
					const uint32_t w = (uint32_t)(grp * kFloats + k * 2048) + 4u * tid;
					next[grp & 1][op][k] = *reinterpret_cast<const float4_t *>(src[op] + (w < words ? w : words - 4u));
				}
		};
		auto store = [&](int grp) __attribute__((always_inline)) {
#pragma unroll
			for (int op = 0; op < 2; ++op)
#pragma unroll
				for (int k = 0; k < kPer; ++k) *reinterpret_cast<float4_t *>(&buf[grp & 1][op][k * 2048 + 4u * tid]) = next[grp & 1][op][k];
		};
		const int it0 = 2 * (wave & 1), ot = wave >> 1;
		float4_t acc[2] = {(float4_t)0.0f, (float4_t)0.0f};
		if (steps > 0) {
			load(0);
			load(1);
			store(0);
		}
#pragma unroll
		for (int grp = 0; grp < kGroups; ++grp) {
			if ((uint32_t)(grp * kTiles) >= steps) break; // uniform
			load(grp + 2);
			block_lds_sync();
			const float4_t *pa = reinterpret_cast<const float4_t *>(buf[grp & 1][0]) + (16 * it0 + r) * 4 + g;
			const float4_t *pd = reinterpret_cast<const float4_t *>(buf[grp & 1][1]) + (16 * ot + r) * 4 + g;
#pragma unroll
			for (int k = 0; k < kTiles; ++k) {
				if ((uint32_t)(grp * kTiles + k) >= steps) break; // uniform
				const float4_t a0 = pa[k * 256], a1 = pa[k * 256 + 64], d = pd[k * 256];
#pragma unroll
				for (int e = 0; e < 4; ++e) {
					acc[0] = mfma4(a0[e], d[e], acc[0]);
					acc[1] = mfma4(a1[e], d[e], acc[1]);
				}
			}
			store(grp + 1); // into the buffer that the group before this one was read from
		}
#pragma unroll
		for (int i = 0; i < 2; ++i) put(pp + l * kWidth * kWidth + (16 * ot + r) * kWidth + 16 * (it0 + i) + 4 * g, acc[i]);
	} else {
		// the output layer: wave w < 4 computes input tile w against the three output rows
		if (wave < 4) {
			const bool live = r < kOut;
			const float *a = acts + (size_t)H * slab + (size_t)nb0 * kWidth + 16 * (16 * wave + r) + 4 * g;
			const float *d = deltas + (size_t)H * slab + (size_t)nb0 * kWidth + 16 * (live ? r : 0) + 4 * g;
			float4_t acc = (float4_t)0.0f;
#pragma unroll 8
			for (uint32_t k = 0; k < steps; ++k) {
				const float4_t av = *reinterpret_cast<const float4_t *>(a + (size_t)k * (16 * kWidth));
				const float4_t dv = *reinterpret_cast<const float4_t *>(d + (size_t)k * (16 * kWidth));
#pragma unroll
				for (int e = 0; e < 4; ++e) acc = mfma4(av[e], live ? dv[e] : 0.0f, acc);
			}
			if (live) put(pp + H * kWidth * kWidth + r * kWidth + 16 * wave + 4 * g, acc);
		}
		__shared__ float sl[256];
		const int t = threadIdx.x;
		float v = 0.0f;
		if (t < 256) {
			for (uint32_t n = nb0 + t; n < nend; n += 256) v += sample_loss[n];
			sl[t] = v;
		}
		__syncthreads();
		for (int s = 128; s > 0; s >>= 1) {
			if (t < s) sl[t] += sl[t + s];
			__syncthreads();
		}
		if (t == 0) pp[WC] = sl[0];
	}
	if (__any(bad) && lane == 0) atomicOr(overflow, 1u);
}

template <int ENC>
__global__ __launch_bounds__(256) void encode_kernel(const float *__restrict__ queries, uint32_t n,
                                                     float *__restrict__ feat) {
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n) return;
	float rec[kQueryFloats];
	load_query(queries + (size_t)i * kQueryFloats, rec);
	float f[kWidth];
	encode_all<ENC>(rec, f);
#pragma unroll
	for (int k = 0; k < kWidth; k += 4)
		*reinterpret_cast<float4 *>(feat + (size_t)i * kWidth + k) = make_float4(f[k], f[k + 1], f[k + 2], f[k + 3]);
}

__global__ __launch_bounds__(256) void sph_kernel(const float *__restrict__ dirs, uint32_t n, float *__restrict__ uv) {
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n) return;
	float o[2];
	sph_encode(dirs[3 * i], dirs[3 * i + 1], dirs[3 * i + 2], o);
	uv[2 * i] = o[0];
	uv[2 * i + 1] = o[1];
}

// One workgroup a CU, and no more than there are tiles.
uint32_t plain_blocks(uint32_t n) {
	const uint32_t tiles = (n + 15) / 16, cus = (uint32_t)device_cu_count();
	return tiles < cus ? tiles : cus;
}

template <int H>
hipError_t plain_infer_h(int enc, const float *q, const uint32_t *dc, uint32_t mc, const float *w, float *rgb,
                         hipStream_t s) {
	const dim3 grid(plain_blocks(mc)), block(64 * kPlainInferWaves);
	switch (enc) {
	case NRC_ENCODING_TRI12: plain_infer_kernel<H, NRC_ENCODING_TRI12><<<grid, block, 0, s>>>(q, dc, mc, w, rgb); break;
	case NRC_ENCODING_SINCOS6: plain_infer_kernel<H, NRC_ENCODING_SINCOS6><<<grid, block, 0, s>>>(q, dc, mc, w, rgb); break;
	default: plain_infer_kernel<H, NRC_ENCODING_UV_SINCOS16><<<grid, block, 0, s>>>(q, dc, mc, w, rgb); break;
	}
	return hipGetLastError();
}

template <int H, int ENC, int LOSS> void plain_fwdbwd_launch(const TrainArgs &a, hipStream_t s) {
	const dim3 grid(plain_blocks(a.max_count < a.clamp ? a.max_count : a.clamp)), block(64 * kPlainWaves);
	plain_fwdbwd_kernel<H, ENC, LOSS><<<grid, block, 0, s>>>(a.records, a.d_count, a.max_count, a.clamp, a.w32,
	                                                          a.state, a.parity, a.acts, a.deltas, a.sample_loss, a.ldn);
}

template <int H, int ENC> void plain_fwdbwd_loss(const TrainArgs &a, hipStream_t s) {
	if (a.loss == NRC_LOSS_L2) plain_fwdbwd_launch<H, ENC, NRC_LOSS_L2>(a, s);
	else plain_fwdbwd_launch<H, ENC, NRC_LOSS_RELATIVE_L2_LUMINANCE>(a, s);
}

template <int H> void plain_gradient_h(const TrainArgs &a, uint32_t nparts, hipStream_t s) {
	switch (a.encoding) {
	case NRC_ENCODING_TRI12: plain_fwdbwd_loss<H, NRC_ENCODING_TRI12>(a, s); break;
	case NRC_ENCODING_SINCOS6: plain_fwdbwd_loss<H, NRC_ENCODING_SINCOS6>(a, s); break;
	default: plain_fwdbwd_loss<H, NRC_ENCODING_UV_SINCOS16>(a, s); break;
	}
	const dim3 grid(H + 1, nparts), block(512);
	plain_dw_kernel<H><<<grid, block, 0, s>>>(a.d_count, a.max_count, a.clamp, a.acts, a.deltas, a.sample_loss, a.ldn,
	                                          a.partials, a.pstride, &a.state->overflow[a.parity]);
}

} // namespace

hipError_t launch_plain_infer(int hidden, int encoding, const float *queries, const uint32_t *d_count,
                              uint32_t max_count, const float *w32, float *rgb, hipStream_t stream) {
	if (max_count == 0) return hipSuccess;
	if (hidden == 5) return plain_infer_h<5>(encoding, queries, d_count, max_count, w32, rgb, stream);
	return plain_infer_h<4>(encoding, queries, d_count, max_count, w32, rgb, stream);
}

hipError_t launch_plain_gradient(const TrainArgs &a, uint32_t *nparts, hipStream_t stream) {
	const uint32_t n = a.max_count < a.clamp ? a.max_count : a.clamp;
	*nparts = (n + kPlainChunk - 1) / kPlainChunk;
	if (*nparts == 0) *nparts = 1;
	if (a.hidden == 5) plain_gradient_h<5>(a, *nparts, stream);
	else plain_gradient_h<4>(a, *nparts, stream);
	return hipGetLastError();
}

hipError_t launch_encode(int encoding, const float *queries, uint32_t n, float *features, hipStream_t stream) {
	if (n == 0) return hipSuccess;
	const dim3 grid((n + 255) / 256), block(256);
	switch (encoding) {
	case NRC_ENCODING_TRI12: encode_kernel<NRC_ENCODING_TRI12><<<grid, block, 0, stream>>>(queries, n, features); break;
	case NRC_ENCODING_SINCOS6: encode_kernel<NRC_ENCODING_SINCOS6><<<grid, block, 0, stream>>>(queries, n, features); break;
	default: encode_kernel<NRC_ENCODING_UV_SINCOS16><<<grid, block, 0, stream>>>(queries, n, features); break;
	}
	return hipGetLastError();
}

hipError_t launch_sph_encode(const float *dirs, uint32_t n, float *uv, hipStream_t stream) {
	if (n == 0) return hipSuccess;
	sph_kernel<<<dim3((n + 255) / 256), dim3(256), 0, stream>>>(dirs, n, uv);
	return hipGetLastError();
}

namespace {
// nrc_inference.comp:50-72: one thread per query.
__global__ __launch_bounds__(256) void composite_kernel(const CompositeArgs a) {
	const uint32_t i = blockIdx.x * 256u + threadIdx.x;
	const uint32_t count = effective_count(a.d_count, a.max_count, a.max_count);
	if (i >= count) return;
	const uint32_t e = a.dst[i];
	if (e == 0xFFFFFFFFu) return;
	const float p0 = a.rgb[(size_t)i * 3], p1 = a.rgb[(size_t)i * 3 + 1], p2 = a.rgb[(size_t)i * 3 + 2];
	const uint32_t v = e >> 1;
	// fields decoded as DecodeNRCEvalDstScreen/Train do (NRCRecord.glsl:24-33): the
	// top field keeps every remaining bit, so an over-wide y or r falls outside the
	// image or the batch and is skipped
	if ((e & 1u) == 0u) { // screen
		const uint32_t x = v & 0x7FFFu, y = v >> 15;
		if (a.bias_factor_r == nullptr || x >= a.width || y >= a.height) return;
		const size_t px = (size_t)y * a.pitch + x;
		float4 *bf = reinterpret_cast<float4 *>(a.bias_factor_r) + px;
		const float4 b = *bf;
		const float2 f = reinterpret_cast<const float2 *>(a.factor_gb)[px];
		*bf = make_float4(mul_add_rn(b.x, b.w, p0), mul_add_rn(b.y, f.x, p1), mul_add_rn(b.z, f.y, p2), 0.0f);
	} else { // train
		const uint32_t b = v & 3u, l = (v >> 2) & 0x3FFFu, r = v >> 16;
		if (a.batches == nullptr) return;
		const uint32_t rr = r < a.batch_stride ? r : a.batch_stride - 1u;
		for (uint32_t j = l; j <= rr && j < a.batch_stride; ++j) {
			const size_t row = (size_t)b * a.batch_stride + j;
			float *t = a.batches + row * kTrainFloats + kQueryFloats;
			const float *f = a.factors + row * 3;
			t[0] = mul_add_rn(t[0], f[0], p0);
			t[1] = mul_add_rn(t[1], f[1], p1);
			t[2] = mul_add_rn(t[2], f[2], p2);
		}
	}
}
} // namespace

hipError_t launch_composite(const CompositeArgs &a, hipStream_t stream) {
	if (a.max_count == 0) return hipSuccess;
	composite_kernel<<<dim3((a.max_count + 255) / 256), dim3(256), 0, stream>>>(a);
	return hipGetLastError();
}

} // namespace nrc
