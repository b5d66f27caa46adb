// The front half of grid self-attention in one pass over the pair tensor (bf16, 128 channels, 4 heads of 32): LayerNorm, the pair
// bias and the four projections,
//     normed = (x - mean) * rstd * gamma + beta (rounded to bf16),   bias[h][i][j] = normed[i][j] . Wb[h],
//     q, k, v, gate [B, 4, N, 32] = normed . Wq, Wk, Wv, Wg,
// for attention along j (B = i, N = j) or, turned, along i (B = j, N = i).  q leaves multiplied by q_scale, rounded once.
// Reference: src/af3_kernels/Attention.py:51-52 and the projections of _attention_impl, src/csrc/dot_product_attention.cpp:275-345.
//
// Bound by memory: a token's 256 bytes come in once and its 1024 + 8 bytes go out (N = 384: 190 MB, 37 us at the rate of a large copy).
// The attention then runs on the shared-bias kernel (four batch rows per wavefront), whose rate the one-kernel form
// (dpa_mfma.hip, FUSED: a workgroup per batch row and head, projections inside) does not reach; the round trip of q, k, v and
// the gate costs less than that difference, and short rows no longer pay a workgroup's projection of all keys.
//
// Work split.  All 512 weight columns stay in LDS (128 KB, in operand order) for a workgroup's whole life: one workgroup of 12 wavefronts per compute
// unit, each walking blocks of 32 consecutive tokens j of a row i on its own, without barriers (with few tokens: workgroups
// of one head each).  LayerNorm works on rows as they
// are loaded (a load is four whole rows, a row sixteen lanes); the normalised rows turn through 2 KB of LDS per wavefront into the B
// operand of out^T = W^T . x^T: channels 64 g + 8 s + 0..7 are contraction slots of step s in half-wave g.  (Loading the operand itself, 16 bytes
// from each of 64 lines per load, refetched lines that the L1 could not hold: N = 128 10.9 us.)  Weight rows are permuted so that a lane's 16
// results are consecutive channels, and a 32 x 32 tile leaves through the same 2 KB as two stores of 1 KB.
#include "mfma_helpers.hpp"

namespace af3 {

namespace {

constexpr int GP_WAVES = 12, GP_C = 128;
constexpr int GP_PATCH = 16 * 8192, GP_WB = GP_PATCH + GP_WAVES * 2048, GP_LDS = GP_WB + 4 * 256;

// sum over the 16 lanes of a DPP row; every lane of the row receives the total
template <int CTRL>
__device__ __forceinline__ float dpp_add(float x) {
	return x + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float row16_sum(float x) {
	x = dpp_add<0xB1>(x);   // quad_perm [1,0,3,2]
	x = dpp_add<0x4E>(x);   // quad_perm [2,3,0,1]
	x = dpp_add<0x141>(x);  // row_half_mirror
	x = dpp_add<0x140>(x);  // row_mirror
	return x;
}

struct grid_project_args {
	const uint16_t* x;
	int64_t         x_stride_i, x_stride_j;   // elements
	const uint16_t *gamma, *beta, *wb;        // [128], [128], [4, 128]
	const uint32_t* w[4];                     // k, v, q, gate: weight^T in panel layout [head][64][32][2]
	uint16_t*       out[4];                   // k, v, q, gate: [B, 4, N, 32] (null: the bias alone)
	uint16_t*       bias;                     // [4, n_i, n_j] (null: the projections alone)
	int             n_i, n_j, turned, split;
	float           eps, q_scale;
};

__global__ void __launch_bounds__(GP_WAVES * 64) __attribute__((amdgpu_waves_per_eu(3))) grid_project_kernel(grid_project_args a) {
	extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int n = lane & 31, half = lane >> 5;

	const int      blocks_per_row = (a.n_j + 31) / 32;
	const int64_t  n_blocks = (int64_t)a.n_i * blocks_per_row;
	// split: this workgroup projects for head blockIdx % 4 alone (a quarter of the weights, four times the workgroups per block)
	const int      h0 = a.split ? (int)(blockIdx.x & 3) : 0, h1 = a.split ? h0 + 1 : a.out[0] ? 4 : 0;
	const int      wgs = a.split ? (int)(gridDim.x >> 2) : (int)gridDim.x, wg = a.split ? (int)(blockIdx.x >> 2) : (int)blockIdx.x;
	const int64_t  step = (int64_t)wgs * GP_WAVES;
	int64_t        u = (int64_t)wave * wgs + wg;   // (first one block per workgroup, then two, ...)
	u32x4 raw[8];   // row 4 k + lane / 16 of the block, channels 8 (lane % 16) ..: one load is four whole rows
	auto  load = [&](int64_t unit) {
		const uint32_t blk = (uint32_t)unit;
		const int      i = (int)(blk / (uint32_t)blocks_per_row), j0 = (int)(blk % (uint32_t)blocks_per_row) * 32;
#pragma unroll
		for(int k = 0; k < 8; k++) {
			const int j = j0 + 4 * k + (lane >> 4) < a.n_j ? j0 + 4 * k + (lane >> 4) : a.n_j - 1;
			raw[k] = *reinterpret_cast<const u32x4*>(a.x + (int64_t)i * a.x_stride_i + (int64_t)j * a.x_stride_j + 8 * (lane & 15));
		}
	};
	if(u < n_blocks) load(u);
	const u32x4 gam = *reinterpret_cast<const u32x4*>(a.gamma + 8 * (lane & 15)), bet = *reinterpret_cast<const u32x4*>(a.beta + 8 * (lane & 15));

	// ---- weights -> LDS: [tile = 4 head + {k, v, q, gate}][step s][lane] x 16 bytes.  Row r of a tile is channel 16 ((r >> 2) & 1) + 4 (r >> 3) + (r & 3)
	// (register i of half-wave g then holds channel 16 g + i); slots j of lane (r, g): input channels 64 g + 8 s + j.
	{
		const int r = n, d = 16 * ((r >> 2) & 1) + 4 * (r >> 3) + (r & 3);
		constexpr int PER_WAVE = (16 * 8 + GP_WAVES - 1) / GP_WAVES;
		u32x4         wr[PER_WAVE];   // (all of a wavefront's pieces under way together: one latency)
#pragma unroll
		for(int k = 0; k < PER_WAVE; k++) {
			const int f = wave + k * GP_WAVES, t = f >> 3, s = f & 7;
			if(t < 4 * h0 || t >= 4 * h1) continue;
			const uint32_t* wp = a.w[t & 3] + (t >> 2) * (GP_C / 2 * 32) + (32 * half + 4 * s) * 32 + d;
			wr[k] = u32x4{wp[0], wp[32], wp[64], wp[96]};
		}
#pragma unroll
		for(int k = 0; k < PER_WAVE; k++)
			if((wave + k * GP_WAVES) >> 3 >= 4 * h0 && (wave + k * GP_WAVES) >> 3 < 4 * h1) *reinterpret_cast<u32x4*>(smem + (wave + k * GP_WAVES) * 1024 + lane * 16) = wr[k];
		for(int c = tid; c < 64; c += GP_WAVES * 64) *reinterpret_cast<u32x4*>(smem + GP_WB + c * 16) = *reinterpret_cast<const u32x4*>(a.wb + c * 8);
	}
	__syncthreads();

	unsigned char* const patch = smem + GP_PATCH + wave * 2048;
	const int            sw_w = (n >> 2) & 3;
	const int            p_wr0 = n * 64 + (((2 * half) ^ sw_w) << 4), p_wr1 = n * 64 + (((2 * half + 1) ^ sw_w) << 4);
	const int            p_row = lane >> 2, p_rd = p_row * 64 + (((lane & 3) ^ ((p_row >> 2) & 3)) << 4);   // (+ 1024: rows 16.., same swizzle)

	for(; u < n_blocks; u += step) {
		const uint32_t blk = (uint32_t)u;
		const int      i = (int)(blk / (uint32_t)blocks_per_row), j0 = (int)(blk % (uint32_t)blocks_per_row) * 32;

		// ---- LayerNorm in registers, a row in sixteen lanes: mean, centred sum of squares, normalise (fp32), round; eight rows at
		// a time then turn through the patch into the B operand: lane (token n, half g), step s: channels 64 g + 8 s .. + 7 ----
		bf16x8 xf[8];
#pragma unroll
		for(int rho = 0; rho < 4; rho++) {
#pragma unroll
			for(int z = 0; z < 2; z++) {
				float v[8];
#pragma unroll
				for(int c = 0; c < 4; c++) v[2 * c] = bf16_bits_to_f32(raw[2 * rho + z][c] & 0xffffu), v[2 * c + 1] = __uint_as_float(raw[2 * rho + z][c] & 0xffff0000u);
				float sum = 0.f, ss = 0.f;
#pragma unroll
				for(int c = 0; c < 8; c++) sum += v[c];
				const float mean = row16_sum(sum) * (1.f / GP_C);
#pragma unroll
				for(int c = 0; c < 8; c++) {
					v[c] -= mean;
					ss = __builtin_fmaf(v[c], v[c], ss);
				}
				const float rstd = __builtin_amdgcn_rsqf(row16_sum(ss) * (1.f / GP_C) + a.eps);
				u32x4       o;
#pragma unroll
				for(int c = 0; c < 4; c++)
					o[c] = pack_bf16x2(__builtin_fmaf(v[2 * c] * rstd, bf16_bits_to_f32(gam[c] & 0xffffu), bf16_bits_to_f32(bet[c] & 0xffffu)),
									   __builtin_fmaf(v[2 * c + 1] * rstd, __uint_as_float(gam[c] & 0xffff0000u), __uint_as_float(bet[c] & 0xffff0000u)));
				const int r = 4 * z + (lane >> 4);   // row within the eight; its 16-byte chunks XOR-swizzled with it
				*reinterpret_cast<u32x4*>(patch + r * 256 + (((lane & 15) ^ r) << 4)) = o;
			}
			__builtin_amdgcn_wave_barrier();
			if((n >> 3) == rho) {
#pragma unroll
				for(int s = 0; s < 8; s++) xf[s] = *reinterpret_cast<const bf16x8*>(patch + (n & 7) * 256 + (((8 * half + s) ^ (n & 7)) << 4));
			}
			__builtin_amdgcn_wave_barrier();
		}
		if(u + step < n_blocks) load(u + step);   // (under way during this block's products)

		// ---- pair bias: every row of the operand is one of the four heads', so that every lane has all four values of its token ----
		if(h0 == 0 && a.bias) {
			f32x16 acc;
#pragma unroll
			for(int k = 0; k < 16; k++) acc[k] = 0.f;
#pragma unroll
			for(int s = 0; s < 8; s++)
				acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8*>(smem + GP_WB + (n & 3) * 256 + half * 128 + s * 16), xf[s], acc, 0, 0, 0);
			if(j0 + n < a.n_j) {
				uint16_t* bp = a.bias + ((int64_t)(2 * half) * a.n_i + i) * a.n_j + j0 + n;
				bp[0] = (uint16_t)f32_to_bf16_bits(half ? acc[2] : acc[0]);
				bp[(int64_t)a.n_i * a.n_j] = (uint16_t)f32_to_bf16_bits(half ? acc[3] : acc[1]);
			}
		}

		// ---- q, k, v, gate: two tiles at a time ----
		const int     left = a.n_j - j0;
		const int64_t tok0 = a.turned ? (int64_t)j0 * 4 * a.n_i + i : (int64_t)i * 4 * a.n_j + j0;      // [B, 4, N]: token j0 of head 0
		const int64_t tok_step = a.turned ? (int64_t)4 * a.n_i : 1, head_step = a.turned ? a.n_i : a.n_j;
#pragma unroll 1
		for(int t = 4 * h0; t < 4 * h1; t += 2) {
			f32x16 acc[2];
#pragma unroll
			for(int k = 0; k < 16; k++) acc[0][k] = 0.f, acc[1][k] = 0.f;
#pragma unroll
			for(int s = 0; s < 8; s++) {
				if(s == 4) __builtin_amdgcn_sched_barrier(0);   // (not all sixteen operands in registers at once)
#pragma unroll
				for(int z = 0; z < 2; z++) acc[z] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8*>(smem + (t + z) * 8192 + s * 1024 + lane * 16), xf[s], acc[z], 0, 0, 0);
			}
			const bool second = (t & 2) != 0;   // tiles q, gate (otherwise k, v)
			const float m0 = second ? a.q_scale : 1.f;
#pragma unroll
			for(int z = 0; z < 2; z++) {
				u32x4 w[2];
#pragma unroll
				for(int k = 0; k < 8; k++) {
					float lo = acc[z][2 * k], hi = acc[z][2 * k + 1];
					if(z == 0) lo *= m0, hi *= m0;
					w[k >> 2][k & 3] = pack_bf16x2(lo, hi);
				}
				*reinterpret_cast<u32x4*>(patch + p_wr0) = w[0];
				*reinterpret_cast<u32x4*>(patch + p_wr1) = w[1];
				__builtin_amdgcn_wave_barrier();   // (a wavefront's LDS operations complete in order; this only holds the compiler)
				uint16_t* const dst = (second ? a.out[2 + z] : a.out[z]) + (tok0 + (t >> 2) * head_step) * 32 + (lane & 3) * 8;
#pragma unroll
				for(int y = 0; y < 2; y++) {
					const u32x4 v = *reinterpret_cast<const u32x4*>(patch + p_rd + y * 1024);
					if(p_row + 16 * y < left) *reinterpret_cast<u32x4*>(dst + (p_row + 16 * y) * tok_step * 32) = v;
				}
				__builtin_amdgcn_wave_barrier();
			}
		}
	}
}

}  // namespace

}  // namespace af3

using namespace af3;

// For the Python entry points' native host side (host.cpp); not part of the ABI.  pair [n_i, n_j, 128] (strides in elements), ln_weight,
// ln_bias [128], proj [4, 128], q/k/v/gate weights in panel layout, all bf16; outputs as in the kernel (q, k, v and gate, or bias, may be null).
extern "C" int af3_grid_project(const void* pair, const int64_t* pair_stride, const void* ln_weight, const void* ln_bias, float eps, const void* proj, const void* wq, const void* wk, const void* wv,
								const void* wg, int64_t n_i, int64_t n_j, int32_t turned, float q_scale, void* q, void* k, void* v, void* gate, void* bias, void* stream) {
	for(const void* p : {pair, ln_weight, ln_bias, proj, wq, wk, wv, wg})
		if(!p) return AF3_ERR_NULL_POINTER;
	const bool projected = q && k && v && gate;
	if(!projected && (!bias || q || k || v || gate)) return AF3_ERR_NULL_POINTER;
	if(n_i <= 0 || n_j <= 0 || n_i > (1 << 20) || n_j > (1 << 20) || n_i * ((n_j + 31) / 32) >= ((int64_t)1 << 31)) return AF3_ERR_BAD_SHAPE;
	for(const void* p : {pair, ln_weight, ln_bias, proj})
		if(reinterpret_cast<uintptr_t>(p) & 15) return AF3_ERR_BAD_ARGUMENT;
	if(pair_stride[0] % 8 || pair_stride[1] % 8) return AF3_ERR_BAD_ARGUMENT;
	grid_project_args a{};
	a.x = static_cast<const uint16_t*>(pair), a.x_stride_i = pair_stride[0], a.x_stride_j = pair_stride[1];
	a.gamma = static_cast<const uint16_t*>(ln_weight), a.beta = static_cast<const uint16_t*>(ln_bias), a.wb = static_cast<const uint16_t*>(proj);
	const void* w[4] = {wk, wv, wq, wg};
	void*       o[4] = {k, v, q, gate};
	for(int t = 0; t < 4; t++) {
		if((reinterpret_cast<uintptr_t>(w[t]) & 3) || (reinterpret_cast<uintptr_t>(o[t]) & 15)) return AF3_ERR_BAD_ARGUMENT;
		a.w[t] = static_cast<const uint32_t*>(w[t]), a.out[t] = static_cast<uint16_t*>(o[t]);
	}
	a.bias = static_cast<uint16_t*>(bias), a.n_i = (int)n_i, a.n_j = (int)n_j, a.turned = turned ? 1 : 0, a.eps = eps, a.q_scale = q_scale;
	const int64_t blocks = n_i * ((n_j + 31) / 32);
	// Few blocks (up to three of the twelve wavefronts of every compute unit): a workgroup per head, which shares the products among four times the
	// wavefronts and loads a quarter of the weights.
	a.split = projected && blocks <= 64 * GP_WAVES ? 1 : 0;
	const int64_t wgs = a.split ? 4 * (blocks < 64 ? blocks : 64) : blocks < 256 ? blocks : 256;
	if(hipFuncSetAttribute(reinterpret_cast<const void*>(grid_project_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, GP_LDS) != hipSuccess) return AF3_ERR_LAUNCH;
	hipLaunchKernelGGL(grid_project_kernel, dim3((unsigned)wgs), dim3(GP_WAVES * 64), GP_LDS, static_cast<hipStream_t>(stream), a);
	return launch_status();
}
