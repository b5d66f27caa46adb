// The four projections of a self-attention block as one product: out[M, N] = x[M, K] . W^T + row, W [N, K] (N = 4K output
// columns, ordered per head k | v | q | gate), the row (the q bias) added in fp32, one rounding to bf16.
// Reference: the four BRGEMMs of self_attention_impl, src/csrc/dot_product_attention.cpp:421-497.
//
// A diffusion step calls this with 60 to 2000 tokens and 384 or 768 channels: 0.03 to 10 GFLOP.  Up to there what bounds the
// call is one round of workgroups (time of one workgroup, not of the chip), and, through a library, the 18 us of host time
// that choosing a solution takes.  Work split: four computing wavefronts (2 x 2) own 64 A tokens x 64 B columns and walk K in
// slabs of 64 channels; four loading wavefronts, one per SIMD, fill a ring of slabs in LDS by loads that write LDS directly.
// (Without them the computing wavefronts stood behind their own loads: 1536 x 3072 x 768 14.4 instead of 11.7 us, 513 x 3072 x
// 768 7.1 instead of 5.9.)  In a slab LDS is the bound: for 128 x 192 columns 80 KB of operand reads and 40 KB of arriving
// data per 768 clocks of matrix work, 0.50 us measured; fetching operands a group ahead, across the barrier, gained nothing.
// The 16-byte chunks of a row (128 bytes) are XOR-swizzled by the lane that fetches them, so that the operand reads of 32
// rows spread over the banks.  out^T = W . x^T on v_mfma_f32_32x32x16_bf16: a lane holds four times four consecutive columns
// of one token, the accumulators start from the row, and the result leaves through a patch of LDS per wavefront as whole
// 16-byte stores.
// us per call, this kernel / hipBLASLt (device time, graph replays), K = 768, N = 3072: M = 64 4.6/5.6, 256 4.9/6.6, 768 7.9/10.0,
// 1024 8.6/11.0, 1536 11.7/12.3, 2048 13.5/15.0, 3840 25.9/22.7; K = 384, N = 1536: 64 3.4/4.9, 1024 4.4/6.8, 2048 6.5/9.2,
// 7680 17.9/22.7.  The library keeps what is larger than that (af3_project_suits).
#include "mfma_helpers.hpp"

namespace af3 {

namespace {

constexpr int SLAB = 64;   // channels per step

template <int A, int B, int NBUF>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) projection_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, const uint16_t* __restrict__ row,
																								   uint16_t* __restrict__ out, int M, int N, int K, int m_tiles, int n_tiles) {
	constexpr int TM = 64 * A, TN = 64 * B, X_BYTES = TM * SLAB * 2, SLAB_BYTES = (TM + TN) * SLAB * 2;
	constexpr int PIECES = (TM + TN) / 8, PER_WAVE = PIECES / 4;   // 1 KB loads (eight rows) of a slab: all, per wavefront
	constexpr int PATCH_ROW = B * 64 + 16;                         // bytes of a token's row in the output patch, padded against bank conflicts
	static_assert(PIECES % 4 == 0 && 4 * 32 * PATCH_ROW <= NBUF * SLAB_BYTES, "pieces divide, the patches fit");
	extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];   // [slab 3][x rows TM | W rows TN][128 bytes]

	// Workgroup -> tile: ids congruent mod 8 run on one XCD; each takes a run of consecutive tiles, column tile slowest, so that
	// an XCD's L2 holds a few column tiles of W and passes x once.
	const int total = m_tiles * n_tiles, per_xcd = (total + 7) / 8;
	const int t = (int)(blockIdx.x & 7) * per_xcd + (int)(blockIdx.x >> 3);
	if((int)(blockIdx.x >> 3) >= per_xcd || t >= total) return;
	const int m0 = (t % m_tiles) * TM, n0 = (t / m_tiles) * TN;

	const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
	const int n = lane & 31, half = lane >> 5;
	const int wm = wave & 1, wn = wave >> 1;   // this wavefront's tokens [32 A wm, ..) and columns [32 B wn, ..) of the tile

	// pieces wave, wave + 4, ...: lane i -> row i / 8 of the piece, chunk position i % 8, which holds chunk (i % 8) ^ (row % 8).
	// Rows past M or N lie past the range: nothing is fetched for them, and what a column of the product made of them is not stored.
	const u32x4    x_rsrc = raw_rsrc(x + (int64_t)m0 * K, (uint32_t)((M - m0) * K * 2));
	const u32x4    w_rsrc = raw_rsrc(w + (int64_t)n0 * K, (uint32_t)((N - n0) * K * 2));
	const int      voff   = (lane >> 3) * K * 2 + (((lane & 7) ^ (lane >> 3)) << 4);
	const uint32_t lds    = lds_addr_of(smem);
	const int slabs = K / SLAB;

	if(wave >= 4) {
		// ---- a loading wavefront ----
		const int ld = wave - 4;
		auto load_slab = [&](int s, int buf) {
#pragma unroll
			for(int i = 0; i < PER_WAVE; i++) {
				const int  j = ld + 4 * i;           // (pieces [0, TM / 8) are x)
				const bool is_x = j < TM / 8;
				const int  r0 = is_x ? j * 8 : j * 8 - TM;
				lds_dma_b128(is_x ? x_rsrc : w_rsrc, lds + buf * SLAB_BYTES + j * 1024, voff + r0 * K * 2 + s * (SLAB * 2));
			}
		};
#pragma unroll
		for(int s = 0; s < NBUF - 1; s++)
			if(s < slabs) load_slab(s, s);
		int bufp = NBUF - 1;   // the buffer of slab s - 1 = slab s + NBUF - 1
		for(int s = 0; s < slabs; s++) {
			// slab s has landed (up to NBUF - 2 younger ones may be under way); behind the barrier every wavefront is done with slab s - 1
			if(s + NBUF - 2 < slabs) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(PER_WAVE * (NBUF - 2)) : "memory");
			else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
			if(s + NBUF - 1 < slabs) load_slab(s + NBUF - 1, bufp);
			bufp = bufp == NBUF - 1 ? 0 : bufp + 1;
		}
		__syncthreads();
		return;
	}

	f32x16 acc[B][A];
#pragma unroll
	for(int b = 0; b < B; b++) {
		f32x16 init;
#pragma unroll
		for(int g4 = 0; g4 < 4; g4++) {   // register i <-> column 8 (i / 4) + 4 half + i % 4
			const int col = n0 + (wn * B + b) * 32 + 8 * g4 + 4 * half;
			u32x2     r   = {0u, 0u};
			if(row && col < N) r = *reinterpret_cast<const u32x2*>(row + col);
			init[4 * g4] = bf16_bits_to_f32(r[0] & 0xffffu), init[4 * g4 + 1] = bf16_bits_to_f32(r[0] >> 16);
			init[4 * g4 + 2] = bf16_bits_to_f32(r[1] & 0xffffu), init[4 * g4 + 3] = bf16_bits_to_f32(r[1] >> 16);
		}
#pragma unroll
		for(int a = 0; a < A; a++) acc[b][a] = init;
	}

	const int sw = n & 7;
	const int x_rd = (wm * A * 32 + n) * 128, w_rd = X_BYTES + (wn * B * 32 + n) * 128;
	int buf = 0;
	for(int s = 0; s < slabs; s++) {
		asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // slab s is in LDS; every wavefront's reads of slab s - 1 have returned
		const unsigned char* const base = smem + buf * SLAB_BYTES;
#pragma unroll
		for(int c = 0; c < SLAB / 16; c++) {
			const int ch = ((2 * c + half) ^ sw) << 4;
			bf16x8    xf[A], wf[B];
#pragma unroll
			for(int a = 0; a < A; a++) xf[a] = *reinterpret_cast<const bf16x8*>(base + x_rd + a * 4096 + ch);
#pragma unroll
			for(int b = 0; b < B; b++) wf[b] = *reinterpret_cast<const bf16x8*>(base + w_rd + b * 4096 + ch);
#pragma unroll
			for(int b = 0; b < B; b++)
#pragma unroll
				for(int a = 0; a < A; a++) acc[b][a] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(wf[b], xf[a], acc[b][a], 0, 0, 0);
		}
		buf = buf == NBUF - 1 ? 0 : buf + 1;
	}
	__syncthreads();   // the slabs are dead: their memory becomes the patches

	unsigned char* const patch = smem + wave * (32 * PATCH_ROW);
	const int            col0  = n0 + wn * B * 32;
#pragma unroll
	for(int a = 0; a < A; a++) {
#pragma unroll
		for(int b = 0; b < B; b++)
#pragma unroll
			for(int g4 = 0; g4 < 4; g4++)
				*reinterpret_cast<u32x2*>(patch + n * PATCH_ROW + b * 64 + g4 * 16 + half * 8) =
					u32x2{pack_bf16x2(acc[b][a][4 * g4], acc[b][a][4 * g4 + 1]), pack_bf16x2(acc[b][a][4 * g4 + 2], acc[b][a][4 * g4 + 3])};
		__builtin_amdgcn_wave_barrier();   // (a wavefront's LDS operations complete in order; this only holds the compiler)
		const int token0 = m0 + (wm * A + a) * 32;
#pragma unroll
		for(int i = 0; i < 2 * B; i++) {   // 32 rows of 4 B chunks
			const int id = lane + 64 * i, r = id / (4 * B), c = id % (4 * B);
			const u32x4 v = *reinterpret_cast<const u32x4*>(patch + r * PATCH_ROW + c * 16);
			if(token0 + r < M && col0 + c * 8 < N) *reinterpret_cast<u32x4*>(out + (int64_t)(token0 + r) * N + col0 + c * 8) = v;
		}
		__builtin_amdgcn_wave_barrier();
	}
}

template <int A, int B, int NBUF>
int launch(const uint16_t* x, const uint16_t* w, const uint16_t* row, uint16_t* out, int M, int N, int K, hipStream_t s) {
	const int    m_tiles = (M + 64 * A - 1) / (64 * A), n_tiles = (N + 64 * B - 1) / (64 * B);
	const size_t smem    = (size_t)NBUF * 64 * (A + B) * SLAB * 2;
	auto         kern    = projection_kernel<A, B, NBUF>;
	if(smem > 64 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) return AF3_ERR_LAUNCH;
	hipLaunchKernelGGL(kern, dim3((unsigned)((m_tiles * n_tiles + 7) / 8 * 8)), dim3(512), smem, s, x, w, row, out, M, N, K, m_tiles, n_tiles);
	return launch_status();
}

}  // namespace

}  // namespace af3

using namespace af3;

// Whether af3_project takes the product: whole slabs of channels, whole 64-column tiles, offsets in 32 bits ...
static bool project_supported(int64_t M, int64_t N, int64_t K) {
	return M > 0 && N > 0 && K > 0 && K % SLAB == 0 && N % 64 == 0 && M * K < (1 << 29) && N * K < (1 << 29) && M < (1 << 22) && N < (1 << 20);
}

// ... and whether it is faster than the library's larger tiles (figures above: the lines cross near 6e9 multiply-adds).
extern "C" int af3_project_suits(int64_t M, int64_t N, int64_t K) { return project_supported(M, N, K) && M * N * K <= (int64_t)6000000000; }

// out[M, N] = x[M, K] . w[N, K]^T + row[N] (row may be null), bf16, dense.  form: 0 = by the rule below, else 10 A + B.
extern "C" int af3_project(const void* x, const void* w, const void* row, void* out, int64_t M, int64_t N, int64_t K, int32_t form, void* stream) {
	if(!x || !w || !out) return AF3_ERR_NULL_POINTER;
	if(!project_supported(M, N, K)) return AF3_ERR_BAD_SHAPE;
	if((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) | reinterpret_cast<uintptr_t>(out) | (row ? reinterpret_cast<uintptr_t>(row) : 0)) & 15) return AF3_ERR_BAD_ARGUMENT;
	const auto *xp = static_cast<const uint16_t*>(x), *wp = static_cast<const uint16_t*>(w), *rp = static_cast<const uint16_t*>(row);
	auto*       op = static_cast<uint16_t*>(out);
	const auto  s  = static_cast<hipStream_t>(stream);
	const auto fits = [&](int tm, int tn) { return ((M + tm - 1) / tm) * ((N + tn - 1) / tn) <= 256; };
	// The smallest tile whose workgroups fit the 256 compute units in one round: what a call takes is the time of one workgroup
	// (fixed part 2.3 us; per slab of 64 channels 0.20, 0.24, 0.33, 0.40, 0.50 us for these five) until there are two rounds.
	if(form == 0) form = fits(64, 64) ? 11 : fits(128, 64) ? 21 : fits(64, 192) ? 13 : fits(128, 128) ? 22 : 23;
	// Three slabs in the ring everywhere.  A fourth asks for more at the start than arrives before it is needed: 64 x 192 columns, four / three, us: 1024 x 3072 x 768
	// 8.96 / 8.61, 2048 x 1536 x 384 6.72 / 6.48, 300 x 1536 x 384 5.24 / 5.02; 128 x 128 columns, 512 x 3072 x 768 8.64 / 8.47.  Two stand still: 11.4 us for the first.
	switch(form) {
	case 11: return launch<1, 1, 3>(xp, wp, rp, op, (int)M, (int)N, (int)K, s);
	case 21: return launch<2, 1, 3>(xp, wp, rp, op, (int)M, (int)N, (int)K, s);
	case 13: return launch<1, 3, 3>(xp, wp, rp, op, (int)M, (int)N, (int)K, s);
	case 22: return launch<2, 2, 3>(xp, wp, rp, op, (int)M, (int)N, (int)K, s);
	case 23: return launch<2, 3, 3>(xp, wp, rp, op, (int)M, (int)N, (int)K, s);
	}
	return AF3_ERR_BAD_ARGUMENT;
}
