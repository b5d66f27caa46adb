// fp32 biased attention on the matrix cores of gfx950: the full-precision path of dot_product_attention_impl<float>
// (reference src/csrc/dot_product_attention.cpp:25-198, dispatch :545-559), for float32 callers who want the 1e-4 tier at
// more than vector-FMA speed.
//
// Products of fp32 numbers on the bf16 matrix instructions.  An fp32 number is the exact sum of three bf16 numbers --
// hi = bf16(x), mid = bf16(x - hi), lo = bf16(x - hi - mid), 3 x 8 significant bits -- and of the nine products of two such
// sums the six largest are kept (hi.hi, hi.mid, mid.hi, mid.mid, hi.lo, lo.hi), accumulated in fp32; the three dropped ones
// are below 2^-23 of the product where the fp32 instructions' is exact (the scheme is published: Henry, Tang, Heinecke, "Leveraging the bfloat16 artificial
// intelligence datatype for higher-precision computations", 2019).  v_mfma_f32_32x32x16_bf16 multiplies 16-deep in 32
// clocks where v_mfma_f32_32x32x2_f32 multiplies 2-deep in 64: six products cost 3/8 of the fp32 instructions' time.
// Errors against 64 bits, relative 2-norm, this form / the fp32 instructions, over 2..64 x 4 x 64..768 x 32, head_dim 4..64 and
// 1 x 4 x 2000 x 32: unit-variance inputs 1.6e-7..4.3e-7 / 2.2e-7..8.2e-7, q times 16 3.9e-7..9.5e-7 / 4.6e-7..1.3e-6, biases
// times 10 1.6e-7..2.3e-7 / 1.9e-7..3.8e-7, biases that grow by 40 along the row 2.1e-7..5.4e-7 / 3.0e-7..5.2e-7 (fewer, deeper
// instructions round the accumulator less often).  Rows whose biases carry an offset of some hundreds or thousands: 0.14 to 1.41
// times the fp32 instructions', by where the offset lies between two powers of two in either domain.
// Measured (64 x 4 x 768 x 32): 234 us with the fp32 instructions (53 % of their peak), 131 to 138 us by card in this form.
//
// Same transposed formulation as the bf16 kernel: S^T[key][q] = K.Q^T, so that in the 32x32
// accumulator layout a lane (q = lane%32, half = lane/32) holds 16 keys of ONE query row
// (register i <-> key 8*(i/4) + 4*half + i%4) and the softmax is an in-lane loop; O^T += V^T.P^T takes
// the probability registers, split into three bf16 terms, directly as its B operand.
//
// Workgroup = NW wavefronts x 32 query rows of one (batch, head); keys in 32-key tiles.  A K or V tile travels global ->
// registers during the matrix work on the tile before and is split on its way into LDS (each value once per workgroup: the
// more wavefronts share a tile the less that costs), double buffered, one barrier per tile.
// Bound: per 32x32 block of logits the matrix pipe works 24 x 32 clocks and the vector ALU about as long (16 exponentials and
// the split of 16 probabilities per lane), so four wavefronts per SIMD (128 registers) overlap the two; 64 x 4 x 768 x 32 runs
// 0.9 PFLOP/s of bf16 instructions, two thirds of what a large bf16 matrix product reaches.
//
// The logit is s + bias, in log2 units (q carries the factor).  p = exp2(fma(bias, log2 e, -m) + s), m the row's softmax
// reference: bias and reference cancel in one rounding before the finished products join them, so a row whose biases carry
// an offset keeps its precision.  (Products accumulated on top of bias minus reference are rounded at that magnitude, up to 30
// where the reference is left behind, once per matrix instruction: up to four times the error at the same speed.)  The reference is
// the running maximum of the first tile; later tiles only check that their row sums have not run away from it (optimistic
// softmax).  A tile that fails the check, the first tile, and every tile of a wavefront that holds a reference of
// extreme magnitude take the exact form: products alone, maximum, rescaling.  Infinities and NaN do not survive the split
// into terms: where a result is not finite the wavefront repeats its walk on the fp32 matrix instructions.
//
// Semantics are the reference harness's (examples/dot_product_attention.py:20-43): a dropped key's
// finished logit is replaced by -1e9, whatever its K row and bias hold, so its weight is exactly 0 unless every key of the row is
// dropped, in which case the row is the mean of V; keys past L weigh 0.
#include "mfma_helpers.hpp"

namespace af3 {
namespace {

constexpr int   F32_KT    = 32;         // keys per tile
constexpr int   F32_MAX_L = 16384;      // tile words and tile list live in LDS
constexpr float DROPPED   = -1.0e9f * LOG2E;   // what masked_fill puts in a dropped key's place, in log2 units
constexpr float F32_FLOOR = -3.0e38f;   // a logit of -inf counts as this, so that a tile of such keys leaves a finite maximum
constexpr float FAST_MAX  = 0x1p20f;    // largest |reference| the fast form takes

__device__ __forceinline__ float other_half(float x) { return __shfl_xor(x, 32); }

// two fp32 values as three pairs of bf16 terms
__device__ __forceinline__ void split3(float x0, float x1, uint32_t& hi, uint32_t& mid, uint32_t& lo) {
	// (the empty asm statements hide where a pair comes from: the compiler would convert each value a second time, alone, rather
	// than take it back out of the pair)
	hi = pack_bf16x2(x0, x1);
	asm("" : "+v"(hi));
	const float r0 = x0 - __uint_as_float(hi << 16), r1 = x1 - __uint_as_float(hi & 0xffff0000u);
	mid = pack_bf16x2(r0, r1);
	asm("" : "+v"(mid));
	lo             = pack_bf16x2(r0 - __uint_as_float(mid << 16), r1 - __uint_as_float(mid & 0xffff0000u));
}

// DP: head_dim padded to 32 or 64.  NW: wavefronts per workgroup.  KS: wavefronts that share a block of 32 query rows, for
// launches with too few blocks to fill the chip: wavefront ks takes tiles ks, ks + KS, ... of the walk, a step of the loop
// moves KS tiles, and the partial (O, m, l) are merged through LDS at the end.
template <int DP, int NW, int KS, bool EVEN>
__global__ void __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(DP == 64 || KS > 1 ? 2 : NW == 4 ? 3 : 4))) dpa_mfma_f32_kernel(af3_dpa_params p, int n_qtiles, int64_t n_groups, int even) {
	constexpr int NC   = DP / 16;             // contraction chunks of K.Q^T
	constexpr int NDB  = DP / 32;             // 32-row blocks of O^T
	constexpr int TERM = F32_KT * DP * 2;     // bytes of one term of a tile
	constexpr int TILE = 3 * TERM;
	constexpr int CPR  = DP / 4;              // 4-column pieces of a row
	constexpr int PCS  = 2 * F32_KT * CPR;    // pieces of a K and a V tile
	constexpr int NQ   = NW / KS;             // blocks of query rows per workgroup
	constexpr int PPT  = PCS * KS / (NW * 64); // pieces per thread and step (a whole number of wavefronts moves a tile)
	constexpr int WPT  = NW / KS;             // wavefronts that move one tile
	static_assert(NW % KS == 0 && PCS % (WPT * 64) == 0, "every thread moves the same number of pieces");

	extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
	// [K tiles of a step x 2][V tiles of a step x 2][live keys of each tile, one bit per key][tile list]
	const int       n_tiles   = (int)((p.L + F32_KT - 1) / F32_KT);
	uint32_t* const live_bits = reinterpret_cast<uint32_t*>(smem + 4 * KS * TILE);
	int16_t* const  live_list = reinterpret_cast<int16_t*>(live_bits + n_tiles);

	// workgroup -> (batch row, head, query tile); consecutive workgroups go round the 8 XCDs, so the
	// query tiles of one (b, h) are kept on one XCD and share its L2 copy of K and V
	// the kernel arguments that the start of a workgroup needs, requested in one batch (otherwise: the launch counts, a wait,
	// the early exit, and only then the fields of p -- memory latencies in a row that a small launch cannot hide)
	asm volatile("" ::"s"(n_qtiles), "s"(n_groups), "s"(p.q), "s"(p.k), "s"(p.v), "s"(p.bias), "s"(p.key_mask), "s"(p.H), "s"(p.L), "s"(p.D), "s"(p.key_mask_stride_b),
				 "s"(p.bias_stride[0]), "s"(p.bias_stride[1]));
	asm volatile("" ::"s"(p.q_stride[0]), "s"(p.q_stride[1]), "s"(p.q_stride[2]), "s"(p.k_stride[0]), "s"(p.k_stride[1]), "s"(p.k_stride[2]), "s"(p.v_stride[0]), "s"(p.v_stride[1]),
				 "s"(p.v_stride[2]));
	// (32-bit divisions: the launcher keeps the grid below 2^31)
	const uint32_t slot = blockIdx.x >> 3, q_div = slot / (uint32_t)n_qtiles, group = q_div * 8 + (blockIdx.x & 7);
	const int      qtile = (int)(slot - q_div * (uint32_t)n_qtiles);
	if(group >= (uint32_t)n_groups) return;
	const int64_t b = group / (uint32_t)p.H, h = group - (uint32_t)b * (uint32_t)p.H;

	const int     tid = threadIdx.x, lane = tid & 63;
	const int     wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int     n = lane & 31, half = lane >> 5;
	const int64_t L = p.L;
	const int     D = (int)p.D;

	// ---- tile mover: thread -> PPT pieces of 4 columns; the first half of the pieces belong to K.  Range-checked loads: rows
	// past L and padded head columns read as zero ----
	const __amdgpu_buffer_rsrc_t k_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(static_cast<const float*>(p.k) + b * p.k_stride[0] + h * p.k_stride[1]), 0,
																			(int)(((L - 1) * p.k_stride[2] + D) * 4), 0x00020000);
	const __amdgpu_buffer_rsrc_t v_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(static_cast<const float*>(p.v) + b * p.v_stride[0] + h * p.v_stride[1]), 0,
																			(int)(((L - 1) * p.v_stride[2] + D) * 4), 0x00020000);
	const int k_row = (int)(p.k_stride[2] * 4), v_row = (int)(p.v_stride[2] * 4);
	// (wavefront w moves pieces of tile w / WPT of a step: the K pieces, then the V pieces)
	const int mv_sub = wave / WPT;
	f32x4     stage[PPT];
	int       m_voff[PPT];
#pragma unroll
	for(int u = 0; u < PPT; u++) {
		const int c = (wave % WPT) * 64 + lane + WPT * 64 * u, row = (c % (PCS / 2)) / CPR, col = (c % CPR) * 4;
		m_voff[u] = col < D ? row * (c < PCS / 2 ? k_row : v_row) + col * 4 : 0x40000000;
	}
	auto fetch_tile = [&](int kt) {
#pragma unroll
		for(int u = 0; u < PPT; u++) {
			const bool is_k = PPT > 1 ? u < PPT / 2 : (wave % WPT) < WPT / 2;  // (wave-uniform: a wavefront's pieces belong to one tensor)
			if(is_k) stage[u] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(k_rsrc, m_voff[u] + kt * (F32_KT * k_row), 0, 0));
			else stage[u] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(v_rsrc, m_voff[u] + kt * (F32_KT * v_row), 0, 0));
		}
	};
	auto store_tile = [&](int buf) {
#pragma unroll
		for(int u = 0; u < PPT; u++) {
			const int  c = (wave % WPT) * 64 + lane + WPT * 64 * u, row = (c % (PCS / 2)) / CPR, col = (c % CPR) * 4;
			const bool is_k = c < PCS / 2;
			const int  chunk = (col >> 3) ^ (is_k ? k_swizzle<DP>(row) : v_swizzle<DP>(row));
			unsigned char* dst = smem + (is_k ? 0 : 2 * KS * TILE) + (buf * KS + mv_sub) * TILE + row * (DP * 2) + chunk * 16 + (col & 4) * 2;
			uint32_t h0, m0, l0, h1, m1, l1;
			split3(stage[u][0], stage[u][1], h0, m0, l0);
			split3(stage[u][2], stage[u][3], h1, m1, l1);
			*reinterpret_cast<u32x2*>(dst)            = u32x2{h0, h1};
			*reinterpret_cast<u32x2*>(dst + TERM)     = u32x2{m0, m1};
			*reinterpret_cast<u32x2*>(dst + 2 * TERM) = u32x2{l0, l1};
		}
	};
	// ---- key-mask bytes, requested first: four keys per lane at any address (the last four of a row that L ends in the middle of are
	// shifted), 256 keys = eight tiles per wavefront and load, four loads under way.  (A byte per lane and a tile per half-wave and load,
	// the list of tiles always compacted, 64-bit divisions: us per call before / now, B x 4 heads x L x 32: 2x128 7.39 / 6.59, 8x384 12.97 / 12.16,
	// 64x256 21.6 / 21.1, 64x768 135.8 / 134.8: there no more than calls differ by.) ----
	const uint8_t* const keep     = p.key_mask ? p.key_mask + b * p.key_mask_stride_b : nullptr;
	const bool           mask_vec = L >= 4;
	const int            n_chunks = (n_tiles * F32_KT + 255) / 256;
	uint32_t             mraw[4];
	auto request_mask = [&](int c0) {
#pragma unroll
		for(int i = 0; i < 4; i++) {
			const int key0 = (c0 + i * NW) * 256 + 4 * lane;
			mraw[i]        = 0x01010101u;
			if(keep && (c0 + i * NW) * 256 < (int)L) mraw[i] = *reinterpret_cast<const u32_bytes*>(keep + (key0 + 4 <= (int)L ? key0 : (int)L - 4));
		}
	};
	if(mask_vec) request_mask(wave);
	const int guess = mv_sub < n_tiles ? mv_sub : n_tiles - 1;
	fetch_tile(guess);  // (the guess that the leading tiles hold live keys: in flight while the mask is read)

	// ---- Q: the B operand of K.Q^T, lane (q = n, g = half): q[q][16c + 8g .. + 7], scaled into log2 units ----
	const int     ks     = wave % KS, wblk = wave / KS;
	const int64_t qrow   = (int64_t)qtile * (NQ * 32) + wblk * 32 + n;
	const bool    row_ok = qrow < L;
	f32x4         qraw[NC][2];
	{
		const float* qp = static_cast<const float*>(p.q) + b * p.q_stride[0] + h * p.q_stride[1] + qrow * p.q_stride[2];
#pragma unroll
		for(int c = 0; c < NC; c++)
#pragma unroll
			for(int e = 0; e < 2; e++) {
				const int d0 = 16 * c + 8 * half + 4 * e;
				qraw[c][e]   = f32x4{0.f, 0.f, 0.f, 0.f};
				if(row_ok && d0 < D) qraw[c][e] = *reinterpret_cast<const f32x4*>(qp + d0);
			}
	}

	const __amdgpu_buffer_rsrc_t b_rsrc = __builtin_amdgcn_make_buffer_rsrc(p.bias ? const_cast<float*>(static_cast<const float*>(p.bias) + h * p.bias_stride[0]) : nullptr, 0,
																			p.bias ? (int)(((L - 1) * p.bias_stride[1] + L) * 4) : 0, 0x00020000);  // (no bias: every load is out of range and reads zero)
	const int b_voff = (int)((row_ok ? qrow : 0) * p.bias_stride[1] * 4) + 16 * half;

	// bias of one tile in accumulator order (register i <-> key 8*(i/4) + 4*half + i%4 of this lane's query row); keys past L: -inf
	auto fetch_bias = [&](int kt, f32x4 (&dst)[4]) {
#pragma unroll
		for(int r4 = 0; r4 < 4; r4++) dst[r4] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(b_rsrc, b_voff + (kt * (F32_KT * 4) + 32 * r4), 0, 0));
		if((int64_t)(kt + 1) * F32_KT > L) {  // (wave-uniform: the row's last tile; what the loads brought for keys past L is not used)
#pragma unroll
			for(int i = 0; i < 16; i++)
				if((int64_t)kt * F32_KT + 8 * (i / 4) + 4 * half + i % 4 >= L) dst[i / 4][i % 4] = -INFINITY;
		}
	};
	f32x4     bias_t[4];  // bias of the tile that comes next
	const int guess_kt = ks < n_tiles ? ks : n_tiles - 1;
	fetch_bias(guess_kt, bias_t);

	// ---- live keys of every tile and the list of tiles with at least one ----
	if(mask_vec) {
		for(int c0 = wave; c0 < n_chunks; c0 += 4 * NW) {
			if(c0 != wave) request_mask(c0);
#pragma unroll
			for(int i = 0; i < 4; i++) {
				const int c = c0 + i * NW;
				if(c >= n_chunks) break;
				// one bit per byte that is not zero, four of them side by side, eight lanes' together in the tile's word
				const uint32_t live = live_bytes(keep_bytes_in_row(mraw[i], c * 256 + 4 * lane + 4 - (int)L));
				int            w    = (int)(((live * 0x01020408u) >> 24) << (4 * (lane & 7)));
				w |= __builtin_amdgcn_update_dpp(0, w, 0xB1, 0xf, 0xf, true);    // lane ^ 1
				w |= __builtin_amdgcn_update_dpp(0, w, 0x4E, 0xf, 0xf, true);    // lane ^ 2
				w |= __builtin_amdgcn_update_dpp(0, w, 0x141, 0xf, 0xf, true);   // mirrored within 8
				if((lane & 7) == 0 && 8 * c + (lane >> 3) < n_tiles) live_bits[8 * c + (lane >> 3)] = (uint32_t)w, live_list[8 * c + (lane >> 3)] = (int16_t)(8 * c + (lane >> 3));
			}
		}
	} else if(wave == 0) {   // (a single tile)
		const unsigned long long bal = __ballot(lane < (int)L && (!keep || keep[lane < (int)L ? lane : 0] != 0));
		if(lane == 0) live_bits[0] = (uint32_t)bal, live_list[0] = 0;
	}
	__syncthreads();
	// the list of the tiles to walk: as it stands if they are the first ones of the row or if no key is live (every tile then), otherwise compacted
	int  nlive = 0;
	bool in_place = true;
	for(int base = 0; base < n_tiles; base += 64) {
		const unsigned long long bal = __ballot(base + lane < n_tiles && live_bits[base + lane] != 0);
		if(bal) in_place = in_place && nlive == base && (bal & (bal + 1)) == 0;
		nlive += __builtin_popcountll(bal);
	}
	if(nlive == 0) nlive = n_tiles;
	if(!in_place) {
		if(wave == 0) {
			int cnt = 0;
			for(int base = 0; base < n_tiles; base += 64) {
				const int  kt     = base + lane;
				const bool keepit = kt < n_tiles && live_bits[kt] != 0;
				const unsigned long long bal = __ballot(keepit);
				const int rank = __builtin_amdgcn_mbcnt_hi((unsigned)(bal >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)bal, 0));
				if(keepit) live_list[cnt + rank] = (int16_t)kt;
				cnt += __builtin_popcountll(bal);
			}
		}
		__syncthreads();
	}

	u32x4 qf[3][NC];
	{
		const float qmul = p.softmax_scale * LOG2E;
#pragma unroll
		for(int c = 0; c < NC; c++)
#pragma unroll
			for(int e = 0; e < 4; e++) {
				const f32x4 w = qraw[c][e >> 1];
				uint32_t    hi, mid, lo;
				split3(w[2 * (e & 1)] * qmul, w[2 * (e & 1) + 1] * qmul, hi, mid, lo);
				qf[0][c][e] = hi, qf[1][c][e] = mid, qf[2][c][e] = lo;
			}
	}
	// DROPPED in the place of a dropped key's finished logit: the tile's word of live keys is wave-uniform, register i's condition
	// is two of its bits, one per half-wave
	auto drop_keys = [&](int kt, f32x16& s) {
		const uint32_t live  = (uint32_t)__builtin_amdgcn_readfirstlane((int)live_bits[kt]);
		const int      past  = (int)((int64_t)(kt + 1) * F32_KT - L);          // keys of this tile that lie past L
		const uint32_t in    = past > 0 ? 0xffffffffu >> past : 0xffffffffu;  // (past < 32)
		if(live == in) return;  // (wave-uniform)
		const uint32_t kept = live | ~in;  // (keys past L keep their -inf)
#pragma unroll
		for(int i = 0; i < 16; i++) {
			const int      k0   = 8 * (i / 4) + i % 4;
			const uint64_t cond = (uint64_t)(uint32_t)((int)(kept << (31 - k0)) >> 31) | (uint64_t)(uint32_t)((int)(kept << (31 - (k0 + 4))) >> 31) << 32;
			float          x    = s[i];
			asm("v_cndmask_b32 %0, %1, %2, %3" : "=v"(x) : "v"(DROPPED), "v"(x), "s"(cond));
			s[i] = x;
		}
	};

	// ---- per-lane LDS read offsets ----
	int k_rd[NC], v_rd[NDB];
#pragma unroll
	for(int c = 0; c < NC; c++) k_rd[c] = n * (DP * 2) + (((2 * c + half) ^ k_swizzle<DP>(n)) << 4);
	{
		const int i16 = lane & 15, G = lane >> 4, row = 4 * (G >> 1) + (i16 >> 2);  // (transposing reads, see dpa_mfma.hip)
#pragma unroll
		for(int db = 0; db < NDB; db++) {
			const int col = 32 * db + 16 * (G & 1) + 4 * (i16 & 3);
			v_rd[db] = 2 * KS * TILE + row * (DP * 2) + (((col >> 3) ^ v_swizzle<DP>(row)) << 4) + (col & 7) * 2;
		}
	}

	auto mfma = [](const u32x4& a, const u32x4& bb, const f32x16& c) -> f32x16 {
		return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, bb), c, 0, 0, 0);
	};
	// s + K.Q^T of the tile in buffer `buf`, smallest products first
	auto products = [&](int buf, f32x16 s) -> f32x16 {
#pragma unroll
		for(int c = 0; c < NC; c++) {
			const unsigned char* kp = smem + buf * TILE + k_rd[c];
			const u32x4 kh = *reinterpret_cast<const u32x4*>(kp), km = *reinterpret_cast<const u32x4*>(kp + TERM), kl = *reinterpret_cast<const u32x4*>(kp + 2 * TERM);
			s = mfma(kl, qf[0][c], s);
			s = mfma(kh, qf[2][c], s);
			s = mfma(km, qf[1][c], s);
			s = mfma(km, qf[0][c], s);
			s = mfma(kh, qf[1][c], s);
			s = mfma(kh, qf[0][c], s);
		}
		return s;
	};

	// ---- online-softmax state (one query row per lane; l_run: this lane's half of the row sum) ----
	float  m_run = -INFINITY, l_run = 0.f;
	f32x16 oacc[NDB];
#pragma unroll
	for(int db = 0; db < NDB; db++)
#pragma unroll
		for(int i = 0; i < 16; i++) oacc[db][i] = 0.f;

	// O^T += V^T.P^T for the tile in buffer `buf`
	auto accumulate = [&](int buf, const f32x16& pr) {
#pragma unroll
		for(int cp = 0; cp < 2; cp++) {
			u32x4 ph, pm, pl;
#pragma unroll
			for(int j = 0; j < 4; j++) {
				uint32_t a, bb, c;
				split3(pr[8 * cp + 2 * j], pr[8 * cp + 2 * j + 1], a, bb, c);
				ph[j] = a, pm[j] = bb, pl[j] = c;
			}
#pragma unroll
			for(int db = 0; db < NDB; db++) {
				u32x4 vf[3];
#pragma unroll
				for(int term = 0; term < 3; term++)
#pragma unroll
					for(int t = 0; t < 2; t++) {
						const s16x4 r = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(smem + v_rd[db] + buf * TILE + term * TERM + (16 * cp + 8 * t) * (DP * 2)));
						const u32x2 rr = __builtin_bit_cast(u32x2, r);
						vf[term][2 * t] = rr[0], vf[term][2 * t + 1] = rr[1];
					}
				oacc[db] = mfma(vf[2], ph, oacc[db]);
				oacc[db] = mfma(vf[0], pl, oacc[db]);
				oacc[db] = mfma(vf[1], pm, oacc[db]);
				oacc[db] = mfma(vf[1], ph, oacc[db]);
				oacc[db] = mfma(vf[0], pm, oacc[db]);
				oacc[db] = mfma(vf[0], ph, oacc[db]);
			}
		}
	};
	bool exact_only = false;  // (wave-uniform)
	// the probabilities of a tile, from its products s, in the exact form, moving the reference to the running maximum
	auto exact_probabilities = [&](int kt, f32x16 s, const f32x4 (&bs)[4]) -> f32x16 {
#pragma unroll
		for(int i = 0; i < 16; i++) {
			s[i] = __builtin_fmaf(bs[i / 4][i % 4], LOG2E, s[i]);
			s[i] = s[i] < F32_FLOOR ? F32_FLOOR : s[i];  // (NaN stays)
		}
		drop_keys(kt, s);
		float mx = -INFINITY;
#pragma unroll
		for(int i = 0; i < 16; i++) {
			if((int64_t)kt * F32_KT + 8 * (i / 4) + 4 * half + i % 4 >= L) s[i] = -INFINITY;
			mx = fmaxf(mx, s[i]);
		}
		mx = fmaxf(mx, other_half(mx));
		const float m_new = fmaxf(m_run, mx);  // finite: every tile has a key below L
		const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
		m_run = m_new;
		l_run *= alpha;
#pragma unroll
		for(int db = 0; db < NDB; db++)
#pragma unroll
			for(int i = 0; i < 16; i++) oacc[db][i] *= alpha;
#pragma unroll
		for(int i = 0; i < 16; i++) s[i] = __builtin_amdgcn_exp2f(s[i] - m_new);  // (the row maximum gets exactly 1)
		exact_only = __ballot(!(fabsf(m_run) <= FAST_MAX)) != 0;
		return s;
	};

	const int n_steps = (nlive + KS - 1) / KS;
	auto tile_at = [&](int i) -> int { return __builtin_amdgcn_readfirstlane((int)live_list[i < nlive ? i : nlive - 1]); };  // (behind the walk's end: its last tile once more, unused)
	const int mv0 = tile_at(mv_sub);
	int       kt  = tile_at(ks);
	if(mv0 != guess) fetch_tile(mv0);
	if(kt != guess_kt) fetch_bias(kt, bias_t);
	store_tile(0);
	__syncthreads();
	auto step = [&](auto first_c, int j) {
		constexpr bool FIRST = decltype(first_c)::value != 0;
		const int buf = FIRST ? 0 : j & 1;
		const int ktn = tile_at((j + 1) * KS + ks);
		fetch_tile(tile_at((j + 1) * KS + mv_sub));  // in flight during the matrix work below
		if(KS == 1 || j * KS + ks < nlive) {  // (wave-uniform)
			f32x16 pr;
			bool   exact = FIRST || exact_only;
			if(!exact) {
#pragma unroll
				for(int i = 0; i < 16; i++) pr[i] = __builtin_fmaf(bias_t[i / 4][i % 4], LOG2E, -m_run);
				fetch_bias(ktn, bias_t);
				f32x16 s;
#pragma unroll
				for(int i = 0; i < 16; i++) s[i] = 0.f;
				s = products(buf * KS + ks, s);
#pragma unroll
				for(int i = 0; i < 16; i++) pr[i] += s[i];
				drop_keys(kt, pr);  // (|m_run| is at most FAST_MAX: weight 0)
				float psum = 0.f;
#pragma unroll
				for(int i = 0; i < 16; i++) {
					pr[i] = __builtin_amdgcn_exp2f(pr[i]);
					psum += pr[i];
				}
				if(__ballot(!(psum < PSUM_LIMIT))) exact = true;  // rare: some probability has run away from the reference (or is not finite)
				else l_run += psum;
			}
			if(exact) {  // (wave-uniform)
				if(!FIRST) fetch_bias(kt, bias_t);  // (once more)
#pragma unroll
				for(int i = 0; i < 16; i++) pr[i] = 0.f;
				pr = exact_probabilities(kt, products(buf * KS + ks, pr), bias_t);
				float psum = 0.f;
#pragma unroll
				for(int i = 0; i < 16; i++) psum += pr[i];
				l_run += psum;
				fetch_bias(ktn, bias_t);
			}
			accumulate(buf * KS + ks, pr);
		}
		store_tile(buf ^ 1);  // that buffer was last read one step ago, before the barrier every wavefront has passed
		__syncthreads();
		kt = ktn;
	};
	even_progress progress(n_steps, EVEN ? even : BY_AGE);
	step(ic<1>{}, 0);
	for(int j = 1; j < n_steps; j++) {
		if constexpr(EVEN) progress.at(j);
		step(ic<0>{}, j);
	}
	// Row numbers from here on come from the lane's number once more, out of the compiler's sight where the loop above has no
	// registers to spare: kept from the start they cost it a fourth wavefront per SIMD.
	int ln = lane;
	if constexpr(KS == 1) {
		ln = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
		asm volatile("" : "+v"(ln));
	}
	const int     on = ln & 31, ohalf = ln >> 5;
	const int64_t orow = (int64_t)qtile * (NQ * 32) + wblk * 32 + on;

	// ---- something is not finite: an infinity or NaN in the inputs (its bf16 terms are an infinity and NaN, and their products
	// are NaN where the formula has an infinity or a weight of zero), a value that rounds up to one, a sum that overflows under a
	// reference left behind.  This wavefront walks its tiles once more, alone, with the fp32 matrix instructions on
	// operands straight from memory and the exact form throughout: what then is not finite is so in the formula. ----
	float finite = l_run * 0.f;  // (0, or NaN)
#pragma unroll
	for(int db = 0; db < NDB; db++)
#pragma unroll
		for(int i = 0; i < 16; i++) finite = __builtin_fmaf(oacc[db][i], 0.f, finite);
	if(__ballot(!(finite == 0.f))) {
		m_run = -INFINITY, l_run = 0.f;
#pragma unroll
		for(int db = 0; db < NDB; db++)
#pragma unroll
			for(int i = 0; i < 16; i++) oacc[db][i] = 0.f;
		const int          cols = (int)p.D, k_bytes = (int)(p.k_stride[2] * 4), v_bytes = (int)(p.v_stride[2] * 4);
		const float        scale = p.softmax_scale * LOG2E;
		const float* const qp = static_cast<const float*>(p.q) + b * p.q_stride[0] + h * p.q_stride[1] + (orow < p.L ? orow : 0) * p.q_stride[2];
#pragma unroll 1
		for(int j = ks; j < nlive; j += KS) {
			kt = tile_at(j);
			fetch_bias(kt, bias_t);
			f32x16 pr;
#pragma unroll
			for(int i = 0; i < 16; i++) pr[i] = 0.f;
#pragma unroll 1
			for(int t = 0; t < DP / 2; t++) {  // A: K[key n][d], B: q[row n][d] of column d = t + DP / 2 half
				const int   d  = t + DP / 2 * ohalf;
				const float kx = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(k_rsrc, d < cols ? (kt * F32_KT + on) * k_bytes + d * 4 : 0x40000000, 0, 0));
				const float qx = d < cols ? qp[d] * scale : 0.f;
				pr = __builtin_amdgcn_mfma_f32_32x32x2f32(kx, qx, pr, 0, 0, 0);
			}
			pr = exact_probabilities(kt, pr, bias_t);
#pragma unroll
			for(int i = 0; i < 16; i++) {  // A: V[key of register i][column n], B: its probability
				l_run += pr[i];
#pragma unroll
				for(int db = 0; db < NDB; db++) {
					const int   col = 32 * db + on;
					const float vx  = __uint_as_float(
						__builtin_amdgcn_raw_buffer_load_b32(v_rsrc, col < cols ? (kt * F32_KT + 8 * (i / 4) + 4 * ohalf + i % 4) * v_bytes + col * 4 : 0x40000000, 0, 0));
					oacc[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(vx, pr[i], oacc[db], 0, 0, 0);
				}
			}
		}
	}
	if constexpr(KS > 1) {
		// ---- merge the partial results of the KS wavefronts of a query block (the tile buffers are dead) ----
		float* const mred = reinterpret_cast<float*>(smem);           // [NW][32] references
		float* const obuf = mred + NW * 32 + wblk * (KS - 1) * (16 * NDB + 1) * 64 + lane;  // [NQ][KS - 1][16 * NDB + 1][64]
		static_assert((NW * 32 + NQ * (KS - 1) * (16 * NDB + 1) * 64) * 4 <= 4 * KS * TILE, "the merge area fits in the tile buffers");
		if(half == 0) mred[wave * 32 + n] = m_run;
		__syncthreads();
		float m_all = mred[wblk * KS * 32 + n];
#pragma unroll
		for(int w = 1; w < KS; w++) m_all = fmaxf(m_all, mred[(wblk * KS + w) * 32 + n]);
		const float f = __builtin_amdgcn_exp2f(m_run - m_all);  // (a wavefront without a tile: m = -inf, factor 0)
		l_run *= f;
#pragma unroll
		for(int db = 0; db < NDB; db++)
#pragma unroll
			for(int i = 0; i < 16; i++) oacc[db][i] *= f;
		if(ks > 0) {
			float* o = obuf + (ks - 1) * (16 * NDB + 1) * 64;
#pragma unroll
			for(int i = 0; i < 16 * NDB; i++) o[i * 64] = oacc[i / 16][i % 16];
			o[16 * NDB * 64] = l_run;
		}
		__syncthreads();
		if(ks > 0) return;
#pragma unroll
		for(int w = 0; w < KS - 1; w++) {
			const float* o = obuf + w * (16 * NDB + 1) * 64;
#pragma unroll
			for(int i = 0; i < 16 * NDB; i++) oacc[i / 16][i % 16] += o[i * 64];
			l_run += o[16 * NDB * 64];
		}
	}

	// ---- epilogue: O^T register i of block db is head column 32*db + 8*(i/4) + 4*half + i%4 ----
	const float l_tot = l_run + other_half(l_run);
	const float inv   = 1.f / l_tot;
	if(orow < p.L) {
		float* const       op = static_cast<float*>(p.out) + b * p.out_stride[0] + h * p.out_stride[1] + orow * p.out_stride[2];
		const float* const gp = p.gate ? static_cast<const float*>(p.gate) + b * p.gate_stride[0] + h * p.gate_stride[1] + orow * p.gate_stride[2] : nullptr;
#pragma unroll
		for(int db = 0; db < NDB; db++)
#pragma unroll
			for(int r4 = 0; r4 < 4; r4++) {
				const int d0 = 32 * db + 8 * r4 + 4 * ohalf;
				if(d0 < p.D) {
					float4 w = {oacc[db][4 * r4] * inv, oacc[db][4 * r4 + 1] * inv, oacc[db][4 * r4 + 2] * inv, oacc[db][4 * r4 + 3] * inv};
					if(gp) {  // out *= sigmoid(gate)
						const float4 g = *reinterpret_cast<const float4*>(gp + d0);
						w.x *= sigmoidf_fast(g.x), w.y *= sigmoidf_fast(g.y), w.z *= sigmoidf_fast(g.z), w.w *= sigmoidf_fast(g.w);
					}
					*reinterpret_cast<float4*>(op + d0) = w;
				}
			}
	}
}

template <int DP, int NW, int KS>
int launch(const af3_dpa_params& p, hipStream_t s) {
	constexpr int QT       = NW / KS * 32;
	const int     n_qtiles = (int)((p.L + QT - 1) / QT);
	const int     n_tiles  = (int)((p.L + F32_KT - 1) / F32_KT);
	const int64_t groups   = p.B * p.H;
	const int64_t grid     = ((groups + 7) / 8) * 8 * n_qtiles;
	if(grid > 0x7fffffff) return AF3_ERR_BAD_SHAPE;
	const size_t smem = (size_t)4 * KS * 3 * F32_KT * DP * 2 + (size_t)n_tiles * 4 + (size_t)n_tiles * 2 + 16;
	const int64_t per_cu = DP == 64 ? 2 : 4;   // workgroups a compute unit holds, by their registers (KS = 1)
	// Wavefronts that are behind on their walk go first (EVEN) where several workgroups stand on a compute unit and walk four tiles and more.  Elsewhere the code costs more than
	// it brings, us without / with it: one workgroup to a compute unit 2 x 4 x 128 x 32 6.33 / 6.41, 5 x 4 x 333 19.8 / 20.1, 32 x 4 x 300 22.5 / 22.7; few tiles
	// 100 x 8 x 22 x 48 13.9 / 14.2, 1 x 4 x 51 x 64 8.14 / 8.31, 100 x 4 x 74 x 8 9.49 / 9.64.
	const int    even = KS == 1 && n_tiles >= 4 ? progress_mode(groups * n_qtiles, 256 * per_cu) : BY_AGE;
	auto         kern = dpa_mfma_f32_kernel<DP, NW, KS, false>;
	if constexpr(KS == 1)
		if(even != BY_AGE) kern = dpa_mfma_f32_kernel<DP, NW, KS, true>;
	if(smem > 64 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) return AF3_ERR_LAUNCH;
	hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(NW * 64), smem, s, p, n_qtiles, groups, even);
	return launch_status();
}

// Launches too small to fill the chip split the key tiles of a query block over two or four wavefronts, as long as their
// workgroups still fit the 256 compute units in one round.  Measured, us (B x 4 heads x L x 32; the form taken is marked):
//                               2x128   2x768   4x768   8x384   8x768  16x384  32x256  16x768  64x256  64x768
//   one wavefront per block      10.4    41.5    41.7    23.1    42.1    23.3    17.4    51.6*   22.3*  131.1*
//   two, 128 query rows           9.1    31.0    31.2    18.6    31.6*   18.8*   14.2*   63.4    26.7   189.7
//   four, 64 query rows           7.6    20.5    20.7*   13.4*   39.8    25.5    19.7    61.2    37.7   238.3
//   four, 32 query rows           7.4*   18.4*   35.1    22.5    52.5    33.2    35.3   105.7    69.6   416.5
// (fp32 matrix instructions, one wavefront per block, before: 2x128 13 us, 64x768 234 us.  With biases joining finished products the forms
// taken measure 2x128 7.4, 8x384 13.0, 32x256 13.2, 16x384 17.4, 16x768 47.7, 64x768 131.6.)  Rows of less than four tiles do
// not gain from a split.
template <int DP>
int launch_dp(const af3_dpa_params& p, hipStream_t s) {
	const int64_t groups = p.B * p.H, tiles = (p.L + F32_KT - 1) / F32_KT;
	auto wgs = [&](int rows) -> int64_t { return groups * ((p.L + rows - 1) / rows); };
	if(tiles >= 4) {
		if constexpr(DP == 32) {
			if(wgs(32) <= 256) return launch<DP, 4, 4>(p, s);
			if(wgs(64) <= 256) return launch<DP, 8, 4>(p, s);
		} else {  // (the tiles of a four-way step do not fit in LDS)
			if(wgs(64) <= 256) return launch<DP, 4, 2>(p, s);
		}
		if(wgs(128) <= 256) return launch<DP, 8, 2>(p, s);
	}
	return launch<DP, 4, 1>(p, s);
}

}  // namespace

// fp32 tensors with 16-byte aligned rows and a head_dim the 32x32 tiles cover; everything else stays on
// the vector-FMA kernel.
bool mfma_f32_eligible(const af3_dpa_params& p) {
	if(p.io_dtype != AF3_F32 || p.mma_dtype != AF3_F32 || p.out_dtype != AF3_F32) return false;
	if(p.bias && p.bias_dtype != AF3_F32) return false;
	if(p.D > 64 || p.D % 4 != 0 || p.L > F32_MAX_L) return false;
	// buffer addressing of one (batch row, head) slab uses 32-bit byte offsets
	const int64_t rows = (p.L + F32_KT - 1) / F32_KT * F32_KT;  // (those of the last tile that lie past L among them)
	if(rows * p.k_stride[2] * 4 >= 0x40000000LL || rows * p.v_stride[2] * 4 >= 0x40000000LL || (p.bias && p.L * p.bias_stride[1] * 4 >= 0x7ff00000LL)) return false;
	if(p.gate && ((reinterpret_cast<uintptr_t>(p.gate) & 15) || p.gate_stride[0] % 4 || p.gate_stride[1] % 4 || p.gate_stride[2] % 4)) return false;
	const void* ptrs[4] = {p.q, p.k, p.v, p.out};
	for(const void* ptr : ptrs)
		if(reinterpret_cast<uintptr_t>(ptr) & 15) return false;
	for(int i = 0; i < 3; i++)
		if(p.q_stride[i] % 4 || p.k_stride[i] % 4 || p.v_stride[i] % 4 || p.out_stride[i] % 4) return false;
	return true;
}

int launch_dpa_mfma_f32(const af3_dpa_params& p, hipStream_t s) { return p.D <= 32 ? launch_dp<32>(p, s) : launch_dp<64>(p, s); }

}  // namespace af3
