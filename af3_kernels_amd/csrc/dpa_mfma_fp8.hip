// fp8 (OCP e4m3) matrix-core attention kernel for gfx950: both products on the e4m3 matrix instructions (64-deep for K.Q^T where
// head_dim allows, 16-deep otherwise) with fp32 accumulation, bf16 bias, bf16 or fp32 output.
//
// The reference has no fp8 path (its e4m3 converters are "not implemented" asserts,
// src/csrc/xsmm_functors.h:218-226); this kernel computes the same formula as
// src/csrc/dot_product_attention.cpp:88-122 on inputs quantised per tensor by
// af3_quantize_fp8_e4m3:
//     q8 = e4m3(q * softmax_scale * sq),  k8 = e4m3(k * sk),  v8t = e4m3(v * sv) transposed to [B,H,D,L]
// with power-of-two scales, so that with alpha = 1/(sq*sk)
//     logits = alpha * (q8 . k8^T) + bias            (natural units)
// Layout is the "transposed" one of the bf16 kernel (dpa_mfma.hip): S^T = K8 . Q8^T with a lane
// holding 16 keys of one query row; the bias rides an identity MFMA
// whose diagonal is 1/alpha (a power of two, exact in bf16), the key mask a third MFMA, in tiles that drop a key;
// P^T = exp(logit - m) * 2^8 is quantised to e4m3 in registers (values in (0, 256], e4m3 tops out at
// 448) and is the B operand of O^T += V8^T . P^T.  The row maximum m is the true running maximum
// (no slack: P must stay below the e4m3 range, and the largest P, exactly 256, is rounded best), the row sum is taken over the quantised P, on the matrix pipe.
//
// What bounds it: the vector port (16 fma, 16 exponentials, 8 packs, a dozen maxima and, while maxima still move, 17 products
// per 32 x 32 logits), then the matrix pipe (256 to 288 clocks), shared by up to four wavefronts per SIMD; everything else must
// stay out of their way:
//   * Key order.  Row r = 8 a + 4 g + e of S^T holds key 16 g + 4 a + e of its 32 keys (K rows, mask entries and the identity are
//     read in that order), so that a lane's 16 keys are consecutive and its V^T operand is ONE 16-byte LDS read.  Chunks are
//     XOR-swizzled: no bank conflicts.  (In natural order V^T took four 4-byte reads of eight-fold conflicts and K 8-byte ones.)
//   * K.Q^T on the 64-deep instruction.  Head_dim up to 32, compensated: a lane's 32 bytes are the K row (lower half-wave) or its
//     residual (upper), so that (k8 | k_lo) meets (q8 | q8) and then (q_lo | 0): 128 clocks instead of the 192 of six 16-deep ones.
//   * Row sums through P.V: where head columns are padded, rows D and D + 4 of the V^T tile are ones, and the sum is a row of O^T.
//   * A stage overlaps the logits of the next 32 keys with the exponentials of these, and leaves P.V to run under the next maxima.
//   * The bias tile of each wavefront travels through LDS as whole 64-byte row segments, by loads that write LDS directly, a tile
//     ahead (16-byte loads from 32 rows per instruction before); rows that start at any element are fetched from the dword
//     below and shifted when read (element by element before).
//   * 39 KB of LDS and 128 registers: four workgroups of four wavefronts per compute unit.
//   * Workgroups in an order that lets batch rows share the bias, tiles in two parts where workgroups are few: see launch8_parts, launch8.
// us per call with its two quantising launches (6 to 13 us), 16 heads of 24, 16-deep products / these forms, workgroups by heads and one part / now:
// 5x1536 89.0/71.3/63.6, 8x1536 133.6/104.9/97.0, 8x1301 (ragged rows) -/101.7/93.2, 8x1000 66.7/54.2/49.7, 5x300 37.9/20.3/17.1, 1x1536 42.1/34.2/26.3 (cards
// differ: 5x1536 63 to 66).  Measured on the way: with the bias streamed once per batch row its loads were 13 us of 57 at 5x1536, the exponentials 4; four workgroups per compute unit instead of three changed nothing, nor did
// pinning the matrix instructions between the exponentials: the vector port is busy three quarters of the time.
#include "mfma_helpers.hpp"

namespace af3 {

namespace {

constexpr int KT8   = 64;    // keys per tile
constexpr int NW8   = 4;     // wavefronts per workgroup (32 query rows each)
constexpr int MAX_L8 = 8192;
constexpr float P_SHIFT = 8.f;  // P is stored as p * 2^8
constexpr int BIAS_HALF8 = 2048 + 128;   // 32 rows x 32 keys of bf16, and one dword per row behind them (rows that start at any element)
constexpr int TILE_FULL = 0x4000;    // flag beside a tile's number: no key of the tile is dropped
typedef __attribute__((ext_vector_type(8))) int i32x8;

__device__ __forceinline__ float max3(float a, float b, float c) {   // (written out: fmaxf quiets its operands first)
	float r;
	asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
	return r;
}

// the maximum of a lane's 16 logits and m, in two chains (one statement: the compiler puts a wait state behind each)
__device__ __forceinline__ float max17(const f32x16& s, float m) {
	float a, b;
	asm("v_max3_f32 %0, %2, %3, %4\n\tv_max3_f32 %1, %5, %6, %7\n\t"
		"v_max3_f32 %0, %0, %8, %9\n\tv_max3_f32 %1, %1, %10, %11\n\t"
		"v_max3_f32 %0, %0, %12, %13\n\tv_max3_f32 %1, %1, %14, %15\n\t"
		"v_max3_f32 %0, %0, %16, %17\n\tv_max3_f32 %0, %0, %1, %18"
		: "=&v"(a), "=&v"(b)
		: "v"(s[0]), "v"(s[1]), "v"(s[2]), "v"(s[3]), "v"(s[4]), "v"(s[5]), "v"(s[6]), "v"(s[7]), "v"(s[8]), "v"(s[9]), "v"(s[10]), "v"(s[11]), "v"(s[12]), "v"(s[13]), "v"(s[14]), "v"(s[15]), "v"(m));
	return a;
}

// DP: head_dim padded to 32 or 64 (bytes per K row in LDS, rows of the V^T tile).
// COMP: compensated logits q8.k8 + q8.k_lo + q_lo.k8 (the residual tensors recover the e4m3 rounding of q and k).
// ONES: head_dim < DP, row sums through P.V; otherwise two 16x16x32 instructions per 32 keys.
// BMODE: 0 = no bias, 1 = element by element (a head's slab beyond 32-bit offsets), 2 = through LDS, rows of whole aligned
// 16-byte chunks, 3 = through LDS, rows that start at any element.
// KS: 1, or the number of parts that the tiles of a block of query rows are dealt to, each with wavefronts and buffers of its own
// (for launches of few workgroups); their sums are merged through LDS at the end.
template <int DP, bool COMP, bool ONES, int BMODE, int KS>
__global__ void __launch_bounds__(KS * NW8 * 64) __attribute__((amdgpu_waves_per_eu(DP == 32 ? 4 : KS == 1 ? 3 : 2))) dpa_mfma_fp8_kernel(af3_dpa_params p, int n_qtiles, int n_units, int per_xcd, int even) {
	constexpr int NDB      = DP / 32;       // 32-row blocks of O^T
	constexpr int K_TILE1  = KT8 * DP;      // bytes of one K tile
	constexpr int K_TILE   = K_TILE1 * (COMP ? 2 : 1);  // hi tile followed by the residual tile
	constexpr int V_TILE   = DP * KT8;      // bytes: [DP rows d][64 keys]
	constexpr int TILE     = K_TILE + V_TILE;
	constexpr int K_LOADS  = K_TILE / 1024, V_LOADS = V_TILE / 1024; // 1 KB wave loads per tile
	constexpr bool RING    = BMODE >= 2, RAGGED = BMODE == 3;

	extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
	// [KS][3][K tile, V^T tile] [two half slots of bias per wavefront] [mask table: bf16 bits per key] [tile flags]
	constexpr int        SLOT_BASE = KS * 3 * TILE;
	constexpr int        MASK_BASE = SLOT_BASE + (RING ? KS * NW8 * 2 * BIAS_HALF8 : 0);
	uint16_t* const      mask_tab  = reinterpret_cast<uint16_t*>(smem + MASK_BASE);
	const int            n_ktiles  = (int)((p.L + KT8 - 1) / KT8);
	uint8_t* const       tile_flags = reinterpret_cast<uint8_t*>(mask_tab + n_ktiles * KT8);   // per tile: bit 0 a live key, bit 1 a key that is not

	// workgroup -> (batch row, head, query tile)
	// the kernel arguments that the start of a workgroup needs, requested in one batch (otherwise: the launch counts, a wait,
	// the early exit, and only then the fields of p -- memory latencies in a row that a small launch cannot hide)
	asm volatile("" ::"s"(n_qtiles), "s"(n_units), "s"(per_xcd), "s"(p.B), "s"(p.q), "s"(p.k), "s"(p.v), "s"(p.bias), "s"(p.key_mask), "s"(p.H), "s"(p.L), "s"(p.D), "s"(p.key_mask_stride_b),
				 "s"(p.bias_stride[0]), "s"(p.bias_stride[1]), "s"(p.device_descales), "s"(p.k_lo));
	asm volatile("" ::"s"(p.q_stride[0]), "s"(p.q_stride[1]), "s"(p.q_stride[2]), "s"(p.k_stride[0]), "s"(p.k_stride[1]), "s"(p.k_stride[2]), "s"(p.v_stride[0]), "s"(p.v_stride[1]),
				 "s"(p.v_stride[2]));
	uint32_t       b_u, h_u, qtile_u;
	const uint32_t xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
	if(per_xcd > 0) {   // blocks of query rows in one run per XCD, the batch rows of a block next to each other
		const uint32_t part = slot / (uint32_t)p.B, block = xcd * (uint32_t)per_xcd + part;
		if(block >= (uint32_t)n_units) return;
		h_u = block / (uint32_t)n_qtiles, qtile_u = block - h_u * (uint32_t)n_qtiles, b_u = slot - part * (uint32_t)p.B;
	} else {   // (batch row, head) pairs dealt to the XCDs, a pair's query tiles next to each other
		const uint32_t part = slot / (uint32_t)n_qtiles, group = part * 8 + xcd;
		if(group >= (uint32_t)n_units) return;
		b_u = group / (uint32_t)p.H, h_u = group - b_u * (uint32_t)p.H, qtile_u = slot - part * (uint32_t)n_qtiles;
	}
	const int64_t b = b_u, h = h_u;
	const int     qtile = (int)qtile_u;

	const int     tid = threadIdx.x, lane = tid & 63;
	const int     wave_all = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wave_all % NW8, part = wave_all / NW8;
	const int     buf0 = part * 3 * TILE;   // this part's first buffer
	const int     n = lane & 31, half = lane >> 5;
	const int64_t L = p.L;
	const int     D = (int)p.D;

	const int64_t qrow   = (int64_t)qtile * (NW8 * 32) + wave * 32 + n;
	const bool    row_ok = qrow < L;
	const int     key_of_row = 16 * ((n >> 2) & 1) + 4 * (n >> 3) + (n & 3);   // the key that row n of S^T holds, of its 32

	// ---- tile loaders (1 KB per wave instruction, straight into LDS) ----
	// K: lane i of a load -> tile row i / (DP/16), chunk position i % (DP/16); V^T: lane i -> row d = i / 4, position i % 4 of
	// its 64 keys.  Positions hold the chunks under the swizzles k_sw, v_sw.  K rows past L repeat row L - 1 (their keys carry the
	// out-of-range mask value); head columns past D are not fetched (the buffers are cleared first: a stale byte there must not be a NaN
	// pattern), nor rows past D of V^T.
	auto k_sw = [](int row) -> int { return DP == 32 ? (row >> 4) & 1 : ((row >> 4) & 1) | (((row >> 2) & 1) << 1); };
	auto v_sw = [](int row) -> int { return (row >> 2) & 3; };
	const uint32_t k_bytes  = (uint32_t)((L - 1) * p.k_stride[2] + D);
	const u32x4    k_rsrc   = raw_rsrc(static_cast<const uint8_t*>(p.k) + b * p.k_stride[0] + h * p.k_stride[1], k_bytes);
	const u32x4    klo_rsrc = raw_rsrc(static_cast<const uint8_t*>(COMP ? p.k_lo : p.k) + b * p.k_stride[0] + h * p.k_stride[1], k_bytes);
	const u32x4    v_rsrc   = raw_rsrc(static_cast<const uint8_t*>(p.v) + b * p.v_stride[0] + h * p.v_stride[1], (uint32_t)(D * p.v_stride[2]));
	constexpr int KCPR = DP / 16;       // 16-byte chunks per K row
	constexpr int KRPI = 1024 / DP;     // K rows per wave load
	constexpr int KPW  = (K_LOADS + NW8 - 1) / NW8, VPW = (V_LOADS + NW8 - 1) / NW8;   // loads per wavefront at most
	constexpr int KV_MIN = K_LOADS / NW8;   // ... and at least (V loads of padded rows only are not issued)
	const uint32_t lds0 = lds_addr_of(smem);
	const int      k_row_bytes = (int)p.k_stride[2];
	int  k_voff[KPW], v_voff[VPW];
	bool k_on[KPW], v_on[VPW];
#pragma unroll
	for(int t = 0; t < KPW; t++) {
		const int j = wave + NW8 * t, r = (COMP ? j % (K_LOADS / 2) : j) * KRPI + lane / KCPR, ch = (lane % KCPR) ^ k_sw(r);
		k_voff[t] = r * k_row_bytes + ch * 16, k_on[t] = j < K_LOADS && ch * 16 < D;
	}
#pragma unroll
	for(int t = 0; t < VPW; t++) {
		const int j = NW8 - 1 - wave + NW8 * t, d = j * 16 + (lane >> 2);   // (from the last wavefront on: the first ones may have one K load more)
		v_voff[t] = d * (int)p.v_stride[2] + (((lane & 3) ^ v_sw(d)) << 4), v_on[t] = j < V_LOADS && d < D;
	}
	auto load_tile = [&](int kt, int buf_off) {
#pragma unroll
		for(int t = 0; t < KPW; t++) {
			const int  j  = wave + NW8 * t;
			const bool lo = COMP && j >= K_LOADS / 2;
			int        o  = k_voff[t] + kt * (KT8 * k_row_bytes);
			if((kt + 1) * KT8 > (int)L) {   // (wave-uniform: the last tile)
				const int over = kt * KT8 + (COMP ? j % (K_LOADS / 2) : j) * KRPI + lane / KCPR - ((int)L - 1);
				if(over > 0) o -= over * k_row_bytes;
			}
			if(k_on[t]) lds_dma_b128(lo ? klo_rsrc : k_rsrc, lds0 + buf_off + j * 1024, o);
		}
#pragma unroll
		for(int t = 0; t < VPW; t++) {
			const int j = NW8 - 1 - wave + NW8 * t;
			if(v_on[t]) lds_dma_b128(v_rsrc, lds0 + buf_off + K_TILE + j * 1024, v_voff[t] + kt * KT8);
		}
	};
	// ---- bias half slots (32 keys each): two loads of sixteen 64-byte row segments, chunk c of row r at position c ^ ((r >> 2) & 3);
	// RAGGED: from the dword that holds a row's first key, plus the dword behind the half of each row (see dpa_mfma.hip) ----
	const uintptr_t b_base = RING ? reinterpret_cast<uintptr_t>(static_cast<const uint16_t*>(p.bias) + h * p.bias_stride[0]) : 0;
	const int       b_odd  = RAGGED ? (int)(b_base & 2) : 0;
	const u32x4     b_rsrc = raw_rsrc(reinterpret_cast<const void*>(b_base - b_odd), RING ? (uint32_t)((((L - 1) * p.bias_stride[1] + L) * 2 + b_odd + 3) & ~3ll) : 0u);
	const int       b_row_bytes = (int)(p.bias_stride[1] * 2), q0 = qtile * (NW8 * 32) + wave * 32;
	const uint32_t  slot_addr   = lds0 + SLOT_BASE + wave_all * (2 * BIAS_HALF8);
	constexpr int   BIAS_LOADS  = RAGGED ? 3 : RING ? 2 : 0;
	int b_voff[2] = {0, 0}, b_tail = 0;
	const int b_chunk = (lane & 3) ^ ((lane >> 4) & 3);   // (row 16 j + lane / 4)
	if constexpr(RING) {
#pragma unroll
		for(int j = 0; j < 2; j++) {
			const int row = q0 + 16 * j + (lane >> 2) < (int)L ? q0 + 16 * j + (lane >> 2) : (int)L - 1;
			b_voff[j]     = ((b_odd + row * b_row_bytes) & (RAGGED ? ~3 : ~0)) + b_chunk * 16;
		}
		const int row = q0 + n < (int)L ? q0 + n : (int)L - 1;
		b_tail        = ((b_odd + row * b_row_bytes) & ~3) + 64;
	}
	auto load_bias = [&](int kt, int sub) {
		if constexpr(!RING) return;
		int off = kt * (KT8 * 2) + sub * 64;
		if(!RAGGED && (kt + 1) * KT8 > (int)L) {   // (wave-uniform: the last tile) chunks past L: the row's last one again
			asm volatile("");   // (kept a branch: as selects it costs every tile six instructions)
			const int over = kt * KT8 + sub * 32 + b_chunk * 8 - ((int)L - 8);
			if(over > 0) off -= over * 2;
		}
#pragma unroll
		for(int j = 0; j < 2; j++) lds_dma_b128(b_rsrc, slot_addr + sub * BIAS_HALF8 + j * 1024, b_voff[j] + off);
		if constexpr(RAGGED)
			if(half == 0) lds_dma_b32(b_rsrc, slot_addr + sub * BIAS_HALF8 + 2048, b_tail + off);
	};

	// ---- requested first: the first tile and its bias (on the guess that the tiles up to it hold live keys), the key-mask bytes, q, the scales.  A workgroup's
	// start is bound by these latencies and by its instructions (a lone wavefront issues one in about 4.5 clocks): hence no barrier
	// in front of the loads, four mask bytes at a time at any address, and no list of tiles but a bit for each.  16 heads of 24, us
	// per call before / after: 1x128 12.3 / 11.7, 5x300 19.1 / 18.4, 2x777 27.1 / 25.9, 8x1301 99.0 / 97.0, 5x1536 70.0 / 69.5 ----
	const int guess = part < n_ktiles ? part : 0;
	load_tile(guess, buf0);
	load_bias(guess, 0);
	load_bias(guess, 1);
	const uint8_t* const keep     = p.key_mask ? p.key_mask + b * p.key_mask_stride_b : nullptr;
	const bool           mask_vec = L >= 4;   // four keys per lane and load at any address (the last four of a row that L ends in the middle of are shifted)
	const int            n_chunks = (n_ktiles * KT8 + 255) / 256;
	uint32_t             mraw[2];
	auto request_mask = [&](int c0) {   // chunk c: keys 256 c + 4 lane .. + 3
#pragma unroll
		for(int i = 0; i < 2; i++) {
			const int key0 = (c0 + i * (KS * NW8)) * 256 + 4 * lane;
			mraw[i]        = 0x01010101u;
			if(keep && (c0 + i * (KS * NW8)) * 256 < (int)L) mraw[i] = *reinterpret_cast<const u32_bytes*>(keep + (key0 + 4 <= (int)L ? key0 : (int)L - 4));
		}
	};
	if(mask_vec) request_mask(wave_all);
	float dq = p.q_descale, dk = p.k_descale, dv = p.v_descale;   // real = stored * descale
	if(p.device_descales) dq = p.device_descales[0], dk = p.device_descales[1], dv = p.device_descales[2];
	// q operands of the 64-deep instruction: lane (q, g = half) holds columns [32 g, ..) of q8 and q_lo (DP = 64), or all 32 columns
	// of q8 in both half-waves (not compensated: in the lower) and of q_lo in the lower (DP = 32); zeros elsewhere
	i32x8 qa, qb;
	{
		const int64_t qoff = b * p.q_stride[0] + h * p.q_stride[1] + qrow * p.q_stride[2];
#pragma unroll
		for(int c = 0; c < 4; c++) {
			const int d0 = (DP == 64 ? 32 * half : 0) + 8 * c;
			u32x2     x = {0u, 0u}, y = {0u, 0u};
			if(row_ok && d0 < D && (DP == 64 || COMP || half == 0)) x = *reinterpret_cast<const u32x2*>(static_cast<const uint8_t*>(p.q) + qoff + d0);
			if(COMP && row_ok && d0 < D && (DP == 64 || half == 0)) y = *reinterpret_cast<const u32x2*>(static_cast<const uint8_t*>(p.q_lo) + qoff + d0);
			qa[2 * c] = (int)x[0], qa[2 * c + 1] = (int)x[1], qb[2 * c] = (int)y[0], qb[2 * c + 1] = (int)y[1];
		}
	}
	// what no load writes of the tiles: head columns past the chunk that holds the last one (zeros: a stale byte there must not be a NaN
	// pattern) and rows from D on of V^T (zeros, and for the row sums e4m3 1.0 in rows D and D + 4)
	if(tid < (DP - D) * (KT8 / 16)) {   // (at most 96)
		const uint32_t w = ONES && ((tid >> 2) & ~4) == 0 ? 0x38383838u : 0u;
#pragma unroll
		for(int buf = 0; buf < 3 * KS; buf++) reinterpret_cast<u32x4*>(smem + buf * TILE + K_TILE + D * KT8)[tid] = u32x4{w, w, w, w};
	}
	if(D <= DP - 16) {
		for(int i = tid; i < KS * 3 * K_TILE / 16; i += KS * NW8 * 64) {
			const int buf = i / (K_TILE / 16), u = i - buf * (K_TILE / 16), row = (u / KCPR) % KT8;
			if((((u % KCPR) ^ k_sw(row)) << 4) >= D) reinterpret_cast<u32x4*>(smem + buf * TILE)[u] = u32x4{0u, 0u, 0u, 0u};
		}
	}

	const float alpha = dq * dk * p.softmax_scale;  // logits = alpha * (q8 . k8) + bias
	const float c_exp = alpha * LOG2E;              // exp(logit - m) = exp2(acc*c_exp - m_acc*c_exp), m_acc in accumulator units

	// ---- key-mask table and tile flags ----
	if(mask_vec) {
		for(int c0 = wave_all; c0 < n_chunks; c0 += 2 * KS * NW8) {
			if(c0 != wave_all) request_mask(c0);
#pragma unroll
			for(int i = 0; i < 2; i++) {
				const int c = c0 + i * (KS * NW8);
				if(c >= n_chunks) break;
				const int key0 = c * 256 + 4 * lane, over = key0 + 4 - (int)L;
				const uint32_t m = keep_bytes_in_row(mraw[i], over), gone = gone_bytes(m);
				if(key0 < n_ktiles * KT8) *reinterpret_cast<u32x2*>(mask_tab + key0) = mask_values_bf16(gone, over);
				const unsigned long long bal = __ballot(m != 0u), baln = __ballot(gone != 0u);   // 16 lanes per tile (keys from L on are gone)
				if(lane < 4 && 4 * c + lane < n_ktiles) tile_flags[4 * c + lane] = (uint8_t)((((bal >> (16 * lane)) & 0xffffull) != 0 ? 1 : 0) | (((baln >> (16 * lane)) & 0xffffull) != 0 ? 2 : 0));
			}
		}
	} else if(wave_all == 0) {   // (a single tile)
		const bool in = lane < (int)L, live = in && (!keep || keep[in ? lane : 0] != 0);
		mask_tab[lane] = live ? (uint16_t)0 : (in ? MASK_DROPPED_BF16 : MASK_OUT_OF_RANGE_BF16);
		const bool any = __ballot(live) != 0;
		if(lane == 0) tile_flags[0] = any ? 3 : 2;
	}
	__syncthreads();
	// the tiles to walk, as bits (at most 128 tiles)
	unsigned long long todo[2], some[2];
#pragma unroll
	for(int i = 0; i < 2; i++) {
		const int f = 64 * i + lane < n_ktiles ? tile_flags[64 * i + lane] : 2;
		todo[i] = __ballot((f & 1) != 0), some[i] = __ballot((f & 2) != 0);
	}
	const bool all_dropped = (todo[0] | todo[1]) == 0;   // no key is live: every tile is walked, the result is the mean over all L keys
	if(all_dropped) todo[0] = __ballot(lane < n_ktiles), todo[1] = __ballot(64 + lane < n_ktiles);
	const int n_todo = __builtin_popcountll(todo[0]) + __builtin_popcountll(todo[1]);
	const int nlive  = (n_todo - part + KS - 1) / KS, n_most = (n_todo + KS - 1) / KS;   // tiles of this part and of the first; they differ by one at most
	int       entry_last = 0, base = 0;
	// (both words chosen between in every step, and maxima in statements of their own: 3x1000 29.0 us, 1x1301 28.5, 8x1536 100.1; so 28.1, 27.6, 98.8)
	auto pop = [&]() -> int {   // the next tile's number and flag; behind the last one: that one again
		if(todo[0] == 0) todo[0] = todo[1], some[0] = some[1], todo[1] = 0, base = 64;   // (once, or behind the last tile)
		if(todo[0] != 0) {
			const int t = __builtin_ctzll(todo[0]);
			entry_last  = (base + t) | ((some[0] >> t) & 1 ? 0 : TILE_FULL);
			todo[0] &= todo[0] - 1;
		}
		return entry_last;
	};
	auto next_entry = [&]() -> int {   // ... of this part
		const int e = pop();
#pragma unroll
		for(int i = 1; i < KS; i++) pop();
		return e;
	};
	for(int i = 0; i < part; i++) pop();

	if(all_dropped) {
#pragma unroll
		for(int i = 0; i < 8; i++) qa[i] = 0, qb[i] = 0;
	}
	// identity fragments scaled by 1/alpha (power of two times 1/softmax_scale folded by the caller: exact in bf16
	// when alpha is a power of two): row n of S^T takes the bias of its key.  Lane (q, g) supplies keys 16 c2 + 8 g + j.
	bf16x8 idf[2];
	{
		const uint32_t one_over_alpha = f32_to_bf16_bits(1.f / alpha);
#pragma unroll
		for(int c2 = 0; c2 < 2; c2++) {
			u32x4     v = {0u, 0u, 0u, 0u};
			const int j = key_of_row - 16 * c2 - 8 * half;
			if(j >= 0 && j < 8) v[j >> 1] = one_over_alpha << ((j & 1) * 16);
			idf[c2] = __builtin_bit_cast(bf16x8, v);
		}
	}
	// mask: a 32x32x8 product, contraction slot 0 = (mask value) x 1.0
	u32x2       maskA = {0u, 0u};
	const u32x2 maskB = {half == 0 ? 0x3F80u : 0u, 0u};

	const bool           has_bias = BMODE != 0 && !all_dropped;
	const unsigned char* bias_row = BMODE == 1 ? static_cast<const unsigned char*>(p.bias) + (h * p.bias_stride[0] + (row_ok ? qrow : 0) * p.bias_stride[1]) * 2 : nullptr;
	// half slot -> the two fragments of 32 keys: lane (n, half), fragment c2: keys 16 c2 + 8 half .. + 7 of query row n
	const int b_rd    = SLOT_BASE + wave_all * (2 * BIAS_HALF8) + n * 64, b_sw = (n >> 2) & 3;
	const int b_shift = RAGGED ? 8 * ((b_odd + (int)(row_ok ? qrow : L - 1) * b_row_bytes) & 2) : 0;
	u32x4     bfrag[2] = {u32x4{0u, 0u, 0u, 0u}, u32x4{0u, 0u, 0u, 0u}};
	auto read_bias = [&](int kt, int sub) {
		if constexpr(BMODE == 0) return;
		if(!has_bias) return;
#pragma unroll
		for(int c2 = 0; c2 < 2; c2++) {
			const int c = 2 * c2 + half;
			if constexpr(RING) bfrag[c2] = *reinterpret_cast<const u32x4*>(smem + b_rd + sub * BIAS_HALF8 + ((c ^ b_sw) << 4));
			if constexpr(RAGGED) {
				const int follow = c + 1 < 4 ? b_rd + (((c + 1) ^ b_sw) << 4) : b_rd - n * 64 + 2048 + n * 4;
				uint32_t  w[5]   = {bfrag[c2][0], bfrag[c2][1], bfrag[c2][2], bfrag[c2][3], *reinterpret_cast<const uint32_t*>(smem + follow + sub * BIAS_HALF8)};
				if(kt == n_ktiles - 1) {  // (wave-uniform) what stands for keys from L on: zero
					const int left = (int)L - (kt * KT8 + 32 * sub + 16 * c2 + 8 * half) + (b_shift >> 4);
#pragma unroll
					for(int j = 0; j < 5; j++) w[j] = left >= 2 * j + 2 ? w[j] : (left == 2 * j + 1 ? w[j] & 0xffffu : 0u);
				}
#pragma unroll
				for(int j = 0; j < 4; j++) bfrag[c2][j] = __builtin_amdgcn_alignbit(w[j + 1], w[j], b_shift);
			}
			if constexpr(BMODE == 1) {
				const uint16_t* bp = reinterpret_cast<const uint16_t*>(bias_row);
#pragma unroll
				for(int j = 0; j < 8; j += 2) {
					const int64_t  key = (int64_t)kt * KT8 + 32 * sub + 16 * c2 + 8 * half + j;
					const uint32_t e0  = row_ok && key < L ? (uint32_t)bp[key] : 0u, e1 = row_ok && key + 1 < L ? (uint32_t)bp[key + 1] : 0u;
					bfrag[c2][j >> 1]  = e0 | (e1 << 16);
				}
			}
		}
	};

	// per-lane LDS read addresses (buffer 0, sub-tile 0).  K: two 16-byte chunks of row key_of_row; DP = 32: of the K row (lower
	// half-wave) or of its residual (upper), DP = 64: columns 32 half .. (the swizzle repeats every 32 rows)
	int k_rd[2], v_rd[2];
#pragma unroll
	for(int i = 0; i < 2; i++) k_rd[i] = key_of_row * DP + (((DP == 64 ? 2 * half + i : i) ^ k_sw(key_of_row)) << 4) + (DP == 32 && COMP && half ? K_TILE1 : 0);
#pragma unroll
	for(int sub = 0; sub < 2; sub++) v_rd[sub] = K_TILE + n * KT8 + (((2 * sub + half) ^ v_sw(n)) << 4);   // (+ 32 KT8 per block of O^T)
	const int mask_rd = MASK_BASE + key_of_row * 2;

	float m_run = -INFINITY, mc = 0.f;  // m_run in accumulator units; mc = m_run*c_exp - P_SHIFT
	// Row sums.  ONES: rows D and D + 4 of V^T are ones, i.e. the sum of exactly the e4m3 weights that enter P.V is in register 4 (D % 32) / 8
	// of both half-waves.  Otherwise on the matrix pipe (as in dpa_mfma.hip): a 16x16x32 MFMA whose A operand is a 0/1 pattern adds
	// the 16 quantised probabilities that a query's two lanes hold of a fragment; register 0 of the result is, in every lane, the running sum of
	// that lane's own query row.  As a B operand of the 16x16x32 shape the P fragment's lane l is column l%16, contraction
	// group l/16, and holds query l%32: groups 0,2 belong to queries 0..15, groups 1,3 to queries 16..31; output register 0
	// of lane l is row 4*(l/16): rows 0 and 8 select the even groups, rows 4 and 12 the odd ones.
	f32x4 lacc = {0.f, 0.f, 0.f, 0.f};
	long  ones_a = 0;
	if constexpr(!ONES) {
		const int  i16 = lane & 15, kg = lane >> 4;
		const bool on  = ((i16 == 0 || i16 == 8) && (kg & 1) == 0) || ((i16 == 4 || i16 == 12) && (kg & 1) == 1);
		const u32x2 w  = {on ? 0x38383838u : 0u, on ? 0x38383838u : 0u};  // e4m3 1.0
		ones_a = __builtin_bit_cast(long, w);
	}
	f32x16 oacc[NDB];
#pragma unroll
	for(int db = 0; db < NDB; db++)
#pragma unroll
		for(int i = 0; i < 16; i++) oacc[db][i] = 0.f;

	auto read_k = [&](int off, int res) -> i32x8 {   // (res: DP = 64, the residual tile)
		const u32x4 lo = *reinterpret_cast<const u32x4*>(smem + off + k_rd[0] + res * K_TILE1), hi = *reinterpret_cast<const u32x4*>(smem + off + k_rd[1] + res * K_TILE1);
		return i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
	};
	auto kq = [&](const i32x8& k, const i32x8& q, const f32x16& c) -> f32x16 { return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(k, q, c, 0, 0, 0, 0, 0, 0); };
	auto bias_mfma = [&](const f32x16& c, int c2) -> f32x16 { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(idf[c2], __builtin_bit_cast(bf16x8, bfrag[c2]), c, 0, 0, 0); };
	auto mask_mfma = [&](const f32x16& c) -> f32x16 {
		return __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(__builtin_bit_cast(s16x4, maskA), __builtin_bit_cast(s16x4, maskB), c, 0, 0, 0);
	};
	auto exp_part = [&](const f32x16& s, u32x2 (&pf)[2], auto i_c) {   // logits 4 I .. 4 I + 3
		constexpr int I = decltype(i_c)::value;
		const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[4 * I], c_exp, -mc)), p1 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[4 * I + 1], c_exp, -mc));
		const float p2 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[4 * I + 2], c_exp, -mc)), p3 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[4 * I + 3], c_exp, -mc));
		int w = __float_as_int(p0);   // (both halves are written)
		w = __builtin_amdgcn_cvt_pk_fp8_f32(p0, p1, w, false);
		w = __builtin_amdgcn_cvt_pk_fp8_f32(p2, p3, w, true);
		pf[I >> 1][I & 1] = (uint32_t)w;
	};

	f32x16 sc;
	// One stage: on entry `sc` holds the finished logits of 32 keys (half SUB of the tile whose V^T tile is at v_off); it leaves those of
	// the next 32 (half 1 - SUB of tile kt_n, K tile at k_off) in `sc` and adds these keys' P.V.  after_bias runs once the bias fragments have been read.
	auto stage = [&](auto sub_c, int kt_n, bool full_n, int k_off, int v_off, auto&& after_bias) {
		constexpr int SUB = decltype(sub_c)::value, SUBN = 1 - SUB;
		const i32x8 ka = read_k(k_off + SUBN * 32 * DP, 0);
		i32x8       kb = ka;
		if constexpr(DP == 64 && COMP) kb = read_k(k_off + SUBN * 32 * DP, 1);
		read_bias(kt_n, SUBN);
		if(!full_n) maskA[0] = *reinterpret_cast<const uint16_t*>(smem + mask_rd + kt_n * (KT8 * 2) + SUBN * 64);
		// online softmax with the true running maximum (in accumulator units)
		// (two chains of three-operand maxima)
		const float mx0 = max17(sc, m_run);
		const auto  sw    = __builtin_amdgcn_permlane32_swap(__float_as_uint(mx0), __float_as_uint(mx0), false, false);
		const float m_new = max3(mx0, __uint_as_float(sw[0]), __uint_as_float(sw[1]));
		if(__ballot(m_new > m_run)) {   // (the first time from -inf: the factor is 0, and nothing has been accumulated)
			const float a = __builtin_amdgcn_exp2f((m_run - m_new) * c_exp);
			if constexpr(!ONES) lacc[0] *= a;
#pragma unroll
			for(int db = 0; db < NDB; db++)
#pragma unroll
				for(int i = 0; i < 16; i++)
					if(!(ONES && db == NDB - 1 && i > 12)) oacc[db][i] *= a;   // (those hold rows of zeros)
			m_run = m_new;
			mc    = m_new * c_exp - P_SHIFT;
		}
		// (the accumulators keep their registers whether or not they were rescaled: the compiler would copy them otherwise)
#pragma unroll
		for(int db = 0; db < NDB; db++) asm volatile("" : "+v"(oacc[db]));
		after_bias();
		u32x2  pf[2];
		f32x16 sn;
#pragma unroll
		for(int i = 0; i < 16; i++) sn[i] = 0.f;
		// One matrix instruction, then a quarter of the exponentials, and so on; the empty asm statements pin that order (matrix
		// intrinsics are values to the compiler and would all be issued in front, each waiting for the one before)
		auto pin = [&](auto i_c) {
			constexpr int I = decltype(i_c)::value;
			float    a_ = sn[0];
			uint32_t b_ = pf[I >> 1][I & 1];
			asm volatile("" : "+v"(a_), "+v"(b_));
			sn[0] = a_, pf[I >> 1][I & 1] = b_;
			__builtin_amdgcn_sched_barrier(0);
		};
		__builtin_amdgcn_sched_barrier(0);
		sn = kq(ka, qa, sn);
		exp_part(sc, pf, ic<0>{});
		pin(ic<0>{});
		if constexpr(COMP && DP == 64) sn = kq(kb, qa, sn);
		if constexpr(COMP) sn = kq(ka, qb, sn);
		exp_part(sc, pf, ic<1>{});
		pin(ic<1>{});
		u32x4 vf[NDB];
#pragma unroll
		for(int db = 0; db < NDB; db++) vf[db] = *reinterpret_cast<const u32x4*>(smem + v_off + v_rd[SUB] + db * 32 * KT8);
		if constexpr(BMODE != 0) sn = bias_mfma(sn, 0);
		exp_part(sc, pf, ic<2>{});
		pin(ic<2>{});
		if constexpr(BMODE != 0) sn = bias_mfma(sn, 1);
		exp_part(sc, pf, ic<3>{});
		pin(ic<3>{});
		if(!full_n) sn = mask_mfma(sn);
		if constexpr(!ONES) {
#pragma unroll
			for(int cp = 0; cp < 2; cp++) lacc = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(ones_a, __builtin_bit_cast(long, pf[cp]), lacc, 0, 0, 0);
		}
		// O^T += V8^T . P^T: contraction slot 8 half + j of chunk cp is key 16 half + 8 cp + j
#pragma unroll
		for(int cp = 0; cp < 2; cp++)
#pragma unroll
			for(int db = 0; db < NDB; db++)
				oacc[db] = __builtin_amdgcn_mfma_f32_32x32x16_fp8_fp8(__builtin_bit_cast(long, u32x2{vf[db][2 * cp], vf[db][2 * cp + 1]}), __builtin_bit_cast(long, pf[cp]), oacc[db], 0, 0, 0);
		sc = sn;
	};

	// ---- prologue: first tile, its first logits; second tile under way ----
	int entry = next_entry(), entry1 = next_entry();
	if((entry & ~TILE_FULL) != guess) {   // (the guess was wrong; loads land in issue order)
		load_tile(entry & ~TILE_FULL, buf0);
		load_bias(entry & ~TILE_FULL, 0);
		load_bias(entry & ~TILE_FULL, 1);
	}
	asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
	{
		const int kt0 = entry & ~TILE_FULL;
		read_bias(kt0, 0);
		asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
		if(nlive > 1) {
			load_tile(entry1 & ~TILE_FULL, buf0 + TILE);
			load_bias(entry1 & ~TILE_FULL, 0);
		}
#pragma unroll
		for(int i = 0; i < 16; i++) sc[i] = 0.f;
		const i32x8 ka = read_k(buf0, 0);
		sc = kq(ka, qa, sc);
		if constexpr(COMP) {
			if constexpr(DP == 64) sc = kq(read_k(buf0, 1), qa, sc);
			sc = kq(ka, qb, sc);
		}
		if constexpr(BMODE != 0) sc = bias_mfma(bias_mfma(sc, 0), 1);
		maskA[0] = *reinterpret_cast<const uint16_t*>(smem + mask_rd + kt0 * (KT8 * 2));
		sc = mask_mfma(sc);
	}
	// Tile `it` is in buffer it % 3.  Order of this wavefront's loads: tile it + 1 (behind the barrier of iteration it - 1), its
	// first half of bias (in the second stage of it - 1), its second half (in the first stage of it), tile it + 2, ...
	int cur = buf0;
	even_progress progress(nlive, even);
	for(int it = 0; it < nlive; it++) {
		progress.at(it);
		const int  kt = entry & ~TILE_FULL, kt1 = entry1 & ~TILE_FULL;
		const int  nxt = cur == buf0 + 2 * TILE ? buf0 : cur + TILE, nxt2 = nxt == buf0 + 2 * TILE ? buf0 : nxt + TILE;
		const bool has1 = it + 1 < nlive, has2 = it + 2 < nlive;
		const int  entry2 = next_entry();
		// the second half of this tile's bias has landed (younger: tile it + 1 and the first half of its bias)
		if(has1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(KV_MIN + BIAS_LOADS) : "memory");
		else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
		stage(ic<0>{}, kt, (entry & TILE_FULL) != 0, cur, cur, [&]() {
			if constexpr(RING)
				if(has1) {
					asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (the half slot has been read)
					load_bias(kt1, 1);
				}
		});
		// tile it + 1 and the first half of its bias have landed (younger: the second half); behind the barrier everyone is done with tile it - 1
		if(has1) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(BIAS_LOADS) : "memory");
		else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
		if(has2) load_tile(entry2 & ~TILE_FULL, nxt2);
		stage(ic<1>{}, kt1, (entry1 & TILE_FULL) != 0, nxt, cur, [&]() {
			if constexpr(RING)
				if(has2) {
					asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
					load_bias(entry2 & ~TILE_FULL, 0);
				}
		});
		entry = entry1, entry1 = entry2, cur = nxt;
	}

	if constexpr(KS > 1) {
		if(nlive < n_most) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");   // (the barrier of the other parts' last tile)
		// the other parts' O, l and m to the first, [wavefront of those][register / 4][lane] x 16 bytes
		constexpr int REGS4 = 4 * NDB + 1;
		static_assert((KS - 1) * NW8 * REGS4 * 1024 <= MASK_BASE, "the partial sums fit the buffers");
		f32x4* const at = reinterpret_cast<f32x4*>(smem) + (part > 0 ? wave_all - NW8 : wave) * (REGS4 * 64) + lane;
		__syncthreads();   // everyone is done with the buffers
		if(part > 0) {
#pragma unroll
			for(int db = 0; db < NDB; db++)
#pragma unroll
				for(int i = 0; i < 4; i++) at[(4 * db + i) * 64] = f32x4{oacc[db][4 * i], oacc[db][4 * i + 1], oacc[db][4 * i + 2], oacc[db][4 * i + 3]};
			at[4 * NDB * 64] = f32x4{m_run, lacc[0], 0.f, 0.f};
		}
		__syncthreads();
		if(part > 0) return;
#pragma unroll
		for(int o = 0; o < KS - 1; o++) {   // (a part without tiles: m = -inf, factor 0)
			const f32x4* const from = at + o * (NW8 * REGS4 * 64);
			const f32x4        ml   = from[4 * NDB * 64];
			const float        m_new = fmaxf(m_run, ml[0]), a = __builtin_amdgcn_exp2f((m_run - m_new) * c_exp), f = __builtin_amdgcn_exp2f((ml[0] - m_new) * c_exp);
			m_run   = m_new;
			lacc[0] = lacc[0] * a + ml[1] * f;
#pragma unroll
			for(int db = 0; db < NDB; db++)
#pragma unroll
				for(int i = 0; i < 4; i++) {
					const f32x4 x = from[(4 * db + i) * 64];
#pragma unroll
					for(int j = 0; j < 4; j++) oacc[db][4 * i + j] = oacc[db][4 * i + j] * a + x[j] * f;
				}
		}
	}
	// epilogue: out = O * dv / l   (l was summed over p * 2^8, the same factor O carries; both half-waves are in it)
	float l_tot = lacc[0];
	if constexpr(ONES) {
		const int i = (D & 31) >> 3;   // 1, 2 or 3: register 4 i of the last block
		l_tot = i == 1 ? oacc[NDB - 1][4] : i == 2 ? oacc[NDB - 1][8] : oacc[NDB - 1][12];
	}
	const float inv = dv / l_tot;
	if(row_ok) {
		const int64_t ooff = b * p.out_stride[0] + h * p.out_stride[1] + qrow * p.out_stride[2];
#pragma unroll
		for(int db = 0; db < NDB; db++)
#pragma unroll
			for(int g4 = 0; g4 < 4; g4++) {
				const int d0 = 32 * db + 8 * g4 + 4 * half;
				if(d0 >= D) continue;
				const float o0 = oacc[db][4 * g4] * inv, o1 = oacc[db][4 * g4 + 1] * inv, o2 = oacc[db][4 * g4 + 2] * inv, o3 = oacc[db][4 * g4 + 3] * inv;
				if(p.out_dtype == AF3_BF16) {
					u32x2 w = {pack_bf16x2(o0, o1), pack_bf16x2(o2, o3)};
					*reinterpret_cast<u32x2*>(static_cast<uint16_t*>(p.out) + ooff + d0) = w;
				} else {
					float4 w = {o0, o1, o2, o3};
					*reinterpret_cast<float4*>(static_cast<float*>(p.out) + ooff + d0) = w;
				}
			}
	}
}

template <int DP, bool COMP, bool ONES, int BMODE, int KS>
int launch8_parts(const af3_dpa_params& p, hipStream_t s) {
	const int     n_qtiles = (int)((p.L + NW8 * 32 - 1) / (NW8 * 32));
	const int     n_ktiles = (int)((p.L + KT8 - 1) / KT8);
	// The batch rows share the bias: with a bias to share, the workgroups of one block of query rows run side by side on one XCD, whose L2
	// then serves all but the first of them.  Fewer than 64 such blocks fill the XCDs unevenly and are dealt by (batch row, head).
	// (16 heads of 24, 1536 rows, us per call, pairs / blocks: 5 batch rows 76.8 / 75.2, 8 106.9 / 102.5; 8 of 1301 102.0 / 100.2.)
	const int64_t n_blocks = p.H * n_qtiles, n_groups = p.B * p.H;
	const int64_t side_by  = (n_blocks + 7) / 8 * 8 * p.B;
	const int64_t per_xcd  = p.bias && p.B > 1 && n_blocks >= 64 && side_by <= 0x7fffffffLL ? (n_blocks + 7) / 8 : 0;
	const int64_t blocks   = per_xcd > 0 ? side_by : (n_groups + 7) / 8 * 8 * n_qtiles;
	if(blocks <= 0 || blocks > 0x7fffffffLL) return AF3_ERR_BAD_SHAPE;
	const size_t smem = (size_t)KS * (3 * (COMP ? 3 : 2) * KT8 * DP + (BMODE >= 2 ? NW8 * 2 * BIAS_HALF8 : 0)) + (size_t)n_ktiles * KT8 * 2 + (size_t)((n_ktiles + 15) & ~15);
	const int64_t by_lds = 160 * 1024 / (int64_t)smem, by_regs = (DP == 32 ? 4 : KS == 1 ? 3 : 2) / KS;   // workgroups a compute unit holds
	const int64_t per_cu = by_lds < 1 ? 1 : by_lds < by_regs ? by_lds : by_regs;
	auto         kern = dpa_mfma_fp8_kernel<DP, COMP, ONES, BMODE, KS>;
	if(smem > 64 * 1024 && hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) return AF3_ERR_LAUNCH;
	hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(KS * NW8 * 64), smem, s, p, n_qtiles, (int)(per_xcd > 0 ? n_blocks : n_groups), (int)per_xcd, progress_mode(n_groups * n_qtiles, 256 * per_cu));
	return launch_status();
}
template <int DP, bool COMP, bool ONES, int BMODE>
int launch8(const af3_dpa_params& p, hipStream_t s) {
	// Launches of few workgroups: two parts.  A lone wavefront of a SIMD takes 1070 clocks for a stage, of which its 175 instructions are 790,
	// two take 1330 for both; from two workgroups per compute unit on there is nothing left to fill, and a part of one or two tiles
	// is not worth its merge.  16 heads of 24, us per call, one part / two: 1x128 11.9/12.0, 1x256 14.1/13.5, 1x512 18.4/16.4, 2x777 25.5/22.9,
	// 1x1536 33.8/27.5, 2x1536 42.5/39.4, 8x512 25.9/25.5, but 8x300 22.6/24.0, 3x1301 50.7/55.0, 3x1536 53.1/56.5.  Four parts are slower than two
	// throughout (1x512 18.2, 1x1536 28.3).  Head_dim above 32 (one such workgroup per compute unit): 16 heads of 48, 1x777 29.2/26.0, 1x1536
	// 40.9/34.3, 2x1200 43.7/49.9.  (Compensated, head_dim 32, rows at any address: 128 registers with 5 spilled in one part, 7 in two;
	// 16 heads of 32, 1x777 31.6/25.0, 1x1491 50.9/37.0, one part throughout 5x1491 89.6 against 79.7 at an aligned 1496.)
	if constexpr(BMODE >= 2) {
		const int64_t n_wg = p.B * p.H * ((p.L + NW8 * 32 - 1) / (NW8 * 32)), n_ktiles = (p.L + KT8 - 1) / KT8;
		if(n_ktiles >= 3 && (n_wg <= 256 || (DP == 32 && n_wg <= 512 && n_ktiles >= 8))) return launch8_parts<DP, COMP, ONES, BMODE, 2>(p, s);
	}
	return launch8_parts<DP, COMP, ONES, BMODE, 1>(p, s);
}
template <int DP, bool COMP, bool ONES>
int launch8_bias(const af3_dpa_params& p, hipStream_t s) {
	if(!p.bias) return launch8<DP, COMP, ONES, 0>(p, s);
	// offsets of a head's bias (and the loads' overhang at its end) fit 32 bits; whole aligned chunks that never straddle the end of a row, or the ragged form
	if(((p.L - 1) * p.bias_stride[1] + p.L) * 2 >= ((int64_t)1 << 31) - 64 * 1024) return launch8<DP, COMP, ONES, 1>(p, s);
	const bool aligned = (reinterpret_cast<uintptr_t>(p.bias) & 15) == 0 && p.bias_stride[0] % 8 == 0 && p.bias_stride[1] % 8 == 0 && p.L % 8 == 0;
	return aligned ? launch8<DP, COMP, ONES, 2>(p, s) : launch8<DP, COMP, ONES, 3>(p, s);
}
template <int DP>
int launch8_form(const af3_dpa_params& p, hipStream_t s) {
	const bool comp = p.q_lo != nullptr && p.k_lo != nullptr;
	if(p.D < DP) return comp ? launch8_bias<DP, true, true>(p, s) : launch8_bias<DP, false, true>(p, s);
	return comp ? launch8_bias<DP, true, false>(p, s) : launch8_bias<DP, false, false>(p, s);
}

}  // namespace

bool mfma_fp8_eligible(const af3_dpa_params& p) {
	if(p.io_dtype != AF3_FP8_E4M3 || p.mma_dtype != AF3_FP8_E4M3) return false;
	if(p.D > 64 || p.D % 8 != 0 || p.L > MAX_L8) return false;
	if(p.bias && p.bias_dtype != AF3_BF16) return false;
	// q rows are read 8 bytes at a time, K / V^T rows in 16-byte chunks at 4-byte aligned offsets
	if((reinterpret_cast<uintptr_t>(p.q) & 7) || (reinterpret_cast<uintptr_t>(p.k) & 3) || (reinterpret_cast<uintptr_t>(p.v) & 15)) return false;
	if((p.q_lo != nullptr) != (p.k_lo != nullptr)) return false;  // both residuals or none
	if((reinterpret_cast<uintptr_t>(p.q_lo) & 7) || (reinterpret_cast<uintptr_t>(p.k_lo) & 3)) return false;
	for(int i = 0; i < 3; i++)
		if(p.q_stride[i] % 8 || p.k_stride[i] % 4 || p.v_stride[i] % 16) return false;
	if(p.L * p.k_stride[2] >= 0x7fffffffLL || p.D * p.v_stride[2] >= 0x7fffffffLL) return false;
	if(p.out_dtype == AF3_BF16) {
		if((reinterpret_cast<uintptr_t>(p.out) & 7) || p.out_stride[0] % 4 || p.out_stride[1] % 4 || p.out_stride[2] % 4) return false;
	} else if((reinterpret_cast<uintptr_t>(p.out) & 15) || p.out_stride[0] % 4 || p.out_stride[1] % 4 || p.out_stride[2] % 4) {
		return false;
	}
	return true;
}

int launch_dpa_mfma_fp8(const af3_dpa_params& p, hipStream_t s) {
	return p.D <= 32 ? launch8_form<32>(p, s) : launch8_form<64>(p, s);
}

}  // namespace af3
