// bf16 matrix-core attention kernel for calls that read their bias in place, once per batch row (single attention with pair bias,
// the token attention of the diffusion transformer, small batches), head_dim up to 48.
//
// Such a launch has few query rows (16 heads of 768: 12288, 12 per SIMD), so the query rows are cut fine and the key axis is cut as
// well: a workgroup owns a strip of NB x 16 query rows of one (batch row, head) -- one to four blocks; 48 rows of 768 make 256 workgroups,
// one per compute unit -- and its wavefronts take the key tiles (32 keys) of the strip in turn.  The NB blocks of 16 rows are NB
// independent chains of one wavefront: they share the tile's K, V and mask operands, and while one block's logits are exponentiated
// the matrix pipe works on its neighbours.  Nothing is shared between wavefronts until the strip's partial sums are added up
// through LDS at the end, so the walk has no barrier: every wavefront's bias, K and V travel by loads that write LDS directly, into
// places of its own, each asked to hold the next tile as soon as it has been read, and are awaited by count.
//
// Logits: S^T[key][q] = K . Q^T on v_mfma_f32_16x16x32_bf16 in two halves of 16 keys, on top of the bias as the matrix pipe adds it
// (a 0/1 selection times the bias rows as they lie in memory: exact), on top of the key mask (the C operand, shared by the strip's
// blocks).  Rows 8 (i / 4) + 4 h + i % 4 of the tile form half h, so that a lane's eight probabilities are eight consecutive keys, the
// order in which ds_read_b64_tr_b16 delivers V^T.  A column of ones in V's padding (or a constant operand) makes the row sums one more
// column of O.
//
// Softmax: the walk subtracts nothing, or, from rows that look masked through their bias, that bias.  Sums that end within
// 2^-60 .. 2^100 with finite results stand (probabilities and sums are floating-point; 2^-60 leaves 66 powers of two below a row's
// largest probability); otherwise the workgroup finds its rows' maxima in a walk of their own and repeats the walk with them (one such
// row in every strip: 7.4 -> 13.4 us at 16 x 768 x 24, 17.7 -> 41 at 1536).
//
// Reference: one (batch, head, query tile) task of src/csrc/dot_product_attention.cpp:88-191.
#include "mfma_helpers.hpp"

namespace af3 {

namespace {

constexpr int      KT_S       = 32;   // keys per tile
// what a dropped key's logit gets: no bias of eight bits brings it near 0, so that the sums of a row without a live key never stand
constexpr float    DROPPED    = MASK_DROPPED - 0x1p88f;

// What the kernel takes, as the launcher lays it out: a workgroup's start is a chain of scalar instructions that no other work covers
// and whose code is fetched cold, so nothing is divided and little is multiplied there.
struct strip_args {
	const char *   q, *k, *v, *bias, *gate;
	const uint8_t* mask;
	char*          out;
	int64_t        q_b, q_h, k_b, k_h, v_b, v_h, bias_h, gate_b, gate_h, mask_b, out_b, out_h;   // bytes
	int32_t        q_row, k_row, v_row, gate_row, out_row;                                         // bytes
	uint32_t       bias_row;
	int32_t        H, L, D, per_chunk, per_quad;   // 2^16 / (D / 8) and / (D / 4), rounded up
	int32_t        out_f32;
	uint32_t       bias_limit;   // two bf16: lower biases, -inf included, become this (0 * inf in the selection product is NaN)
	float          scale;
};

// A workgroup's LDS, all of it dynamic, as the kernel and its launcher see it:
// [tiles and constants of each wavefront | partial sums (in the same place, later)] [q, as the matrix instructions take it | rows' maxima (later)] [a flag] [key-mask tables: 128 B per tile]
template <int NB, int KIND, bool ANY, int NW>
struct strip_lds {
	static constexpr int KS = KIND == 2 ? 2 : 1;       // contraction steps of 32 head columns
	static constexpr int NV = KIND == 2 ? 3 : 2;       // 1 KB loads of a K or V tile
	static constexpr int R  = NB * 16;                 // query rows of the strip
	static constexpr int NT = ANY ? (NB + 3) / 4 : 0;  // loads of the dwords that follow the rows of a tile's bias (64 rows each)
	static constexpr int PC = KIND == 2 ? 52 : 36;     // floats of a row's partial sums
	static constexpr int WAVE   = 2 * NB * 1024 + 2 * NV * 1024 + 2 * NT * 256 + 32;   // of a wavefront's own: two tiles of the bias, one of K and of V, constants
	static constexpr int Q_ROW  = KS * 64 + 16;
	static constexpr int TILES = NW * WAVE, PARTS = NW * R * PC * 4, Q_AT = TILES > PARTS ? TILES : PARTS;
	static constexpr int FLAG_AT = Q_AT + (KIND == 1 ? 2 : 1) * R * Q_ROW, MASK_AT = FLAG_AT + 16;
	static_assert(NW * R * 4 <= R * Q_ROW, "the rows' maxima of all wavefronts take no more than q did");
	static constexpr int bytes(int L) { return MASK_AT + ((L + KT_S - 1) / KT_S + NW) * 128; }
	static_assert(bytes(MAX_L_MFMA) <= 160 * 1024, "every length that reaches this kernel fits a compute unit");
};

// KIND: 0 = head_dim up to 24 (row sums in V's column 24), 1 = 32, 2 = 40 and 48 (two contraction steps).  Grid: x = head (with a multiple of 8 heads the strips of one head share an XCD and
// its L2 copy of K and V), y = strip, z = batch row.  EVEN: wavefronts that are behind on their walk go first (goes_evenly).
template <int NB, int KIND, bool ANY, int NW, bool EVEN>
__global__ void __launch_bounds__(NW * 64) __attribute__((amdgpu_waves_per_eu(2, 2))) dpa_strip_bf16_kernel(strip_args p) {
	using lds = strip_lds<NB, KIND, ANY, NW>;
	static_assert(NB <= 4, "the walk has four slots a tile");
	constexpr int KS = lds::KS, NV = lds::NV, NT = lds::NT, R = lds::R, PC = lds::PC, WAVE_LDS = lds::WAVE, Q_AT = lds::Q_AT, Q_ROW = lds::Q_ROW, MASK_AT = lds::MASK_AT;
	constexpr int ND = KIND == 2 ? 3 : 2;       // blocks of 16 head columns of V
	constexpr int NO = KIND == 0 ? ND : ND + 1; // ... of O: the row sums in a block of their own, or in column 24
	constexpr bool LO = KIND == 1;              // q's second term meets K in matrix instructions of its own
	constexpr int SUM_COL = KIND == 0 ? 24 : 16 * ND;
	extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
	float* const s_max = reinterpret_cast<float*>(smem + Q_AT);   // (q is in registers by then)
	int* const   s_bad = reinterpret_cast<int*>(smem + lds::FLAG_AT);   // [0]: rows whose sums do not stand; [1]: how many wavefronts took references from samples, + 2^8 for each that took one below a dropped key's logit, + 2^16 if its tiles hold a live key; [2]: wavefronts whose tiles do (second walk)

	asm volatile("" ::"s"(p.q), "s"(p.k), "s"(p.v), "s"(p.bias), "s"(p.mask), "s"(p.q_h), "s"(p.k_h), "s"(p.v_h), "s"(p.bias_h), "s"(p.q_row), "s"(p.k_row), "s"(p.v_row), "s"(p.bias_row), "s"(p.H),
				 "s"(p.L), "s"(p.D), "s"(p.per_chunk), "s"(p.scale));
	const int h = blockIdx.x, strip = blockIdx.y, b = blockIdx.z;
	const int L = p.L, D = p.D;
	const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int i16 = lane & 15, g = lane >> 4;
	const int n_tiles = (L + KT_S - 1) / KT_S;
	const char* const    kp   = p.k + b * p.k_b + h * p.k_h;
	const char* const    vp   = p.v + b * p.v_b + h * p.v_h;
	const char* const    qp   = p.q + b * p.q_b + h * p.q_h;
	const char* const    bias = p.bias + h * p.bias_h;
	const uint8_t* const keep = p.mask + b * p.mask_b;
	const bool           masked = p.mask != nullptr;
	const int            ks2 = p.k_row, vs2 = p.v_row;

	// ---- requests that the compiler waits for: q (a thread takes a 16-byte chunk of a row of the strip, padding included: what the
	// range checks keep out is zero), and the key mask of this wavefront's tiles (wave, wave + NW, ...) ----
	constexpr int QN = (R * 4 * KS + NW * 64 - 1) / (NW * 64);
	const int DC = D >> 3;   // 16-byte chunks of a q, K or V row
	auto q_chunk = [&](int ch) __attribute__((always_inline)) { return ch < DC ? ch : ch - DC; };   // (chunk DC + c of an operand: the second term of chunk c)
	const __amdgpu_buffer_rsrc_t q_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(qp), 0, (L - 1) * p.q_row + D * 2, 0x00020000);
	u32x4 qraw[QN];
#pragma unroll
	for(int j = 0; j < QN; j++) {
		const int i = tid + j * NW * 64, ch = i % (4 * KS);
		qraw[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(q_rsrc, q_chunk(ch) < DC ? (strip * R + i / (4 * KS)) * p.q_row + q_chunk(ch) * 16 : 0x40000000, 0, 0));
	}
	const int last_k0 = L - KT_S, my_all = (n_tiles - wave + NW - 1) / NW;   // (0 or less: no tile)
	const __amdgpu_buffer_rsrc_t m_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(keep), 0, masked ? L : 0, 0x00020000);
	// lane = key of a tile, the upper half-wave that of this wavefront's next tile
	const int mask_key = (wave + (lane >> 5) * NW) * KT_S + (lane & 31);
	auto load_mask = [&](int j) __attribute__((always_inline)) {   // (a lane whose key lies at or beyond L looks at the key it stands for in the last tile, moved forward)
		const int key = mask_key + j * (2 * NW * KT_S), over = (key | 31) + 1 - L;
		return (uint32_t)(uint8_t)__builtin_amdgcn_raw_buffer_load_b8(m_rsrc, over > 0 ? key - over : key, 0, 0);
	};
	uint32_t m_first[2] = {load_mask(0), load_mask(1)};

	// ---- loads that write LDS directly.  A wavefront's tiles are its own: nothing but its own waits orders them.  The last tile of a
	// length that is no multiple of 32 starts at key L - 32; its first keys, seen before, are masked out of it. ----
	const int b_base = wave * WAVE_LDS, k_base = b_base + 2 * NB * 1024, v_base = k_base + NV * 1024, t_base = v_base + NV * 1024, const_base = t_base + 2 * NT * 256;
	// K: place i of half h holds key 8 (i / 4) + 4 h + i % 4; with 2, 4 or 6 chunks a row the chunks of some rows are swapped, so that the 16 rows
	// of a fragment read always meet 16 different places of the banks
	const int  swap_shift = DC == 4 ? 2 : 3, swap_mask = DC == 4 ? 3 : DC & 1 ? 0 : 1;
	auto key_at = [](int place) __attribute__((always_inline)) { return 8 * ((place >> 2) & 3) + 4 * (place >> 4) + (place & 3); };
	int k_off[NV], v_off[NV];
#pragma unroll
	for(int j = 0; j < NV; j++) {
		const int  idx = 64 * j + lane, row = (idx * p.per_chunk) >> 16, ch = idx - row * DC;   // idx / DC
		const bool in  = idx < 32 * DC;
		k_off[j] = in ? key_at(row) * ks2 + ((ch ^ (((row & 15) >> swap_shift) & swap_mask)) << 4) : 0x40000000;   // (out of range: nothing is fetched)
		v_off[j] = in ? row * vs2 + ch * 16 : 0x40000000;
	}
	// The bias travels as whole 64-byte pieces of 16 rows; of rows past L nothing is fetched that the head's slab does not hold, and
	// what they compute stays in their own columns of every product.  Where rows start at any element (ANY) a piece is fetched from the
	// dword that holds its first element, the dword behind it separately, and shifted when it is read.
	const int odd_row = ANY ? (int)((p.bias_row >> 1) & 1) : 0, odd_base = ANY ? (int)((reinterpret_cast<uintptr_t>(bias) >> 1) & 1) : 0;
	const int b_off = (strip * R + (lane >> 2)) * (int)p.bias_row + odd_base * 2 + (((lane & 3) ^ ((lane >> 4) & 3)) << 4), b_step = 16 * (int)p.bias_row;
	const int t_off = ANY ? (strip * R + lane) * (int)p.bias_row + odd_base * 2 + 64 : 0;
	const uint32_t k_bytes = (L - 1) * ks2 + D * 2, v_bytes = (L - 1) * vs2 + D * 2, b_bytes = ((uint32_t)(L - 1) * p.bias_row + L * 2 + odd_base * 2 + 3) & ~3u;
	u32x4 k_rsrc = raw_rsrc(kp, k_bytes), v_rsrc = raw_rsrc(vp, v_bytes), b_rsrc = raw_rsrc(bias - odd_base * 2, b_bytes);
	const uint32_t lds0 = lds_addr_of(smem);
	auto load_k = [&](int k0) __attribute__((always_inline)) {
		const int at = k0 * ks2;
#pragma unroll
		for(int j = 0; j < NV; j++) lds_dma_b128(k_rsrc, lds0 + k_base + j * 1024, k_off[j] + at);
	};
	auto load_v = [&](int k0) __attribute__((always_inline)) {
		const int at = k0 * vs2;
#pragma unroll
		for(int j = 0; j < NV; j++) lds_dma_b128(v_rsrc, lds0 + v_base + j * 1024, v_off[j] + at);
	};
	auto load_b = [&](int k0, int half, int c) __attribute__((always_inline)) {
		const int at = b_off + (c * b_step + 2 * k0);
		lds_dma_b128(b_rsrc, lds0 + b_base + half + c * 1024, ANY ? at & ~3 : at);
	};
	auto load_t = [&](int k0, int half) __attribute__((always_inline)) {   // half: as for the bias
#pragma unroll
		for(int j = 0; j < NT; j++) lds_dma_b32(b_rsrc, lds0 + t_base + (half ? NT * 256 : 0) + j * 256, (t_off + (4 * j * b_step + 2 * k0)) & ~3);
	};
	const int k0_first = wave * KT_S < last_k0 ? wave * KT_S : last_k0;
	auto load_first = [&]() __attribute__((always_inline)) {
		load_k(k0_first);
#pragma unroll
		for(int c = 0; c < NB; c++) load_b(k0_first, 0, c);
		load_t(k0_first, 0);
		load_v(k0_first);
	};
	load_first();

	// ---- constants in LDS: zeros, and V's column of ones ----
	const int ZEROS_AT = const_base, ONES_AT = const_base + 16;
	auto fill = [&]() __attribute__((always_inline)) {
		if(lane < 8) *reinterpret_cast<uint32_t*>(smem + const_base + 4 * lane) = lane == 4 ? 0x3F80u : 0u;
	};
	fill();
	if(tid < 3) s_bad[tid] = 0;

	// ---- per-lane constants ----
	u32x4 sel[2];   // half h of the tile's keys: row i picks key 8 (i / 4) + 4 h + i % 4
	const int k_row = key_at(i16);
#pragma unroll
	for(int hf = 0; hf < 2; hf++)
#pragma unroll
		for(int j = 0; j < 4; j++) {
			const int at = k_row + 4 * hf - 8 * g - 2 * j;   // element 2 j + at of this lane's eight
			sel[hf][j] = at == 0 ? 0x3F80u : at == 1 ? 0x3F800000u : 0u;
		}
	const u32x4 ones    = {0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
	int k_rd[KS][2], v_rd[ND][2];
#pragma unroll
	for(int st = 0; st < KS; st++)
#pragma unroll
		for(int hf = 0; hf < 2; hf++) {
			const int ch = 4 * st + g;
			k_rd[st][hf] = q_chunk(ch) < DC ? k_base + (16 * hf + i16) * (DC * 16) + ((q_chunk(ch) ^ ((i16 >> swap_shift) & swap_mask)) << 4) : ZEROS_AT;
		}
#pragma unroll
	for(int d = 0; d < ND; d++)
#pragma unroll
		for(int u = 0; u < 2; u++) {
			const int col = 16 * d + 4 * (i16 & 3);
			v_rd[d][u] = col < D ? v_base + (8 * g + 4 * u + (i16 >> 2)) * (DC * 16) + col * 2 : KIND == 0 && col == 24 ? ONES_AT : ZEROS_AT;
		}
	const int mask_base = MASK_AT + wave * ((n_tiles + NW - 1) / NW) * 128;
	const int m_rd = mask_base + g * 32;   // this lane's eight keys; + 128 per tile of this wavefront
	const int sh0 = ((odd_base + odd_row * i16) & 1) << 4;
	const int t_rd = g < 3 ? b_base + i16 * 64 + (((g + 1) ^ ((i16 >> 2) & 3)) << 4) : t_base + i16 * 4;   // the dword behind this lane's eight elements
	const int t_half = g < 3 ? NB * 1024 : NT * 256, t_blk = g < 3 ? 1024 : 64;
	const int b_rd = b_base + i16 * 64 + ((g ^ ((i16 >> 2) & 3)) << 4);
	const int s_row = lane < R ? lane : R - 1, s_rd = b_base + s_row * 64 + (((s_row >> 2) & 3) << 4) + 2;   // one bias (the first or second of this wavefront's first tile) of each row
	const unsigned s_low = strip * R + s_row < L ? 0xC200u : 0xFFFFu;   // -32 (of rows past L: none is lower)

	// q to LDS, scaled, as two bf16 terms as far as there is room: the second one of the first columns takes the columns behind head_dim, where
	// K's operand repeats those columns, or (head_dim 32: none) all of it goes through matrix instructions of its own.  (Rounded once, the
	// rms error against 64 bits was 1 to 8 % above that of the one-row kernel, whose reference makes a row's largest weight exactly
	// 1; now, one-row kernel / here: 37 x 4 x 37 x 32 8.2e-4 / 7.5e-4, 16 heads of 24 x 768 2.8e-4 / 2.7e-4, 16 heads of 48 x 128 5.4e-4 / 5.4e-4.  The second terms cost nothing, at head_dim
	// 32 3 % of a call.)
	// A column's two terms have one sign, and neither is zero unless q is (or is smaller than 2^-102): the first is truncated, the second a 2^-24th of it above the rest, so
	// that an infinity in K makes the infinity of the formula of both, never infinity minus infinity or 0 times infinity.
	const uint32_t first = LO || tid % (4 * KS) >= DC || tid % (4 * KS) + DC < 4 * KS ? 0xffff0000u : ~0u;   // (a column without a second term is rounded)
#pragma unroll
	for(int j = 0; j < QN; j++) {
		const int i = tid + j * NW * 64, row = i / (4 * KS), ch = i % (4 * KS);
		u32x4     hi, lo;
#pragma unroll
		for(int e = 0; e < 4; e++) {
			const uint32_t raw = qraw[j][e];
			const float    x = bf16_bits_to_f32(raw & 0xffffu) * p.scale, y = bf16_bits_to_f32(raw >> 16) * p.scale;
			const float    xh = __uint_as_float(__float_as_uint(x) & first), yh = __uint_as_float(__float_as_uint(y) & first);
			hi[e] = pack_bf16x2(xh, yh), lo[e] = pack_bf16x2(__builtin_fmaf(xh, -0x1.fffffep-1f, x), __builtin_fmaf(yh, -0x1.fffffep-1f, y));
		}
		if(i < R * 4 * KS) {
			*reinterpret_cast<u32x4*>(smem + Q_AT + row * Q_ROW + ch * 16) = ch < DC ? hi : lo;
			if constexpr(LO) *reinterpret_cast<u32x4*>(smem + Q_AT + (R + row) * Q_ROW + ch * 16) = lo;
		}
	}

	// ---- key-mask table of this wavefront's tiles: what is added to a key's logits.  Tiles behind the last one with a live key are not walked. ----
	int  my_n = my_all > 0 ? 1 : 0;
	for(int j = 0; 2 * j < my_all; j++) {
		const uint32_t m = (j == 0 ? m_first[0] : j == 1 ? m_first[1] : load_mask(j)) | (masked ? 0u : 1u);
		const int      i = 2 * j + (lane >> 5), seen = ((wave + NW * i) * KT_S + KT_S) - L;   // seen: keys of the last tile that the one before has covered
		if(i < my_all) *reinterpret_cast<float*>(smem + mask_base + i * 128 + (lane & 31) * 4) = (lane & 31) < seen ? MASK_OUT_OF_RANGE : m ? 0.f : DROPPED;
		const unsigned long long bal = __ballot(m != 0u);
		if(bal) my_n = (bal >> 32) && 2 * j + 1 < my_all ? 2 * j + 2 : 2 * j + 1;
	}
	asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
	const unsigned long long low = __ballot(*reinterpret_cast<const uint16_t*>(smem + s_rd) > s_low);   // (bf16 bits; negative NaN as well)
	__syncthreads();   // q
	bf16x8 qf[NB][KS], ql[NB];   // (ql: LO only)
#pragma unroll
	for(int c = 0; c < NB; c++)
#pragma unroll
		for(int s = 0; s < KS; s++) {
			qf[c][s] = *reinterpret_cast<const bf16x8*>(smem + Q_AT + (16 * c + i16) * Q_ROW + s * 64 + g * 16);
			if constexpr(LO) ql[c] = *reinterpret_cast<const bf16x8*>(smem + Q_AT + (R + 16 * c + i16) * Q_ROW + g * 16);
		}

	auto read_k = [&](bf16x8 (&kf)[2][KS], f32x4 (&mk)[2], int i) __attribute__((always_inline)) {   // i: of this wavefront's tiles
#pragma unroll
		for(int hf = 0; hf < 2; hf++) {
			mk[hf] = *reinterpret_cast<const f32x4*>(smem + m_rd + i * 128 + hf * 16);
#pragma unroll
			for(int st = 0; st < KS; st++) kf[hf][st] = *reinterpret_cast<const bf16x8*>(smem + k_rd[st][hf]);
		}
	};
	auto read_v = [&](bf16x8 (&vf)[ND], int seen) __attribute__((always_inline)) {   // seen: keys of the last tile that the one before has covered
#pragma unroll
		for(int d = 0; d < ND; d++) {
			u32x4 w;
#pragma unroll
			for(int u = 0; u < 2; u++) {
				const u32x2 r = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(smem + v_rd[d][u])));
				w[2 * u] = r[0], w[2 * u + 1] = r[1];
			}
			if(seen > 0) {   // (their weights are 0, but 0 times an infinity is not)
#pragma unroll
				for(int j = 0; j < 4; j++) w[j] &= (8 * g + 2 * j < seen ? 0u : 0xffffu) | (8 * g + 2 * j + 1 < seen ? 0u : 0xffff0000u);
			}
			vf[d] = __builtin_bit_cast(bf16x8, w);
		}
	};
	struct bias_piece {
		u32x4    w;
		uint32_t next;
		int      sh;
	};
	auto read_b = [&](int half, int c, int k0) __attribute__((always_inline)) {
		bias_piece r;
		r.w = *reinterpret_cast<const u32x4*>(smem + b_rd + half + c * 1024);
		if constexpr(ANY) r.next = *reinterpret_cast<const uint32_t*>(smem + t_rd + (half ? t_half : 0) + c * t_blk), r.sh = sh0 ^ ((k0 & 1) << 4);
		return r;
	};
	auto mfma = [](const bf16x8& a, const bf16x8& bb, const f32x4& c) __attribute__((always_inline)) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bb, c, 0, 0, 0); };
	auto live_keys = [&]() __attribute__((always_inline)) {   // whether this wavefront's tiles hold any
		bool any = false;
		for(int i = lane; i < my_all * KT_S; i += 64) any = any || *reinterpret_cast<const float*>(smem + mask_base + i * 4) == 0.f;
		return __ballot(any) != 0;
	};
	uint32_t limit = p.bias_limit;
	auto clamped = [&](const bias_piece& raw) __attribute__((always_inline)) {
		u32x4 w;
#pragma unroll
		for(int j = 0; j < 4; j++) {
			const uint32_t lo = raw.w[j];
			w[j] = bias_limited(ANY ? __builtin_amdgcn_alignbit(j < 3 ? raw.w[j < 3 ? j + 1 : 3] : raw.next, lo, raw.sh) : lo, limit);
		}
		return __builtin_bit_cast(bf16x8, w);
	};
	auto wait_loads = [](auto n_c) __attribute__((always_inline)) { asm volatile("s_waitcnt vmcnt(%0)" ::"n"(decltype(n_c)::value) : "memory"); };

	// Padded queries masked through the bias would leave the range and have their strips walked three times.  A wavefront that finds a row's
	// bias below -32 at the head of its first tile looks at two more of each row, one of them the row's own (rows masked but for their
	// neighbourhood show themselves there), and takes the larger for a reference where both are that low.  (Other wavefronts of the strip
	// come to the same answer or, where they had no reason to look, to a count that does not match at the end.)  us per call, one-row kernel /
	// without this / with it: 16 heads of 24 x 768, the last tenth of the rows at -1e9 9.6 / 13.1 / 7.8 (ordinary rows 9.7 / 7.4 / 7.4, rows that
	// see 64 neighbours - / 7.3 / 7.5), x 1536 19.1 / 31.7 / 18.3, 37 x 4 x 37 x 32 5.6 / 8.3 / 5.5.
	f32x4 o[NB][NO];
	float m_ref[NB];   // what the walk with references (REF) takes off this lane's query row of each block
	int   ref = 0;
	if(__builtin_expect(low != 0 && my_n > 0, 0)) {
		int row = strip * R + s_row;
		asm volatile("" : "+v"(row));   // (none of this is prepared at the start)
		const bool     in  = row < L;
		const int      far = in ? row + (L >> 1) : 0, at = in ? row * (int)p.bias_row : 0;
		const uint32_t r0 = *reinterpret_cast<const uint16_t*>(bias + (uint32_t)(at + (in ? row : 0) * 2)), r1 = *reinterpret_cast<const uint16_t*>(bias + (uint32_t)(at + (far < L ? far : far - L) * 2));
		const uint32_t lim = p.bias_limit & 0xffffu;   // (as the walk takes them)
		float          m = fmaxf(bf16_bits_to_f32(r0 < lim ? r0 : lim), bf16_bits_to_f32(r1 < lim ? r1 : lim));
		m   = in && m < -32.f ? m : 0.f;
		ref = __builtin_amdgcn_readfirstlane(__ballot(m < 0.f) != 0);
		int count = 1;
		if(__ballot(m < DROPPED)) {   // (there a dropped key's logit is no lower than the others': all keys count, and sums without a live key may look as if they stood)
			my_n  = my_all;
			count = live_keys() ? 0x10101 : 0x101;
		}
#pragma unroll
		for(int c = 0; c < NB; c++) m_ref[c] = __shfl(m, 16 * c + i16);
		if(ref && lane == 0) atomicAdd(s_bad + 1, count);
	}
	auto walk = [&](auto ref_c) __attribute__((always_inline)) {
		constexpr bool REF = decltype(ref_c)::value;
#pragma unroll
		for(int c = 0; c < NB; c++)
#pragma unroll
			for(int d = 0; d < NO; d++) o[c][d] = f32x4{0.f, 0.f, 0.f, 0.f};
		if(my_n > 0) {
			// k0_0, k0_1, k0_2: first keys of the tile in work and of the two after it.  A tile that does not exist is asked of a buffer of no
			// bytes: nothing is fetched, and the waits keep their counts.
			int k0_0 = k0_first, k0_1 = k0_0 + NW * KT_S, k0_2 = k0_1 + NW * KT_S;
			k0_1 = k0_1 < last_k0 ? k0_1 : last_k0, k0_2 = k0_2 < last_k0 ? k0_2 : last_k0;
			bf16x8 kf[2][KS], vf[ND];
			f32x4  mk[2], s[2];
			u32x4  pprev = {0u, 0u, 0u, 0u};
#pragma unroll
			for(int d = 0; d < ND; d++) vf[d] = __builtin_bit_cast(bf16x8, pprev);
			read_k(kf, mk, 0);
			bias_piece b_next = read_b(0, 0, k0_0);   // the bias of the next slot's logits
			{
				const bf16x8 bb = clamped(b_next);
#pragma unroll
				for(int hf = 0; hf < 2; hf++) {
					s[hf] = mfma(__builtin_bit_cast(bf16x8, sel[hf]), bb, mk[hf]);
#pragma unroll
					for(int st = 0; st < KS; st++) s[hf] = mfma(kf[hf][st], qf[0][st], s[hf]);
					if constexpr(LO) s[hf] = mfma(kf[hf][0], ql[0], s[hf]);
				}
			}
			if constexpr(NB > 1) b_next = read_b(0, 1, k0_0);
			b_rsrc[2] = my_n > 1 ? b_bytes : 0u;
#pragma unroll
			for(int c = 0; c < NB; c++) load_b(k0_1, NB * 1024, c);
			load_t(k0_1, NB * 1024);
			asm volatile("" ::"v"(s[0]), "v"(s[1]));   // (K's operands have been read)
			k_rsrc[2] = my_n > 1 ? k_bytes : 0u;
			load_k(k0_1);
			// One slot = one block of 16 query rows x 32 keys: P.V of the slot before (c_prev), logits of the next one (c_next, bias
			// bn, K operands kn) and this slot's exponentials, a matrix instruction in front of each slice of the vector work.
#define AF3_PIN(x)                         \
	{                                      \
		auto px_ = x;                      \
		asm volatile("" : "+v"(px_));      \
		x = px_;                           \
	}
			auto slot = [&](auto c_c, const bias_piece& b_next, const bf16x8 (&kf)[2][KS], const f32x4 (&mk)[2], const bf16x8 (&vf)[ND]) __attribute__((always_inline)) {
				constexpr int C = decltype(c_c)::value, CN = (C + 1) % NB, CP = (C + NB - 1) % NB;
				const bf16x8  bb = clamped(b_next);
				f32x4 sn[2];
				u32x4 pc;
				auto ex = [&](auto i_c) __attribute__((always_inline)) {   // two probabilities of this slot
					constexpr int I = decltype(i_c)::value;
					pc[I] = pack_bf16x2(__builtin_amdgcn_exp2f(s[I >> 1][(I & 1) * 2] * LOG2E), __builtin_amdgcn_exp2f(s[I >> 1][(I & 1) * 2 + 1] * LOG2E));
				};
				const bf16x8 pp = __builtin_bit_cast(bf16x8, pprev);
				if constexpr(REF) {   // (from the finished logit: where all keys are dropped, all are equal)
#pragma unroll
					for(int e = 0; e < 4; e++) s[0][e] -= m_ref[C], s[1][e] -= m_ref[C];
				}
				__builtin_amdgcn_sched_barrier(0);
				o[CP][0] = mfma(vf[0], pp, o[CP][0]);
				if constexpr(LO) sn[0] = mfma(__builtin_bit_cast(bf16x8, sel[0]), bb, mfma(kf[0][0], ql[CN], mk[0]));
				else sn[0] = mfma(__builtin_bit_cast(bf16x8, sel[0]), bb, mk[0]);
				ex(ic<0>{});
				AF3_PIN(pc[0]); AF3_PIN(sn[0][0]);
				__builtin_amdgcn_sched_barrier(0);
				o[CP][1] = mfma(vf[1], pp, o[CP][1]);
				if constexpr(LO) sn[1] = mfma(__builtin_bit_cast(bf16x8, sel[1]), bb, mfma(kf[1][0], ql[CN], mk[1]));
				else sn[1] = mfma(__builtin_bit_cast(bf16x8, sel[1]), bb, mk[1]);
				ex(ic<1>{});
				AF3_PIN(pc[1]); AF3_PIN(sn[1][0]);
				__builtin_amdgcn_sched_barrier(0);
				if constexpr(KIND == 2) o[CP][2] = mfma(vf[2], pp, o[CP][2]);
				sn[0] = mfma(kf[0][0], qf[CN][0], sn[0]);
				ex(ic<2>{});
				AF3_PIN(pc[2]); AF3_PIN(sn[0][0]);
				__builtin_amdgcn_sched_barrier(0);
				if constexpr(KIND > 0) o[CP][ND] = mfma(__builtin_bit_cast(bf16x8, ones), pp, o[CP][ND]);
				sn[1] = mfma(kf[1][0], qf[CN][0], sn[1]);
				ex(ic<3>{});
				AF3_PIN(pc[3]); AF3_PIN(sn[1][0]);
				__builtin_amdgcn_sched_barrier(0);
				if constexpr(KS == 2) {
					sn[0] = mfma(kf[0][1], qf[CN][1], sn[0]);
					sn[1] = mfma(kf[1][1], qf[CN][1], sn[1]);
				}
				s[0] = sn[0], s[1] = sn[1], pprev = pc;
			};
			// One tile t: K's operands are in kf, V and the biases in LDS, the logits of block 0 in s, block 1's bias in b_next; K of tile
			// t + 1 and its biases are there or on their way.  Each place in LDS is asked to hold the tile after it as soon as it has been read: bias block c
			// (tile t + 2) in slot c, V (t + 1) in slot 1, K and the biases' last dwords (t + 2) at the end.  The waits count the loads younger than what is read next.
			int half = 0;
			int i = 0;
			even_progress progress(my_n, EVEN && my_n > 2 ? EVENLY : BY_AGE);
			auto tile = [&]() __attribute__((always_inline)) {
				if constexpr(EVEN) progress.at(i);
				const int other = NB * 1024 - half;
				constexpr int K_SLOT = NB > 2 ? NB - 2 : NB - 1;
				v_rsrc[2] = i + 1 < my_n ? v_bytes : 0u;
				b_rsrc[2] = i + 2 < my_n ? b_bytes : 0u;
				k_rsrc[2] = i + 2 < my_n ? k_bytes : 0u;
				bf16x8 kf_next[2][KS], vf_now[ND];
				f32x4  mk_next[2];
				auto one = [&](auto c_c) __attribute__((always_inline)) {
					constexpr int C = decltype(c_c)::value;
					if constexpr(C < NB) {
						// (LDS is read a slot before the matrix instructions that need it)
						if constexpr(C == 0) {
							wait_loads(ic<(NB > 2 ? NB - 2 + NT + NV : NB > 1 ? NV : 0)>{});   // V (t) and bias blocks 0 and 1 of t + 1
							read_v(vf_now, (wave + NW * i) * KT_S - k0_0);
						}
						if constexpr(C == K_SLOT && NB > 1) wait_loads(ic<(NB > 2 ? NB - 2 + (NB > 3 ? NV : 0) : 1)>{});   // K (t + 1)
						if constexpr(C == K_SLOT) read_k(kf_next, mk_next, i + 1 < my_n ? i + 1 : 0);
						bias_piece b_after;
						if constexpr(NB == 1) b_next = read_b(other, 0, k0_1);
						else b_after = read_b(C + 2 < NB ? half : other, (C + 2) % NB, C + 2 < NB ? k0_0 : k0_1);
						if constexpr(NB > 1) load_b(k0_2, half, C);
						if constexpr(C == 1) {
							asm volatile("" ::"v"(vf_now[0]), "v"(vf_now[ND - 1]));
							load_v(k0_1);
						}
						if constexpr(C == 0 && NB == 1) slot(c_c, b_next, kf_next, mk_next, vf);
						else if constexpr(C == 0) slot(c_c, b_next, kf, mk, vf);
						else if constexpr(C == NB - 1) slot(c_c, b_next, kf_next, mk_next, vf_now);
						else slot(c_c, b_next, kf, mk, vf_now);
						if constexpr(NB > 1) b_next = b_after;
						if constexpr(C == NB - 1) {
							asm volatile("" ::"v"(kf_next[0][0]), "v"(kf_next[1][0]), "v"(kf_next[0][KS - 1]), "v"(kf_next[1][KS - 1]));   // (have been read)
							if constexpr(NB == 1) {
								asm volatile("" ::"v"(vf_now[0]), "v"(vf_now[ND - 1]));
								load_v(k0_1);
								load_b(k0_2, half, 0);
							}
							load_t(k0_2, half);
							load_k(k0_2);
						}
					}
				};
				one(ic<0>{}), one(ic<1>{}), one(ic<2>{}), one(ic<3>{});
				half = other;
				i++, k0_0 = k0_1, k0_1 = k0_2, k0_2 = k0_2 + NW * KT_S < last_k0 ? k0_2 + NW * KT_S : last_k0;
#pragma unroll
				for(int d = 0; d < ND; d++) vf[d] = vf_now[d];
#pragma unroll
				for(int hf = 0; hf < 2; hf++) {
					mk[hf] = mk_next[hf];
#pragma unroll
					for(int st = 0; st < KS; st++) kf[hf][st] = kf_next[hf][st];
				}
			};
			do tile();
			while(i < my_n);
			const bf16x8 pp = __builtin_bit_cast(bf16x8, pprev);
#pragma unroll
			for(int d = 0; d < ND; d++) o[NB - 1][d] = mfma(vf[d], pp, o[NB - 1][d]);
			if constexpr(KIND > 0) o[NB - 1][ND] = mfma(__builtin_bit_cast(bf16x8, ones), pp, o[NB - 1][ND]);
		}
	};

	// ---- the wavefronts' partial sums, added up by all threads: four head columns of a row per thread and trip; optional output
	// gate (out *= sigmoid(gate)), any row and head strides.  Results leave before it is known whether they stand. ----
	auto merge = [&]() __attribute__((always_inline)) {   // whether they do not
		asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // (no load may still be writing LDS)
		__syncthreads();   // (they lie over the tiles)
		float* const part = reinterpret_cast<float*>(smem) + wave * (R * PC) + i16 * PC + 4 * g;
#pragma unroll
		for(int c = 0; c < NB; c++)
#pragma unroll
			for(int d = 0; d < NO; d++)
				if(d < ND || g == 0) *reinterpret_cast<f32x4*>(part + c * 16 * PC + d * 16) = o[c][d];
		__syncthreads();
		const int    q4    = D >> 2, items = R * q4;
		const float* parts = reinterpret_cast<const float*>(smem);
		bool bad = false;
		for(int it = tid; it < items; it += NW * 64) {
			const int row = (it * p.per_quad) >> 16, d0 = (it - row * q4) * 4, qrow = strip * R + row;
			if(qrow >= L) continue;
			u32x2 gw = {0u, 0u};
			if(p.gate) gw = *reinterpret_cast<const u32x2*>(p.gate + b * p.gate_b + h * p.gate_h + (int64_t)qrow * p.gate_row + d0 * 2);
			f32x4 t = *reinterpret_cast<const f32x4*>(parts + row * PC + d0);
			float l = parts[row * PC + SUM_COL];
#pragma unroll
			for(int w = 1; w < NW; w++) t += *reinterpret_cast<const f32x4*>(parts + w * (R * PC) + row * PC + d0), l += parts[w * (R * PC) + row * PC + SUM_COL];
			bad = bad || !(l > 0x1p-60f && l * 0x1p28f + ((t[0] + t[1]) + (t[2] + t[3])) * 0.f < __builtin_inff());
			const float inv = 1.f / l;
#pragma unroll
			for(int e = 0; e < 4; e++) t[e] *= inv;
			if(p.gate) {
				t[0] *= sigmoidf_fast(bf16_bits_to_f32(gw[0] & 0xffffu)), t[1] *= sigmoidf_fast(bf16_bits_to_f32(gw[0] >> 16));
				t[2] *= sigmoidf_fast(bf16_bits_to_f32(gw[1] & 0xffffu)), t[3] *= sigmoidf_fast(bf16_bits_to_f32(gw[1] >> 16));
			}
			char* const at = p.out + b * p.out_b + h * p.out_h + (int64_t)qrow * p.out_row;
			if(p.out_f32) *reinterpret_cast<f32x4*>(at + d0 * 4) = t;
			else *reinterpret_cast<u32x2*>(at + d0 * 2) = u32x2{pack_bf16x2(t[0], t[1]), pack_bf16x2(t[2], t[3])};
		}
		if(__ballot(bad) && lane == 0) s_bad[0] = 1;
		__syncthreads();
		const int some = __builtin_amdgcn_readfirstlane(s_bad[0]), looked = __builtin_amdgcn_readfirstlane(s_bad[1]);
		return (some | looked) != 0 && (some != 0 || (looked & 0xff) != (n_tiles < NW ? n_tiles : NW) || (looked > 0xff && looked < 0x10000));
	};

	if(ref) walk(std::true_type{});
	else walk(std::false_type{});
	if(!merge()) return;

	// ---- rare: the rows' maxima, then the walk again, over all tiles (a row without a live key needs them).  A batch row without a live
	// key yields the mean over all L keys whatever the dropped logits are: q and the bias (every one is limited to 0) are left out (16 heads of
	// 24 x 768 12.1 us instead of 7.1, x 1536 31.8 instead of 17.1). ----
	my_n = my_all > 0 ? my_all : 0;
	if(live_keys() && lane == 0) atomicAdd(s_bad + 2, 1);
	__syncthreads();
	if(__builtin_amdgcn_readfirstlane(s_bad[2]) == 0) {
		limit = 0;
#pragma unroll
		for(int c = 0; c < NB; c++) {
#pragma unroll
			for(int s = 0; s < KS; s++) qf[c][s] = __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u});
			if constexpr(LO) ql[c] = qf[c][0];
		}
	}
	fill();
	k_rsrc[2] = k_bytes, v_rsrc[2] = v_bytes, b_rsrc[2] = b_bytes;
	float mx[NB];
#pragma unroll
	for(int c = 0; c < NB; c++) mx[c] = -__builtin_inff();
	for(int i = 0; i < my_all; i++) {
		const int at = (wave + NW * i) * KT_S, k0 = at < last_k0 ? at : last_k0;
		load_k(k0);
#pragma unroll
		for(int c = 0; c < NB; c++) load_b(k0, 0, c);
		load_t(k0, 0);
		wait_loads(ic<0>{});
		bf16x8 kf[2][KS];
		f32x4  mk[2];
		read_k(kf, mk, i);
#pragma unroll
		for(int c = 0; c < NB; c++) {
			const bf16x8 bb = clamped(read_b(0, c, k0));
#pragma unroll
			for(int hf = 0; hf < 2; hf++) {
				f32x4 s = mfma(__builtin_bit_cast(bf16x8, sel[hf]), bb, mk[hf]);
#pragma unroll
				for(int st = 0; st < KS; st++) s = mfma(kf[hf][st], qf[c][st], s);
				if constexpr(LO) s = mfma(kf[hf][0], ql[c], s);
				mx[c] = fmaxf(fmaxf(fmaxf(mx[c], s[0]), s[1]), fmaxf(s[2], s[3]));
			}
		}
		asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (read before the next tile's loads write there)
	}
#pragma unroll
	for(int c = 0; c < NB; c++) {
		mx[c] = fmaxf(mx[c], __shfl_xor(mx[c], 16));
		mx[c] = fmaxf(mx[c], __shfl_xor(mx[c], 32));
		if(g == 0) s_max[wave * R + 16 * c + i16] = mx[c];
	}
	__syncthreads();
#pragma unroll
	for(int c = 0; c < NB; c++) {
		float m = s_max[16 * c + i16];
#pragma unroll
		for(int w = 1; w < NW; w++) m = fmaxf(m, s_max[w * R + 16 * c + i16]);
		m_ref[c] = m;
	}
	__syncthreads();
	load_first();
	wait_loads(ic<0>{});
	walk(std::true_type{});
	merge();
}

}  // namespace

// A strip's wavefronts meet only at its end; served by age, those that share a SIMD end one after the other.  With few tiles to a wavefront the code of the even walk costs
// more than it brings (the kernel's time is its instructions), and the forms for those have none of it.  Where one strip of eight wavefronts fills a compute unit, the older
// wavefront of a SIMD takes the tile more where there is one: with one to four of the eight wavefronts so, going by age is what ends them together.  Even / by age, 8 heads of 24,
// tiles: 18 to 20 1.00-1.01, 21 to 24 0.99-1.00, 25 to 28 1.02, 29 to 32 0.99-1.00, 33 to 36 1.03, 37 to 44 0.98-0.99; of 48 the same; 16 heads of 24 (odd rows) 18 to 20 1.01, 21 to
// 24 0.97-0.98, 25 to 28 0.99-1.00, 29 to 32 0.96-0.97; from there on two strips of four wavefronts share a compute unit: more than two tiles to a wavefront are enough, 3 rows x
// 264 x 48 6.98 us by age, 6.82 even, 4 x 264 x 24 6.54 / 6.41, 5 x 271 x 48 8.94 / 8.61, 4 x 320 x 48 8.59 / 8.44, 2 x 8 x 1105 x 24 13.2 / 12.7, one row of 16 x 1105 16.6 / 16.7.  Strips of one
// block have no more than two tiles, and head_dim 25 to 32 comes as triangles of few tokens.
constexpr bool may_go_evenly(int nb, int kind) { return nb > 1 && kind != 1; }
static bool goes_evenly(int64_t L, int nw) {
	const int64_t tiles = (L + KT_S - 1) / KT_S;
	return nw == 4 ? tiles > 8 : tiles > 36 || (tiles > 20 && (tiles - 1) % 8 >= 4);
}

template <int NB, int KIND, bool ANY, int NW>
static int launch_strip_n(const af3_dpa_params& p, hipStream_t s) {
	using lds = strip_lds<NB, KIND, ANY, NW>;
	constexpr int R    = lds::R;
	const int     smem = lds::bytes((int)p.L);
	auto          kern = dpa_strip_bf16_kernel<NB, KIND, ANY, NW, false>;
	if constexpr(may_go_evenly(NB, KIND))
		if(goes_evenly(p.L, NW)) kern = dpa_strip_bf16_kernel<NB, KIND, ANY, NW, true>;
	if(smem > 64 * 1024) {   // beyond the default limit: raise it for this kernel (the call costs the host 0.7 us)
		if(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, smem) != hipSuccess) return AF3_ERR_LAUNCH;
	}
	const int  out_size = p.out_dtype == AF3_F32 ? 4 : 2;
	strip_args a{};
	a.q = static_cast<const char*>(p.q), a.q_b = p.q_stride[0] * 2, a.q_h = p.q_stride[1] * 2, a.q_row = (int)p.q_stride[2] * 2;
	a.k = static_cast<const char*>(p.k), a.k_b = p.k_stride[0] * 2, a.k_h = p.k_stride[1] * 2, a.k_row = (int)p.k_stride[2] * 2;
	a.v = static_cast<const char*>(p.v), a.v_b = p.v_stride[0] * 2, a.v_h = p.v_stride[1] * 2, a.v_row = (int)p.v_stride[2] * 2;
	a.gate = static_cast<const char*>(p.gate), a.gate_b = p.gate_stride[0] * 2, a.gate_h = p.gate_stride[1] * 2, a.gate_row = p.gate ? (int)p.gate_stride[2] * 2 : 0;
	a.bias = static_cast<const char*>(p.bias), a.bias_h = p.bias_stride[0] * 2, a.bias_row = (uint32_t)(p.bias_stride[1] * 2);
	a.mask = p.key_mask, a.mask_b = p.key_mask_stride_b;
	a.out = static_cast<char*>(p.out), a.out_b = p.out_stride[0] * out_size, a.out_h = p.out_stride[1] * out_size, a.out_row = (int)p.out_stride[2] * out_size;
	a.H = (int)p.H, a.L = (int)p.L, a.D = (int)p.D, a.out_f32 = p.out_dtype == AF3_F32, a.scale = p.softmax_scale;
	a.bias_limit = (uint32_t)p.reserved;
	const int dc = (int)p.D / 8;
	a.per_chunk = (65536 + dc - 1) / dc, a.per_quad = (65536 + 2 * dc - 1) / (2 * dc);   // (exact below 192 and 1536)
	hipLaunchKernelGGL(kern, dim3((unsigned)p.H, (unsigned)((p.L + R - 1) / R), (unsigned)p.B), dim3(NW * 64), smem, s, a);
	return launch_status();
}

namespace {
struct strip_form {
	int nb, nw;   // blocks of 16 query rows, wavefronts; nb = 0: none
};
bool bias_rows_anywhere(const af3_dpa_params& p) { return (reinterpret_cast<uintptr_t>(p.bias) & 3) || p.bias_stride[0] % 2 || p.bias_stride[1] % 2 || p.L % 2; }

// The lowest strip whose workgroups are all resident at once (a second round pays the start again): eight wavefronts and one workgroup
// per compute unit, or four and two where three blocks are not enough or the row has so few tiles that eight would idle.  Measured, us per
// call in a graph replay, one batch row of 16 heads (the kernel of dpa_mfma.hip / here):
//   head_dim 24   L  64        128       256       384       512       640       768       896         1024        1280        1536
//                 4.8 / 4.1  5.5 / 4.1  5.7 / 4.7  6.6 / 5.2  6.8 / 5.7  8.9 / 6.4  9.6 / 7.2  10.3 / 9.3  11.2 / 10.4  17.0 / 14.7  19.2 / 17.9
//   head_dim 48      5.4 / 4.3  6.3 / 4.5  7.2 / 5.2  8.0 / 6.0  8.8 / 6.5  10.3 / 7.9  11.2 / 8.8  12.0 / 11.1  13.5 / 12.6  19.0 / 17.9  21.9 / 21.3
// and beyond that, in two rounds, 22.1 / 29.3 and 25.9 / 33.7 at 1792.  Rows at any address (one more load and LDS read per piece):
//   head_dim 24   L  65        257       385       513        769         1025         1153         1281         1491
//                 5.8 / 4.2  7.3 / 5.5  7.4 / 6.0  8.6 / 6.9  10.2 / 8.8  15.9 / 15.3  16.5 / 17.7  18.9 / 20.4  20.5 / 22.1
//   head_dim 48   L  65        257       385       513         769          1023         1155         1291         1491
//                 6.6 / 4.6  7.7 / 6.3  8.6 / 7.0  10.1 / 8.5  11.8 / 10.9  14.6 / 13.9  20.6 / 21.2  22.3 / 23.6  25.0 / 26.2
// (769 to 1023 there: four blocks on 256 registers, 6 of them spilled.)
// Few heads: 4 x 2048 x 24 23.7 / 10.6, 2 x 1500 x 48 29.8 / 8.7, 2 x 7871 x 48 269 / 72, 3 x 8192 x 48 262 / 199.  Batches that read in place:
// 37 x 4 x 37 x 32 5.6 / 5.1, 2 x 16 x 512 x 24 8.5 / 7.1, 5 x 16 x 128 x 48 6.9 / 5.8.
strip_form strip_form_of(const af3_dpa_params& p) {
	const bool any = bias_rows_anywhere(p);
	auto wgs = [&](int nb) { return p.B * p.H * ((p.L + 16 * nb - 1) / (16 * nb)); };
	if(p.L <= 256)
		for(int nb = 1; nb <= 3; nb++)
			if(wgs(nb) <= 256) return {nb, 4};
	for(int nb = 1; nb <= (any ? 4 : 3); nb++)
		if(wgs(nb) <= 256) return {nb, 8};
	// (two workgroups per compute unit read K and V twice: not where their rows lie scattered, as in a packed projection)
	if(p.k_stride[2] > p.D || p.v_stride[2] > p.D || (any && p.L > 1152)) return {0, 0};
	for(int nb = 2; nb <= 3; nb++)
		if(wgs(nb) <= 512) return {nb, 4};
	return {0, 0};
}

template <int KIND, bool ANY>
int launch_strip(const af3_dpa_params& p, const strip_form& f, hipStream_t s) {
	switch(f.nb * 10 + f.nw) {
		case 14: return launch_strip_n<1, KIND, ANY, 4>(p, s);
		case 24: return launch_strip_n<2, KIND, ANY, 4>(p, s);
		case 34: return launch_strip_n<3, KIND, ANY, 4>(p, s);
		case 18: return launch_strip_n<1, KIND, ANY, 8>(p, s);
		case 28: return launch_strip_n<2, KIND, ANY, 8>(p, s);
		case 38: return launch_strip_n<3, KIND, ANY, 8>(p, s);
		default:
			if constexpr(ANY) return launch_strip_n<4, KIND, ANY, 8>(p, s);
			return AF3_ERR_BAD_SHAPE;
	}
}
}  // namespace

// The call as mfma_bf16_eligible has checked it (p.reserved: the limit of its biases, two bf16), its bf16 bias read in place: head_dim that leaves the mask and the reference their
// padding columns, at least one whole tile of keys, offsets of 31 bits, and a form whose workgroups fit in one round.
bool mfma_strip_wanted(const af3_dpa_params& p) {
	if(p.D > 48 || p.L < KT_S || !p.bias || p.bias_dtype != AF3_BF16 || p.B > 65535 || p.H > 65535) return false;
	const int64_t limit = 0x40000000;
	for(int64_t s : {p.q_stride[2], p.k_stride[2], p.v_stride[2], p.gate ? p.gate_stride[2] : 0, p.out_stride[2] * 2})
		if((p.L + 64) * s * 2 >= limit) return false;
	return (p.L + 64) * p.bias_stride[1] * 2 < limit && strip_form_of(p).nb > 0;
}

int launch_dpa_strip(const af3_dpa_params& p, hipStream_t s) {
	const strip_form f = strip_form_of(p);
	const bool       any = bias_rows_anywhere(p);
	auto go = [&](auto kind_c) {
		constexpr int KIND = decltype(kind_c)::value;
		return any ? launch_strip<KIND, true>(p, f, s) : launch_strip<KIND, false>(p, f, s);
	};
	return p.D <= 24 ? go(ic<0>{}) : p.D <= 32 ? go(ic<1>{}) : go(ic<2>{});
}

}  // namespace af3
