// bf16 matrix-core attention kernel for batched calls whose batch rows share one bias (triangle / grid attention):
// out[b] = softmax(q[b].k[b]^T*scale + bias, mask[b]).v[b] with bias [H, L, L] common to all b.
//
// The reference walks (batch, head, query tile) tasks and re-reads the bias tile for every batch row
// (src/csrc/dot_product_attention.cpp:88-110).  Here a wavefront owns one block of 32 query rows of one head for FOUR
// batch rows at once and walks the key axis once for all four: a 32 x 32 bias tile is loaded once, as fp32 already
// laid out like the matrix core's accumulator, and is the C operand of the first K.Q^T instruction of each of the
// four rows -- the bias add costs no instruction at all and a quarter of the loads.  The four rows are four
// independent dependence chains: while the vector ALU exponentiates the logits of one row, the matrix pipe computes
// the logits of the next row and the P.V product of the previous one.
//
// Per 32 x 32 block of logits: 2 MFMA K.Q^T (+ bias through C), 1 MFMA key mask and softmax reference, 2 MFMA
// V^T.P^T, 2 half-size MFMA row sums; 16 v_exp_f32 and 8 v_cvt_pk_bf16_f32 -- the arithmetic of dpa_mfma.hip's log2
// variant (same transposed layout, same optimistic softmax reference, same mask constants) without its two bias
// MFMAs.
//
// Work split.  Workgroup = NW wavefronts = NW blocks of 32 query rows of one (group of 4 batch rows, head).  K and V
// tiles (32 keys x 4 batch rows) are staged in LDS by loads that write LDS directly, three buffers deep, and shared
// by the NW wavefronts; one workgroup barrier per tile, i.e. per four blocks of logits of every wavefront.  A workgroup may
// walk several query tiles of its group and head one behind the other without coming to rest (plan_chunks).
#include "mfma_helpers.hpp"

namespace af3 {

namespace {

constexpr int KT_R   = 32;                 // keys per tile
constexpr int NBUF_R = 3;                  // tile buffers
constexpr int TILE_R = KT_R * 32 * 2;      // bytes of one tensor's tile of one batch row (head_dim padded to 32)
constexpr int MAX_L_ROWS = 4096;           // mask table: 8 bytes per key for the four rows
constexpr float BIAS_FLOOR = -0x1p17f;     // lowest value the rewritten bias holds (log2 units)

// ---- bias prepass ---------------------------------------------------------------------------------------------------
// Workspace layout: [H][query block of 32][key tile of 32][load 4][lane 64] x 16 bytes = the accumulator layout of
// v_mfma_f32_32x32x16: lane (q = lane%32, g = lane/32), register 4*ld + e  <->  key 32*t + 8*ld + 4*g + e.
// Values are fp32 bias * log2 e; zero outside the L x L corner; -inf, NaN and anything below -2^17 become -2^17: such an
// entry still gets weight exactly 0 beside any ordinary logit, a row made of nothing else still comes out uniform, and a
// softmax reference that starts there (a row whose first keys are all masked through the bias) leaves the logits that
// follow their fp32 precision to within 2^-6.
template <bool BIAS_F32>
__global__ void __launch_bounds__(256) bias_rows_prepass_kernel(const void* __restrict__ bias, f32x4* __restrict__ ws, int64_t H, int64_t L, int64_t stride_h, int64_t stride_q,
																  int n_qblocks, int n_tiles) {
	// one workgroup per (head, query block, key tile) and trip: the index arithmetic (divisions) is per workgroup, on the
	// scalar unit, not per thread; the launcher keeps the number of units below 2^31
	const uint32_t units = (uint32_t)(H * n_qblocks * (int64_t)n_tiles);
	const int      lane = threadIdx.x & 63, ld = threadIdx.x >> 6;
	for(uint32_t u = blockIdx.x; u < units; u += gridDim.x) {
		const int64_t  i  = (int64_t)u * 256 + threadIdx.x;
		const int      t  = (int)(u % (uint32_t)n_tiles);
		const uint32_t t2 = u / (uint32_t)n_tiles;
		const int      qb = (int)(t2 % (uint32_t)n_qblocks);
		const int64_t  h  = t2 / (uint32_t)n_qblocks;
		const int64_t row  = (int64_t)qb * 32 + (lane & 31);
		const int64_t key  = (int64_t)t * KT_R + 8 * ld + 4 * (lane >> 5);
		float         f[4] = {0.f, 0.f, 0.f, 0.f};
		if(row < L) {
			const int64_t off = h * stride_h + row * stride_q + key;
			if(BIAS_F32) {
				const float* bp = static_cast<const float*>(bias) + off;
				if(key + 4 <= L) {
					const f32x4 raw = *reinterpret_cast<const f32x4_any*>(bp);
					f[0] = raw[0], f[1] = raw[1], f[2] = raw[2], f[3] = raw[3];
				} else {
#pragma unroll
					for(int e = 0; e < 4; e++)
						if(key + e < L) f[e] = bp[e];
				}
			} else {
				const uint16_t* bp = static_cast<const uint16_t*>(bias) + off;
				if(key + 4 <= L) {
					const u32x2 raw = *reinterpret_cast<const u32x2_any*>(bp);
					f[0] = bf16_bits_to_f32(raw[0] & 0xffffu), f[1] = bf16_bits_to_f32(raw[0] >> 16);
					f[2] = bf16_bits_to_f32(raw[1] & 0xffffu), f[3] = bf16_bits_to_f32(raw[1] >> 16);
				} else {
#pragma unroll
					for(int e = 0; e < 4; e++)
						if(key + e < L) f[e] = bf16_bits_to_f32(bp[e]);
				}
			}
		}
		f32x4 o;
#pragma unroll
		for(int e = 0; e < 4; e++) o[e] = fmaxf(f[e] * LOG2E, BIAS_FLOOR);  // (fmaxf returns the other operand for NaN)
		ws[i] = o;
	}
}

// ROWS: batch rows per wavefront (2, 3 or 4); a workgroup is always four wavefronts = 128 query rows, and wavefront w < ROWS
// fetches the K and V tiles of batch row w.
// BMODE: 0 = no bias (C operand zero); 1 = bias from the rewritten fp32 workspace, one 4 KB fragment per tile through this
// wavefront's LDS slot; 2 = bf16 bias read in place (no workspace: for batches too small to pay for the rewrite), four
// 8-byte loads per lane and tile, converted to the accumulator layout in registers; 3 = bf16 bias read in place through LDS: the
// 32 x 32 tile of this wavefront's query block travels as two 1 KB loads of whole 64-byte row segments straight into one of
// two 2 KB halves of the wavefront's slot, a tile ahead of its conversion (needs 16-byte aligned rows; a quarter of mode
// 2's cache-line requests, whose lanes each fetch from a row of their own).
// The launch covers batch rows [b_first, b_first + b_count) in groups of ROWS.
// GATE: out *= sigmoid(gate) in the epilogue.
// MULTI: workgroups may walk several query tiles; per XCD the first n_chunked (group, head) pairs are cut into n_chunks workgroups of q_chunk query tiles, the
// others into workgroups of one.  Launches of single query tiles take the form without: with the code of the longer walk in it (10 KB more, scalar and,
// with four rows, 7 vector registers spilled) they took, us, that code in / out: 512 x 4 x 128 x 32 25.2 / 23.9, 1024 38.4 / 37.0, 1536 50.2 / 47.4, 1000 x 4 x 64 x 32
// 26.4 / 24.9, 512 x 8 x 256 x 32 on packed rows 110.1 / 94.5.  With four rows and a bias staged in place the longer walk spills 7 vector registers, stored once per
// workgroup and read back in the careful walk alone; every form of it holds 12 to 113 scalar registers in vector lanes.
// Whether there is such a form.  Four batch rows and their gates do not fit the registers between two query tiles (14 spilled ones: the
// grid block of 768 tokens 637 -> 655 us; with one query tile to a workgroup 633), the in-place form has not been given it.
constexpr bool several_query_tiles(int rows, int bmode, bool gate) { return bmode != 2 && !(gate && rows == 4); }
template <int ROWS, int BMODE, bool GATE, bool MULTI>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) dpa_rows_bf16_kernel(af3_dpa_params p, int n_qtiles, int64_t n_groups, int64_t b_first, int64_t b_count, int q_chunk,
																										   int n_chunks, int n_chunked, int even) {
	static_assert(ROWS >= 2 && ROWS <= 4, "two to four row chains per wavefront");
	static_assert(!MULTI || several_query_tiles(ROWS, BMODE, GATE), "no such form");
	constexpr int  NW       = 4;
	constexpr bool HAS_BIAS = BMODE != 0, SLOT = BMODE == 1, DIRECT = BMODE == 2, STAGED = BMODE == 3;
	constexpr int  BUF_R    = ROWS * 2 * TILE_R;                    // one buffer: [row][K tile | V tile]
	constexpr int  SLOT_BASE = NBUF_R * BUF_R;                      // per-wavefront bias slots (4 KB each)
	constexpr int  MASK_BASE = SLOT_BASE + (SLOT || STAGED ? NW * 4096 : 0);
	extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
	// [buffer 3][batch row 4][K tile 2 KB | V tile 2 KB] [bias slot 4 KB per wavefront] [mask table: (tiles + 1) x 4 rows x 32 keys, bf16 bits]
	const int64_t L        = p.L;
	const int     D        = (int)p.D;
	const int     n_t_all  = (int)((L + KT_R - 1) / KT_R);
	uint16_t* const mask_tab = reinterpret_cast<uint16_t*>(smem + MASK_BASE);
	__shared__ int  s_last[4];  // index of the last live key + 1 of each batch row (0: every key dropped)
	__shared__ uint32_t s_again;  // query tiles of which some wavefront's walk has to be repeated carefully
	__shared__ int  s_first[4]; // index of the first key tile of each batch row that holds a live key

	// ---- workgroup -> (group of batch rows, head, query tile): all query tiles of one (group, head) get ids congruent
	// mod 8, i.e. the same XCD (they share that XCD's L2 copy of K and V), and an XCD only sees heads xcd % H (for H | 8),
	// so its share of the bias workspace stays L2-resident across the whole batch.
	// The kernel arguments that the start of a workgroup needs, requested in one batch (the compiler would fetch the launch
	// counts, wait, test the early exit, and only then request the fields of p, in two more batches: three memory latencies
	// in a row that the wavefronts of a small launch stand through).
	asm volatile("" ::"s"(n_qtiles), "s"(n_groups), "s"(b_first), "s"(b_count), "s"(q_chunk), "s"(n_chunks), "s"(n_chunked), "s"(p.q), "s"(p.k), "s"(p.v), "s"(p.bias), "s"(p.key_mask), "s"(p.workspace), "s"(p.H), "s"(p.L),
				 "s"(p.D), "s"(p.key_mask_stride_b), "s"(p.bias_stride[0]), "s"(p.bias_stride[1]));
	asm volatile("" ::"s"(p.q_stride[0]), "s"(p.q_stride[1]), "s"(p.q_stride[2]), "s"(p.k_stride[0]), "s"(p.k_stride[1]), "s"(p.k_stride[2]), "s"(p.v_stride[0]), "s"(p.v_stride[1]),
				 "s"(p.v_stride[2]));
	// (32-bit divisions: a 64-bit one is 150 instructions, i.e. 700 clocks of a start that waits for them)
	const uint32_t slot = blockIdx.x >> 3, chunked = MULTI ? (uint32_t)n_chunked * (uint32_t)n_chunks : 0u;
	const bool     single = !MULTI || slot >= chunked;
	const uint32_t s_rel = single ? slot - chunked : slot, parts = single ? (uint32_t)n_qtiles : (uint32_t)n_chunks, q_div = s_rel / parts;
	const uint32_t group = (q_div + (MULTI && single ? (uint32_t)n_chunked : 0u)) * 8 + (blockIdx.x & 7);
	if(group >= (uint32_t)n_groups) return;
	const int chunk = single ? 1 : q_chunk, qtile0 = (int)(s_rel - q_div * parts) * chunk;
	const int n_q   = !MULTI ? 1 : qtile0 + chunk <= n_qtiles ? chunk : n_qtiles - qtile0;   // query tiles of this workgroup
	const int64_t g = group / (uint32_t)p.H, h = group - (uint32_t)g * (uint32_t)p.H;
	const int64_t b0 = b_first + g * ROWS, b_end = b_first + b_count;   // (rows past b_end repeat the last one and are not stored)

	const int tid = threadIdx.x, lane = tid & 63;
	const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
	const int n = lane & 31, half = lane >> 5;

	// The start of a workgroup is bound by the number of its instructions (a wavefront issues one in about 4.5 clocks) and by one memory
	// latency; of the 25 k clocks around the walk of 12 tiles at L = 384 it was half.  Hence 32-bit divisions, a mask table written four keys
	// at a time without a length-specific unroll, its last and first live key from ballots, and everything that needs no other
	// wavefront's data in front of the barrier.  H = 4, D = 32: L = 384, B = 384 62.8 -> 61.5 us, L = 768 392 -> 386, L = 1491 (mask rows at
	// odd addresses, once read byte by byte) 2713 -> 2590.
	// ---- key-mask bytes of batch row `wave`, requested before anything else: four keys per lane and load at any address (the last four of
	// a row that L ends in the middle of are shifted), up to 2048 keys in flight ----
	const bool           mask_vec = L >= 4;
	const int64_t        mask_row = b0 + (wave < ROWS ? wave : 0) < b_end ? b0 + (wave < ROWS ? wave : 0) : b_end - 1;
	const uint8_t* const keep     = p.key_mask ? p.key_mask + mask_row * p.key_mask_stride_b : nullptr;
	constexpr int MASK_CHUNKS = 8;
	uint32_t      mraw[MASK_CHUNKS];
	auto load_mask = [&](int c) -> uint32_t {   // chunk c: keys 256 c + 4 lane .. + 3, as they lie in memory
		const int key0 = 256 * c + 4 * lane;
		return *reinterpret_cast<const u32_bytes*>(keep + (key0 + 4 <= (int)L ? key0 : (int)L - 4));
	};
	auto mask_of = [&](int c, uint32_t w) -> uint32_t { return keep_bytes_in_row(w, 256 * c + 4 * lane + 4 - (int)L); };
	auto request_mask = [&](int c0) {
#pragma unroll
		for(int c = 0; c < MASK_CHUNKS; c++) {
			mraw[c] = 0x01010101u;
			if(keep && 256 * (c0 + c) < (int)L) mraw[c] = load_mask(c0 + c);
		}
	};
	if(mask_vec && wave < ROWS) request_mask(0);

	// ---- zero the tile buffers when a load can leave parts of them unwritten (padded head columns, rows past L):
	// stale LDS contents there must be finite ----
	if(D != 32 || L % KT_R != 0) {
		for(int i = tid; i < NBUF_R * BUF_R / 16; i += NW * 64) reinterpret_cast<u32x4*>(smem)[i] = u32x4{0u, 0u, 0u, 0u};
		__syncthreads();
	}

	if(STAGED && L % KT_R != 0) {  // (chunks past L are never fetched: what the slots hold there must be finite)
		for(int i = tid; i < NW * 4096 / 16; i += NW * 64) reinterpret_cast<u32x4*>(smem + SLOT_BASE)[i] = u32x4{0u, 0u, 0u, 0u};
		__syncthreads();
	}

	// ---- per-lane constants ----
	const int64_t row00 = (int64_t)qtile0 * (NW * 32) + wave * 32;   // this wavefront's first query row
	const int     my_q  = row00 + (int64_t)(n_q - 1) * (NW * 32) < L ? n_q : n_q - 1;   // query tiles in which it has rows: all, or all but the last
	int n_t = 1;   // key tiles to walk: known once the key masks are read; the first tile is always walked

	// ---- tile and bias loaders: loads that write LDS directly (no registers, invisible to the compiler's wait counting;
	// every wait for them below is explicit).  This wavefront fetches K and V of batch row `wave`: four 1 KB pieces per
	// tile (K rows 0-15, 16-31, V rows 0-15, 16-31; lane i -> tile row i/4, 16-byte chunk i%4, K chunks swizzled), and
	// the four 1 KB pieces of its own bias fragment.  Lanes of padded head columns carry an offset beyond the buffer's
	// range: the hardware fetches nothing for them. ----
	const int64_t b_ld   = b0 + wave < b_end ? b0 + wave : b_end - 1;
	const bool    loader = wave < ROWS;  // (wave-uniform)
	const u32x4   k_rsrc = raw_rsrc(static_cast<const uint16_t*>(p.k) + b_ld * p.k_stride[0] + h * p.k_stride[1], (uint32_t)(((L - 1) * p.k_stride[2] + D) * 2));
	const u32x4   v_rsrc = raw_rsrc(static_cast<const uint16_t*>(p.v) + b_ld * p.v_stride[0] + h * p.v_stride[1], (uint32_t)(((L - 1) * p.v_stride[2] + D) * 2));
	const int     ld_row = lane >> 2, ld_pc = lane & 3;
	const int     k_chunk = ld_pc ^ k_swizzle<32>(ld_row);
	const int     k_voff  = k_chunk * 8 < D ? (int)(ld_row * p.k_stride[2] * 2) + k_chunk * 16 : 0x40000000;
	const int     v_voff  = ld_pc * 8 < D ? (int)(ld_row * p.v_stride[2] * 2) + ld_pc * 16 : 0x40000000;
	const int     k_tile_stride = (int)(KT_R * p.k_stride[2] * 2), v_tile_stride = (int)(KT_R * p.v_stride[2] * 2);
	const int     k_pc_stride = (int)(16 * p.k_stride[2] * 2), v_pc_stride = (int)(16 * p.v_stride[2] * 2);
	const uint32_t lds_tiles = lds_addr_of(smem) + wave * (2 * TILE_R);
	auto load_tile = [&](int t, int buf_off) {   // (for tiles that will be walked only: nothing is in flight when the kernel ends)
		if(!loader) return;
		lds_dma_b128(k_rsrc, lds_tiles + buf_off, k_voff + t * k_tile_stride);
		lds_dma_b128(k_rsrc, lds_tiles + buf_off + 1024, k_voff + (t * k_tile_stride + k_pc_stride));
		lds_dma_b128(v_rsrc, lds_tiles + buf_off + TILE_R, v_voff + t * v_tile_stride);
		lds_dma_b128(v_rsrc, lds_tiles + buf_off + TILE_R + 1024, v_voff + (t * v_tile_stride + v_pc_stride));
	};
	// (The arguments of what happens once or twice per query tile are loaded again where they are used: kept through the walk, they are spilled.)
	using args_t = const __attribute__((address_space(4))) af3_dpa_params*;
	auto args = []() __attribute__((always_inline)) -> args_t {
		args_t a = (args_t)__builtin_amdgcn_kernarg_segment_ptr();
		asm volatile("" : "+s"(a));
		return a;
	};
	// Output gate: the 2 ROWS pieces of this wavefront's gate rows (16 query rows of a batch row, 1 KB each) go into the tile buffers
	// that the last two tiles leave free -- the places of tiles n_t and n_t + 1, requested where those tiles would be -- and are
	// read in the epilogue.  (Loaded there, they exposed a memory latency per workgroup: 36 of 448 us at 768 x 4 x 768 x 32, 9 of 81 at 384.)
	auto load_gate = [&](int part, int buf_off, int i) {
		if constexpr(!GATE) return;
		const args_t a = args();
#pragma unroll
		for(int j = 0; j < ROWS; j++) {
			const int     k = part * ROWS + j, r = k >> 1;
			const int64_t br = b0 + r < b_end ? b0 + r : b_end - 1, row = row00 + i * (NW * 32) + 16 * (k & 1) + (lane >> 2);
			const u32x4   g_rsrc = raw_rsrc(static_cast<const uint16_t*>(a->gate) + br * a->gate_stride[0] + h * a->gate_stride[1], (uint32_t)(((L - 1) * a->gate_stride[2] + D) * 2));
			lds_dma_b128(g_rsrc, lds_addr_of(smem) + buf_off + (wave * ROWS + j) * 1024, (lane & 3) * 8 < D && row < L ? (int)(row * a->gate_stride[2] * 2) + (lane & 3) * 16 : 0x7FFF0000);
		}
	};
	auto load_tile_or_gate = [&](int t, int buf_off, int i) {
		if(t < n_t) load_tile(t, buf_off);
		else load_gate(t - n_t, buf_off, i);
	};
	// bias fragment of key tile t: 4 KB of this (head, query block)'s slab of the workspace -> this wavefront's slot
	// (i: query tile of the workgroup, here and below; its blocks are NW slabs further on)
	const int     n_qblocks = (int)((L + 31) / 32);
	const int64_t qb        = (int64_t)qtile0 * NW + wave;
	const int64_t qbc       = qb < n_qblocks ? qb : n_qblocks - 1;  // (blocks past the end only hold rows >= L)
	const u32x4   ws_rsrc   = raw_rsrc(SLOT ? static_cast<const unsigned char*>(p.workspace) + ((h * n_qblocks + qbc) * n_t_all) * 4096 : nullptr,
									   SLOT ? (uint32_t)((n_qblocks - qbc) * n_t_all) * 4096u : 0u);
	const int      ws_voff  = lane * 16, ws_step = NW * n_t_all * 4096;
	const uint32_t lds_slot = lds_addr_of(smem) + SLOT_BASE + wave * 4096;
	auto load_bias = [&](int t, int i) {
		if(!SLOT) return;
		const int off = i * ws_step + t * 4096;
#pragma unroll
		for(int pc = 0; pc < 4; pc++) lds_dma_b128(ws_rsrc, lds_slot + pc * 1024, ws_voff + (off + pc * 1024));
	};
	// direct mode: this lane's four 8-byte pieces of a tile's bias, bias[h][q][32 t + 8 ld + 4 half .. + 3] (bf16), through a
	// range-checked buffer over the head's slab; pieces whose keys lie at or beyond L are sent out of range and read as zero
	// (workgroups of this mode take one query tile)
	[[maybe_unused]] u32x2 braw[4] = {u32x2{0u, 0u}, u32x2{0u, 0u}, u32x2{0u, 0u}, u32x2{0u, 0u}};
	const int64_t qrow_b = row00 + n < L ? row00 + n : L - 1;
	const __amdgpu_buffer_rsrc_t bd_rsrc = __builtin_amdgcn_make_buffer_rsrc(
		DIRECT ? const_cast<uint16_t*>(static_cast<const uint16_t*>(p.bias)) + h * p.bias_stride[0] : nullptr, 0, DIRECT ? (int)(((L - 1) * p.bias_stride[1] + L) * 2) : 0, 0x00020000);
	const int bd_voff = (int)((qrow_b * p.bias_stride[1] + 4 * half) * 2);
	// staged mode: lane i of load j fetches 16 bytes of row 16 j + i / 4 of the tile; the chunk it fetches is the one that
	// belongs at its place under the swizzle (chunk c of row r sits at position c ^ ((r >> 2) & 3): the fragment reads of 32
	// rows then spread over the banks).  Rows past L and chunks whose keys lie at or beyond L are out of the buffer's range or
	// hold other biases (their results are not stored, those keys carry the out-of-range mask value).
	const u32x4 st_rsrc = raw_rsrc(STAGED ? static_cast<const uint16_t*>(p.bias) + h * p.bias_stride[0] : nullptr, STAGED ? (uint32_t)(((L - 1) * p.bias_stride[1] + L) * 2) : 0u);
	int st_voff[2] = {0, 0};
	int st_key[2]  = {0, 0};  // first key (within a tile) of the chunk this lane fetches
	const int st_step = STAGED ? (int)(NW * 32 * p.bias_stride[1] * 2) : 0;
	if constexpr(STAGED) {
#pragma unroll
		for(int j = 0; j < 2; j++) {
			const int     r   = 16 * j + (lane >> 2), c = (lane & 3) ^ ((r >> 2) & 3);
			const int64_t row = row00 + r;
			st_voff[j] = n_q > 1 || row < L ? (int)(row * p.bias_stride[1] * 2) + c * 16 : (int)((L - 1) * p.bias_stride[1] * 2) + c * 16;
			st_key[j]  = c * 8;
		}
	}
	auto load_bias_staged = [&](int t, int i, int parity) {
		if(!STAGED) return;
#pragma unroll
		for(int j = 0; j < 2; j++) lds_dma_b128(st_rsrc, lds_slot + (parity & 1) * 2048 + j * 1024, t * KT_R + st_key[j] < L ? st_voff[j] + (i * st_step + t * (KT_R * 2)) : 0x40000000);
	};
	auto load_bias_direct = [&](int t) {
		if(!DIRECT) return;
#pragma unroll
		for(int ld = 0; ld < 4; ld++) {
			const bool in = t * KT_R + 8 * ld + 4 * half < L;
			braw[ld] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(bd_rsrc, in ? bd_voff + ld * 16 : 0x40000000, t * (KT_R * 2), 0));
		}
	};
	// q rows, gate rows and output rows of this wavefront's 32 rows of query tile i: per batch row a buffer that starts at the first of them and
	// ends with row L - 1 (rows past it read zero and are not stored).  The addresses move along in scalar registers; lane offsets are
	// made anew where they are used, from a lane number that the compiler cannot keep (it would hold a dozen registers through the walk).
	auto lane_now = []() -> int {
		int l;
		asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
		return l;
	};
	const int      n_rows = (int)(b_end - b0 < ROWS ? b_end - b0 : ROWS);   // batch rows of this group
	auto rows_left = [&](int i) -> int {   // (at most 32)
		const int64_t left = L - row00 - i * (NW * 32);
		return left < 0 ? 0 : left < 32 ? (int)left : 32;
	};
	auto buffer_of = [&](const void* base, int64_t row_stride, int rows, int el) -> __amdgpu_buffer_rsrc_t {   // (31 row strides fit 31 bits: mfma_rows_eligible)
		return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, rows > 0 ? ((rows - 1) * (int)row_stride + D) * el : 0, 0x00020000);
	};
	u32x4 qraw[ROWS][2];
	const uint16_t* q_row = nullptr;
	int64_t         q_sb = 0;
	int             q_sr = 0;   // (strides of batch rows and of query rows)
	auto request_q = [&](auto r_c, int i) {   // (batch rows in their order)
		constexpr int r  = decltype(r_c)::value;
		if constexpr(r < ROWS) {
			if constexpr(r == 0) {
				const args_t a = args();
				q_sb = a->q_stride[0], q_sr = (int)a->q_stride[2];
				q_row = static_cast<const uint16_t*>(a->q) + b0 * q_sb + h * a->q_stride[1] + (row00 + i * (NW * 32)) * q_sr;
			} else q_row += r < n_rows ? q_sb : 0;   // (rows past the last repeat it)
			const __amdgpu_buffer_rsrc_t rsrc = buffer_of(q_row, q_sr, rows_left(i), 2);
			const int l = lane_now(), d0 = 8 * (l >> 5), voff = ((l & 31) * q_sr + d0) * 2;
#pragma unroll
			for(int c = 0; c < 2; c++) qraw[r][c] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, 16 * c + d0 < D ? voff + 32 * c : 0x7FFF0000, 0, 0));
		}
	};

	// ---- everything the walk needs before its first step is requested here in one go, so that the workgroup pays one
	// memory latency, not a chain of them: the first K and V tiles, the first bias fragment (straight into LDS)
	// and the raw q rows ----
	load_tile(0, 0);
	load_bias(0, 0);
	load_bias_direct(0);
	load_bias_staged(0, 0, 0);
	request_q(ic<0>{}, 0), request_q(ic<1>{}, 0), request_q(ic<2>{}, 0), request_q(ic<3>{}, 0);

	// ---- key-mask table: entry = additive mask value of (tile, batch row, key) as bf16 bits; wavefront w fills row w ----
	const int n_keys_tab = (n_t_all + 1) * KT_R;
	if(wave < ROWS) {
		const int r    = wave;
		int       last = 0, first = -1;   // (wave-uniform)
		if(mask_vec) {
			auto write_chunk = [&](int c, uint32_t m) {
				const int key0 = 256 * c + 4 * lane;
				if(key0 >= n_keys_tab) return;
				*reinterpret_cast<u32x2*>(mask_tab + ((key0 >> 5) * ROWS + r) * 32 + (key0 & 31)) = mask_values_bf16(gone_bytes(m), key0 + 4 - (int)L);
			};
			for(int c0 = 0; 256 * c0 < n_keys_tab; c0 += MASK_CHUNKS) {
				if(c0 > 0) request_mask(c0);
#pragma unroll
				for(int c = 0; c < MASK_CHUNKS; c++) {
					if(256 * (c0 + c) >= n_keys_tab) break;
					const uint32_t           mc  = mask_of(c0 + c, mraw[c]);
					const unsigned long long bal = __ballot(mc != 0u);   // a lane's four keys of chunk c lie in tile 8 c + lane / 8
					if(bal) {
						const int      top = 63 - __builtin_clzll(bal);
						const uint32_t m   = __builtin_amdgcn_readlane(mc, top);
						last               = 256 * (c0 + c) + 4 * top + ((31 - __builtin_clz(m)) >> 3) + 1;
						if(first < 0) first = 8 * (c0 + c) + (__builtin_ctzll(bal) >> 3);
					}
					write_chunk(c0 + c, mc);
				}
			}
			// A batch row without any live key yields the mean over all L keys (masked_fill(-1e9) + softmax in
			// examples/dot_product_attention.py:37-39): its keys count as live, and q and the bias are dropped for it
			// below, so that all its logits are exactly equal.
			if(last == 0)
				for(int c = 0; 256 * c < n_keys_tab; c++) write_chunk(c, 0x01010101u);
		} else {
			for(int base = 0; base < n_keys_tab; base += 64) {
				const int  key  = base + lane;
				const bool in   = key < L;
				const bool live = in && (!keep || keep[in ? key : 0] != 0);
				if(key < n_keys_tab) mask_tab[((key >> 5) * ROWS + r) * 32 + (key & 31)] = live ? (uint16_t)0 : (in ? MASK_DROPPED_BF16 : MASK_OUT_OF_RANGE_BF16);
				const unsigned long long bal = __ballot(live);
				if(bal) last = base + 64 - __builtin_clzll(bal);
				if(bal && first < 0) first = (base + __builtin_ctzll(bal)) / KT_R;
			}
			if(last == 0)   // (as above)
				for(int key = lane; key < n_keys_tab; key += 64) mask_tab[((key >> 5) * ROWS + r) * 32 + (key & 31)] = key < L ? (uint16_t)0 : MASK_OUT_OF_RANGE_BF16;
		}
		if(lane == 0) s_last[r] = last, s_first[r] = first;
	}
	if(tid == 0) s_again = 0;
	// Operands of the mask MFMA (v_mfma_f32_32x32x8_bf16: four contraction slots per half-wave, two registers per operand).
	// A (per key): slot 0 = the key's mask value (from the table, zero-extended), slots 2 and 3 = 1.0.
	// B (per query): slot 0 = 1.0, slots 2 and 3 = -m_hi and -m_lo, the softmax reference of this lane's query row as two
	// bf16 terms (16 significant bits).  Lanes of the upper half-wave supply slots 4..7: their B is zero, so whatever
	// finite value their A holds contributes nothing.
	u32x2 maskA = {0u, 0x3F803F80u};
	u32x2 maskB[ROWS];

	// ---- per-lane LDS read offsets inside a (buffer, batch row) block ----
	int k_rd[2];
#pragma unroll
	for(int c = 0; c < 2; c++) k_rd[c] = n * 64 + (((2 * c + half) ^ k_swizzle<32>(n)) << 4);
	// V^T fragment reads (ds_read_b64_tr_b16): lane l: i = l%16, G = l/16 supplies the 8-byte chunk at tile row
	// base + 4*(G/2) + i/4, column 16*(G%2) + 4*(i%4); it receives 4 keys of column l%32.
	int v_rd;
	{
		const int i16 = lane & 15, G = lane >> 4;
		const int row = 4 * (G >> 1) + (i16 >> 2), col = 16 * (G & 1) + 4 * (i16 & 3);
		v_rd = TILE_R + row * 64 + (col >> 3) * 16 + (col & 7) * 2;
	}
	const int mask_rd = MASK_BASE + n * 2;               // + ((tile * ROWS + row) * 32) * 2
	const int slot_rd = SLOT_BASE + wave * 4096 + lane * 16;  // + 1024 per group of four accumulator registers

	// Row sums on the matrix pipe (see dpa_mfma.hip): a 16x16x32 MFMA whose A operand is this 0/1 pattern leaves, in
	// register 0 of every lane, the sum of the 16 packed probabilities of that lane's own query row over both half-waves.
	u32x4 ones_a;
	{
		const int      i16 = lane & 15, kg = lane >> 4;
		const bool     on  = ((i16 == 0 || i16 == 8) && (kg & 1) == 0) || ((i16 == 4 || i16 == 12) && (kg & 1) == 1);
		const uint32_t w   = on ? 0x3F803F80u : 0u;
		ones_a = u32x4{w, w, w, w};
	}

	// Q fragments (B operand of S^T = K.Q^T): lane (q = n, g = half) holds q[q][16c + 8g .. +7], scaled by
	// softmax_scale * log2 e in fp32 and rounded once to bf16 (the reference rounds the scaled q too,
	// src/csrc/dot_product_attention.cpp:95-98).
	bf16x8 qf[ROWS][2];
	auto convert_q = [&](auto r_c) {
		constexpr int r = decltype(r_c)::value;
		if constexpr(r < ROWS) {
			const float qmul = args()->softmax_scale * LOG2E;
#pragma unroll
			for(int c = 0; c < 2; c++) {
				u32x4 sc4;
#pragma unroll
				for(int j = 0; j < 4; j++) {
					const uint32_t w = qraw[r][c][j];
					sc4[j] = pack_bf16x2(bf16_bits_to_f32(w & 0xffffu) * qmul, bf16_bits_to_f32(w >> 16) * qmul);
				}
				asm volatile("" : "+v"(sc4));   // (here, not where it is used: the wait for the loads would then take in younger tile loads)
				qf[r][c] = __builtin_bit_cast(bf16x8, sc4);
			}
		}
	};
	convert_q(ic<0>{}), convert_q(ic<1>{}), convert_q(ic<2>{}), convert_q(ic<3>{});
	asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wavefront's pieces of the first tile and its bias fragment have landed
	__syncthreads();                                    // the mask table and the first tile are complete
	// keys behind the last live key of every row carry weight 0 and are not walked; a row without live keys needs them all
	// The softmax reference of a batch row is fixed by the first tile that holds a live key of that row (a tile of dropped
	// keys says nothing about the row's logits): tiles up to the last such tile over the group's rows (normally tile 0 alone)
	// run the variant of the tile code that can do so.
	int  l_eff = 0, t_force_max = 0;
	bool dropped[ROWS];
	uint32_t first_tiles = 0;   // byte r: the first tile of batch row r that holds a live key (at most 128 tiles)
#pragma unroll
	for(int r = 0; r < ROWS; r++) {
		const int last = __builtin_amdgcn_readfirstlane(s_last[r]);
		dropped[r]     = last == 0;
		const int need = dropped[r] ? (int)L : last;
		l_eff          = need > l_eff ? need : l_eff;
		const int ft   = dropped[r] ? 0 : __builtin_amdgcn_readfirstlane(s_first[r]);
		first_tiles |= (uint32_t)ft << (8 * r);
		t_force_max    = ft > t_force_max ? ft : t_force_max;
	}
	n_t = (l_eff + KT_R - 1) / KT_R;
	if(n_q > 1 && n_t < 2) n_t = 2;   // (several query tiles: the walk of one requests two tiles of the next; keys behind the last live one weigh 0)

	// a batch row without live keys gets q = 0
	auto drop_q = [&]() {
#pragma unroll
		for(int r = 0; r < ROWS; r++)
			if(dropped[r]) qf[r][0] = qf[r][1] = __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u});
	};
	drop_q();
	// ---- online-softmax state: one query row per lane and batch row (the two half-waves hold disjoint keys) ----
	float  m_ref[ROWS];   // reference maximum, log2 units, exactly m_hi + m_lo of two bf16 values
	float  lsum[ROWS];    // the row sum (complete: the same value in both half-waves)
	float  rs_prev;       // the previous step's share of it (quick walk)
	f32x16 oacc[ROWS];

	// Move the reference of batch row R for every query whose maximum is not within REF_SLACK of it (all queries when
	// `force`), rescale what has been accumulated and re-express s relative to the new reference.
	auto rereference = [&](auto r_c, f32x16& s, bool force) {
		constexpr int R = decltype(r_c)::value;
		float mx = fmaxf(fmaxf(s[0], s[1]), s[2]);
#pragma unroll
		for(int i = 3; i < 15; i += 2) mx = fmaxf(fmaxf(mx, s[i]), s[i + 1]);
		mx = half_swap_max(fmaxf(mx, s[15]));
		// s already has m_ref subtracted (by the mask MFMA)
		// (forced: the row's first tile with a live key.  Every query then has a logit above the mask constants, the new
		// reference is its maximum, and that key's probability is exactly 1: the row sum can no longer flush to zero however
		// negative the row's biases are.  Tiles in front of it hold dropped keys only: their probabilities are exactly 0
		// against the initial reference 0, and nothing has been accumulated when the reference moves.)
		const bool  need   = (force && mx > -0x1p99f) || mx > REF_SLACK;
		const float m_want = m_ref[R] + mx;
		const float m_hi   = bf16_bits_to_f32(f32_to_bf16_bits(need ? m_want : m_ref[R]));
		const float m_lo   = bf16_bits_to_f32(f32_to_bf16_bits((need ? m_want : m_ref[R]) - m_hi));
		const float m_new  = m_hi + m_lo;  // exactly what the mask MFMA will subtract (unchanged when !need)
		const float delta  = m_new - m_ref[R];
		const float alpha  = force ? 1.f : __builtin_amdgcn_exp2f(-delta);  // nothing is accumulated yet when forced
#pragma unroll
		for(int i = 0; i < 16; i++) s[i] -= delta;
		m_ref[R] = m_new;
		if(half == 0) maskB[R][1] = f32_to_bf16_bits(-m_hi) | (f32_to_bf16_bits(-m_lo) << 16);
		lsum[R] *= alpha;
#pragma unroll
		for(int i = 0; i < 16; i++) oacc[R][i] *= alpha;
	};
	// The quick walk's first tile: every batch row has a live key in it, nothing is accumulated, and each query's reference is the
	// maximum of its logits.  The mask instruction once more, without mask values, subtracts it.
	auto first_reference = [&](auto r_c, f32x16& s) {
		constexpr int R = decltype(r_c)::value;
		float mx = fmaxf(fmaxf(s[0], s[1]), s[2]);
#pragma unroll
		for(int i = 3; i < 15; i += 2) mx = fmaxf(fmaxf(mx, s[i]), s[i + 1]);
		mx = half_swap_max(fmaxf(mx, s[15]));
		const float neg_hi = __uint_as_float(pack_bf16x2(0.f, -mx));   // (the high half is the rounded value; the low one is zero)
		const float neg_lo = -mx - neg_hi;
		if(half == 0) maskB[R][1] = pack_bf16x2(neg_hi, neg_lo);
		const u32x2 ones = {0u, 0x3F803F80u};
		s = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(__builtin_bit_cast(s16x4, ones), __builtin_bit_cast(s16x4, maskB[R]), s, 0, 0, 0);
	};
	auto exp_part = [&](const f32x16& s, u32x4 (&pf)[2], auto i0_c, auto n_c) {
		constexpr int I0 = decltype(i0_c)::value, N = decltype(n_c)::value;
#pragma unroll
		for(int i = I0; i < I0 + N; i += 2) pf[i >> 3][(i & 7) >> 1] = pack_bf16x2(__builtin_amdgcn_exp2f(s[i]), __builtin_amdgcn_exp2f(s[i + 1]));
	};
	auto read_kfrag = [&](int addr) -> u32x4 { return *reinterpret_cast<const u32x4*>(smem + addr); };
	auto rowsum     = [&](const f32x4& c, const u32x4& pf) -> f32x4 { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, ones_a), __builtin_bit_cast(bf16x8, pf), c, 0, 0, 0); };
	auto mask_mfma  = [&](const f32x16& c, const u32x2& b) -> f32x16 {
		return __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(__builtin_bit_cast(s16x4, maskA), __builtin_bit_cast(s16x4, b), c, 0, 0, 0);
	};

	// Pipeline registers: S^T of the current step, P^T and V^T fragments of the previous one, K fragments of the next
	// one, and the bias fragment of the tile the next step belongs to (accumulator order: the C operand of that step's
	// first K.Q^T instruction).
	f32x16 sc, bias_frag;
	u32x4  kf[2];
	u32x4  pprev[2], vprev[2];
#pragma unroll
	for(int i = 0; i < 16; i++) bias_frag[i] = 0.f;
	// the next tile's bias fragment -> registers: from the slot, or (direct mode) from the raw bf16 pieces loaded a tile ago:
	// clamped from below like the workspace's values (packed unsigned minimum: -2^16 and everything beyond it, -inf and
	// -NaN patterns included), widened to fp32 and scaled by log2 e
	auto next_bias_fragment = [&](int parity) {  // (staged mode: which half of the slot holds it)
		// (The old fragment is named once more behind its last reader: the registers it occupied then are the only free block of
		// 16 when the new one is defined, so the fragment keeps its place from tile to tile.  Without this the compiler lets
		// that reader's result overwrite the old fragment, puts the new one elsewhere and copies 16 registers per tile.)
		if constexpr(HAS_BIAS) asm volatile("" ::"v"(bias_frag));
		if constexpr(SLOT) {
#pragma unroll
			for(int ld = 0; ld < 4; ld++) {
				const f32x4 v = *reinterpret_cast<const f32x4*>(smem + slot_rd + ld * 1024);
				bias_frag[4 * ld] = v[0], bias_frag[4 * ld + 1] = v[1], bias_frag[4 * ld + 2] = v[2], bias_frag[4 * ld + 3] = v[3];
			}
		} else if constexpr(DIRECT || STAGED) {
			const uint32_t lim = 0xC780C780u;
			if constexpr(STAGED) {  // this lane's four 8-byte pieces, keys 8 ld + 4 half .. + 3 of row n: chunk ld at its swizzled place
#pragma unroll
				for(int ld = 0; ld < 4; ld++)
					braw[ld] = *reinterpret_cast<const u32x2*>(smem + SLOT_BASE + wave * 4096 + (parity & 1) * 2048 + n * 64 + ((ld ^ ((n >> 2) & 3)) << 4) + half * 8);
			}
#pragma unroll
			for(int ld = 0; ld < 4; ld++)
#pragma unroll
				for(int j = 0; j < 2; j++) {
					const uint32_t raw = braw[ld][j];
					const uint32_t w   = bias_limited(raw, lim);
					bias_frag[4 * ld + 2 * j]     = __uint_as_float(w << 16) * LOG2E;
					bias_frag[4 * ld + 2 * j + 1] = __uint_as_float(w & 0xffff0000u) * LOG2E;
				}
		}
	};

	// One step = one 32 x 32 block of logits of batch row R.  On entry `sc` holds its finished S^T, `pprev` / `vprev`
	// belong to the previous step (batch row R-1, or row 3 of the previous tile) and `kf` holds the K fragments of the
	// next step.  The step alternates matrix instructions of three independent chains with slices of its vector work
	//     matrix pipe                                            vector ALU
	//     O^T[R-1] += V^T . P^T (previous step, 2 instructions)   exp2 / pack of this step, two logits per slice
	//     S^T of the next step (K.Q^T + bias, mask: 3)
	//     row sum of this step (2 half-size instructions)
	// so that no instruction waits for the one issued just before it, and leaves S^T(next) in `sc`, P^T in `pprev`, this
	// step's V^T fragments in `vprev`, the K fragments of the step after the next in `kf`.
	// k_addr2: LDS byte address of the K tile of the step after the next; m_addr: (per lane) of the next step's mask
	// entries; v_addr: of this step's V tile; hook(i): run behind the i-th matrix instruction of the step (i = 0..4; 1 is the
	// first K.Q^T instruction of the next step).
	// FIRST: a leading tile, in which a row that meets its first live key (`force`, wave-uniform) fixes its softmax reference.  CAREFUL: the walk that tests every step's row
	// sums, and whose batch rows may lack live keys (they then take no bias: a wave-uniform branch that the quick walk does not carry).
	auto step = [&](auto r_c, auto first_c, auto careful_c, bool force, int k_addr2, int m_addr, int v_addr, auto&& behind_reference, auto&& hook) {
		constexpr int  R = decltype(r_c)::value, RN = (R + 1) % ROWS, RP = (R + ROWS - 1) % ROWS;
		constexpr bool FIRST = decltype(first_c)::value != 0, CAREFUL = decltype(careful_c)::value != 0;
		if constexpr(FIRST && CAREFUL) rereference(r_c, sc, force);
		else if constexpr(FIRST) first_reference(r_c, sc);
		behind_reference();
		maskA[0] = *reinterpret_cast<const uint16_t*>(smem + m_addr);
		u32x4  pcur[2];
		f32x16 sn;
		f32x4  rs = {0.f, 0.f, 0.f, 0.f};
		if constexpr(!CAREFUL) lsum[RP] += rs_prev;
		// The order below is the order the instructions are meant to issue in: one matrix instruction, then a slice of the
		// vector work, so that consecutive matrix instructions belong to different chains.  Matrix intrinsics are pure
		// values to the compiler and would drift to wherever their consumers are; each slice therefore ends with an empty
		// asm statement that names what the slice produced and the operand the next slice's matrix instruction waits for
		// (asm statements keep their order, and so does everything that feeds or reads them), followed by a scheduling barrier.
#define AF3_PIN2(a, b)                                \
	{                                                 \
		auto pa_ = a;                                 \
		auto pb_ = b;                                 \
		asm volatile("" : "+v"(pa_), "+v"(pb_));      \
		a = pa_, b = pb_;                             \
	}                                                 \
	__builtin_amdgcn_sched_barrier(0)
#define AF3_PIN3(a, b, c)                                        \
	{                                                            \
		auto pa_ = a;                                            \
		auto pb_ = b;                                            \
		auto pc_ = c;                                            \
		asm volatile("" : "+v"(pa_), "+v"(pb_), "+v"(pc_));      \
		a = pa_, b = pb_, c = pc_;                               \
	}                                                            \
	__builtin_amdgcn_sched_barrier(0)
		__builtin_amdgcn_sched_barrier(0);
		oacc[RP] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, vprev[0]), __builtin_bit_cast(bf16x8, pprev[0]), oacc[RP], 0, 0, 0);
		hook(ic<0>{});
		exp_part(sc, pcur, ic<0>{}, ic<2>{});
		AF3_PIN3(oacc[RP][0], pcur[0][0], kf[0][0]);
		{
			f32x16 z;
#pragma unroll
			for(int i = 0; i < 16; i++) z[i] = 0.f;
			bool with_bias = HAS_BIAS;
			if constexpr(CAREFUL) with_bias = HAS_BIAS && !dropped[RN];  // (wave-uniform)
			if(with_bias) sn = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kf[0]), qf[RN][0], bias_frag, 0, 0, 0);
			else sn = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kf[0]), qf[RN][0], z, 0, 0, 0);
		}
		hook(ic<1>{});
		exp_part(sc, pcur, ic<2>{}, ic<2>{});
		AF3_PIN3(sn[0], pcur[0][1], pprev[1][0]);
		oacc[RP] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, vprev[1]), __builtin_bit_cast(bf16x8, pprev[1]), oacc[RP], 0, 0, 0);
		// V^T fragments of this step for the next step's P.V, now that the previous ones are consumed
#pragma unroll
		for(int cp = 0; cp < 2; cp++)
#pragma unroll
			for(int t = 0; t < 2; t++) {
				const s16x4 rr = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(smem + v_addr + v_rd + (16 * cp + 8 * t) * 64));
				const u32x2 r2 = __builtin_bit_cast(u32x2, rr);
				vprev[cp][2 * t] = r2[0], vprev[cp][2 * t + 1] = r2[1];
			}
		hook(ic<2>{});
		exp_part(sc, pcur, ic<4>{}, ic<2>{});
		AF3_PIN3(oacc[RP][0], pcur[0][2], kf[1][0]);
		sn = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kf[1]), qf[RN][1], sn, 0, 0, 0);
		// K fragments of the step after the next, now that the next step's are consumed
		kf[0] = read_kfrag(k_addr2 + k_rd[0]);
		kf[1] = read_kfrag(k_addr2 + k_rd[1]);
		hook(ic<3>{});
		exp_part(sc, pcur, ic<6>{}, ic<2>{});
		AF3_PIN2(sn[0], pcur[0][3]);
		rs = rowsum(rs, pcur[0]);
		hook(ic<4>{});
		exp_part(sc, pcur, ic<8>{}, ic<4>{});
		AF3_PIN3(rs[0], pcur[1][0], pcur[1][1]);
		{
			uint32_t ma_ = maskA[0];
			asm volatile("" : "+v"(ma_));
			maskA[0] = ma_;
		}
		sn = mask_mfma(sn, maskB[RN]);
		exp_part(sc, pcur, ic<12>{}, ic<4>{});
		AF3_PIN3(sn[0], pcur[1][2], pcur[1][3]);
#undef AF3_PIN2
#undef AF3_PIN3
		rs = rowsum(rs, pcur[1]);
		if constexpr(CAREFUL) {
			// This step's sum stays below 32 * 2^REF_SLACK while every probability respects the reference, so the test also
			// catches a single probability near or beyond the limit (inf, NaN).
			if(__ballot(!(rs[0] < PSUM_LIMIT))) {  // rare
				rereference(r_c, sc, false);
				exp_part(sc, pcur, ic<0>{}, ic<16>{});
				rs = rowsum(f32x4{0.f, 0.f, 0.f, 0.f}, pcur[0]);
				rs = rowsum(rs, pcur[1]);
			}
			lsum[R] += rs[0];
		} else {
			rs_prev = rs[0];   // (added a step later: nothing waits for the matrix pipe here)
		}
		sc       = sn;
		pprev[0] = pcur[0];
		pprev[1] = pcur[1];
	};

	// What remains of query tile i's batch row R when its last product is in: divide by the row sum, gate, store.  GATE_LDS: the gate rows wait
	// in LDS.  BF16: the output is known to be bf16.  The stores go through a range-checked buffer and are always four to a lane (columns
	// from D on lie out of its range): the wait in the tile that follows counts them.
	uint32_t redo[ROWS];   // query tiles of batch row r whose sums do not stand: walked again carefully
#pragma unroll
	for(int r = 0; r < ROWS; r++) redo[r] = 0u;
	u32x2           graw[4];   // gate values of a batch row, as request_gate leaves them
	const uint16_t* gate_ptr = nullptr;
	auto request_gate = [&](auto r_c, int i) {   // (batch rows in their order)
		constexpr int R = decltype(r_c)::value;
		if constexpr(GATE && R < ROWS) {
			const args_t a = args();
			if constexpr(R == 0) gate_ptr = static_cast<const uint16_t*>(a->gate) + b0 * a->gate_stride[0] + h * a->gate_stride[1] + (row00 + i * (NW * 32)) * a->gate_stride[2];
			else gate_ptr += R < n_rows ? a->gate_stride[0] : 0;
			const __amdgpu_buffer_rsrc_t rsrc = buffer_of(gate_ptr, a->gate_stride[2], rows_left(i), 2);
			const int l = lane_now(), voff = ((l & 31) * (int)a->gate_stride[2] + 4 * (l >> 5)) * 2;
#pragma unroll
			for(int g4 = 0; g4 < 4; g4++) graw[g4] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(rsrc, 8 * g4 < D ? voff + 16 * g4 : 0x7FFF0000, 0, 0));
		}
	};
	unsigned char* out_row = nullptr;
	int64_t        out_sb = 0;
	int            out_sr = 0, out_el = 2;   // (bytes from batch row to batch row, elements from query row to query row, bytes per element)
	auto finish_row = [&](auto r_c, auto careful_c, auto gate_lds_c, auto bf16_c, int i, [[maybe_unused]] int gate_buf0, [[maybe_unused]] int gate_buf1) {   // (batch rows in their order)
		constexpr int  R = decltype(r_c)::value;
		constexpr bool CAREFUL = decltype(careful_c)::value != 0, GATE_LDS = decltype(gate_lds_c)::value != 0, BF16 = decltype(bf16_c)::value != 0;
		if constexpr(R < ROWS) {
			const int rows = rows_left(i);
			bool      keep_row = R < n_rows;   // (wave-uniform)
			if constexpr(!CAREFUL) {
				// Sums that end below the careful walk's limit have stayed below it throughout: the results are the careful walk's.  Beyond it
				// they stand all the same if they stay below 2^100 and the results are finite.
				if(__ballot(!(lsum[R] < PSUM_LIMIT))) {   // rare
					const int n_ = lane_now() & 31;
					float     t = lsum[R] * 0x1p28f;   // (infinite from 2^100 on)
#pragma unroll
					for(int k = 0; k < 16; k++) t = fmaf(oacc[R][k], 0.f, t);
					if(__ballot(n_ < rows && !(t < __builtin_inff()))) {
						redo[R] |= 1u << i;
						keep_row = false;
						if(lane_now() == 0) atomicOr(&s_again, 1u << i);
					}
				}
			} else {
				keep_row = keep_row && ((redo[R] >> i) & 1u) != 0;
			}
			if constexpr(R == 0) {
				const args_t a = args();
				if(!BF16) out_el = a->out_dtype == AF3_BF16 ? 2 : 4;
				const int es = BF16 ? 2 : out_el;
				out_sb = a->out_stride[0] * es, out_sr = (int)a->out_stride[2];
				out_row = static_cast<unsigned char*>(a->out) + (b0 * a->out_stride[0] + h * a->out_stride[1] + (row00 + i * (NW * 32)) * out_sr) * es;
			} else out_row += out_sb;
			const int es = BF16 ? 2 : out_el;
			const __amdgpu_buffer_rsrc_t rsrc = buffer_of(out_row, out_sr, keep_row ? rows : 0, es);
			const int l = lane_now(), half_ = l >> 5, n_ = l & 31, voff = (n_ * out_sr + 4 * half_) * es;
			// (a Newton step behind the reciprocal: half an ulp, as the division)
			const float r0 = __builtin_amdgcn_rcpf(lsum[R]), inv = __builtin_fmaf(r0, __builtin_fmaf(-lsum[R], r0, 1.f), r0);
			if constexpr(GATE && GATE_LDS) {
				const int gk = 2 * R + (n_ >> 4);   // this query row's piece of the gate
				const unsigned char* const gate_row = smem + (gk < ROWS ? gate_buf0 : gate_buf1) + (wave * ROWS + (gk < ROWS ? gk : gk - ROWS)) * 1024 + (n_ & 15) * 64 + half_ * 8;
#pragma unroll
				for(int g4 = 0; g4 < 4; g4++) graw[g4] = *reinterpret_cast<const u32x2*>(gate_row + g4 * 16);
			}
			auto columns = [&](int g4) {
				float o[4];
#pragma unroll
				for(int e = 0; e < 4; e++) o[e] = oacc[R][4 * g4 + e] * inv;
				if constexpr(GATE) {
					const u32x2 gw = graw[g4];
					o[0] *= sigmoidf_fast(bf16_bits_to_f32(gw[0] & 0xffffu)), o[1] *= sigmoidf_fast(bf16_bits_to_f32(gw[0] >> 16));
					o[2] *= sigmoidf_fast(bf16_bits_to_f32(gw[1] & 0xffffu)), o[3] *= sigmoidf_fast(bf16_bits_to_f32(gw[1] >> 16));
				}
				if(BF16 || es == 2)
					__builtin_amdgcn_raw_buffer_store_b64(u32x2{pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3])}, rsrc, 8 * g4 < D ? voff + 16 * g4 : 0x7FFF0000, 0, 0);
				else __builtin_amdgcn_raw_buffer_store_b128(u32x4{__float_as_uint(o[0]), __float_as_uint(o[1]), __float_as_uint(o[2]), __float_as_uint(o[3])}, rsrc, voff + 32 * g4, 0, 0);
			};
			// (head_dim 8 to 24 leave blocks of columns out; with all four gated and stored 2000 x 8 x 64 x 8 with a gate took 81.9 us, 300 x 8 x 300 x 8 80.4, so 69.5 and
			// 72.8; between query tiles no branch: the compiler's count of what is in flight would lose the stores)
			columns(0);
			if(BF16 || D > 8) columns(1);
			if(BF16 || D > 16) {
				columns(2);
				if(BF16 || D > 24) columns(3);
			}
			lsum[R] = 0.f;
#pragma unroll
			for(int k = 0; k < 16; k++) oacc[R][k] = 0.f;
		}
	};

	// One tile: ROWS steps.  The seq-th tile of the workgroup (tile t of query tile i) sits in buffer seq % 3.  In front of the last-but-one step the loads issued one tile
	// earlier (tile t + 1 and its bias fragment: the youngest loads this wavefront has in flight) are awaited and a barrier
	// publishes tile t + 1 -- that step fetches K fragments from it -- and tells that every wavefront is done with tile
	// t - 1, whose buffer tile t + 2 then overwrites.  That step's first matrix instruction is the last reader of bias
	// fragment t: behind it the fragment registers take fragment t + 1, and the slot (once those reads have returned: the
	// last step's first matrix instruction waits for them) or the raw-piece registers are refilled with fragment t + 2.
	//
	// Several query tiles of one head and the same batch rows: K, V and the masks stay, so the ring of tiles runs on -- behind the last
	// tile come the first two again -- and so do the four chains.  The last tile's steps (LAST) request the next query tile's q rows
	// as their predecessors' last readers pass, row r in step r and row 0 ROWS - 1 steps ahead of its first use; the next query tile's first tile (FIRST_NEXT) finishes and
	// stores a batch row's results between the step's new reference and its exponentials.  A workgroup of one query tile spends 26 k clocks of its 79 k
	// (L = 768) in front of its walk and behind it; from query tile to query tile it is 6 k.
	// The hand-written waits in front of the barriers let what was issued behind the awaited loads stay in flight.  The compiler's own, for q rows and gates, do not count the
	// loads that write LDS and so take in the next tile's, which are a step old by then.  With everything requested and awaited in front of those loads (they a step later, q
	// rows converted and the gates of two rows requested in LAST) no wait did, in the same time: us, so / here: 384 x 4 x 384 x 32 58.3 / 58.1, with a gate 63.3 / 63.7,
	// 768 374.1 / 373.9, 1491 2564 / 2558, 300 x 16 x 384 x 24 172.6 / 167.9, and 4 registers more spilled.
	// (INNER: a MIDDLE tile with two more of its query tile behind it; it asks nothing about what is to be requested.)
	enum { MIDDLE = 0, FIRST = 1, LAST = 2, FIRST_NEXT = 3, CAREFUL_MIDDLE = 4, CAREFUL_FIRST = 5, INNER = -1 };
	// more: this wavefront walks another query tile behind this one; more_wg: the workgroup does
	auto tile = [&](auto kind_c, int t, int i, int seq, bool more, bool more_wg, int buf, int bufn, int bufnn) {
		constexpr int  KIND = decltype(kind_c)::value;
		constexpr auto first_c = ic<(KIND == FIRST || KIND == FIRST_NEXT || KIND == CAREFUL_FIRST) ? 1 : 0>{};
		constexpr auto careful_c = ic<(KIND >= CAREFUL_MIDDLE) ? 1 : 0>{};
		asm volatile("" : "+s"(t));   // (offsets of known tiles would be kept in registers, or spilled, through the walk)
		const int m0 = mask_rd + t * (ROWS * 64);
		// what is requested in this tile: the tile after the next
		int tn = t + 2, tb = t + 2, ib = i;
		if constexpr(KIND != INNER) {
			if(tn >= n_t && more_wg) tn -= n_t;
			if(tb >= n_t && more) tb -= n_t, ib = i + 1;
		}
		auto one = [&](auto r_c) {
			constexpr int R = decltype(r_c)::value;
			if constexpr(R < ROWS) {
				constexpr int R1 = R + 1, R2 = R + 2;                        // the next step and the one after it ...
				const int     k2 = (R2 >= ROWS ? bufn : buf) + (R2 % ROWS) * (2 * TILE_R);   // ... may belong to the next tile
				const int     m1 = KIND == LAST && R1 == ROWS ? mask_rd : m0 + R1 * 64;      // (row ROWS of tile t is row 0 of tile t + 1)
				const int     vc = buf + R * (2 * TILE_R);
				const bool    fr = KIND == CAREFUL_FIRST && t == (int)((first_tiles >> (8 * (R < ROWS ? R : 0))) & 0xffu);
				if constexpr(KIND == LAST) {
					request_q(r_c, i + 1);   // (row R: its last reader was the step before this one)
					if constexpr(R1 == ROWS) {
						convert_q(ic<0>{});
						maskB[0][1] = 0u;
						request_gate(ic<0>{}, i);
					}
				}
				// (between the new reference's matrix instruction and the exponentials that wait for it)
				auto finish = [&]() {
					if constexpr(KIND == FIRST_NEXT) {
						finish_row(r_c, ic<0>{}, ic<0>{}, ic<1>{}, i - 1, 0, 0);
						request_gate(ic<R1>{}, i - 1);
						if constexpr(R1 < ROWS) {
							convert_q(ic<R1>{});
							maskB[R1][1] = 0u;
						}
					}
					if constexpr(R == ROWS - 2) {
						// (with two rows the V^T fragments of tile t - 1 may still be on their way: they are consumed in this step; with more
						// rows an earlier step of this tile has consumed them)
						// (what was issued behind the awaited loads may stay in flight: the q rows of the steps so far, or the stores of finished rows)
						constexpr int YOUNGER = KIND == LAST ? 2 * (ROWS - 1) : KIND == FIRST_NEXT ? (GATE ? 8 : 4) * (ROWS - 1) : 0;
						if constexpr(ROWS == 2) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
						asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(YOUNGER) : "memory");
					}
				};
				if constexpr(R == ROWS - 2) {
					step(r_c, first_c, careful_c, fr, k2, m1, vc, finish, [&](auto s_c) {
						constexpr int S = decltype(s_c)::value;
						if constexpr(S == 1) {
							if constexpr(KIND == INNER) load_tile(tn, bufnn);
							else load_tile_or_gate(tn, bufnn, i);
							next_bias_fragment(seq + 1);
							if(KIND == INNER || tb < n_t) load_bias_direct(tb), load_bias_staged(tb, ib, seq);   // (into the half that held this tile's fragment, read a tile ago)
						}
					});
				} else if constexpr(R == ROWS - 1) {
					step(r_c, first_c, careful_c, fr, k2, m1, vc, finish, [&](auto s_c) {
						constexpr int S = decltype(s_c)::value;
						if constexpr(S == 1)
							if(KIND == INNER || tb < n_t) load_bias(tb, ib);   // (behind this step's first K.Q^T instruction, which has waited for the slot's reads)
					});
				} else {
					step(r_c, first_c, careful_c, fr, k2, m1, vc, finish, [](auto) {});
				}
			}
		};
		one(ic<0>{}), one(ic<1>{}), one(ic<2>{}), one(ic<3>{});
	};
	// the second tile and bias fragment, S^T of the first step, K fragments of the second (tile 0 and bias fragment 0 of query tile i are complete)
	auto prologue = [&](auto careful_c, int i) {
		constexpr bool CAREFUL = decltype(careful_c)::value != 0;
#pragma unroll
		for(int r = 0; r < ROWS; r++) {
			m_ref[r] = 0.f;
			lsum[r]  = 0.f;
			maskB[r] = u32x2{half == 0 ? 0x3F80u : 0u, 0u};
#pragma unroll
			for(int k = 0; k < 16; k++) oacc[r][k] = 0.f;
		}
		rs_prev  = 0.f;
		pprev[0] = pprev[1] = vprev[0] = vprev[1] = u32x4{0u, 0u, 0u, 0u};
		next_bias_fragment(0);  // fragment 0 -> registers
		asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
		load_tile_or_gate(1, BUF_R, i);
		if(n_t > 1) load_bias(1, i), load_bias_direct(1), load_bias_staged(1, i, 1);
		f32x16 s0;
#pragma unroll
		for(int k = 0; k < 16; k++) s0[k] = (HAS_BIAS && !(CAREFUL && dropped[0])) ? bias_frag[k] : 0.f;
#pragma unroll
		for(int c = 0; c < 2; c++) s0 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, read_kfrag(k_rd[c])), qf[0][c], s0, 0, 0, 0);
		maskA[0] = *reinterpret_cast<const uint16_t*>(smem + mask_rd);
		sc = mask_mfma(s0, maskB[0]);
		kf[0] = read_kfrag(2 * TILE_R + k_rd[0]);
		kf[1] = read_kfrag(2 * TILE_R + k_rd[1]);
	};
	auto last_product = [&]() {   // the last step's P.V product (the last batch row)
		lsum[ROWS - 1] += rs_prev;
		oacc[ROWS - 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, vprev[0]), __builtin_bit_cast(bf16x8, pprev[0]), oacc[ROWS - 1], 0, 0, 0);
		oacc[ROWS - 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, vprev[1]), __builtin_bit_cast(bf16x8, pprev[1]), oacc[ROWS - 1], 0, 0, 0);
	};
	auto next_buf = [](int buf) { return buf == (NBUF_R - 1) * BUF_R ? 0 : buf + BUF_R; };
	// a wavefront none of whose query rows exist (L % 128 != 0, the last query tile) fetches its batch row's tiles, keeps the barriers' count --
	// one per tile -- and leaves the vector and matrix pipes to others
	auto load_only = [&](int buf) {   // (tiles 0 and 1 are requested)
		int bufnn = next_buf(next_buf(buf));
		for(int t = 0; t < n_t; t++) {
			asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
			if(t + 2 < n_t) load_tile(t + 2, bufnn);
			bufnn = next_buf(bufnn);
		}
	};
	// The key axis is walked without a look at the row sums on the way (a test per step made the wavefront wait for the matrix pipe
	// and kept the step's logits alive behind it: 768 x 4 x 768 x 32 408 -> 392 us without, 1491 2837 -> 2713, 384 64.9 -> 62.8).  Sums
	// that end below the careful walk's limit have stayed below it throughout: the results are the careful walk's.  Beyond it they
	// stand all the same if the sums stay below 2^100 and the results are finite (probabilities and sums are floating-point: a
	// reference left behind costs them no digits).  Otherwise the whole workgroup -- its wavefronts fetch tiles for one another --
	// walks that query tile once more, carefully, and a workgroup with a batch row without a live key, or without one in its first tile, walks all of them so.
	bool careful = t_force_max > 0;
#pragma unroll
	for(int r = 0; r < ROWS; r++) careful = careful || dropped[r];   // (the same in every wavefront of the workgroup)
	uint32_t again = 0xffffffffu >> (32 - n_q);
	if(!careful) {
		int buf = 0, seq = 0;
		if(my_q > 0) {
			prologue(ic<0>{}, 0);
			bool more = my_q > 1, more_wg = n_q > 1;
			tile(ic<FIRST>{}, 0, 0, 0, more, more_wg, 0, BUF_R, 2 * BUF_R);
			buf = BUF_R, seq = 1;
			int i = 0;
			even_progress progress(n_q * n_t, even);
			for(;;) {
				const int t_end = more ? n_t - 1 : n_t;
				int       t = 1;
				for(; t < n_t - 2; t++) {
					const int bufn = next_buf(buf), bufnn = next_buf(bufn);
					progress.at(seq);
					tile(ic<INNER>{}, t, i, seq, more, more_wg, buf, bufn, bufnn);
					buf = bufn, seq++;
				}
				for(; t < t_end; t++) {
					const int bufn = next_buf(buf), bufnn = next_buf(bufn);
					tile(ic<MIDDLE>{}, t, i, seq, more, more_wg, buf, bufn, bufnn);
					buf = bufn, seq++;
				}
				if(!MULTI || !more) break;
				{
					const int bufn = next_buf(buf), bufnn = next_buf(bufn);
					tile(ic<LAST>{}, n_t - 1, i, seq, true, true, buf, bufn, bufnn);
					buf = bufn, seq++, i++;
				}
				more = i + 1 < my_q, more_wg = i + 1 < n_q;
				{
					const int bufn = next_buf(buf), bufnn = next_buf(bufn);
					tile(ic<FIRST_NEXT>{}, 0, i, seq, more, more_wg, buf, bufn, bufnn);
					buf = bufn, seq++;
				}
			}
			last_product();
			asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the gate rows)
			const int gate0 = buf, gate1 = next_buf(buf);
			auto finish_last = [&](auto r_c) {
				if(!GATE || my_q == n_q) finish_row(r_c, ic<0>{}, ic<1>{}, ic<0>{}, i, gate0, gate1);
				else request_gate(r_c, i), finish_row(r_c, ic<0>{}, ic<0>{}, ic<0>{}, i, 0, 0);   // (the workgroup walks on: its tile buffers are in use)
			};
			finish_last(ic<0>{}), finish_last(ic<1>{}), finish_last(ic<2>{}), finish_last(ic<3>{});
		} else {
			if(n_t > 1) load_tile(1, BUF_R);
		}
		if(my_q < n_q) {
			load_only(buf);
			asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load may still be writing LDS when the workgroup's allocation is released
		}
		asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
		again = (uint32_t)__builtin_amdgcn_readfirstlane((int)*(volatile uint32_t*)&s_again);
		if(again == 0u) return;
	} else {
#pragma unroll
		for(int r = 0; r < ROWS; r++) redo[r] = again;
	}
	// ---- the careful walk of the query tiles in `again` (rare) ----
	bool fresh = careful;   // the start's requests serve the first query tile
	while(again) {
		const int i = __builtin_ctz(again);
		again &= again - 1;
		if(!fresh || i > 0) {
			__syncthreads();   // (every wavefront has left the tiles of the walk before)
			load_tile(0, 0);
			load_bias(0, i);
			load_bias_direct(0);
			load_bias_staged(0, i, 0);
			request_q(ic<0>{}, i), request_q(ic<1>{}, i), request_q(ic<2>{}, i), request_q(ic<3>{}, i);
			convert_q(ic<0>{}), convert_q(ic<1>{}), convert_q(ic<2>{}), convert_q(ic<3>{});
			drop_q();
			asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
			__syncthreads();
		}
		fresh = false;
		if(i >= my_q) {
			if(n_t > 1) load_tile(1, BUF_R);
			load_only(0);
			asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
			continue;
		}
		prologue(ic<1>{}, i);
		int buf = 0, t = 0;
		for(; t <= t_force_max; t++) {   // (more than one trip where some row's leading tiles hold dropped keys only)
			const int bufn = next_buf(buf), bufnn = next_buf(bufn);
			tile(ic<CAREFUL_FIRST>{}, t, i, t, false, false, buf, bufn, bufnn);
			buf = bufn;
		}
		for(; t < n_t; t++) {
			const int bufn = next_buf(buf), bufnn = next_buf(bufn);
			tile(ic<CAREFUL_MIDDLE>{}, t, i, t, false, false, buf, bufn, bufnn);
			buf = bufn;
		}
		last_product();
		asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load may still be writing LDS when the workgroup's allocation is released
		const int gate0 = buf, gate1 = next_buf(buf);
		finish_row(ic<0>{}, ic<1>{}, ic<1>{}, ic<0>{}, i, gate0, gate1), finish_row(ic<1>{}, ic<1>{}, ic<1>{}, ic<0>{}, i, gate0, gate1), finish_row(ic<2>{}, ic<1>{}, ic<1>{}, ic<0>{}, i, gate0, gate1), finish_row(ic<3>{}, ic<1>{}, ic<1>{}, ic<0>{}, i, gate0, gate1);
	}
}

int64_t rows_ws_bytes(const af3_dpa_params& p) {
	const int64_t n_qblocks = (p.L + 31) / 32, n_t_all = (p.L + KT_R - 1) / KT_R;
	return p.H * n_qblocks * n_t_all * 4096;
}

// The bf16 bias can be read in place when its rows start on 8-byte boundaries, keys come in whole groups of four and the
// slab of one head fits 32-bit byte offsets.
bool direct_bias_ok(const af3_dpa_params& p) {
	return p.bias && p.bias_dtype == AF3_BF16 && p.L % 4 == 0 && (reinterpret_cast<uintptr_t>(p.bias) & 7) == 0 && p.bias_stride[0] % 4 == 0 && p.bias_stride[1] % 4 == 0 &&
		   ((p.L - 1) * p.bias_stride[1] + p.L) * 2 < 0x40000000LL;
}

// ... and through LDS, in whole 16-byte chunks of whole rows, when rows start on 16-byte boundaries and keys come in groups of eight.
bool staged_bias_ok(const af3_dpa_params& p) {
	return direct_bias_ok(p) && p.L % 8 == 0 && (reinterpret_cast<uintptr_t>(p.bias) & 15) == 0 && p.bias_stride[0] % 8 == 0 && p.bias_stride[1] % 8 == 0;
}

// Staging the bf16 bias costs each step 8 vector instructions (widening it) that the fp32 workspace does not -- about 5 % of
// the kernel's time -- the workspace a prepass over the whole bias (about 3 us + 0.46 us per MB read and written) and twice
// the bytes per tile.  Staged / workspace, us, prepass included: 32 x 16 x 1536 x 24 245 / 299, 64 x 4 x 768 x 32 50 / 55,
// 200 119 / 124, 256 132 / 131, 288 177 / 182, 512 263 / 257, 768 390 / 379, 384 x 4 x 384 x 32 60.2 / 60.3, 560 102 / 104, 640 102 / 101, 1024 160 / 156.
// The prepass is worth its time from about 224 + 2.4e8 / (H L^2) batch rows on (the second term: its fixed cost against the
// time of one batch row).
constexpr int64_t STAGED_MAX_B_SMALL = 128;  // below this the kernel is taken for launches the one-row kernel would otherwise serve
static bool staged_preferred(const af3_dpa_params& p) {
	if(!staged_bias_ok(p)) return false;
	const double x = (double)p.H * (double)p.L * (double)p.L;
	return (double)p.B < 224.0 + 2.44e8 / x;
}

// 0 = no bias, 1 = through the rewritten workspace, 2 = read in place (3: through LDS), -1 = this kernel cannot serve the call.
int rows_bias_mode(const af3_dpa_params& p) {
	if(!p.bias) return 0;
	const bool ws_ok = p.workspace && p.workspace_bytes >= rows_ws_bytes(p) && (reinterpret_cast<uintptr_t>(p.workspace) & 15) == 0;
	if(staged_preferred(p)) return 3;
	if(p.B >= 16 && ws_ok) return 1;
	if(direct_bias_ok(p)) return staged_bias_ok(p) ? 3 : 2;
	return ws_ok ? 1 : -1;
}

// Lines of 128 bytes that a key's K and V rows lie in, as a sum over `count` of its heads and neighbours: one to a key where rows follow one another or K and V of a
// head share a line, two where they are views of [.., heads, 32] or of a packed projection, more where rows straddle lines.
struct kv_lines {
	int64_t sum = 0, count = 0;
	bool    apart = true;   // K's lines hold nothing of V
};
kv_lines lines_of_a_key(const af3_dpa_params& p) {
	if(p.k_stride[2] == p.D && p.v_stride[2] == p.D) return {1, 1, false};
	kv_lines n;
	for(int64_t h = 0; h < p.H && h < 8; h++)
		for(int64_t key = 0; key < p.L && key < 4; key++) {
			const uint64_t k = reinterpret_cast<uintptr_t>(p.k) + (h * p.k_stride[1] + key * p.k_stride[2]) * 2, v = reinterpret_cast<uintptr_t>(p.v) + (h * p.v_stride[1] + key * p.v_stride[2]) * 2;
			const uint64_t k0 = k / 128, k1 = (k + p.D * 2 - 1) / 128, v0 = v / 128, v1 = (v + p.D * 2 - 1) / 128;
			const bool     meet = k0 <= v1 && v0 <= k1;
			n.sum += meet ? (k1 > v1 ? k1 : v1) - (k0 < v0 ? k0 : v0) + 1 : k1 - k0 + v1 - v0 + 2;
			n.apart = n.apart && !meet;
			n.count++;
		}
	return n;
}

// How many query tiles a workgroup walks.  Its start and its end (masks, first tiles, q, the stores' way out) are paid once, but workgroups of several
// query tiles come in fewer rounds of the 64 an XCD holds (two per compute unit), and query tiles that are walked one behind the other read K and V
// from the L2 at different times, where neighbours read them together.  So a divisor of the number of query tiles: the smallest of those that leave whole rounds or a last
// one more than nine tenths full, else of two and three that leave one more than four fifths full; else, from two rounds of single tiles on (three tiles to a head 1.75; eight and
// more 3, nine 5, where single ones would not make whole rounds), two (three of three and nine), and what would be the last round ends in single tiles.
// Time of single tiles = 1, by rounds of them: two tiles to a head, in twos 1.5 1.02-1.03, 1.62 0.89-0.94, 1.75 0.91-0.95, 2 0.89-0.97, 2.9 0.97; ending in single ones 1.5
// 1.04-1.07, 1.62 1.01-1.04, 2.6-2.9 0.92-0.99, 5-6.9 0.93-1.02; three, in threes 2.5-2.6 0.92-0.93, 2.7-3 0.92-0.97, 4.9 1.03, 5.5 0.95-0.98; ending in single ones 1.4-1.6
// 1.03-1.18, 1.7 0.99-1.02, 1.8-2 0.94-0.99, 2.5-2.6 1.03-1.06, 4.9-6.8 0.94-1.00; four, in twos 1.6-1.75 0.94-1.00, 1.9-2 0.95-0.99, 2.6-3 1.0-1.07; ending in single ones
// 1.5-1.75 1.00-1.06, 2.6-3 0.90-0.99, 5-7 0.95-1.01; in fours 2.6-3 1.04-1.13, 3.6 0.90-0.92 (in twos 0.94), 4 0.98 (0.96); six, in twos 1.7 0.92-1.00, 1.9 0.94-0.99, 5.6 0.92-0.95;
// ending 1.4-1.7 1.02-1.13, 2.6-6.8 0.94-1.00; eight and ten alike, but ending 2.5-2.8 0.97-1.05 and whole rounds of single ones 5 1.05-1.08; nine, in threes 2.8-3 0.98-1.00, ending 1.7-3.1 1.03-1.13, 3.5-4.5 0.98-1.04, 5-20 0.94-1.00.
// Five go as 2 2 1, in one round (0.95-0.97) or, where the bias is not staged in place and single tiles would not make whole rounds, from three on, ending in single tiles
// (3.75 0.95, 4.7 0.95-0.98, 5.5-6.8 0.95-0.99; whole rounds of single ones 3 1.01-1.05, 5 1.02-1.03; staged 0.99-1.05; 2 2 1 throughout 1.01-1.07).  Seven, eleven and thirteen stay single: 832 507 us, in twos / threes / fours 535 / 521 / 565, 896 608 / 618 / 621 / 637, 300 x 4 x 1600 x 32 637 / 655 / 660 / 726; eleven
// as 3 3 3 2 0.99-1.10.  us, one query tile each / so, one card, L x 4 x L x 32: 300 41.8 / 40.9, 384 62.4 / 57.7, 512 131.6 / 122.2, 768 393.8 / 377.3, 1024 874 / 841,
// 1491 2643 / 2564; 2048 x 4 x 256 x 32 165.9 / 162.1, 512 x 4 x 768 x 24 242.6 / 234.3; larger chunks of more query tiles: 1491 in chunks of 12 3521, of 6 2802, of 3 2704.
// Every tile that a workgroup walks behind the first fetches K and V once more, in whole lines.  Where a line holds rows of other heads too, that costs more than it saves
// unless so many workgroups still walk a head side by side that its lines are fetched no oftener than those of dense rows are when one workgroup walks all its tiles.
// us, one tile each / in chunks: [.., 4 heads, 32] 384 67.1 / 83.6 (all three in one workgroup), 512 142.5 / 135.5 (two of four), 768 445.0 / 431.0 (three of six),
// packed 512 157.8 / 144.8, 1000 994 / 1016 (four of eight) / 956 (two), 640 273 / 280 (2 2 1); 8 heads 512 x 256 90.8 / 116.7 (both); k | v of a head in whole lines 384
// 64.6 / 62.2, 1000 x 4 x 150 63.9 / 53.4, across lines 300 x 4 x 500 x 24 98.9 / 94.0 (two of four).  Rows apart from V's that lie across lines gain by no chunk (head_dim 24, packed
// 512 x 4 x 512 149.9 / 158.9 in twos, 904 x 8 x 904 1335 / 1507), nor from 9 heads on does anything but whole lines (packed 300 x 16 x 384 x 24 239.6 / 371.2, 128 x 16 x 512 x 32
// 137.9 / 149.2, 64 x 32 x 512 145.6 / 173.6, k | v across lines 128 x 16 x 512 x 24 141 / 147, 256 x 16 x 1232 x 24 1494 / 1582; with 8, packed 256 x 512 x 32 138.9 / 142.4, 200 x 512
// 126.2 / 120.9, 128 x 1024 234.6 / 235.7), nor 2 2 1 (128 x 8 x 531 x 24 99.0 / 102.9); ending in single tiles they gain from three rounds on.
void plan_chunks(const af3_dpa_params& p, int bmode, int n_qtiles, int64_t per_xcd, int& chunk, int& parts, int64_t& chunked) {
	constexpr int64_t SLOTS = 64;
	const int64_t tiles = per_xcd * n_qtiles;
	if(tiles <= SLOTS) return;   // (one round as it is)
	const kv_lines lines = lines_of_a_key(p);
	const bool     five  = n_qtiles == 5;
	if(lines.sum > lines.count && (five || p.H > 8 || (lines.apart && lines.sum > 2 * lines.count))) return;
	auto few_fetches = [&](int c) { return c * lines.sum <= n_qtiles * lines.count; };
	auto fullness    = [&](int c) {   // of the last round: 2, 1 or 0
		const int64_t last = per_xcd * ((n_qtiles + c - 1) / c) % SLOTS;
		return last == 0 || last > SLOTS * 9 / 10 ? 2 : last > SLOTS * 4 / 5 && c < 4 ? 1 : 0;
	};
	int c = five ? 2 : 1;
	for(int i = lines.apart ? 3 : 4; i >= 2; i--)
		if(n_qtiles % i == 0 && few_fetches(i) && (c == 1 || fullness(i) >= fullness(c))) c = i;
	if(c == 1) return;
	const bool whole  = fullness(c) > 0 && (!five || per_xcd * 3 <= SLOTS);
	const bool partial = tiles % SLOTS > 0 && tiles % SLOTS <= SLOTS * 9 / 10;   // the last round of single ones
	const bool enough  = five ? bmode != 3 && partial && tiles >= SLOTS * 3 : n_qtiles == 3 ? tiles * 4 >= SLOTS * 7 : c == 3 ? partial && tiles >= SLOTS * 5 :
						 n_qtiles >= 8 ? partial && tiles >= SLOTS * 3 : tiles >= SLOTS * (lines.apart ? 3 : 2);
	if(!whole && !enough) return;
	chunk = c, parts = (n_qtiles + c - 1) / c;
	chunked = whole ? per_xcd : per_xcd - (SLOTS + n_qtiles - 1) / n_qtiles;
}

// How a launch over b_count batch rows in groups of `rows` is laid out.
struct rows_launch {
	int     n_qtiles, chunk, parts, even;
	int64_t n_groups, per_xcd, chunked, blocks;
};
rows_launch lay_out(const af3_dpa_params& p, int rows, int bmode, int64_t b_count) {
	rows_launch l{};
	l.n_qtiles = (int)((p.L + 127) / 128), l.n_groups = ((b_count + rows - 1) / rows) * p.H, l.per_xcd = (l.n_groups + 7) / 8;
	l.chunk = 1, l.parts = l.n_qtiles;
	if(several_query_tiles(rows, bmode, p.gate != nullptr) && p.out_dtype == AF3_BF16) plan_chunks(p, bmode, l.n_qtiles, l.per_xcd, l.chunk, l.parts, l.chunked);
	l.blocks = (l.chunked * l.parts + (l.per_xcd - l.chunked) * l.n_qtiles) * 8;
	// Workgroups of several query tiles go evenly whatever the last round holds: it consists of single tiles or is nearly whole.  us, by age / evenly / by the rule for
	// single ones, L x 4 x L x 32: 300 40.3 / 40.0 / 40.5, 384 60.3 / 59.2 / 58.8, 400 86.8 / 87.4 / 87.7, 440 103.6 / 105.0 / 104.3, 500 121.5 / 119.1 / 118.8,
	// 600 210.4 / 209.7 / 208.6, 660 286.5 / 279.9 / 286.3, 768 388.2 / 376.8 / 380.2, 960 735 / 725 / 724, 1216 1433 / 1419 / 1436, 1300 1864 / 1831 / 1834, 1491 2576 / 2586 / 2583;
	// 5 x 16 x 2000 x 24 83.1 / 78.4 / 79.0, 12 x 16 x 1536 97.3 / 98.6 / 96.0, 16 x 16 x 1536 134.9 / 130.7 / 131.6.  Single tiles, by age / evenly: less than a round 64 x 4 x 384 x 32
	// 15.9 / 14.9, 150 x 4 x 384 x 32 27.4 / 26.4, 24 x 4 x 768 25.0 / 23.5, 80 x 4 x 768 45.1 / 44.3, of it half or less 16 x 4 x 384 11.1 / 11.3; many rounds: the grid block
	// of 512 tokens 246 / 252, 832 511.5 / 514.9; few with a short last one, by age / evenly / the last one first: 32 x 4 x 1300 84.8 / 88.1 / 83.9, 104 x 4 x 640 packed
	// 51.0 / 52.3 / 50.3, 520 x 4 x 128 20.0 / 20.0 / 19.9.
	l.even = l.chunked > 0 ? EVENLY : l.blocks <= 3 * 512 ? progress_mode(l.blocks, 512) : BY_AGE;
	return l;
}

template <int ROWS, int BMODE>
int launch_rows(const af3_dpa_params& p, int64_t b_first, int64_t b_count, hipStream_t s) {
	const rows_launch l = lay_out(p, ROWS, BMODE, b_count);
	if(l.blocks <= 0 || l.blocks > 0x7fffffffLL) return AF3_ERR_BAD_SHAPE;
	const size_t n_t_all = (size_t)((p.L + KT_R - 1) / KT_R);
	const size_t smem    = (size_t)NBUF_R * ROWS * 2 * TILE_R + (BMODE == 1 || BMODE == 3 ? 4 * 4096 : 0) + (n_t_all + 1) * ROWS * 32 * 2;
	auto         kern    = p.gate ? dpa_rows_bf16_kernel<ROWS, BMODE, true, false> : dpa_rows_bf16_kernel<ROWS, BMODE, false, false>;
	if(l.chunked > 0) {
		if constexpr(several_query_tiles(ROWS, BMODE, true))
			if(p.gate) kern = dpa_rows_bf16_kernel<ROWS, BMODE, true, true>;
		if constexpr(several_query_tiles(ROWS, BMODE, false))
			if(!p.gate) kern = dpa_rows_bf16_kernel<ROWS, BMODE, false, true>;
	}
	if(smem > 63 * 1024) {   // (the kernel's static words take 1 KB of the 64 that need no asking: smem's alignment)
		if(hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem) != hipSuccess) return AF3_ERR_LAUNCH;
	}
	hipLaunchKernelGGL(kern, dim3((unsigned)l.blocks), dim3(256), smem, s, p, l.n_qtiles, l.n_groups, b_first, b_count, l.chunk, l.parts, (int)l.chunked, l.even);
	return launch_status();
}

template <int BMODE>
int launch_rows_n(int rows, const af3_dpa_params& p, int64_t b_first, int64_t b_count, hipStream_t s) {
	return rows == 4 ? launch_rows<4, BMODE>(p, b_first, b_count, s) : rows == 3 ? launch_rows<3, BMODE>(p, b_first, b_count, s) : launch_rows<2, BMODE>(p, b_first, b_count, s);
}

}  // namespace

// Shapes the kernel takes: what dpa_mfma.hip's kernel takes (mfma_bf16_eligible, checked by the caller), and in addition
// head_dim <= 32, at least two batch rows, a length whose mask table fits beside the tile buffers, 16-byte aligned gate rows.
bool mfma_rows_eligible(const af3_dpa_params& p) {
	if(p.D > 32 || p.B < 2 || p.L > MAX_L_ROWS) return false;
	constexpr int64_t MAX_ROW_STRIDE = 1 << 24;   // (elements: 32 rows of q, gate or out are addressed with 32-bit byte offsets)
	if(p.q_stride[2] >= MAX_ROW_STRIDE || p.out_stride[2] >= MAX_ROW_STRIDE || (p.gate && p.gate_stride[2] >= MAX_ROW_STRIDE)) return false;
	if(p.gate && ((reinterpret_cast<uintptr_t>(p.gate) & 15) || p.gate_stride[0] % 8 || p.gate_stride[1] % 8 || p.gate_stride[2] % 8)) return false;
	return true;
}

// Workspace the call would use: none when the bias is better read in place (few batch rows).
int64_t mfma_rows_workspace_bytes(const af3_dpa_params& p) {
	if(!p.bias) return 0;
	if(staged_preferred(p) || (p.B < 16 && direct_bias_ok(p))) return 0;
	return rows_ws_bytes(p);
}

bool mfma_rows_can_serve(const af3_dpa_params& p) { return mfma_rows_eligible(p) && rows_bias_mode(p) >= 0; }

// Fewer than 128 batch rows whose bias this kernel can stage in place: the one-row kernel would first rewrite the whole bias
// into its workspace (a pass that so few rows do not amortise) and then stream the rewritten copy once per row; here each
// group of rows streams the original once.  Measured (one-row kernel with its rewrite / this kernel, us): 2 x 16 x 1536 x 24
// 61 / 38, 5 x 16 x 1536 x 24 79 / 67, 12 x 16 x 1536 x 24 139 / 109, 5 x 16 x 768 x 24 32 / 28, 8 x 4 x 2048 x 32 62 / 50,
// 12 x 4 x 384 x 32 21 / 17, 8 x 4 x 768 x 32 21 / 21, 16 x 4 x 768 x 32 26 / 22, 48 x 4 x 768 x 32 45 / 40,
// 16 x 16 x 1536 x 24 172 / 149, 40 x 4 x 384 x 32 22 / 18.  Not for long rows in so few workgroups that most compute units
// would stay empty (2 x 4 x 1536 x 32: 48 workgroups, 30 / 37 us: the one-row kernel splits the key axis of such rows).
bool mfma_rows_suits_a_small_batch(const af3_dpa_params& p) {
	if(!p.bias || p.B >= STAGED_MAX_B_SMALL || !staged_bias_ok(p)) return false;
	const int64_t wgs = ((p.B + 3) / 4) * p.H * ((p.L + 127) / 128);
	return wgs >= 64 || p.L < 1024;
}

// The batch is cut into groups of `rows` batch rows per wavefront, the remainder into groups of two or three (a
// remainder of one borrows from the last full group); every group of one launch has the same number of rows.  Four
// rows share a bias tile best, but what counts is how evenly the workgroups fill the GPU's 512 slots (two per
// compute unit): the launch time is about (rounds of 512 workgroups) x (rows per group) x (cost per row, which grows
// as fewer rows share a tile: measured 1 : 1.075 : 1.09 for 4 : 3 : 2 rows), and the cheapest plan is taken.  For a
// small batch the cheapest plan is often ONE launch whose last group is short (its missing rows repeat the last batch
// row and are not stored): launches run one after the other, so 3 + 2 rows in two launches of half-empty rounds take
// the time of five rows, the same five rows as 3 + (2 and a repeated one) in one launch the time of three.
static bool cut_batch(const af3_dpa_params& p, int64_t (&count)[3], int (&rows_of)[3]) {
	const int64_t B = p.B, per_row_wgs = p.H * ((p.L + 127) / 128);
	auto plan = [&](int rows, int64_t (&count)[3], int (&rows_of)[3]) -> double {
		static const double cost_per_row[5] = {0, 0, 1.09, 1.075, 1.0};
		int64_t full = B / rows, rem = B % rows;
		int     n    = 0;
		if(rem == 1 && rows > 2) {
			if(full >= 1) full -= 1, rem += rows;  // e.g. 4 + 1 -> 3 + 2
			else return 1e30;
		} else if(rem == 1) {
			return 1e30;  // (rows == 2 and an odd batch: another plan serves it)
		}
		if(full > 0) count[n] = full * rows, rows_of[n] = rows, n++;
		if(rem == 5) count[n] = 3, rows_of[n] = 3, n++, count[n] = 2, rows_of[n] = 2, n++;
		else if(rem == 4) count[n] = 2, rows_of[n] = 2, n++, count[n] = 2, rows_of[n] = 2, n++;   // (rows == 3: 3 + 1 -> 2 + 2)
		else if(rem > 0) count[n] = rem, rows_of[n] = (int)rem, n++;
		for(int i = n; i < 3; i++) count[i] = 0, rows_of[i] = 0;
		double t = 0;
		for(int i = 0; i < n; i++) {
			const int64_t wgs = ((count[i] + rows_of[i] - 1) / rows_of[i]) * per_row_wgs;
			t += (double)((wgs + 511) / 512) * rows_of[i] * cost_per_row[rows_of[i]];
		}
		return t;
	};
	for(int i = 0; i < 3; i++) count[i] = 0, rows_of[i] = 0;
	double  best = 1e30;
	for(int rows = 4; rows >= 2; rows--) {
		int64_t c[3];
		int     r[3];
		const double t = plan(rows, c, r);
		if(t < best * 0.999) {
			best = t;
			for(int i = 0; i < 3; i++) count[i] = c[i], rows_of[i] = r[i];
		}
		if(B % rows != 0) {   // one launch, last group short
			static const double cost_per_row[5] = {0, 0, 1.09, 1.075, 1.0};
			const int64_t wgs = ((B + rows - 1) / rows) * per_row_wgs;
			const double  t1  = (double)((wgs + 511) / 512) * rows * cost_per_row[rows];
			if(t1 < best * 0.999) {
				best = t1;
				count[0] = B, rows_of[0] = rows;
				count[1] = count[2] = 0, rows_of[1] = rows_of[2] = 0;
			}
		}
	}
	return best < 1e30;
}

int launch_dpa_mfma_rows(const af3_dpa_params& p, hipStream_t s) {
	const int mode = rows_bias_mode(p);
	if(mode < 0) return AF3_ERR_BAD_ARGUMENT;
	if(mode == 1) {
		const bool     bf32      = p.bias_dtype == AF3_F32;
		const int      n_qblocks = (int)((p.L + 31) / 32), n_t_all = (int)((p.L + KT_R - 1) / KT_R);
		const int64_t  total     = p.H * n_qblocks * (int64_t)n_t_all * 256;
		if(total / 256 >= ((int64_t)1 << 31)) return AF3_ERR_BAD_SHAPE;  // (the prepass counts its units in 32 bits)
		const unsigned g         = (unsigned)((total + 255) / 256 > 65536 ? 65536 : (total + 255) / 256);
		if(bf32)
			hipLaunchKernelGGL(bias_rows_prepass_kernel<true>, dim3(g), dim3(256), 0, s, p.bias, static_cast<f32x4*>(p.workspace), p.H, p.L, p.bias_stride[0], p.bias_stride[1],
							   n_qblocks, n_t_all);
		else
			hipLaunchKernelGGL(bias_rows_prepass_kernel<false>, dim3(g), dim3(256), 0, s, p.bias, static_cast<f32x4*>(p.workspace), p.H, p.L, p.bias_stride[0], p.bias_stride[1],
							   n_qblocks, n_t_all);
		const int rc = launch_status();
		if(rc != AF3_OK) return rc;
	}
	int64_t count[3];
	int     rows_of[3];
	if(!cut_batch(p, count, rows_of)) return AF3_ERR_BAD_SHAPE;  // (B == 1 is not eligible)
	int64_t done = 0;
	for(int i = 0; i < 3; i++) {
		if(count[i] == 0) continue;
		const int rc = mode == 0 ? launch_rows_n<0>(rows_of[i], p, done, count[i], s) : mode == 1 ? launch_rows_n<1>(rows_of[i], p, done, count[i], s) : mode == 2 ? launch_rows_n<2>(rows_of[i], p, done, count[i], s) : launch_rows_n<3>(rows_of[i], p, done, count[i], s);
		if(rc != AF3_OK) return rc;
		done += count[i];
	}
	return AF3_OK;
}

int mfma_rows_plan(const af3_dpa_params& p, int64_t (&plan)[3][6]) {
	int64_t count[3];
	int     rows_of[3], n = 0;
	const int mode = rows_bias_mode(p);
	if(mode < 0 || !cut_batch(p, count, rows_of)) return 0;
	for(int i = 0; i < 3; i++) {
		if(count[i] == 0) continue;
		const rows_launch l = lay_out(p, rows_of[i], mode, count[i]);
		const int64_t     what[6] = {rows_of[i], mode, count[i], l.chunked > 0 ? l.chunk : 1, l.chunked * 8 < l.n_groups ? l.chunked * 8 : l.n_groups, l.even};
		for(int j = 0; j < 6; j++) plan[n][j] = what[j];
		n++;
	}
	return n;
}

}  // namespace af3
