// Device helpers shared by the matrix-core attention kernels (dpa_mfma.hip, dpa_mfma_rows.hip, dpa_strip.hip, dpa_mfma_fp8.hip, dpa_mfma_f32.hip).
#pragma once
#include <type_traits>

#include "common.hpp"

namespace af3 {

constexpr int   KT         = 64;       // keys per tile (dpa_mfma.hip)
constexpr int   MAX_L_MFMA = 8192;     // mask table (4 B/key) and tile list live in LDS
constexpr float REF_SLACK  = 12.f;     // log2 units: a moved reference sits this close to the row maximum
constexpr float PSUM_LIMIT = 0x1p30f;  // per-lane row-sum bound that triggers the rare path

typedef __attribute__((ext_vector_type(2))) __bf16   bf16x2;
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;
typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
// vectors at any element's address (global memory takes them; the compiler must be told not to split the access)
typedef __attribute__((ext_vector_type(4), aligned(2))) uint32_t u32x4_any;
typedef __attribute__((ext_vector_type(2), aligned(2))) uint32_t u32x2_any;
typedef __attribute__((ext_vector_type(4), aligned(4))) float    f32x4_any;
typedef __attribute__((aligned(1))) uint32_t u32_bytes;
typedef __attribute__((ext_vector_type(2))) unsigned short u16x2;
template <int V>
using ic = std::integral_constant<int, V>;

// Wavefronts that share a SIMD are served oldest first: of four equal workgroups of a compute unit that start together the first is done after little more
// than half the time (32, 41, 49 and 57 us in the fp8 kernel at 5 x 16 x 1536 x 24) and the last one walks its end alone, which keeps no pipe busy.  A
// wavefront that lowers its priority with every quarter of its walk lets those behind it catch up; they end together ...
struct even_progress {   // from: EVENLY, BY_AGE or the first workgroup that goes before all others (below)
	int quarter, next, level;
	__device__ __forceinline__ even_progress(int steps, int from) : quarter((steps + 3) >> 2), next(from < 0 ? quarter : 0x7fffffff), level(3) {
		if(from < 0 || (from != 0x7fffffff && (int)blockIdx.x >= from)) __builtin_amdgcn_s_setprio(3);
	}
	__device__ __forceinline__ void at(int step) {   // (wave-uniform)
		if(step >= next) {
			next += quarter, level--;
			if(level == 2) __builtin_amdgcn_s_setprio(2);
			else if(level == 1) __builtin_amdgcn_s_setprio(1);
			else __builtin_amdgcn_s_setprio(0);
		}
	}
};
// ... in launches of whole rounds of workgroups, or with a last one that is more than half full.  Workgroups that end together leave a short last round nothing to
// overlap with: there the earlier rounds go by age, so that places come free one after the other, and the workgroups of the last round, the last to
// start, go before all others on their SIMD.  By rounds (1024 workgroups each), us, of the fp32 kernel (B x 4 x 768 x 32) by age / evenly: 0.94 85.7 / 82.4,
// 1.03 106.0 / 112.2, 1.69 149.0 / 145.3, 1.88 166.3 / 160.9, 3.0 258.0 / 251.4; by age / last round first: 1.03 105.3 / 97.8, 1.13 105.8 / 99.3;
// evenly / last round first: 1.31 120.0 / 119.7, 1.41 123.1 / 122.8, 1.5 128.0 / 127.1, 1.69 149.3 / 149.3, 1.78 155.0 / 163.8, 1.88 159.6 / 171.7,
// 2.34 205.6 / 202.2, 2.58 221.0 / 225.5.  Of the fp8 kernel (B x 16 x 1536 x 24) by age / evenly: 0.94 68.6 / 64.4; by age / last round first: 1.13 81.6 / 76.1,
// 2.25 139.4 / 137.3; evenly / last round first: 1.31 92.0 / 90.5, 1.5 96.5 / 95.7, 1.88 116.7 / 123.3, 2.44 152.3 / 148.1.
constexpr int EVENLY = -1, BY_AGE = 0x7fffffff;
// (A launch of at most half a round has no earlier round: its wavefronts keep the priority that every other kernel's have.  The padding of a grid lies at its end, so
// that the last round begins where its real workgroups do, or a few behind.)
inline int progress_mode(int64_t workgroups, int64_t slots) {   // EVENLY, BY_AGE or the first workgroup of the last round
	if(workgroups * 2 <= slots) return BY_AGE;
	const int64_t last = workgroups % slots;
	return last == 0 || last * 2 > slots ? EVENLY : (int)(workgroups - last);
}

// ---- LDS layout -----------------------------------------------------------------------------
// K tile: [KT rows][DP cols] bf16; the 16-byte chunks of a row are XOR-swizzled so that the 8
// lanes served in one LDS cycle of a ds_read_b128 (8 consecutive rows, same logical chunk) hit
// distinct banks.  The swizzle only depends on row % 8.
template <int DP>
__device__ __forceinline__ int k_swizzle(int row) {
	return (DP == 32) ? ((row >> 1) & 3) : (row & 7);
}
// V tile: [KT rows][DP cols] bf16 row-major; for DP = 64 the two 64-byte halves of a row are
// swapped on odd rows (keeps the transposed reads of 8 rows x 64 B spread over all banks).
template <int DP>
__device__ __forceinline__ int v_swizzle(int row) {  // in 16-byte chunks
	return (DP == 64) ? ((row & 1) << 2) : 0;
}

__device__ __forceinline__ float half_swap_max(float x) {
	// lanes l and l^32 exchange; v_permlane32_swap swaps the upper half of one operand with the
	// lower half of the other, so (x, x) yields {low|low} and {high|high}.
	auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
	return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// ---- key masks, four keep bytes to a word ----
// what a load at `key + 4 <= L ? key : L - 4` brought for keys from `key` on, `over` = key + 4 - L: zeros from L on
__device__ __forceinline__ uint32_t keep_bytes_in_row(uint32_t m, int over) {
	if(over > 0) m = over < 4 ? m >> (8 * over) : 0u;
	return m;
}
// 1 in the bytes that are not zero, and in those that are
__device__ __forceinline__ uint32_t live_bytes(uint32_t m) { return ((((m & 0x7f7f7f7fu) + 0x7f7f7f7fu) | m) >> 7) & 0x01010101u; }
__device__ __forceinline__ uint32_t gone_bytes(uint32_t m) { return (~(((m & 0x7f7f7f7fu) + 0x7f7f7f7fu) | m) >> 7) & 0x01010101u; }
// the additive mask values of four keys, as bf16
__device__ __forceinline__ u32x2 mask_values_bf16(uint32_t gone, int over) {
	constexpr uint32_t OUT = MASK_OUT_OF_RANGE_BF16;   // keys from L on
	uint32_t           lo = ((gone & 1u) | ((gone & 0x100u) << 8)) * MASK_DROPPED_BF16, hi = (((gone >> 16) & 1u) | ((gone >> 24) << 16)) * MASK_DROPPED_BF16;
	if(over > 0) {
		lo = over <= 2 ? lo : over == 3 ? (lo & 0xffffu) | (OUT << 16) : OUT | (OUT << 16);
		hi = over == 1 ? (hi & 0xffffu) | (OUT << 16) : OUT | (OUT << 16);
	}
	return u32x2{lo, hi};
}
// two biases, limited from below: as unsigned numbers every negative bf16 beyond the limit, -inf and negative NaN included, is larger
__device__ __forceinline__ uint32_t bias_limited(uint32_t x, uint32_t lim) {
	return __builtin_bit_cast(uint32_t, __builtin_elementwise_min(__builtin_bit_cast(u16x2, x), __builtin_bit_cast(u16x2, lim)));
}

// 16 bytes per lane from a raw buffer straight into LDS (lane i lands at lds_addr + 16*i).  Written as
// inline assembly on purpose: the compiler makes every LDS read that follows an LDS-direct load it
// knows about wait for vmcnt(0), which exposes the whole latency of every tile load when only one or
// two wavefronts share a SIMD.  Loads issued here are invisible to it; the kernel orders them itself
// (explicit s_waitcnt vmcnt before the barrier that publishes a tile).  rsrc and lds_addr must be
// wave-uniform.  The whole byte offset travels in the vector operand, which the hardware range-checks
// against the buffer size: a lane whose offset is past the end fetches nothing from memory.
// M0 (the LDS base of the load) is written behind the compiler's back.  It cannot be declared: the compiler treats
// M0 as a reserved register and answers an "m0" clobber with a warning that it is ignored.  What keeps this safe is
// that nothing else in this file makes the compiler use M0 -- no LDS-direct builtins, no indirect register indexing,
// no message or GWS instructions -- and gfx950's LDS instructions do not read it.
__device__ __forceinline__ void lds_dma_b128(const u32x4& rsrc, uint32_t lds_addr, int voff) {
	asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds_addr), "v"(voff), "s"(rsrc) : "memory");
}
// ... 4 bytes per lane (lane i lands at lds_addr + 4*i)
__device__ __forceinline__ void lds_dma_b32(const u32x4& rsrc, uint32_t lds_addr, int voff) {
	asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, 0 offen lds" ::"s"(lds_addr), "v"(voff), "s"(rsrc) : "memory");
}
__device__ __forceinline__ u32x4 raw_rsrc(const void* base, uint32_t bytes) {
	const uint64_t a = reinterpret_cast<uint64_t>(base);
	return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a), (uint32_t)__builtin_amdgcn_readfirstlane((int)((uint32_t)(a >> 32) & 0xFFFFu)),
				 (uint32_t)__builtin_amdgcn_readfirstlane((int)bytes), 0x00020000u};
}
__device__ __forceinline__ uint32_t lds_addr_of(const void* ptr) {
	return (uint32_t)(uintptr_t)((__attribute__((address_space(3))) const void*)ptr);
}

}  // namespace af3
