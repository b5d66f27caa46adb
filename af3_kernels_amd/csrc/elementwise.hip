// Vectorised element-wise kernels: dtype casts, per-tensor fp8 scaling, pad and VNNI repack.
//
// Casts replace tpp::ConvertTPP and the AVX-512 converters of the reference
// (src/csrc/xsmm_functors.h:139-145, :838-885).  The e4m3 path has no reference behaviour to
// follow (src/csrc/xsmm_functors.h:218-226 asserts "not implemented"); it implements OCP e4m3fn
// with round-to-nearest-even and saturation, which is what gfx950's v_cvt_pk_fp8_f32 does.
#include <algorithm>
#include <type_traits>

#include "common.hpp"

namespace af3 {

constexpr int EW_THREADS = 256;

static inline unsigned ew_blocks(int64_t work_items, int64_t cap = 256 * 64) {
	int64_t b = (work_items + EW_THREADS - 1) / EW_THREADS;
	if(b < 1) b = 1;
	return (unsigned)(b > cap ? cap : b);
}

// ---- f32 <-> bf16 ----------------------------------------------------------------------------
__global__ void __launch_bounds__(EW_THREADS) cvt_f32_bf16_kernel(const float* __restrict__ src, uint16_t* __restrict__ dst, int64_t n) {
	const int64_t stride = (int64_t)gridDim.x * EW_THREADS;
	const int64_t nvec   = n >> 3;
	const bool    vec    = ((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 15) == 0;
	int64_t       done   = 0;
	if(vec) {
		for(int64_t i = (int64_t)blockIdx.x * EW_THREADS + threadIdx.x; i < nvec; i += stride) {
			const float4 a = reinterpret_cast<const float4*>(src)[2 * i], c = reinterpret_cast<const float4*>(src)[2 * i + 1];
			u32x4        o = {pack_bf16x2(a.x, a.y), pack_bf16x2(a.z, a.w), pack_bf16x2(c.x, c.y), pack_bf16x2(c.z, c.w)};
			reinterpret_cast<u32x4*>(dst)[i] = o;
		}
		done = nvec << 3;
	}
	for(int64_t i = done + (int64_t)blockIdx.x * EW_THREADS + threadIdx.x; i < n; i += stride) dst[i] = (uint16_t)f32_to_bf16_bits(src[i]);
}

__global__ void __launch_bounds__(EW_THREADS) cvt_bf16_f32_kernel(const uint16_t* __restrict__ src, float* __restrict__ dst, int64_t n) {
	const int64_t stride = (int64_t)gridDim.x * EW_THREADS;
	const int64_t nvec   = n >> 3;
	const bool    vec    = ((reinterpret_cast<uintptr_t>(src) | reinterpret_cast<uintptr_t>(dst)) & 15) == 0;
	int64_t       done   = 0;
	if(vec) {
		for(int64_t i = (int64_t)blockIdx.x * EW_THREADS + threadIdx.x; i < nvec; i += stride) {
			const u32x4 a = reinterpret_cast<const u32x4*>(src)[i];
			float4      lo = {bf16_bits_to_f32(a[0] & 0xffffu), bf16_bits_to_f32(a[0] >> 16), bf16_bits_to_f32(a[1] & 0xffffu), bf16_bits_to_f32(a[1] >> 16)};
			float4      hi = {bf16_bits_to_f32(a[2] & 0xffffu), bf16_bits_to_f32(a[2] >> 16), bf16_bits_to_f32(a[3] & 0xffffu), bf16_bits_to_f32(a[3] >> 16)};
			reinterpret_cast<float4*>(dst)[2 * i]     = lo;
			reinterpret_cast<float4*>(dst)[2 * i + 1] = hi;
		}
		done = nvec << 3;
	}
	for(int64_t i = done + (int64_t)blockIdx.x * EW_THREADS + threadIdx.x; i < n; i += stride) dst[i] = bf16_bits_to_f32(src[i]);
}

// ---- e4m3 -> f32 / bf16 ----------------------------------------------------------------------
template <bool TO_BF16>
__global__ void __launch_bounds__(EW_THREADS) cvt_e4m3_kernel(const uint8_t* __restrict__ src, void* __restrict__ dst, int64_t n) {
	const int64_t stride = (int64_t)gridDim.x * EW_THREADS;
	const int64_t nvec   = n >> 2;
	const bool    vec    = ((reinterpret_cast<uintptr_t>(src) & 3) | (reinterpret_cast<uintptr_t>(dst) & 15)) == 0;
	int64_t       done   = 0;
	if(vec) {
		for(int64_t i = (int64_t)blockIdx.x * EW_THREADS + threadIdx.x; i < nvec; i += stride) {
			const uint32_t w  = reinterpret_cast<const uint32_t*>(src)[i];
			const auto     lo = __builtin_amdgcn_cvt_pk_f32_fp8(w, false);
			const auto     hi = __builtin_amdgcn_cvt_pk_f32_fp8(w, true);
			if(TO_BF16) {
				u32x2 o = {pack_bf16x2(lo[0], lo[1]), pack_bf16x2(hi[0], hi[1])};
				reinterpret_cast<u32x2*>(dst)[i] = o;
			} else {
				float4 o = {lo[0], lo[1], hi[0], hi[1]};
				reinterpret_cast<float4*>(dst)[i] = o;
			}
		}
		done = nvec << 2;
	}
	for(int64_t i = done + (int64_t)blockIdx.x * EW_THREADS + threadIdx.x; i < n; i += stride) {
		const float f = __builtin_amdgcn_cvt_pk_f32_fp8((uint32_t)src[i], false)[0];
		if(TO_BF16) static_cast<uint16_t*>(dst)[i] = (uint16_t)f32_to_bf16_bits(f);
		else static_cast<float*>(dst)[i] = f;
	}
}

// ---- e5m2 (OCP float8 e5m2: fp16's exponent range with two mantissa bits; infinities and NaN like IEEE) ---------------
// fp32 -> e5m2 bits, round to nearest even straight from fp32 (one rounding), overflow to infinity: what torch.float8_e5m2
// does.  (The reference's AVX-512 helper _mm_convert_ps_bf8, src/csrc/xsmm_functors.h:214-217, rounds to fp16 first and then
// drops the low mantissa byte, i.e. rounds twice, the second time towards zero.)
__device__ __forceinline__ uint32_t f32_to_e5m2_bits(float f) {
	uint32_t       u    = __float_as_uint(f);
	const uint32_t sign = (u >> 24) & 0x80u;
	u &= 0x7fffffffu;
	uint32_t r;
	if(u >= (143u << 23)) r = u > 0x7f800000u ? 0x7fu : 0x7cu;          // |x| >= 2^16, infinity, NaN
	else if(u < (113u << 23)) r = __float_as_uint(__uint_as_float(u) + __uint_as_float(134u << 23)) - (134u << 23);   // below 2^-14: the adder rounds to the subnormal grid 2^-16
	else r = (u + ((uint32_t)(15 - 127) << 23) + 0xfffffu + ((u >> 21) & 1u)) >> 21;
	return r | sign;
}

template <bool SRC_BF16>
__global__ void __launch_bounds__(EW_THREADS) cvt_to_e5m2_kernel(const void* __restrict__ src, uint8_t* __restrict__ dst, int64_t n) {
	const int64_t stride = (int64_t)gridDim.x * EW_THREADS;
	const int64_t nvec   = n >> 2;
	const bool    vec    = ((reinterpret_cast<uintptr_t>(src) & (SRC_BF16 ? 7 : 15)) | (reinterpret_cast<uintptr_t>(dst) & 3)) == 0;
	int64_t       done   = 0;
	if(vec) {
		for(int64_t i = (int64_t)blockIdx.x * EW_THREADS + threadIdx.x; i < nvec; i += stride) {
			float f[4];
			if(SRC_BF16) {
				const u32x2 w = static_cast<const u32x2*>(src)[i];
				f[0] = bf16_bits_to_f32(w[0] & 0xffffu), f[1] = bf16_bits_to_f32(w[0] >> 16), f[2] = bf16_bits_to_f32(w[1] & 0xffffu), f[3] = bf16_bits_to_f32(w[1] >> 16);
			} else {
				const float4 w = static_cast<const float4*>(src)[i];
				f[0] = w.x, f[1] = w.y, f[2] = w.z, f[3] = w.w;
			}
			reinterpret_cast<uint32_t*>(dst)[i] = f32_to_e5m2_bits(f[0]) | (f32_to_e5m2_bits(f[1]) << 8) | (f32_to_e5m2_bits(f[2]) << 16) | (f32_to_e5m2_bits(f[3]) << 24);
		}
		done = nvec << 2;
	}
	for(int64_t i = done + (int64_t)blockIdx.x * EW_THREADS + threadIdx.x; i < n; i += stride)
		dst[i] = (uint8_t)f32_to_e5m2_bits(SRC_BF16 ? bf16_bits_to_f32(static_cast<const uint16_t*>(src)[i]) : static_cast<const float*>(src)[i]);
}

// e5m2 -> f32 / bf16: the byte is the upper half of the fp16 pattern of the same value (src/csrc/xsmm_functors.h:211-213);
// exact in both targets (two mantissa bits)
template <bool TO_BF16>
__global__ void __launch_bounds__(EW_THREADS) cvt_e5m2_kernel(const uint8_t* __restrict__ src, void* __restrict__ dst, int64_t n) {
	const int64_t stride = (int64_t)gridDim.x * EW_THREADS;
	for(int64_t i = (int64_t)blockIdx.x * EW_THREADS + threadIdx.x; i < n; i += stride) {
		const _Float16 h = __builtin_bit_cast(_Float16, (uint16_t)((uint16_t)src[i] << 8));
		const float    f = (float)h;
		if(TO_BF16) static_cast<uint16_t*>(dst)[i] = (uint16_t)f32_to_bf16_bits(f);
		else static_cast<float*>(dst)[i] = f;
	}
}

// maximum over a wavefront, in every lane: without the cross-lane network of LDS, whose six passes are a chain of 700 clocks
__device__ __forceinline__ float wave_max(float a) {
	auto dpp = [&](auto ctrl) { a = fmaxf(a, __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(a), decltype(ctrl)::value, 0xf, 0xf, true))); };
	dpp(std::integral_constant<int, 0xB1>{});    // lane ^ 1
	dpp(std::integral_constant<int, 0x4E>{});    // lane ^ 2
	dpp(std::integral_constant<int, 0x141>{});   // mirrored within 8
	dpp(std::integral_constant<int, 0x140>{});   // mirrored within 16
	const auto x = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(a), false, false);
	a            = fmaxf(__uint_as_float(x[0]), __uint_as_float(x[1]));
	const auto y = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(a), false, false);
	return fmaxf(__uint_as_float(y[0]), __uint_as_float(y[1]));
}

// ---- per-tensor amax -------------------------------------------------------------------------
// 16-byte loads, wave then workgroup reduction, one atomic per workgroup (a few hundred atomics on
// the one result word instead of one per wavefront).
// maximum of |src[i]| over this workgroup's grid-stride share; valid in thread 0
template <bool SRC_BF16>
__device__ __forceinline__ float block_amax(const void* __restrict__ src, int64_t n) {
	__shared__ float part[EW_THREADS / 64];
	const int64_t stride = (int64_t)gridDim.x * EW_THREADS, tid0 = (int64_t)blockIdx.x * EW_THREADS + threadIdx.x;
	constexpr int PER  = SRC_BF16 ? 8 : 4;  // elements per 16-byte load
	const bool    vec  = (reinterpret_cast<uintptr_t>(src) & 15) == 0;
	const int64_t nvec = vec ? n / PER : 0;
	float         a    = 0.f;  // fmaxf drops NaN operands: a NaN element does not poison the scale
	// four loads under way at a time (one memory latency for all): trips past the end repeat the thread's first element
	for(int64_t i = tid0; i < nvec; i += 4 * stride) {
		u32x4 w[4];
#pragma unroll
		for(int u = 0; u < 4; u++) w[u] = static_cast<const u32x4*>(src)[i + u * stride < nvec ? i + u * stride : i];
#pragma unroll
		for(int u = 0; u < 4; u++)
#pragma unroll
			for(int j = 0; j < 4; j++) {
				if(SRC_BF16) a = fmaxf(a, fmaxf(fabsf(bf16_bits_to_f32(w[u][j] & 0xffffu)), fabsf(bf16_bits_to_f32(w[u][j] >> 16))));
				else a = fmaxf(a, fabsf(__uint_as_float(w[u][j])));
			}
	}
	for(int64_t i = nvec * PER + tid0; i < n; i += stride) {
		const float f = SRC_BF16 ? bf16_bits_to_f32(static_cast<const uint16_t*>(src)[i]) : static_cast<const float*>(src)[i];
		a = fmaxf(a, fabsf(f));
	}
	a = wave_max(a);
	if((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = a;
	__syncthreads();
	if(threadIdx.x == 0)
		for(int w = 1; w < EW_THREADS / 64; w++) a = fmaxf(a, part[w]);
	return a;
}

template <bool SRC_BF16>
__global__ void __launch_bounds__(EW_THREADS) amax_kernel(const void* __restrict__ src, int64_t n, float* amax_out) {
	const float a = block_amax<SRC_BF16>(src, n);
	// non-negative floats order like their bit patterns
	if(threadIdx.x == 0) atomicMax(reinterpret_cast<unsigned int*>(amax_out), __float_as_uint(a));
}

// Three tensors in one launch (blockIdx.y), every workgroup storing its partial maximum: no atomics,
// nothing to clear beforehand.  partials: [3][AMAX3_BLOCKS].
constexpr int AMAX3_BLOCKS = 256;
struct Amax3Args {
	const void* src[3];
	int64_t     n[3];
};
template <bool SRC_BF16>
__global__ void __launch_bounds__(EW_THREADS) amax3_kernel(Amax3Args a, float* __restrict__ partials) {
	const int   t = blockIdx.y;
	const float m = block_amax<SRC_BF16>(a.src[t], a.n[t]);
	if(threadIdx.x == 0) partials[t * AMAX3_BLOCKS + blockIdx.x] = m;
}

// scale = 2^floor(log2(448 / (amax*pre_scale))); the power of two keeps every descale product exact.
__device__ __forceinline__ float fp8_pow2_scale(float amax, float pre_scale) {
	const float a = amax * fabsf(pre_scale);
	if(!(a > 0.f) || !(a < INFINITY)) return 1.f;
	int e;
	frexpf(448.f / a, &e);             // 448/a = m * 2^e with m in [0.5, 1)  ->  floor(log2) = e - 1
	e = e - 1;
	e = e > 120 ? 120 : (e < -120 ? -120 : e);
	return ldexpf(1.f, e);
}

// multiplier(): pre_scale * scale, called once, behind the first loads (what it takes to find the scale runs under their latency)
template <bool SRC_BF16, typename Multiplier>
__device__ __forceinline__ void quantize_e4m3_body(const void* __restrict__ src, uint8_t* __restrict__ dst, int64_t rows, int64_t cols, int64_t src_row_stride,
													 int transpose, int64_t rows_per_matrix, int64_t dst_row_stride, Multiplier multiplier,
													 uint8_t* __restrict__ dst_lo) {
	float         mul    = 0.f;
	const int64_t stride = (int64_t)gridDim.x * EW_THREADS;
	auto          ld     = [&](int64_t r, int64_t c) -> float {
        const int64_t i = r * src_row_stride + c;
        const float   f = SRC_BF16 ? bf16_bits_to_f32(static_cast<const uint16_t*>(src)[i]) : static_cast<const float*>(src)[i];
        return fminf(fmaxf(f * mul, -448.f), 448.f);
	};
	// residual word: e4m3 of (scaled value - decoded hi), the rounding error of hi at the same scale
	auto residual = [&](float f0, float f1, float f2, float f3, uint32_t hi) -> uint32_t {
		const auto lo01 = __builtin_amdgcn_cvt_pk_f32_fp8(hi, false), lo23 = __builtin_amdgcn_cvt_pk_f32_fp8(hi, true);
		uint32_t   w    = 0;
		w = __builtin_amdgcn_cvt_pk_fp8_f32(f0 - lo01[0], f1 - lo01[1], w, false);
		w = __builtin_amdgcn_cvt_pk_fp8_f32(f2 - lo23[0], f3 - lo23[1], w, true);
		return w;
	};
	if(!transpose && src_row_stride == cols && dst_row_stride == cols && (reinterpret_cast<uintptr_t>(src) & 15) == 0 && (reinterpret_cast<uintptr_t>(dst) & 7) == 0 &&
	   (!dst_lo || (reinterpret_cast<uintptr_t>(dst_lo) & 7) == 0) && rows * cols < ((int64_t)1 << 31)) {
		// dense rows on both sides: the tensor is one run of elements; one thread = 8 consecutive elements (16- or 2 x 16-byte
		// loads, 8-byte stores), no index arithmetic beyond the running offset
		const int total8 = (int)((rows * cols) >> 3), step = (int)stride;
		constexpr int NV = SRC_BF16 ? 1 : 2;
		u32x4         w[NV], w_next[NV];
		auto          load = [&](int i, u32x4 (&to)[NV]) {
#pragma unroll
			for(int u = 0; u < NV; u++) to[u] = static_cast<const u32x4*>(src)[NV * (i < total8 ? i : 0) + u];   // (total8 > 0, or the loop does not run)
		};
		const int i0 = (int)(blockIdx.x * EW_THREADS + threadIdx.x);
		if(total8 > 0) load(i0, w_next);
		mul = multiplier();
		for(int i = i0; i < total8; i += step) {
			float f[8];
#pragma unroll
			for(int u = 0; u < NV; u++) w[u] = w_next[u];
			load(i < total8 - step ? i + step : 0, w_next);
			if constexpr(SRC_BF16) {
#pragma unroll
				for(int j = 0; j < 4; j++) f[2 * j] = bf16_bits_to_f32(w[0][j] & 0xffffu), f[2 * j + 1] = bf16_bits_to_f32(w[0][j] >> 16);
			} else {
#pragma unroll
				for(int j = 0; j < 4; j++) f[j] = __uint_as_float(w[0][j]), f[4 + j] = __uint_as_float(w[NV - 1][j]);
			}
#pragma unroll
			for(int j = 0; j < 8; j++) f[j] = fminf(fmaxf(f[j] * mul, -448.f), 448.f);
			uint32_t w0 = 0, w1 = 0;
			w0 = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], w0, false), w0 = __builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], w0, true);
			w1 = __builtin_amdgcn_cvt_pk_fp8_f32(f[4], f[5], w1, false), w1 = __builtin_amdgcn_cvt_pk_fp8_f32(f[6], f[7], w1, true);
			reinterpret_cast<u32x2*>(dst)[i] = u32x2{w0, w1};
			if(dst_lo) reinterpret_cast<u32x2*>(dst_lo)[i] = u32x2{residual(f[0], f[1], f[2], f[3], w0), residual(f[4], f[5], f[6], f[7], w1)};
		}
		// (a tail of 4 elements when rows * cols is not a multiple of 8: cols % 4 == 0 is checked by the launcher)
		if(((rows * cols) & 7) && blockIdx.x == 0 && threadIdx.x == 0) {
			const int64_t e0 = (rows * cols) & ~(int64_t)7;
			const float   f0 = ld(0, e0), f1 = ld(0, e0 + 1), f2 = ld(0, e0 + 2), f3 = ld(0, e0 + 3);
			uint32_t      w  = 0;
			w = __builtin_amdgcn_cvt_pk_fp8_f32(f0, f1, w, false), w = __builtin_amdgcn_cvt_pk_fp8_f32(f2, f3, w, true);
			*reinterpret_cast<uint32_t*>(dst + e0) = w;
			if(dst_lo) *reinterpret_cast<uint32_t*>(dst_lo + e0) = residual(f0, f1, f2, f3, w);
		}
	} else if(!transpose) {
		// one thread = 4 consecutive columns of one row (cols % 4 == 0 is checked by the launcher)
		mul = multiplier();
		const int64_t cq = cols >> 2, total = rows * cq;
		for(int64_t i = (int64_t)blockIdx.x * EW_THREADS + threadIdx.x; i < total; i += stride) {
			const int64_t r = i / cq, c = (i % cq) << 2;
			const float   f0 = ld(r, c), f1 = ld(r, c + 1), f2 = ld(r, c + 2), f3 = ld(r, c + 3);
			uint32_t      w = 0;
			w = __builtin_amdgcn_cvt_pk_fp8_f32(f0, f1, w, false);
			w = __builtin_amdgcn_cvt_pk_fp8_f32(f2, f3, w, true);
			*reinterpret_cast<uint32_t*>(dst + r * dst_row_stride + c) = w;
			if(dst_lo) *reinterpret_cast<uint32_t*>(dst_lo + r * dst_row_stride + c) = residual(f0, f1, f2, f3, w);
		}
	} else {
		// one thread = 4 consecutive rows of one column, written as 4 consecutive bytes of dst[matrix][col][row..row+3];
		// rows past the end of a matrix quantise to zero, and the whole padded length of every output row
		// (dst_row_stride, a multiple of 4) is written, so the destination needs no clearing beforehand
		const int64_t rq = dst_row_stride >> 2, n_mat = rows / rows_per_matrix, total = n_mat * rq * cols;
		// (index arithmetic in 32 bits when the count allows: 64-bit divisions cost several times the rest of the body)
		auto element = [&](auto i, auto cols_i, auto rq_i) {
			const auto    c    = i % cols_i;
			const auto    r4   = (i / cols_i) % rq_i;
			const int64_t mat  = i / (cols_i * rq_i);
			const int64_t r    = mat * rows_per_matrix + ((int64_t)r4 << 2);
			const int64_t left = rows_per_matrix - ((int64_t)r4 << 2);
			const float   f0 = left > 0 ? ld(r, c) : 0.f, f1 = left > 1 ? ld(r + 1, c) : 0.f, f2 = left > 2 ? ld(r + 2, c) : 0.f, f3 = left > 3 ? ld(r + 3, c) : 0.f;
			uint32_t      w   = 0;
			w = __builtin_amdgcn_cvt_pk_fp8_f32(f0, f1, w, false);
			w = __builtin_amdgcn_cvt_pk_fp8_f32(f2, f3, w, true);
			*reinterpret_cast<uint32_t*>(dst + (mat * cols + c) * dst_row_stride + ((int64_t)r4 << 2)) = w;
			if(dst_lo) *reinterpret_cast<uint32_t*>(dst_lo + (mat * cols + c) * dst_row_stride + ((int64_t)r4 << 2)) = residual(f0, f1, f2, f3, w);
		};
		if(SRC_BF16 && cols % 8 == 0 && src_row_stride % 8 == 0 && (reinterpret_cast<uintptr_t>(src) & 15) == 0 && total < ((int64_t)1 << 29) && stride < ((int64_t)1 << 30)) {
			// bf16 rows of whole 16-byte chunks: one thread = 4 consecutive rows x 8 consecutive columns (four 16-byte loads, eight
			// 4-byte stores).  Consecutive lanes take consecutive row quads, so each store instruction of a wavefront writes 256
			// consecutive bytes of one output row; consecutive wavefronts take the column blocks of the same 64 row quads, so
			// the rows they share are fetched by one compute unit (in different workgroups they would be fetched once per XCD).
			const uint32_t cb_n = (uint32_t)(cols >> 3), rq_u = (uint32_t)rq, rq_b = (rq_u + 63) >> 6, items = (uint32_t)n_mat * rq_b * cb_n * 64;
			bool first = true;
			for(uint32_t i = blockIdx.x * EW_THREADS + threadIdx.x; i < items; i += (uint32_t)stride) {
				const uint32_t wi = i >> 6, cb = wi % cb_n, r4 = ((wi / cb_n) % rq_b) * 64 + (i & 63);
				const int64_t  mat = wi / (cb_n * rq_b), r = mat * rows_per_matrix + ((int64_t)r4 << 2), left = rows_per_matrix - ((int64_t)r4 << 2);
				u32x4          w[4];
#pragma unroll
				for(int k = 0; k < 4; k++) {
					w[k] = u32x4{0u, 0u, 0u, 0u};
					if(left > k) w[k] = *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(src) + (r + k) * src_row_stride + (cb << 3));
				}
				if(first) mul = multiplier();   // (a wavefront's lanes run the same trips: items is a multiple of 64)
				first = false;
				if(r4 >= rq_u) continue;
				uint8_t* const d0 = dst + (mat * cols + (cb << 3)) * dst_row_stride + ((int64_t)r4 << 2);
#pragma unroll
				for(int j = 0; j < 8; j++) {
					float f[4];
#pragma unroll
					for(int k = 0; k < 4; k++) {
						const float x = bf16_bits_to_f32((j & 1) ? (w[k][j >> 1] >> 16) : (w[k][j >> 1] & 0xffffu));
						f[k]          = left > k ? fminf(fmaxf(x * mul, -448.f), 448.f) : 0.f;
					}
					uint32_t o = 0;
					o = __builtin_amdgcn_cvt_pk_fp8_f32(f[0], f[1], o, false);
					o = __builtin_amdgcn_cvt_pk_fp8_f32(f[2], f[3], o, true);
					*reinterpret_cast<uint32_t*>(d0 + j * dst_row_stride) = o;
					if(dst_lo) *reinterpret_cast<uint32_t*>(dst_lo + (d0 - dst) + j * dst_row_stride) = residual(f[0], f[1], f[2], f[3], o);
				}
			}
		} else if(total < ((int64_t)1 << 31) && stride < ((int64_t)1 << 30)) {
			mul = multiplier();
			for(uint32_t i = blockIdx.x * EW_THREADS + threadIdx.x; i < (uint32_t)total; i += (uint32_t)stride) element(i, (uint32_t)cols, (uint32_t)rq);
		} else {
			mul = multiplier();
			for(int64_t i = (int64_t)blockIdx.x * EW_THREADS + threadIdx.x; i < total; i += stride) element(i, cols, rq);
		}
	}
}

template <bool SRC_BF16>
__global__ void __launch_bounds__(EW_THREADS) quantize_e4m3_kernel(const void* __restrict__ src, uint8_t* __restrict__ dst, int64_t rows, int64_t cols,
																	 int64_t src_row_stride, int transpose, int64_t rows_per_matrix, int64_t dst_row_stride,
																	 float pre_scale, const float* amax, float* descale_out, uint8_t* __restrict__ dst_lo) {
	const float scale = fp8_pow2_scale(*amax, pre_scale);
	if(blockIdx.x == 0 && threadIdx.x == 0 && descale_out) *descale_out = 1.f / scale;
	quantize_e4m3_body<SRC_BF16>(src, dst, rows, cols, src_row_stride, transpose, rows_per_matrix, dst_row_stride, [&]() { return pre_scale * scale; }, dst_lo);
}

// q, k and v of one attention call in one launch (blockIdx.y): q and k as they are (plus residuals),
// v transposed; each wavefront folds its tensor's partial maxima from amax3_kernel for itself, under the latency of its first loads.
// (Short launches: what they wait for counts.  With the maxima folded by shuffles and through LDS before the first load, and one load at a
// time in both launches, us for the two: 1x16x128x24 6.5 / now 6.2, 2x16x777x24 9.1 / 8.4, 5x16x1536x24 14.0 / 13.3.)
struct Quant3Args {
	const void* src[3];
	uint8_t*    dst[3];
	uint8_t*    dst_lo[3];
	int64_t     rows, cols, rows_per_matrix, v_row_stride;
	float       pre_scale[3];
};
template <bool SRC_BF16>
__global__ void __launch_bounds__(EW_THREADS) quantize3_kernel(Quant3Args a, const float* __restrict__ partials, float* __restrict__ descales) {
	const int t = blockIdx.y;
	static_assert(AMAX3_BLOCKS == 4 * 64, "four partial maxima per lane: every wavefront folds them for itself");
	typedef __attribute__((ext_vector_type(4), aligned(4))) float f32x4_any;   // (the caller's floats start at any of them)
	const f32x4 m4 = *reinterpret_cast<const f32x4_any*>(partials + t * AMAX3_BLOCKS + 4 * (threadIdx.x & 63));
	auto multiplier = [&]() -> float {
		const float scale = fp8_pow2_scale(wave_max(fmaxf(fmaxf(m4[0], m4[1]), fmaxf(m4[2], m4[3]))), a.pre_scale[t]);
		if(blockIdx.x == 0 && threadIdx.x == 0) descales[t] = 1.f / scale;
		return a.pre_scale[t] * scale;
	};
	const bool tr = t == 2;
	quantize_e4m3_body<SRC_BF16>(a.src[t], a.dst[t], a.rows, a.cols, a.cols, tr ? 1 : 0, a.rows_per_matrix, tr ? a.v_row_stride : a.cols, multiplier, a.dst_lo[t]);
}

// ---- pad / repack ----------------------------------------------------------------------------
struct PadDims {
	int     ndim;
	int64_t src_shape[AF3_PAD_MAX_DIMS], src_stride[AF3_PAD_MAX_DIMS], dst_shape[AF3_PAD_MAX_DIMS];
};

template <typename T>
__global__ void __launch_bounds__(EW_THREADS) pad_nd_kernel(const T* __restrict__ src, T* __restrict__ dst, PadDims d, int64_t total, T fill) {
	const int64_t stride = (int64_t)gridDim.x * EW_THREADS;
	for(int64_t i = (int64_t)blockIdx.x * EW_THREADS + threadIdx.x; i < total; i += stride) {
		int64_t rem = i, soff = 0;
		bool    in  = true;
		for(int a = d.ndim - 1; a >= 0; a--) {
			const int64_t c = rem % d.dst_shape[a];
			rem /= d.dst_shape[a];
			in = in && c < d.src_shape[a];
			soff += c * d.src_stride[a];
		}
		dst[i] = in ? src[soff] : fill;
	}
}

__global__ void __launch_bounds__(EW_THREADS) vnni_repack_kernel(const uint16_t* __restrict__ src, uint16_t* __restrict__ dst, int64_t M, int64_t N, int64_t blk) {
	const int64_t stride = (int64_t)gridDim.x * EW_THREADS, total = M * N;
	for(int64_t o = (int64_t)blockIdx.x * EW_THREADS + threadIdx.x; o < total; o += stride) {
		// o = panel*M*blk + i*blk*2 + j*2 + k   (src/csrc/xsmm_functors.h:2100-2111 applied per panel, tools.cpp:171-173)
		const int64_t panel = o / (M * blk), rem = o % (M * blk);
		const int64_t i = rem / (2 * blk), j = (rem % (2 * blk)) >> 1, k = rem & 1;
		dst[o] = src[(2 * i + k) * N + panel * blk + j];
	}
}

}  // namespace af3

using namespace af3;

extern "C" int af3_convert(const void* src, int32_t sd, void* dst, int32_t dd, int64_t n, void* stream) {
	if(n < 0) return AF3_ERR_BAD_SHAPE;
	if(n == 0) return AF3_OK;
	if(!src || !dst) return AF3_ERR_NULL_POINTER;
	hipStream_t s = static_cast<hipStream_t>(stream);
	if(sd == AF3_F32 && dd == AF3_BF16)
		hipLaunchKernelGGL(cvt_f32_bf16_kernel, dim3(ew_blocks((n + 7) / 8)), dim3(EW_THREADS), 0, s, static_cast<const float*>(src), static_cast<uint16_t*>(dst), n);
	else if(sd == AF3_BF16 && dd == AF3_F32)
		hipLaunchKernelGGL(cvt_bf16_f32_kernel, dim3(ew_blocks((n + 7) / 8)), dim3(EW_THREADS), 0, s, static_cast<const uint16_t*>(src), static_cast<float*>(dst), n);
	else if(sd == AF3_FP8_E4M3 && dd == AF3_F32)
		hipLaunchKernelGGL(cvt_e4m3_kernel<false>, dim3(ew_blocks((n + 3) / 4)), dim3(EW_THREADS), 0, s, static_cast<const uint8_t*>(src), dst, n);
	else if(sd == AF3_FP8_E4M3 && dd == AF3_BF16)
		hipLaunchKernelGGL(cvt_e4m3_kernel<true>, dim3(ew_blocks((n + 3) / 4)), dim3(EW_THREADS), 0, s, static_cast<const uint8_t*>(src), dst, n);
	else if(sd == AF3_F32 && dd == AF3_FP8_E5M2)
		hipLaunchKernelGGL(cvt_to_e5m2_kernel<false>, dim3(ew_blocks((n + 3) / 4)), dim3(EW_THREADS), 0, s, src, static_cast<uint8_t*>(dst), n);
	else if(sd == AF3_BF16 && dd == AF3_FP8_E5M2)
		hipLaunchKernelGGL(cvt_to_e5m2_kernel<true>, dim3(ew_blocks((n + 3) / 4)), dim3(EW_THREADS), 0, s, src, static_cast<uint8_t*>(dst), n);
	else if(sd == AF3_FP8_E5M2 && dd == AF3_F32)
		hipLaunchKernelGGL(cvt_e5m2_kernel<false>, dim3(ew_blocks(n)), dim3(EW_THREADS), 0, s, static_cast<const uint8_t*>(src), dst, n);
	else if(sd == AF3_FP8_E5M2 && dd == AF3_BF16)
		hipLaunchKernelGGL(cvt_e5m2_kernel<true>, dim3(ew_blocks(n)), dim3(EW_THREADS), 0, s, static_cast<const uint8_t*>(src), dst, n);
	else
		return AF3_ERR_BAD_DTYPE;
	return launch_status();
}

extern "C" int af3_amax(const void* src, int32_t sd, int64_t n, float* amax_out, void* stream) {
	if(n < 0) return AF3_ERR_BAD_SHAPE;
	if(!amax_out || (n > 0 && !src)) return AF3_ERR_NULL_POINTER;
	if(n == 0) return AF3_OK;
	hipStream_t s = static_cast<hipStream_t>(stream);
	if(sd == AF3_F32) hipLaunchKernelGGL(amax_kernel<false>, dim3(ew_blocks((n + 7) / 8, 512)), dim3(EW_THREADS), 0, s, src, n, amax_out);
	else if(sd == AF3_BF16) hipLaunchKernelGGL(amax_kernel<true>, dim3(ew_blocks((n + 7) / 8, 512)), dim3(EW_THREADS), 0, s, src, n, amax_out);
	else return AF3_ERR_BAD_DTYPE;
	return launch_status();
}

extern "C" int af3_quantize_fp8_e4m3(const void* src, int32_t sd, void* dst, int64_t rows, int64_t cols, int64_t src_row_stride, int32_t transpose_last2,
									 int64_t rows_per_matrix, int64_t dst_row_stride, float pre_scale, const float* amax, float* descale_out, void* dst_residual,
									 void* stream) {
	if(rows < 0 || cols < 0) return AF3_ERR_BAD_SHAPE;
	if(!amax) return AF3_ERR_NULL_POINTER;
	if(rows == 0 || cols == 0) return AF3_OK;
	if(!src || !dst) return AF3_ERR_NULL_POINTER;
	if(src_row_stride < cols) return AF3_ERR_BAD_STRIDE;
	if(transpose_last2) {
		if(rows_per_matrix <= 0 || rows % rows_per_matrix != 0) return AF3_ERR_BAD_ARGUMENT;
		if(dst_row_stride < (rows_per_matrix + 3) / 4 * 4 || dst_row_stride % 4 != 0) return AF3_ERR_BAD_STRIDE;
	} else {
		if(cols % 4 != 0) return AF3_ERR_BAD_ARGUMENT;
		if(dst_row_stride < cols || dst_row_stride % 4 != 0) return AF3_ERR_BAD_STRIDE;
	}
	if((reinterpret_cast<uintptr_t>(dst) & 3) || (reinterpret_cast<uintptr_t>(dst_residual) & 3)) return AF3_ERR_BAD_ARGUMENT;
	hipStream_t    s = static_cast<hipStream_t>(stream);
	const unsigned g = ew_blocks(rows * cols / 4);
	if(sd == AF3_F32)
		hipLaunchKernelGGL(quantize_e4m3_kernel<false>, dim3(g), dim3(EW_THREADS), 0, s, src, static_cast<uint8_t*>(dst), rows, cols, src_row_stride, (int)transpose_last2,
						   rows_per_matrix, dst_row_stride, pre_scale, amax, descale_out, static_cast<uint8_t*>(dst_residual));
	else if(sd == AF3_BF16)
		hipLaunchKernelGGL(quantize_e4m3_kernel<true>, dim3(g), dim3(EW_THREADS), 0, s, src, static_cast<uint8_t*>(dst), rows, cols, src_row_stride, (int)transpose_last2,
						   rows_per_matrix, dst_row_stride, pre_scale, amax, descale_out, static_cast<uint8_t*>(dst_residual));
	else
		return AF3_ERR_BAD_DTYPE;
	return launch_status();
}

extern "C" int af3_quantize_qkv_fp8_e4m3(const void* q, const void* k, const void* v, int32_t sd, int64_t B, int64_t H, int64_t L, int64_t D, float q_pre_scale, void* q8,
										void* k8, void* v8t, int64_t v8t_row_stride, void* q_lo, void* k_lo, float* descales, float* scratch, void* stream) {
	if(B <= 0 || H <= 0 || L <= 0 || D <= 0) return AF3_ERR_BAD_SHAPE;
	if(!q || !k || !v || !q8 || !k8 || !v8t || !descales || !scratch) return AF3_ERR_NULL_POINTER;
	if(D % 4 != 0) return AF3_ERR_BAD_ARGUMENT;
	if(v8t_row_stride < (L + 3) / 4 * 4 || v8t_row_stride % 4 != 0) return AF3_ERR_BAD_STRIDE;
	if(sd != AF3_F32 && sd != AF3_BF16) return AF3_ERR_BAD_DTYPE;
	for(const void* ptr : {(const void*)q8, (const void*)k8, (const void*)v8t, (const void*)q_lo, (const void*)k_lo})
		if(reinterpret_cast<uintptr_t>(ptr) & 3) return AF3_ERR_BAD_ARGUMENT;
	hipStream_t   s = static_cast<hipStream_t>(stream);
	const int64_t n = B * H * L * D;
	Amax3Args     aa;
	aa.src[0] = q, aa.src[1] = k, aa.src[2] = v;
	aa.n[0] = aa.n[1] = aa.n[2] = n;
	Quant3Args qa;
	qa.src[0] = q, qa.src[1] = k, qa.src[2] = v;
	qa.dst[0] = static_cast<uint8_t*>(q8), qa.dst[1] = static_cast<uint8_t*>(k8), qa.dst[2] = static_cast<uint8_t*>(v8t);
	qa.dst_lo[0] = static_cast<uint8_t*>(q_lo), qa.dst_lo[1] = static_cast<uint8_t*>(k_lo), qa.dst_lo[2] = nullptr;
	qa.rows = B * H * L, qa.cols = D, qa.rows_per_matrix = L, qa.v_row_stride = v8t_row_stride;
	qa.pre_scale[0] = q_pre_scale, qa.pre_scale[1] = qa.pre_scale[2] = 1.f;
	// (quantise: a thread of the dense paths takes 8 elements per trip.  One trip per thread up to two workgroups per compute unit
	// and tensor -- few elements in few workgroups of four trips each took 4.7 us --, four trips beyond, so that the three tensors'
	// workgroups, each of which first folds its tensor's partial maxima, are all resident at once for the usual sizes)
	const int64_t qb = ew_blocks(n / 32, 1024);
	const dim3    ga(AMAX3_BLOCKS, 3), gq((unsigned)(qb >= 512 ? qb : std::min<int64_t>(ew_blocks(n / 8, 1024), 512)), 3);
	if(sd == AF3_F32) {
		hipLaunchKernelGGL(amax3_kernel<false>, ga, dim3(EW_THREADS), 0, s, aa, scratch);
		hipLaunchKernelGGL(quantize3_kernel<false>, gq, dim3(EW_THREADS), 0, s, qa, scratch, descales);
	} else {
		hipLaunchKernelGGL(amax3_kernel<true>, ga, dim3(EW_THREADS), 0, s, aa, scratch);
		hipLaunchKernelGGL(quantize3_kernel<true>, gq, dim3(EW_THREADS), 0, s, qa, scratch, descales);
	}
	return launch_status();
}

extern "C" int af3_pad_nd(const void* src, void* dst, int32_t ndim, const int64_t* src_shape, const int64_t* src_strides, const int64_t* dst_shape,
						  int32_t elem_size, uint32_t fill_bits, void* stream) {
	if(ndim < 1 || ndim > AF3_PAD_MAX_DIMS) return AF3_ERR_BAD_SHAPE;
	if(!src_shape || !src_strides || !dst_shape) return AF3_ERR_NULL_POINTER;
	PadDims d;
	d.ndim = ndim;
	int64_t total = 1, src_total = 1;
	for(int a = 0; a < ndim; a++) {
		if(src_shape[a] < 0 || dst_shape[a] < src_shape[a]) return AF3_ERR_BAD_SHAPE;
		if(src_strides[a] < 0) return AF3_ERR_BAD_STRIDE;
		d.src_shape[a] = src_shape[a], d.src_stride[a] = src_strides[a], d.dst_shape[a] = dst_shape[a];
		total *= dst_shape[a];
		src_total *= src_shape[a];
	}
	if(total == 0) return AF3_OK;
	if(!dst || (src_total > 0 && !src)) return AF3_ERR_NULL_POINTER;
	hipStream_t    s = static_cast<hipStream_t>(stream);
	const unsigned g = ew_blocks(total);
	if(elem_size == 4)
		hipLaunchKernelGGL(pad_nd_kernel<uint32_t>, dim3(g), dim3(EW_THREADS), 0, s, static_cast<const uint32_t*>(src), static_cast<uint32_t*>(dst), d, total, fill_bits);
	else if(elem_size == 2)
		hipLaunchKernelGGL(pad_nd_kernel<uint16_t>, dim3(g), dim3(EW_THREADS), 0, s, static_cast<const uint16_t*>(src), static_cast<uint16_t*>(dst), d, total, (uint16_t)fill_bits);
	else if(elem_size == 1)
		hipLaunchKernelGGL(pad_nd_kernel<uint8_t>, dim3(g), dim3(EW_THREADS), 0, s, static_cast<const uint8_t*>(src), static_cast<uint8_t*>(dst), d, total, (uint8_t)fill_bits);
	else
		return AF3_ERR_BAD_DTYPE;
	return launch_status();
}

extern "C" int af3_vnni_repack_bf16(const void* src, void* dst, int64_t M, int64_t N, int64_t blk, void* stream) {
	if(M <= 0 || N <= 0) return AF3_ERR_BAD_SHAPE;
	if(!src || !dst) return AF3_ERR_NULL_POINTER;
	if(blk == 0) blk = N;
	// the reference asserts N % BLK_SZ == 0 and exits (src/csrc/tools.cpp:167); here it is an error code
	if(blk < 0 || N % blk != 0 || (M & 1)) return AF3_ERR_BAD_ARGUMENT;
	hipLaunchKernelGGL(vnni_repack_kernel, dim3(ew_blocks(M * N)), dim3(EW_THREADS), 0, static_cast<hipStream_t>(stream), static_cast<const uint16_t*>(src),
					   static_cast<uint16_t*>(dst), M, N, blk);
	return launch_status();
}
