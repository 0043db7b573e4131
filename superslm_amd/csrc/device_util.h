// Device helpers shared by the kernel files: vector types, wave reductions, segment views, the packed
// weight layout's addressing.
#pragma once

#include "kernels.h"

namespace sslm {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v16i __attribute__((ext_vector_type(16)));

// Row maxima travel as 32-bit magnitudes: |v| saturated at 2^32 - 2, so that 2^32 - 1 (kBad32)
// is free to mark a refusal somewhere in the row.  Every consumer rejects a maximum above 2^31
// (the funnel's accepted domain), so the saturation changes no outcome.
constexpr uint32_t kBad32 = 0xffffffffu;

__device__ __forceinline__ uint32_t sat_abs_u32(int64_t v) {
	uint64_t a = v < 0 ? (uint64_t)0 - (uint64_t)v : (uint64_t)v;
	return a > 0xfffffffeull ? 0xfffffffeu : (uint32_t)a;
}

// sat_abs_u32 of a row maximum held in a non-negative double
__device__ __forceinline__ uint32_t sat_u32_d(double m) { return (uint32_t)fmin(m, 4294967294.0); }

__device__ __forceinline__ int32_t sat_i32(int64_t v) {
	return v > kI32Max ? kI32Max : (v < kI32Min ? kI32Min : (int32_t)v);
}

__device__ __forceinline__ v4i load16(const int8_t* p) { return *(const v4i*)p; }

__device__ __forceinline__ uint32_t dpp_max16(uint32_t v) {
	// row_ror:8, 4, 2, 1 -- every lane of the 16-lane row ends with the row maximum
	uint32_t w = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, false);
	v = w > v ? w : v;
	w = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xf, 0xf, false);
	v = w > v ? w : v;
	w = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x122, 0xf, 0xf, false);
	v = w > v ? w : v;
	w = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x121, 0xf, 0xf, false);
	return w > v ? w : v;
}

// maximum / sum over each 16-lane row, in every lane of it
__device__ __forceinline__ int32_t row16_max(int32_t v) { return (int32_t)(dpp_max16((uint32_t)v ^ 0x80000000u) ^ 0x80000000u); }
template <int CTRL>
__device__ __forceinline__ int64_t row16_rot(int64_t v) {
	const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)v, CTRL, 0xf, 0xf, false);
	const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)((uint64_t)v >> 32), CTRL, 0xf, 0xf, false);
	return (int64_t)((uint64_t)hi << 32 | lo);
}
__device__ __forceinline__ int64_t row16_sum(int64_t v) {
	v += row16_rot<0x128>(v);
	v += row16_rot<0x124>(v);
	v += row16_rot<0x122>(v);
	return v + row16_rot<0x121>(v);
}

// The fields of segment `si` (wave-uniform) that the decode GEMV epilogue uses, selected with
// constant indices so they stay scalar kernel-argument loads.
struct SegView {
	int32_t n_begin, mode, ld_out;
	void* out;
	uint32_t* maxpart;
	const int32_t* fold;
	const int64_t* bias;
	const int8_t* lora_b;
	const int32_t* lora_dfold;
	const int8_t* lora_u;
};

__device__ __forceinline__ SegView seg_view(const Epilogue& e, int si) {
	const Segment& s = si == 0 ? e.seg[0] : (si == 1 ? e.seg[1] : e.seg[2]);
	return SegView{s.n_begin, s.mode, s.ld_out, s.out, s.maxpart, s.fold, s.bias, s.lora_b, s.lora_dfold, s.lora_u};
}

// segment of the 16-column tile starting at column c0 (bounds are multiples of 16), with
// constant indices so the fields stay scalar kernel-argument loads
__device__ __forceinline__ int tile_segment(const Epilogue& e, int c0) {
	return (e.nseg > 1 && c0 >= e.seg[0].n_end) ? ((e.nseg > 2 && c0 >= e.seg[1].n_end) ? 2 : 1) : 0;
}

// lane `lane`'s 16 bytes of chunk 0, half 0 of `tile` in a packed decode copy (k_gemv_pk)
__device__ __forceinline__ const int8_t* pk_lane(const int8_t* wp, int tile, int C, int lane) {
	return wp + (size_t)tile * C * 2048 + lane * 16;
}

// A block reduction's result is the same in every lane; saying so (readfirstlane) lets the
// compiler keep it, and the scalar scale plans computed from it, in scalar registers.
__device__ __forceinline__ uint64_t uni_u64(uint64_t v) {
	const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
	const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
	return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ int64_t uni_i64(int64_t v) { return (int64_t)uni_u64((uint64_t)v); }

// 32-bit wave reductions: a 16-lane rotate butterfly (DPP) leaves every lane with its row's
// result, and the four row results are read as scalars -- the value comes back wave-uniform.
__device__ __forceinline__ uint32_t wave_max32(uint32_t v) {
	v = dpp_max16(v);
	const uint32_t a = __builtin_amdgcn_readlane(v, 0), b = __builtin_amdgcn_readlane(v, 16);
	const uint32_t c = __builtin_amdgcn_readlane(v, 32), d = __builtin_amdgcn_readlane(v, 48);
	return max(max(a, b), max(c, d));
}

__device__ __forceinline__ int32_t wave_sum32(int32_t v) {
	v += __builtin_amdgcn_update_dpp(0, v, 0x128, 0xf, 0xf, false);  // row_ror:8
	v += __builtin_amdgcn_update_dpp(0, v, 0x124, 0xf, 0xf, false);  // row_ror:4
	v += __builtin_amdgcn_update_dpp(0, v, 0x122, 0xf, 0xf, false);  // row_ror:2
	v += __builtin_amdgcn_update_dpp(0, v, 0x121, 0xf, 0xf, false);  // row_ror:1
	return __builtin_amdgcn_readlane(v, 0) + __builtin_amdgcn_readlane(v, 16) + __builtin_amdgcn_readlane(v, 32) +
	       __builtin_amdgcn_readlane(v, 48);
}

}  // namespace sslm
