// The decode layer of a few sequences in fewer launches: funnels run inside the packed GEMV that reads
// their codes.
//
//   k_funnel_gemv   (M <= 4) context funnel                -> o GEMV (raw)
//   k_residual_gemv (M = 1)  o funnel, residual, norm      -> gate|up GEMV (funnel epilogue)
//   k_act_gemv      (M <= 4) activation funnel             -> down GEMV (raw split-K planes)
//   k_residual_gemv (M = 1)  down funnel, residual, norm   -> the next layer's q|k|v GEMV (general epilogue)
//
// What bounds such a layer is its chain of dependent launches: a row kernel is 4-8 us of latency
// during which the weights of the next GEMV, which depend on nothing, sit unread.  Every block here
// issues its first weight tiles and then derives the rows it multiplies by itself: a row is a few
// thousand values that come from L2, so 100-250 blocks computing it alike costs less than handing it
// from one launch to the next, and the chain runs while the weights stream in.  The repeated rows
// are what ends this: at three sequences residual + norm inside gate|up took 19.0 us against 7.7 + 7.4,
// while the shorter funnels still gain (ctx + o 6.0 against 4.5 + 3.7, act + down 7.6 against 4.8 + 4.5);
// at 16 rows every block would requantize 16 rows and the funnels lose too.
// A layer of hidden 1536, intermediate 8960, one sequence: 61 -> 47 us.
//
// The arithmetic is that of k_funnel, k_residual_norm, k_mlp_act_s2 and k_gemv_pk / k_gemv_sk, element by
// element; block 0 writes the rows' codes, scales and refusals where those kernels do.  A row that is
// refused, or was before, multiplies as zeros and reports nothing further.  (k_funnel_gemv: a block that
// reads head_status after block 0 has resolved it multiplies the row as any other.  Either product is
// dropped: every later kernel leaves a refused row by its status word.)
#include <hip/hip_runtime.h>

#include <algorithm>

#include "device_util.h"

namespace sslm {

constexpr int kCW = 4;  // waves that split K in k_residual_gemv / k_funnel_gemv

// K chunks [wave CPW, + CPW) of the A operand from the block's codes in LDS ([M][ld] bytes): lane
// (ri, grp) reads row ri at 128 c + {0, 64} + 16 grp; rows past M and chunks past C are zero.
template <int CPW>
__device__ __forceinline__ void take_rows(const int8_t* s_x, int ld, int M, int C, int wave, int lane, v4i (&x)[CPW][2]) {
	const int ri = lane & 15, grp = lane >> 4;
	const v4i z = v4i{0, 0, 0, 0};
	const int8_t* row = s_x + min(ri, M - 1) * ld + grp * 16;
#pragma unroll
	for (int i = 0; i < CPW; ++i) {
		const int c = wave * CPW + i, cc = min(c, C - 1);
		const v4i a = *(const v4i*)(row + cc * 128), b = *(const v4i*)(row + cc * 128 + 64);
		const bool ok = ri < M && c < C;
		x[i][0] = ok ? a : z;
		x[i][1] = ok ? b : z;
	}
}

// maximum / sum over the block's NW waves (one barrier; `slots`: an entry per wave)
template <int NW>
__device__ __forceinline__ uint32_t row_max(uint32_t v, uint32_t* slots) {
	v = wave_max32(v);
	if ((threadIdx.x & 63) == 0) slots[threadIdx.x >> 6] = v;
	__syncthreads();
	v = slots[0];
#pragma unroll
	for (int i = 1; i < NW; ++i) v = max(v, slots[i]);
	return __builtin_amdgcn_readfirstlane(v);
}
template <int NW>
__device__ __forceinline__ int32_t row_sum(int32_t v, int32_t* slots) {
	v = wave_sum32(v);
	if ((threadIdx.x & 63) == 0) slots[threadIdx.x >> 6] = v;
	__syncthreads();
	v = 0;
#pragma unroll
	for (int i = 0; i < NW; ++i) v += slots[i];
	return __builtin_amdgcn_readfirstlane(v);
}

// Projection funnel -> residual reconcile -> RMSNorm of one row (k_residual_norm with a raw projection of
// at most RS planes, no LoRA, no bias), then its GEMV (k_gemv_pk).  The row is a serial chain per
// thread, so eight waves share it (four waves, six elements a thread: gate|up of hidden 1536 in 13.4 us, eight:
// 11.8; k_residual_norm + k_gemv_pk took 7.7 + 7.2); for the GEMV
// they form two groups of four that split K as k_gemv_pk does and take the block's tiles in turn.
// Every tile's partial sums meet in LDS behind one barrier, and a thread finishes one column.
// One row only: two rows on eight waves or four on sixteen took 17-19 us with gate|up, where the row
// kernel and k_gemv_pk take 15.
template <int NT, int CPW, bool FUNNEL, int RS>
__global__ __launch_bounds__(512) void k_residual_gemv(GemmArgs g, sslm_launch::ResidualArgs a) {
	constexpr int NW = 8, RT = 64 * NW, EP = (4 * CPW * 128 + RT - 1) / RT;  // waves, threads, elements a thread
	constexpr int TG = NW / kCW, NI = (NT + TG - 1) / TG;                    // tile groups, tiles per group
	constexpr int LDX = 4 * CPW * 128 + 16;
	static_assert(NT * 16 <= RT, "a thread per column");
	// tiles issued ahead of the row's chain: all of a group's where they fit the registers beside it
	constexpr int PD = NI * CPW <= 12 ? NI : (NI < 2 ? NI : 2);
	__shared__ __attribute__((aligned(16))) int8_t s_x[1][LDX];
	__shared__ int32_t red[NI][NW][16];
	__shared__ uint32_t s_m[3][NW];
	__shared__ int32_t s_s[NW];
	const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
	const int ri = lane & 15, grp = lane >> 4, kw = wave & 3, tg = wave >> 2;
	const int C = g.K >> 7, T = (g.N + 15) / 16, H = a.H;
	const int rl = threadIdx.x;
	const bool lead = blockIdx.x == 0;
	// ---- the row's loads, then the first tiles' weights ----
	const int slot = a.tok[0].slot;
	const int sidx = a.stream_idx[0], oidx = a.out_idx[0];
	const Scale bin = a.branch_in[0];
	const Scale ss = a.stream_scale[sidx];
	const int32_t status0 = a.status[slot];
	const int32_t* prow = a.raw.part;
	const size_t plane = (size_t)a.raw.ld;
	const int8_t* srow = a.stream + (size_t)sidx * H;
	const int32_t* fold = a.raw.epi.seg[0].fold;
	uint32_t acc[EP];
	int32_t fo[EP][3], sv[EP], gn[EP];
#pragma unroll
	for (int k = 0; k < EP; ++k) {
		const int e = min(rl + k * RT, H - 1);
		sv[k] = srow[e];
		gn[k] = a.gain[e];
		acc[k] = 0;
#pragma unroll
		for (int s2 = 0; s2 < RS; ++s2) {
			const uint32_t x = (uint32_t)prow[(size_t)(RS == 1 ? 0 : min(s2, a.raw.splits - 1)) * plane + e];
			acc[k] += (RS == 1 || s2 < a.raw.splits) ? x : 0u;  // the true sum fits int32; partials wrap harmlessly
		}
		fo[k][0] = fold[3 * e];
		fo[k][1] = fold[3 * e + 1];
		fo[k][2] = fold[3 * e + 2];
	}
	// the column this thread finishes (threads past NT * 16 none) and its epilogue parameters
	const Epilogue& e = g.epi;
	const int q = min(rl >> 4, NT - 1), tile_q = (int)blockIdx.x + q * (int)gridDim.x, j = tile_q * 16 + (rl & 15);
	const bool fin = rl < NT * 16 && tile_q < T && j < g.N;
	// the segment is a lane's own (a wave holds four tiles): fields by constant index
	const int si = tile_segment(e, min(tile_q, T - 1) * 16);
#define SSLM_SEG_FIELD(f) (si == 0 ? e.seg[0].f : (si == 1 ? e.seg[1].f : e.seg[2].f))
	const int jj = min(j, g.N - 1) - SSLM_SEG_FIELD(n_begin), mode = SSLM_SEG_FIELD(mode);
	void* const sout = SSLM_SEG_FIELD(out);
	uint32_t* const smax = SSLM_SEG_FIELD(maxpart);
	const int32_t* const fp = SSLM_SEG_FIELD(fold) + 3 * jj;
	const int64_t* const sbias = SSLM_SEG_FIELD(bias);
#undef SSLM_SEG_FIELD
	const int32_t f0 = fp[0], f1 = fp[1], f2 = fp[2];
	const int64_t bias = FUNNEL ? 0 : *(sbias ? sbias + jj : (const int64_t*)g.wp);
	struct Slot {
		v4i b[CPW][2];
	};
	Slot S[PD];
	// the i-th tile of this wave's group (past the block's last: one that it loads anyway)
	auto tile_of = [&](int i) {
		const int qi = i * TG + tg;
		return (int)blockIdx.x + (qi < NT ? qi : max(qi - TG, 0) % NT) * (int)gridDim.x;
	};
	auto load_w = [&](int i, Slot& d) {
		const int8_t* tp = pk_lane(g.wp, min(tile_of(i), T - 1), C, lane);
#pragma unroll
		for (int c2 = 0; c2 < CPW; ++c2) {
			const int c = min(kw * CPW + c2, C - 1);
			d.b[c2][0] = load16(tp + (size_t)c * 2048);
			d.b[c2][1] = load16(tp + (size_t)c * 2048 + 1024);
		}
	};
#pragma unroll
	for (int i = 0; i < PD; ++i) load_w(i, S[i]);
	// ---- the branch funnel ----
	int32_t bv[EP];
	uint32_t mx = 0;
#pragma unroll
	for (int k = 0; k < EP; ++k) {
		const int32_t v = fold_bounded((int32_t)acc[k], fold_consts(fo[k][0], fo[k][1], fo[k][2]));
		bv[k] = rl + k * RT < H ? v : 0;
		mx = max(mx, (uint32_t)(bv[k] < 0 ? -bv[k] : bv[k]));
	}
	mx = row_max<NW>(mx, s_m[0]);
	FunnelPlan bp{}, rp{}, np{};
	// Any block may report a bias refusal of the layer after a.layer at its end, before a late block (block
	// 0 too, which commits this layer's row) has read the word: only refusals up to a.layer count here.
	bool ok = !refused_through(status0, a.layer);
	int32_t st = funnel_plan(mx, &bin, 1, a.branch_site, &bp);
	if (st == kOk && !fits_i32(ss.m)) st = kCarriedScaleMantissaOutOfDomain;
	if (ok && st != kOk) {
		if (lead && rl == 0) set_status(a.status, slot, a.layer, st);
		ok = false;
	}
	// ---- residual: the landed value of each branch code ----
	const int64_t r_h = reciprocal_fast(ok ? ss.m : ((int64_t)1 << 30)), kx = composed_exponent(bp.out.e, ss.e);
	const double lf = landing_scale(bp.out.m, r_h, kx).f;
	const double bf = bp.f;
	int32_t c[EP];
#pragma unroll
	for (int k = 0; k < EP; ++k) c[k] = ok ? requant_code_f(bv[k], bf) : 0;
	double w[EP], mxd = 0.0;
#pragma unroll
	for (int k = 0; k < EP; ++k) {
		w[k] = rl + k * RT < H ? residual_land(c[k], bp.out.m, r_h, kx, lf) + (double)sv[k] : 0.0;
		mxd = fmax(mxd, fabs(w[k]));
	}
	mx = row_max<NW>(mxd == (double)INFINITY ? kBad32 : sat_u32_d(mxd), s_m[1]);
	st = mx == kBad32 ? kResidualReconciliationMagnitudeOutOfDomain : funnel_plan(mx, &ss, 1, a.res_site, &rp);
	if (ok && st != kOk) {
		if (lead && rl == 0) set_status(a.status, slot, a.layer, st);
		ok = false;
	}
	const double rf = rp.f;
	int32_t sq = 0;
	int8_t* out = a.out_stream + (size_t)oidx * H;
#pragma unroll
	for (int k = 0; k < EP; ++k) {
		c[k] = ok ? requant_code_d(w[k], rf) : 0;
		sq += c[k] * c[k];
		if (lead && ok && rl + k * RT < H) out[rl + k * RT] = (int8_t)c[k];
	}
	if (lead && ok && rl == 0) a.out_stream_scale[oidx] = rp.out;
	// ---- RMSNorm (rmsnorm_regs) ----
	sq = row_sum<NW>(sq, s_s);
	const double rd = (double)rms_root(sq, H), inv = rcp_est(rd);
	mxd = 0.0;
#pragma unroll
	for (int k = 0; k < EP; ++k) {
		w[k] = norm_qd(c[k], rd, inv) * (double)gn[k];
		mxd = fmax(mxd, fabs(w[k]));
	}
	mx = row_max<NW>(sat_u32_d(mxd), s_m[2]);
	st = funnel_plan(mx, nullptr, 0, a.norm_site, &np);
	if (ok && st != kOk) {
		if (lead && rl == 0) set_status(a.status, slot, a.layer, st);
		ok = false;
	}
	const double nf = np.f;
#pragma unroll
	for (int k = 0; k < EP; ++k) {
		const int el = rl + k * RT;
		const int8_t v = ok ? requant_code_d(w[k], nf) : (int8_t)0;
		if (el < LDX) s_x[0][el] = v;
		if (lead && ok && el < H) a.norm_out[el] = v;
	}
	const int64_t rcp = fits_i32(np.out.m) ? reciprocal_fast(np.out.m) : 0;
	if (lead && ok && rl == 0) {
		a.norm_scale[0] = np.out;
		if (a.norm_recip) a.norm_recip[0] = rcp;
	}
	__syncthreads();
	// ---- GEMV: row 0 of the A operand; the other rows are zero ----
	v4i x[CPW][2];
	take_rows<CPW>(s_x[0], LDX, 1, C, kw, lane, x);
#pragma unroll
	for (int i = 0; i < NI; ++i) {
		Slot& cur = S[i % PD];
		v4i ac = v4i{0, 0, 0, 0};
#pragma unroll
		for (int c2 = 0; c2 < CPW; ++c2) {
			ac = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[c2][0], cur.b[c2][0], ac, 0, 0, 0);
			ac = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[c2][1], cur.b[c2][1], ac, 0, 0, 0);
		}
		if (i + PD < NI) load_w(i + PD, cur);
		if (grp == 0) red[i][wave][ri] = ac[0];  // accumulator lanes 0..15 hold token 0
	}
	__syncthreads();
	if (rl >= NT * 16) return;
	int32_t tot = 0;
#pragma unroll
	for (int wv = 0; wv < kCW; ++wv) tot += red[q / TG][(q % TG) * kCW + wv][rl & 15];
	if (FUNNEL) {  // |tot| <= 127^2 K < 2^29 for K <= 4096: the bounded fold applies
		const int32_t val = fold_bounded(tot, fold_consts(f0, f1, f2));
		const uint32_t mabs = dpp_max16(fin ? (uint32_t)(val < 0 ? -val : val) : 0u);
		if (fin) ((int32_t*)sout)[jj] = val;
		if ((rl & 15) == 0 && tile_q < T) smax[(size_t)tile_q * kPartLd] = mabs;
		return;
	}
	int64_t val = apply_fold((int64_t)tot, f0, f1, f2);
	if (sbias) {
		int64_t term;
		if (bias_term(bias, rcp, np.out.e, val, &term)) val += term;
		else if (fin && ok) set_status(e.status, slot, e.layer, kBiasReconcileProductOutOfDomain);
	}
	const uint32_t mabs = dpp_max16(fin && mode == kSegFunnel ? sat_abs_u32(val) : 0u);
	if (fin) {
		if (mode == kSegWide) ((int64_t*)sout)[jj] = val;
		else ((int32_t*)sout)[jj] = sat_i32(val);
	}
	if (mode == kSegFunnel && smax && (rl & 15) == 0 && tile_q < T) smax[(size_t)tile_q * kPartLd] = mabs;
}

// Context funnel of M rows (k_funnel with head statuses, no incoming scale) -> o GEMV, raw sums, one
// 16-column tile per block.  Every wave derives every row's plan from the NH <= 64 per-head maxima.
template <int MR, int CPW>
__global__ __launch_bounds__(64 * kCW) void k_funnel_gemv(GemmArgs g, sslm_launch::FunnelArgs a) {
	constexpr int LDX = 4 * CPW * 128 + 16;
	__shared__ __attribute__((aligned(16))) int8_t s_x[MR][LDX];
	__shared__ v4i red[kCW][64];
	const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
	const int ri = lane & 15, grp = lane >> 4, M = a.M, N = a.N, C = g.K >> 7, tile = blockIdx.x;
	int32_t st0[MR], hs[MR], slot[MR];
	uint32_t pm[MR];
	int2 fv[MR][CPW];
#pragma unroll
	for (int r = 0; r < MR; ++r) {
		const int t = min(r, M - 1);
		slot[r] = a.tok[t].slot;
		st0[r] = a.status[slot[r]];
		hs[r] = a.head_status[slot[r]];
		pm[r] = a.maxpart[(size_t)min(lane, a.ntiles - 1) * kPartLd + t];
#pragma unroll
		for (int k = 0; k < CPW; ++k)
			fv[r][k] = *(const int2*)(a.f + (size_t)t * a.ld_f + min(2 * ((int)threadIdx.x + k * 64 * kCW), N - 2));
	}
	v4i b[CPW][2];
	const int8_t* tp = pk_lane(g.wp, tile, C, lane);
#pragma unroll
	for (int c2 = 0; c2 < CPW; ++c2) {
		const int c = min(wave * CPW + c2, C - 1);
		b[c2][0] = load16(tp + (size_t)c * 2048);
		b[c2][1] = load16(tp + (size_t)c * 2048 + 1024);
	}
#pragma unroll
	for (int r = 0; r < MR; ++r) {
		if (r >= M) break;
		const bool lead = blockIdx.x == 0;
		FunnelPlan plan{};
		const uint32_t mx = wave_max32(pm[r]);
		const bool ref = hs[r] != kHeadStatusNone;
		const int32_t st = funnel_plan(mx, nullptr, 0, a.site, &plan);
		const bool ok = st0[r] == 0 && !ref && st == kOk;
		if (lead && threadIdx.x == 0) {
			if (ref) {  // resolve the attention's first refusing head into the status
				set_status(a.status, slot[r], a.layer, hs[r] & 0xff);
				a.head_status[slot[r]] = kHeadStatusNone;
			} else if (st0[r] == 0 && st != kOk) {
				set_status(a.status, slot[r], a.layer, st);
			}
			if (ok) a.out_scale[r] = plan.out;
		}
		const double f = plan.f;
#pragma unroll
		for (int k = 0; k < CPW; ++k) {
			const int e = 2 * ((int)threadIdx.x + k * 64 * kCW);
			if (e >= N) continue;
			const char2 v = ok ? make_char2((char)requant_code_f(fv[r][k].x, f), (char)requant_code_f(fv[r][k].y, f)) : make_char2(0, 0);
			*(char2*)&s_x[r][e] = v;
			if (lead && ok) *(char2*)(a.out + (size_t)r * N + e) = v;
		}
	}
	__syncthreads();
	v4i x[CPW][2];
	take_rows<CPW>(s_x[0], LDX, M, C, wave, lane, x);
	v4i ac = v4i{0, 0, 0, 0};
#pragma unroll
	for (int c2 = 0; c2 < CPW; ++c2) {
		ac = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[c2][0], b[c2][0], ac, 0, 0, 0);
		ac = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[c2][1], b[c2][1], ac, 0, 0, 0);
	}
	red[wave][lane] = ac;
	__syncthreads();
	const int j = tile * 16 + ri, tk = grp * 4 + wave;
	int32_t tot = 0;
#pragma unroll
	for (int wv = 0; wv < kCW; ++wv) tot += ((const int32_t*)&red[wv][lane])[wave];
	if (j < g.N && tk < M) g.epi.raw_out[(size_t)tk * g.N + j] = tot;
}

// Activation funnel of M rows over the sliced SiLU's products and slice maxima (k_mlp_act_s2) -> down
// GEMV in split-K planes (k_gemv_sk's split: 8 waves of CPW chunks).  A block requantizes its own K
// range of the rows; the blocks of tile group 0 write those codes, the first of them the scales.
template <int MR, int NTB, int CPW>
__global__ __launch_bounds__(512) void k_act_gemv(GemmArgs g, sslm_launch::ActArgs a, int slices) {
	constexpr int W = 8, SPAN = W * CPW * 128, LDX = SPAN + 16;
	__shared__ __attribute__((aligned(16))) int8_t s_x[MR][LDX];
	__shared__ int32_t sum[NTB][MR][16];
	const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
	const int ri = lane & 15, grp = lane >> 4, M = a.M, I = a.I;
	const int C = g.K >> 7, T = (g.N + 15) / 16, split = blockIdx.y;
	const int c0 = split * W * CPW, c1 = min(C, c0 + W * CPW), k0 = c0 * 128, kn = (c1 - c0) * 128;
	const int tile0 = blockIdx.x * NTB;
	int32_t st0[MR], slot[MR];
	uint32_t mx[MR];
	Scale gs[MR][2];
	int2 pv[MR][CPW];
#pragma unroll
	for (int r = 0; r < MR; ++r) {
		const int t = min(r, M - 1);
		slot[r] = a.tok[t].slot;
		st0[r] = a.status[slot[r]];
		gs[r][0] = a.gu_scale[2 * t];
		gs[r][1] = a.gu_scale[2 * t + 1];
		mx[r] = a.act_maxpart[(size_t)min(lane, slices - 1) * kPartLd + t];
#pragma unroll
		for (int k = 0; k < CPW; ++k)
			pv[r][k] = *(const int2*)(a.prod + (size_t)t * I + k0 + min(2 * ((int)threadIdx.x + k * 512), kn - 2));
	}
	v4i b[NTB][CPW][2];
#pragma unroll
	for (int tt = 0; tt < NTB; ++tt) {
		const int8_t* tp = pk_lane(g.wp, min(tile0 + tt, T - 1), C, lane);
#pragma unroll
		for (int i = 0; i < CPW; ++i) {
			const int c = min(c0 + wave * CPW + i, c1 - 1);
			b[tt][i][0] = load16(tp + (size_t)c * 2048);
			b[tt][i][1] = load16(tp + (size_t)c * 2048 + 1024);
		}
	}
	for (int i = threadIdx.x; i < NTB * MR * 16; i += 512) (&sum[0][0][0])[i] = 0;
#pragma unroll
	for (int r = 0; r < MR; ++r) {
		if (r >= M) break;
		const bool lead = blockIdx.x == 0;
		FunnelPlan plan{};
		const int32_t st = funnel_plan(wave_max32(mx[r]), gs[r], 2, a.act_site, &plan);
		const bool ok = st0[r] == 0 && st == kOk;
		if (lead && split == 0 && threadIdx.x == 0) {
			if (st0[r] == 0 && st != kOk) set_status(a.status, slot[r], a.layer, st);
			if (ok) a.act_scale[r] = plan.out;
		}
		const double f = plan.f;
#pragma unroll
		for (int k = 0; k < CPW; ++k) {
			const int e = 2 * ((int)threadIdx.x + k * 512);
			if (e >= kn) continue;
			const char2 v = ok ? make_char2((char)requant_code_f(pv[r][k].x, f), (char)requant_code_f(pv[r][k].y, f)) : make_char2(0, 0);
			*(char2*)&s_x[r][e] = v;
			if (lead && ok) *(char2*)(a.act + (size_t)r * I + k0 + e) = v;
		}
	}
	__syncthreads();
	v4i x[CPW][2];
	take_rows<CPW>(s_x[0], LDX, M, c1 - c0, wave, lane, x);
#pragma unroll
	for (int tt = 0; tt < NTB; ++tt) {
		v4i ac = v4i{0, 0, 0, 0};
#pragma unroll
		for (int i = 0; i < CPW; ++i) {
			ac = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[i][0], b[tt][i][0], ac, 0, 0, 0);
			ac = __builtin_amdgcn_mfma_i32_16x16x64_i8(x[i][1], b[tt][i][1], ac, 0, 0, 0);
		}
		if (grp == 0) {  // accumulator lanes 0..15 hold tokens 0..3
#pragma unroll
			for (int v = 0; v < MR; ++v) atomicAdd(&sum[tt][v][ri], ac[v]);
		}
	}
	__syncthreads();
	int32_t* plane = g.split_part + (size_t)split * g.M * g.N;
	for (int i = threadIdx.x; i < NTB * MR * 16; i += 512) {
		const int tt = i / (MR * 16), rem = i - tt * MR * 16, tk = rem >> 4, j = (tile0 + tt) * 16 + (rem & 15);
		if (tk < M && j < g.N) plane[(size_t)tk * g.N + j] = sum[tt][tk][rem & 15];
	}
}

}  // namespace sslm

namespace sslm_launch {

// chunks per wave of the four-wave kernels: 0 when none covers C
static int chain_cpw(int C) {
	for (int w : {2, 3, 4, 7})
		if (C <= kCW * w) return w;
	return 0;
}
// tiles per block of the q|k|v and gate|up launches
static int chain_nt(int T, bool funnel) {
	const int need = (T + device_cus() - 1) / device_cus();
	if (!funnel) return need <= 1 ? 1 : (need == 2 ? 2 : 0);
	for (int nt : {2, 3, 5, 10})
		if (need <= nt) return nt;
	return 0;
}
static int act_cpw(int C) { return (C + 63) / 64; }  // k_gemv_sk's: 8 waves, at most kMaxRawSplits planes
static int act_ntb(int N, int splits) {
	const int need = ((N + 15) / 16 * splits + device_cus() - 1) / device_cus();
	for (int n : {2, 4, 7})
		if (need <= n) return n;
	return 0;
}

// Rows past kChainRows and the second to fourth row's residual: the header's figures.  The other limits are
// what the kernels hold, not lines between two measured forms: k_act_gemv writes the split-K planes
// that the down GEMV has past I = 4096 only (up to there it runs unsplit in k_gemv_pk); a wave reads one maximum per
// lane (NH); an adapter's u = A x needs the codes in memory before the GEMV that k_funnel_gemv and
// k_act_gemv derive them in, so the caller takes no layer with an adapter here.
bool decode_chain_ok(int M, int H, int NH, int KVH, int I) {
	if (M < 1 || M > kChainRows || H % 128 || I % 128 || I <= 4096 || NH > 64) return false;
	const int C = H / 128, cpw = chain_cpw(C), ac = act_cpw(I / 128), planes = packed_planes(M, H, I);
	if (cpw == 0 || (H + 15) / 16 > device_cus()) return false;
	if (M == 1 && (!chain_nt((H + 2 * KVH + 15) / 16, false) || !chain_nt((2 * I + 15) / 16, true))) return false;
	return planes >= 1 && ac >= 1 && ac <= 3 && planes == (I / 128 + 8 * ac - 1) / (8 * ac) && act_ntb(H, planes) != 0;
}

template <int CPW>
static bool launch_residual_cpw(const GemmArgs& g, const ResidualArgs& a, bool funnel, int nt, dim3 grid, hipStream_t s) {
	const dim3 block(512);
	if (!funnel) {
		if (nt == 1) hipLaunchKernelGGL((k_residual_gemv<1, CPW, false, kMaxRawSplits>), grid, block, 0, s, g, a);
		else hipLaunchKernelGGL((k_residual_gemv<2, CPW, false, kMaxRawSplits>), grid, block, 0, s, g, a);
		return true;
	}
	switch (nt) {
#define X(N) \
	case N: hipLaunchKernelGGL((k_residual_gemv<N, CPW, true, 1>), grid, block, 0, s, g, a); return true;
		X(2) X(3) X(5) X(10)
#undef X
	}
	return false;
}

void residual_gemv(const GemmArgs& g, const ResidualArgs& a, hipStream_t s) {
	const int T = (g.N + 15) / 16, cpw = chain_cpw(g.K / 128);
	bool funnel = true;
	for (int i = 0; i < g.epi.nseg; ++i) funnel = funnel && g.epi.seg[i].mode == kSegFunnel && !g.epi.seg[i].bias;
	const int nt = chain_nt(T, funnel);
	const dim3 grid(nt ? (T + nt - 1) / nt : 1);
	bool ok = nt && g.wp && a.raw.part && a.gain && a.M == 1 && g.M == 1 && a.H == g.K &&
	          (funnel ? a.raw.splits == 1 : a.raw.splits <= kMaxRawSplits);
	if (ok) {
		switch (cpw) {
#define X(W) \
	case W: ok = launch_residual_cpw<W>(g, a, funnel, nt, grid, s); break;
			X(2) X(3) X(4) X(7)
#undef X
			default: ok = false;
		}
	}
	if (!ok) throw LaunchRefused{"residual_gemv"};
}

void funnel_gemv(const GemmArgs& g, const FunnelArgs& a, hipStream_t s) {
	const dim3 grid((g.N + 15) / 16), block(64 * kCW);
	if (!g.wp || !g.epi.raw_out || !a.head_status || a.incoming || a.ntiles > 64 || a.M != g.M || a.N != g.K || a.M > kChainRows)
		throw LaunchRefused{"funnel_gemv"};
	switch (chain_cpw(g.K / 128)) {
#define X(W)                                                                                      \
	case W:                                                                                       \
		if (a.M == 1) hipLaunchKernelGGL((k_funnel_gemv<1, W>), grid, block, 0, s, g, a);          \
		else hipLaunchKernelGGL((k_funnel_gemv<4, W>), grid, block, 0, s, g, a);                   \
		return;
		X(2) X(3) X(4) X(7)
#undef X
	}
	throw LaunchRefused{"funnel_gemv"};
}

template <int MR, int NTB>
static bool launch_act_ntb(const GemmArgs& g, const ActArgs& a, int slices, int cpw, hipStream_t s) {
	const dim3 grid(((g.N + 15) / 16 + NTB - 1) / NTB, g.splits), block(512);
	switch (cpw) {
#define X(W) \
	case W: hipLaunchKernelGGL((k_act_gemv<MR, NTB, W>), grid, block, 0, s, g, a, slices); return true;
		X(1) X(2) X(3)
#undef X
	}
	return false;
}

void act_gemv(const GemmArgs& g, const ActArgs& a, hipStream_t s) {
	const int C = g.K / 128, cpw = act_cpw(C), slices = act_slices(a.I);
	bool ok = g.wp && g.split_part && a.M == g.M && a.M <= kChainRows && a.I == g.K && slices <= 64 &&
	          cpw >= 1 && g.splits == (C + 8 * cpw - 1) / (8 * cpw);
	if (ok) {
		switch (act_ntb(g.N, g.splits)) {
#define X(N) \
	case N: ok = a.M == 1 ? launch_act_ntb<1, N>(g, a, slices, cpw, s) : launch_act_ntb<4, N>(g, a, slices, cpw, s); break;
			X(2) X(4) X(7)
#undef X
			default: ok = false;
		}
	}
	if (!ok) throw LaunchRefused{"act_gemv"};
}

}  // namespace sslm_launch
