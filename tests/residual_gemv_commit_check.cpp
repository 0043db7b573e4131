// sslm_launch::residual_gemv in its q|k|v form (one row: down funnel, residual, norm of layer l, then the
// q|k|v GEMV of layer l + 1) with the slot's status word as other blocks of the launch, or earlier
// launches, may have left it.  A refusal of layer l + 1 -- which any block of this launch may report before a
// late block has read the word -- must not keep layer l's stream row, its scale and its norm from
// being written; a refusal of layer l or before must.  Every case is set by the host before the launch.
// Prints "ok" and exits 0 when every case agrees.
#include <hip/hip_runtime.h>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "kernels.h"

using namespace sslm;
using namespace sslm_launch;

constexpr int H = 256, KVH = 128, N = H + 2 * KVH, kLayer = 3;

static void ck(hipError_t e, const char* what) {
	if (e == hipSuccess) return;
	printf("%s: %s\n", what, hipGetErrorString(e));
	exit(2);
}
template <typename T>
static T* dev(const std::vector<T>& v) {
	T* p = nullptr;
	ck(hipMalloc(&p, v.size() * sizeof(T)), "hipMalloc");
	ck(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice), "upload");
	return p;
}
template <typename T>
static std::vector<T> host(const T* p, size_t n) {
	std::vector<T> v(n);
	ck(hipMemcpy(v.data(), p, n * sizeof(T), hipMemcpyDeviceToHost), "read back");
	return v;
}

struct Outcome {
	std::vector<int8_t> stream, norm;
	std::vector<Scale> scale, norm_scale;
	std::vector<int64_t> recip, kv;
	std::vector<int32_t> q;
	int32_t status;
	bool same_rows(const Outcome& o) const {
		return stream == o.stream && norm == o.norm && recip == o.recip &&
		       !memcmp(scale.data(), o.scale.data(), sizeof(Scale)) &&
		       !memcmp(norm_scale.data(), o.norm_scale.data(), sizeof(Scale));
	}
};

int main() {
	std::mt19937_64 rng(5);
	auto uni = [&](int64_t lo, int64_t hi) { return lo + (int64_t)(rng() % (uint64_t)(hi - lo + 1)); };
	std::vector<int32_t> raw(H), gain(H), fold(3 * N, 0), rfold(3 * H, 0);
	std::vector<int8_t> stream(H), wp(packed_bytes(N, H));
	uint32_t mx = 0;
	for (int j = 0; j < H; ++j) {
		raw[j] = (int32_t)uni(-(1 << 20), 1 << 20);
		gain[j] = (int32_t)uni(-127, 127);
		stream[j] = (int8_t)uni(-127, 127);
		rfold[3 * j + 1] = (int32_t)uni(1LL << 30, (1LL << 31) - 1);
		rfold[3 * j + 2] = (int32_t)uni(0, 3);
		const int32_t v = fold_bounded(raw[j], fold_consts(0, rfold[3 * j + 1], rfold[3 * j + 2]));
		mx = std::max(mx, (uint32_t)(v < 0 ? -v : v));
	}
	for (int j = 0; j < N; ++j) {
		fold[3 * j + 1] = (int32_t)uni(1LL << 30, (1LL << 31) - 1);
		fold[3 * j + 2] = (int32_t)uni(0, 3);
	}
	for (auto& b : wp) b = (int8_t)uni(-127, 127);
	// the stream's scale a power of two above the branch's, so that the landed codes stay in range
	const Scale in{1LL << 30, -37}, site{1518500250, -45};
	FunnelPlan bp;
	if (funnel_plan(mx, &in, 1, site, &bp) != kOk) return printf("the branch is refused\n"), 2;
	const Scale ss{1288490189, bp.out.e + 1};

	ResidualArgs a{};
	a.M = 1;
	a.H = H;
	a.tok = dev(std::vector<TokenInfo>(1, TokenInfo{0, 0, 0}));
	a.raw.part = dev(raw);
	a.raw.splits = 1;
	a.raw.ld = H;
	a.raw.epi.nseg = 1;
	a.raw.epi.seg[0].n_end = H;
	a.raw.epi.seg[0].fold = dev(rfold);
	a.branch_in = dev(std::vector<Scale>(1, in));
	a.branch_site = site;
	a.stream = dev(stream);
	const int32_t* zero = dev(std::vector<int32_t>(1, 0));
	a.stream_idx = zero;
	a.out_idx = zero;
	a.stream_scale = dev(std::vector<Scale>(1, ss));
	a.res_site = Scale{1082196484, -37};
	a.out_stream = dev(std::vector<int8_t>(H));
	a.out_stream_scale = dev(std::vector<Scale>(1));
	a.gain = dev(gain);
	// puts the norm's carried exponent near -71: a bias code b reconciles to about b 2^10, refused past int64
	a.norm_site = Scale{1082196484, -96};
	a.norm_out = dev(std::vector<int8_t>(H));
	a.norm_scale = dev(std::vector<Scale>(1));
	a.norm_recip = dev(std::vector<int64_t>(1));
	a.layer = kLayer;
	int32_t* status = dev(std::vector<int32_t>(1, 0));
	a.status = status;

	GemmArgs g{};
	g.wp = dev(wp);
	g.w = g.wp;
	g.M = 1;
	g.N = N;
	g.K = g.lda = H;
	g.epi.tok = a.tok;
	g.epi.status = status;
	g.epi.layer = kLayer + 1;
	g.epi.nseg = 3;
	int32_t* q = dev(std::vector<int32_t>(H));
	uint32_t* qmax = dev(std::vector<uint32_t>((size_t)N / 16 * kPartLd));
	int64_t* kv = dev(std::vector<int64_t>(2 * KVH));
	const int32_t* dfold = dev(fold);
	// a bias that every reconcile accepts, and one that every reconcile refuses
	const int64_t* mild = dev(std::vector<int64_t>(N, 12345));
	const int64_t* wild = dev(std::vector<int64_t>(N, 1LL << 62));
	const int begin[4] = {0, H, H + KVH, N};
	for (int i = 0; i < 3; ++i) {
		Segment& s = g.epi.seg[i];
		s.n_begin = begin[i];
		s.n_end = begin[i + 1];
		s.mode = i ? kSegWide : kSegFunnel;
		s.out = i ? (void*)(kv + (i - 1) * KVH) : (void*)q;
		s.ld_out = i ? 2 * KVH : H;
		s.maxpart = i ? nullptr : qmax;
		s.fold = dfold + 3 * begin[i];
	}
	if (!decode_chain_ok(1, H, 4, KVH, 4352)) return printf("the shape is not taken\n"), 2;

	auto run = [&](int32_t word, const int64_t* bias) {
		for (int i = 0; i < 3; ++i) g.epi.seg[i].bias = bias + begin[i];
		ck(hipMemset(a.out_stream, 0x55, H), "fill");
		ck(hipMemset(a.out_stream_scale, 0x55, sizeof(Scale)), "fill");
		ck(hipMemset(a.norm_out, 0x55, H), "fill");
		ck(hipMemset(a.norm_scale, 0x55, sizeof(Scale)), "fill");
		ck(hipMemset(a.norm_recip, 0x55, 8), "fill");
		ck(hipMemcpy(status, &word, 4, hipMemcpyHostToDevice), "status");
		residual_gemv(g, a, nullptr);
		ck(hipGetLastError(), "launch");
		ck(hipDeviceSynchronize(), "kernel");
		return Outcome{host(a.out_stream, H), host(a.norm_out, H), host(a.out_stream_scale, 1), host(a.norm_scale, 1),
		               host(a.norm_recip, 1), host(kv, 2 * KVH), host(q, H), host(status, 1)[0]};
	};
	int bad = 0;
	auto expect = [&](bool ok, const char* what) {
		if (!ok) printf("FAIL %s\n", what), ++bad;
	};
	const Outcome clean = run(0, mild);
	Outcome none = clean;
	memset(none.stream.data(), 0x55, H);
	memset(none.norm.data(), 0x55, H);
	memset(none.scale.data(), 0x55, sizeof(Scale));
	memset(none.norm_scale.data(), 0x55, sizeof(Scale));
	memset(none.recip.data(), 0x55, 8);
	expect(clean.status == 0, "the clean row is refused");
	expect(clean.stream != none.stream && clean.norm != none.norm, "the clean row is not written");
	for (int later = kLayer + 1; later < kLayer + 3; ++later) {
		const int32_t word = status_word(later, kBiasReconcileProductOutOfDomain);
		const Outcome o = run(word, mild);
		expect(o.same_rows(clean), "a later layer's refusal kept the row from being committed");
		expect(o.q == clean.q && o.kv == clean.kv, "a later layer's refusal changed the projection");
		expect(o.status == word, "a later layer's refusal was overwritten");
	}
	for (int l : {0, kLayer - 1, kLayer}) {
		const int32_t word = status_word(l, kChainInputOutOfDomain);
		const Outcome o = run(word, mild);
		expect(o.same_rows(none), "a refused row was written");
		expect(o.status == word, "a refusal was overwritten");
	}
	const Outcome w = run(0, wild);
	expect(w.status == status_word(kLayer + 1, kBiasReconcileProductOutOfDomain), "the bias refusal is not reported");
	expect(w.same_rows(clean), "the bias refusal kept the row from being committed");
	if (bad) return 1;
	printf("ok\n");
	return 0;
}
