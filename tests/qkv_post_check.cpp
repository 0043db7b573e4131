// sslm_launch::qkv_post at every spread of a row over its threads (up to three slots evenly, past that by
// kind), with rows a thread, a wave or a slot short of full, against the same steps one value at a time on the
// host: fold, bias, landing by the 128-bit form, q funnel, RoPE.  Inputs: fold outputs, or raw planes (one,
// three, eight; with and without a bias); outputs: the pool, or a prefill span's staging rows.
// Prints "ok" and exits 0 when every case agrees.
#include <hip/hip_runtime.h>
#include <cstdio>
#include <cstring>
#include <random>
#include <vector>

#include "kernels.h"

using namespace sslm;
using namespace sslm_launch;

constexpr int kM = 5, kCap = 8;

static void ck(hipError_t e, const char* what) {
	if (e == hipSuccess) return;
	printf("%s: %s\n", what, hipGetErrorString(e));
	exit(2);
}
static std::vector<void*> g_dev;
template <typename T>
static T* dev(const std::vector<T>& v) {
	T* p = nullptr;
	ck(hipMalloc(&p, v.size() * sizeof(T)), "hipMalloc");
	ck(hipMemcpy(p, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice), "upload");
	g_dev.push_back(p);
	return p;
}
template <typename T>
static std::vector<T> host(const T* p, size_t n) {
	std::vector<T> v(n);
	ck(hipMemcpy(v.data(), p, n * sizeof(T), hipMemcpyDeviceToHost), "read back");
	return v;
}

struct Shape {
	int H, NKV, D;
};

static int g_bad = 0;

static void run(const Shape& sh, int planes, bool bias, bool staged) {
	const int H = sh.H, D = sh.D, KVH = sh.NKV * D, N = H + 2 * KVH, pairs = D / 2;
	printf("case H=%d KVH=%d D=%d planes=%d bias=%d staged=%d\n", H, KVH, D, planes, bias, staged);
	fflush(stdout);
	std::mt19937_64 rng(H * 131 + KVH * 7 + planes * 3 + bias);
	auto uni = [&](int64_t lo, int64_t hi) { return lo + (int64_t)(rng() % (uint64_t)(hi - lo + 1)); };
	// ---- inputs ----
	const std::vector<Scale> ns(kM, Scale{1288490189, -50});
	std::vector<int64_t> recip(kM, reciprocal_div(ns[0].m));
	std::vector<int64_t> val((size_t)kM * N);  // the projection's values, before the landing and the funnel
	std::vector<int32_t> part, fold(3 * N, 0);
	std::vector<int64_t> b(N);
	for (int j = 0; j < N; ++j) {
		fold[3 * j] = uni(0, 40) == 0;
		fold[3 * j + 1] = (int32_t)uni(1LL << 30, (1LL << 31) - 1);
		fold[3 * j + 2] = (int32_t)uni(0, 4);
		b[j] = uni(-(1LL << 31), 1LL << 31);  // terms up to 2^21
	}
	if (planes) {
		part.resize((size_t)planes * kM * N);
		for (auto& x : part) x = (int32_t)uni(-(1 << 22), 1 << 22);
		for (int t = 0; t < kM; ++t)
			for (int j = 0; j < N; ++j) {
				int64_t acc = 0;
				for (int s = 0; s < planes; ++s) acc += part[((size_t)s * kM + t) * N + j];
				int64_t v = apply_fold(acc, fold[3 * j], fold[3 * j + 1], fold[3 * j + 2]), term = 0;
				if (bias) {
					if (!bias_term(b[j], recip[t], ns[t].e, v, &term)) printf("a bias is refused\n"), exit(2);
					v += term;
				}
				val[(size_t)t * N + j] = v;
			}
	} else {
		for (int t = 0; t < kM; ++t)
			for (int j = 0; j < N; ++j) val[(size_t)t * N + j] = uni(-(1 << 22), 1 << 22);
	}
	std::vector<int64_t> rt[2], et[2];  // K, V
	for (int kind = 0; kind < 2; ++kind)
		for (int h = 0; h < sh.NKV; ++h) {
			rt[kind].push_back(uni((1LL << 31) + 1, 1LL << 32));
			et[kind].push_back(ns[0].e + 13 + h % 5);  // codes around +-127: some clamp
		}
	std::vector<int64_t> cs((size_t)kCap * pairs), sn((size_t)kCap * pairs);
	for (auto& x : cs) x = uni(-(1LL << 30), 1LL << 30);
	for (auto& x : sn) x = uni(-(1LL << 30), 1LL << 30);
	std::vector<TokenInfo> tok(kM);
	for (int t = 0; t < kM; ++t) tok[t] = staged ? TokenInfo{1 + t, 0, 0} : TokenInfo{(3 * t + 1) % kCap, t, kM - 1 - t};
	const Scale site{1518500250, -45};
	// ---- the launch ----
	QkvPostArgs a{};
	a.M = kM;
	a.H = H;
	a.NH = H / D;
	a.NKV = sh.NKV;
	a.D = D;
	a.cap = kCap;
	a.tok = dev(tok);
	a.in_scale = dev(ns);
	a.q_site = site;
	a.r_t_k = dev(rt[0]);
	a.e_t_k = dev(et[0]);
	a.r_t_v = dev(rt[1]);
	a.e_t_v = dev(et[1]);
	a.rope_cos = dev(cs);
	a.rope_sin = dev(sn);
	if (planes) {
		a.raw.part = dev(part);
		a.raw.splits = planes;
		a.raw.ld = N;
		a.raw.epi.nseg = 3;
		const int32_t* df = dev(fold);
		const int64_t* db = bias ? dev(b) : nullptr;
		const int begin[4] = {0, H, H + KVH, N};
		for (int i = 0; i < 3; ++i) {
			a.raw.epi.seg[i].n_begin = begin[i];
			a.raw.epi.seg[i].n_end = begin[i + 1];
			a.raw.epi.seg[i].fold = df + 3 * begin[i];
			a.raw.epi.seg[i].bias = db ? db + begin[i] : nullptr;
		}
		a.raw.epi.in_recip = dev(recip);
		a.raw.epi.in_scale = a.in_scale;
	} else {
		std::vector<int32_t> q((size_t)kM * H);
		std::vector<int64_t> kv((size_t)kM * 2 * KVH);
		std::vector<uint32_t> mx((size_t)H / 16 * kPartLd, 0);
		for (int t = 0; t < kM; ++t) {
			for (int j = 0; j < H; ++j) {
				const int64_t v = val[(size_t)t * N + j];
				q[(size_t)t * H + j] = (int32_t)v;
				uint32_t& m = mx[(size_t)(j / 16) * kPartLd + t];
				m = std::max(m, (uint32_t)(v < 0 ? -v : v));
			}
			for (int j = 0; j < 2 * KVH; ++j) kv[(size_t)t * 2 * KVH + j] = val[(size_t)t * N + H + j];
		}
		a.q_f = dev(q);
		a.q_maxpart = dev(mx);
		a.kv_f = dev(kv);
	}
	const size_t block = (size_t)2 * 2 * kCap * KVH;  // two layers of K and V
	int8_t* pool = dev(std::vector<int8_t>(kM * block, 0x55));
	int8_t* stage = dev(std::vector<int8_t>((size_t)kM * 2 * KVH, 0x55));
	uint32_t* sat_stage = dev(std::vector<uint32_t>(kM, 0));
	a.kv_pool = pool;
	a.block_bytes = (int64_t)block;
	a.layer = 1;
	a.q_rot = dev(std::vector<int8_t>((size_t)kM * H, 0x55));
	a.q_scale = dev(std::vector<Scale>(kM));
	a.sat = dev(std::vector<unsigned long long>(kM, 0));
	a.status = dev(std::vector<int32_t>(kM, 0));
	if (staged) {
		a.kv_stage = stage;
		a.sat_stage = sat_stage;
	}
	qkv_post(a, nullptr);
	ck(hipGetLastError(), "launch");
	ck(hipDeviceSynchronize(), "kernel");
	// ---- the same on the host ----
	std::vector<int8_t> wq((size_t)kM * H), wpool(kM * block, 0x55), wstage((size_t)kM * 2 * KVH, 0x55);
	std::vector<Scale> wscale(kM);
	std::vector<uint64_t> wsat(kM, 0);
	for (int t = 0; t < kM; ++t) {
		const int64_t* v = &val[(size_t)t * N];
		const int64_t pos = tok[t].pos;
		uint64_t mx = 0;
		for (int j = 0; j < H; ++j) mx = std::max(mx, (uint64_t)(v[j] < 0 ? -v[j] : v[j]));
		FunnelPlan plan;
		if (funnel_plan(mx, &ns[t], 1, site, &plan) != kOk) printf("the q row is refused\n"), exit(2);
		wscale[t] = plan.out;
		for (int p = 0; p < H / 2; ++p) {
			int64_t x, y;
			rope_pair(requant_code_f(v[2 * p], plan.f), requant_code_f(v[2 * p + 1], plan.f), (int32_t)cs[pos * pairs + p % pairs],
			          (int32_t)sn[pos * pairs + p % pairs], &x, &y);
			wq[(size_t)t * H + 2 * p] = (int8_t)clamp_code(x);
			wq[(size_t)t * H + 2 * p + 1] = (int8_t)clamp_code(y);
		}
		for (int kind = 0; kind < 2; ++kind)
			for (int p = 0; p < KVH / 2; ++p) {
				const int h = 2 * p / D, i = p % pairs;
				const int64_t k = composed_exponent(ns[t].e, et[kind][h]);
				int64_t c[2];
				for (int u = 0; u < 2; ++u) {
					bool clamped, exceeded;
					c[u] = clamp_code(landing_rescale(v[H + kind * KVH + 2 * p + u], ns[t].m, rt[kind][h], k, &clamped, &exceeded));
					wsat[t] += clamped;
				}
				if (kind == 0) {
					int64_t x, y;
					rope_pair((int32_t)c[0], (int32_t)c[1], (int32_t)cs[pos * pairs + i], (int32_t)sn[pos * pairs + i], &x, &y);
					c[0] = clamp_code(x);
					c[1] = clamp_code(y);
				}
				int8_t* dst = staged ? &wstage[(size_t)t * 2 * KVH + kind * KVH + 2 * p]
				                     : &wpool[tok[t].block * block + (2 + kind) * (size_t)kCap * KVH + ((size_t)h * kCap + pos) * D + 2 * i];
				dst[0] = (int8_t)c[0];
				dst[1] = (int8_t)c[1];
			}
	}
	auto expect = [&](bool ok, const char* what) {
		if (!ok) printf("FAIL %s\n", what), ++g_bad;
	};
	uint64_t clamps = 0;
	for (uint64_t s : wsat) clamps += s;
	expect(clamps > 0 && clamps < (uint64_t)kM * 2 * KVH, "the inputs clamp some values, not all");
	expect(host(a.status, kM) == std::vector<int32_t>(kM, 0), "status");
	expect(host(a.q_rot, (size_t)kM * H) == wq, "q codes");
	const auto qs = host(a.q_scale, kM);
	expect(!memcmp(qs.data(), wscale.data(), kM * sizeof(Scale)), "q scales");
	expect(host(pool, kM * block) == wpool, "pool");
	expect(host(stage, (size_t)kM * 2 * KVH) == wstage, "staging rows");
	const auto s0 = host(a.sat, kM);
	const auto s1 = host(sat_stage, kM);
	for (int t = 0; t < kM; ++t) {
		expect(s0[t] == (staged ? 0 : wsat[t]), "clamp counts");
		expect(s1[t] == (staged ? wsat[t] : 0), "staged clamp counts");
	}
	for (void* p : g_dev) ck(hipFree(p), "hipFree");
	g_dev.clear();
}

int main() {
	// slots of q and of K and V at 512 threads (pairs past a full slot)
	const Shape shapes[] = {
	    {128, 2, 32},                  // one slot, partly filled
	    {896, 2, 64}, {1536, 2, 128},  // two: 576 pairs, 1,024
	    {2048, 8, 64},                 // three, full
	    {1984, 16, 64}, {1088, 32, 64},  // (2, 2), (2, 4)
	    {3008, 8, 64}, {3072, 8, 128},   // (3, 1), (3, 2)
	    {3584, 4, 128}, {4032, 9, 64}, {4096, 31, 64},  // (4, 1), (4, 2), (4, 4)
	    {4160, 9, 64}, {8192, 8, 256},   // (8, 2), (8, 4)
	};
	for (const Shape& sh : shapes) {
		for (int planes : {0, 1, 3, 8}) run(sh, planes, planes == 1 || planes == 3, planes != 3);
		run(sh, 0, false, false);
	}
	if (g_bad) return 1;
	printf("ok\n");
	return 0;
}
