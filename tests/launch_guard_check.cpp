// Host-only check of the launch wrappers' guards (no GPU needed): a GEMM launch without a complete
// output and row launches that no kernel instance covers must throw sslm_launch::LaunchRefused
// before anything is enqueued.  Linked against libsslm_hip.so; prints "ok" on success.
#include <cstdio>

#include "../superslm_amd/csrc/kernels.h"

using namespace sslm_launch;

template <typename F>
static bool refuses(F&& f) {
	try {
		f();
	} catch (const LaunchRefused&) {
		return true;
	}
	return false;
}

int main() {
	int bad = 0;
	auto expect = [&](bool ok, const char* what) {
		if (!ok) {
			printf("FAIL %s\n", what);
			++bad;
		}
	};
	GemmArgs g{};
	g.M = 16;
	g.N = 256;
	g.K = 1024;
	g.lda = 1024;
	expect(refuses([&] { gemm(g, nullptr); }), "gemm without any output");
	g.epi.nseg = 1;
	g.epi.seg[0].n_begin = 0;
	g.epi.seg[0].n_end = 128;  // does not cover N
	int32_t f[4];
	int32_t fold[12];
	g.epi.seg[0].out = f;
	g.epi.seg[0].fold = fold;
	expect(refuses([&] { gemm(g, nullptr); }), "gemm whose segments stop short of N");
	g.epi.seg[0].n_end = 256;
	g.epi.seg[0].fold = nullptr;
	expect(refuses([&] { gemm(g, nullptr); }), "gemm segment without fold parameters");
	g.epi.seg[0].fold = fold;
	g.epi.seg[0].n_begin = 16;
	expect(refuses([&] { gemm(g, nullptr); }), "gemm segments not starting at column 0");
	g.epi.nseg = kMaxSeg + 1;
	expect(refuses([&] { gemm(g, nullptr); }), "gemm with too many segments");

	RowNormArgs rn{};
	expect(refuses([&] { rmsnorm(rn, 1, 1 << 20, nullptr, nullptr, 0, nullptr); }), "rmsnorm row too long");
	FunnelArgs fa{};
	fa.M = 1;
	fa.N = 1 << 20;
	expect(refuses([&] { funnel(fa, nullptr); }), "funnel row too long");
	ResidualArgs ra{};
	ra.M = 1;
	ra.H = 1 << 20;
	expect(refuses([&] { residual_norm(ra, nullptr); }), "residual row too long");
	ActArgs aa{};
	aa.M = 1;
	aa.I = 1 << 22;
	expect(refuses([&] { mlp_act(aa, nullptr); }), "mlp_act row too long");
	AttnArgs at{};
	at.M = 1;
	at.NH = 1;
	at.NKV = 1;
	at.D = 48;
	at.cap = 16;
	expect(refuses([&] { attention_decode(at, nullptr); }), "attention head_dim without an instance");
	QkvPostArgs qa{};
	qa.M = 1;
	qa.H = 1 << 20;
	expect(refuses([&] { qkv_post(qa, nullptr); }), "qkv_post row too long");
	// the fused decode attention past 64 rows: where a packed GEMV writes the projection and the grouped
	// kernel (caps from 1,024) runs in one round of one block per CU (256 without a GPU)
	const int cus = device_cus();
	expect(decode_fused_ok(64, 3584, 4, 512, 4608, true) && decode_fused_ok(64, 3584, 4, 512, 4608, false), "fused, 64 rows");
	expect(!decode_fused_ok(65, 3584, 4, 512, 4608, true) && !decode_fused_ok(128, 3584, 4, 512, 64, true), "not fused, depth");
	expect(decode_fused_ok(65, 1536, 2, 256, 1024, true) && decode_fused_ok(cus / 2, 1536, 2, 256, 1024, true), "fused, one round");
	expect(!decode_fused_ok(65, 1536, (cus + 64) / 65, 256, 1024, true), "not fused, two rounds of the grouped kernel");
	expect(decode_fused_ok(128, 1024, 16, 1024, 512, true), "fused, one block per head");
	expect(!decode_fused_ok(65, 1536, 2, 256, 1024, false) && !decode_fused_ok(129, 1536, 1, 128, 1024, true), "not fused, no packed launch");
	// the sliced SiLU up to 64 rows
	ActArgs sl{};
	sl.I = 8960;
	sl.prod = &f[0];
	sl.act_maxpart = (uint32_t*)f;
	sl.gu_scale = (Scale*)fold;
	sl.M = 64;
	expect(mlp_act_sliced_ok(sl), "sliced SiLU, 64 rows");
	sl.M = 65;
	expect(!mlp_act_sliced_ok(sl), "no sliced SiLU, 65 rows");
	// direct loads to LDS at ragged depths only from rows of 16-byte alignment
	GemmArgs al{};
	al.K = al.lda = 208;
	for (int off = 0; off < 32; ++off) {
		al.a = (const int8_t*)(uintptr_t)(4096 + off);
		al.w = (const int8_t*)(uintptr_t)8192;
		expect(gemm_lds_loads_ok(al) == (off % 16 == 0), "alignment of the activations");
		al.a = (const int8_t*)(uintptr_t)4096;
		al.w = (const int8_t*)(uintptr_t)(8192 + off);
		expect(gemm_lds_loads_ok(al) == (off % 16 == 0), "alignment of the weights");
	}
	if (bad) return 1;
	printf("ok\n");
	return 0;
}
