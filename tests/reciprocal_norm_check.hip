// Device check of the double-estimate forms of superslm_amd/csrc/int_math.h whose GPU branch starts from a
// hardware estimate, which no host check compiles:
// - reciprocal_norm, the reciprocal every funnel plan uses: for every normalized divisor dn in
//   [2^30, 2^31) equal to reciprocal_div (round_half_up(2^62 / dn), the value the reference's
//   corrected-Newton DynamicScaleReciprocal returns, src/intmath.cpp:303-333), which the host tests pin
//   against the oracle; and the plan's factor f equal to 127 r 2^-(62-s);
// - rcp_est: within 2^-40 of 1 / d for every integer d in [1, 2^24];
// - rms_root: for every row length h in [1, 2^13], the largest r with r^2 h <= ss 2^32 (at least 1), over
//   sums ss spread evenly, and at and beside those where the root steps;
// - norm_qd on rcp_est: floor(v 2^32 / root) for every code v and every root in [1, 2^23].
// Prints each mismatch count; exit status 0 only when all are zero.
#include <hip/hip_runtime.h>
#include <cstdio>
#include "int_math.h"
using namespace sslm;

struct Count {
	unsigned long long bad;
	long long first;  // smallest failing argument
};

__device__ void report(Count* c, unsigned long long nb, long long fb) {
	if (nb) {
		atomicAdd(&c->bad, nb);
		atomicMin(&c->first, fb);
	}
}

#define FOR_ALL(i, n) for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < (n); i += (int64_t)gridDim.x * blockDim.x)
#define MISS(x) (++nb, fb = fb < (x) ? fb : (x))

__global__ void k_recip(Count* c) {
	const int64_t base = (int64_t)1 << 30;
	unsigned long long nb = 0;
	long long fb = (long long)1 << 40;
	FOR_ALL(i, base) {
		const int64_t dn = base + i;
		const int64_t r = reciprocal_div(dn);
		if (reciprocal_norm(dn) != r) MISS(dn);
		// the plan of a maximum that normalizes to dn, at one of the 32 shifts (dn's low bits dropped)
		const int sh = (int)(i & 31);
		FunnelPlan p;
		const uint64_t d = sh < 31 ? (uint64_t)dn >> sh : (uint64_t)1 << 31;
		int s;
		const int64_t nd = normalize_scale((int64_t)d, &s);
		if (funnel_plan(d, nullptr, 0, Scale{(int64_t)1 << 30, -40}, &p) != kOk || p.s != s || p.r != reciprocal_div(nd) ||
		    p.f != ldexp((double)(p.r * 127), p.s - 62))
			MISS(dn);
	}
	report(c, nb, fb);
}

__global__ void k_rcp_est(Count* c) {
	unsigned long long nb = 0;
	long long fb = (long long)1 << 40;
	FOR_ALL(i, (int64_t)1 << 24) {
		const double d = (double)(i + 1);
		if (!(fabs(fma(rcp_est(d), d, -1.0)) <= 0x1p-40)) MISS(i + 1);
	}
	report(c, nb, fb);
}

// r is the root of ss / h
__device__ bool is_root(int64_t r, int64_t ss, int64_t h) {
	const int64_t n = ss << 32;
	if (n < h) return r == 1;
	return r >= 1 && r * r * h <= n && (r + 1) * (r + 1) * h > n;
}
constexpr int kSums = 4096;  // sums per row length, of each kind
__global__ void k_rms_root(Count* c) {
	unsigned long long nb = 0;
	long long fb = (long long)1 << 40;
	FOR_ALL(i, (int64_t)8192 * kSums) {
		const int64_t h = i / kSums + 1, j = i % kSums, top = h << 14;
		auto check = [&](int64_t ss) {
			if (ss >= 0 && ss <= top && !is_root(rms_root((int32_t)ss, (int32_t)h), ss, h)) MISS(h);
		};
		check(j);
		check(top * j / (kSums - 1));
		const int64_t r = ((int64_t)1 << 23) * (j + 1) / kSums;  // the first sum whose root is r, and its neighbours
		const int64_t s0 = (r * r * h + 0xffffffffll) >> 32;
		for (int64_t d = -2; d <= 2; ++d) check(s0 + d);
	}
	report(c, nb, fb);
}

__global__ void k_norm(Count* c) {
	unsigned long long nb = 0;
	long long fb = (long long)1 << 40;
	FOR_ALL(i, (int64_t)1 << 23) {
		const int64_t root = i + 1;
		const double rd = (double)root, inv = rcp_est(rd);
		for (int v = -128; v < 128; ++v) {
			const int64_t q = (int64_t)norm_qd(v, rd, inv), n = (int64_t)v * 4294967296ll;
			if (!(q * root <= n && n < (q + 1) * root)) MISS(root);
		}
	}
	report(c, nb, fb);
}

static int run(const char* what, void (*k)(Count*)) {
	Count* c;
	Count z{0, (long long)1 << 40};
	if (hipMalloc(&c, sizeof z) != hipSuccess || hipMemcpy(c, &z, sizeof z, hipMemcpyHostToDevice) != hipSuccess) return 2;
	k<<<8192, 256>>>(c);
	if (hipGetLastError() != hipSuccess || hipDeviceSynchronize() != hipSuccess) return 2;
	if (hipMemcpy(&z, c, sizeof z, hipMemcpyDeviceToHost) != hipSuccess || hipFree(c) != hipSuccess) return 2;
	printf("%s: %llu mismatches\n", what, z.bad);
	if (z.bad) printf("first mismatch at %lld\n", z.first);
	fflush(stdout);
	return z.bad != 0;
}

int main() {
	int rc = run("reciprocal_norm and plan factor over every dn in [2^30, 2^31)", k_recip);
	if (rc < 2) rc |= run("rcp_est over every d in [1, 2^24]", k_rcp_est);
	if (rc < 2) rc |= run("rms_root over every h in [1, 2^13]", k_rms_root);
	if (rc < 2) rc |= run("norm_qd over every code and root in [1, 2^23]", k_norm);
	return rc;
}
