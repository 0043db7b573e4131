"""GEMMs whose depth K is a multiple of 16 but not of 128 (the last 128-deep step is partly past K), and
launches of few large tiles (64 x 64 tiles with the funnel epilogue): raw int32 sums against exact
integer products, and GEMM + fold + requant against the oracle, at the edges of rows, columns and K."""
import numpy as np
import pytest

from superslm_amd.device import Device
from test_gpu_gemm import IN_SCALE, SITE, _lib

pytestmark = pytest.mark.gpu


def _inputs(m, n, k):
    rng = np.random.default_rng(m * 7919 + n * 31 + k)
    a = rng.integers(-127, 128, size=(m, k), dtype=np.int8)
    w = rng.integers(-127, 128, size=(n, k), dtype=np.int8)
    fold = np.zeros((n, 3), dtype=np.int32)
    fold[:, 0] = rng.random(n) < 0.02
    fold[:, 1] = rng.integers(1 << 30, 1 << 31, size=n, dtype=np.int64).astype(np.int32)
    fold[:, 2] = rng.integers(8, 21, size=n, dtype=np.int32)
    return a, w, fold


@pytest.mark.parametrize("m,n,k", [(1, 16, 16), (5, 33, 48), (16, 20000, 144), (17, 250, 1552), (33, 528, 624), (64, 77, 4080),
                                   (65, 79, 48), (100, 208, 240), (129, 1000, 1040), (257, 384, 112), (512, 272, 208),
                                   (300, 16512, 272)])
def test_ragged_raw_exact(m, n, k, hip_lib):
    L = _lib(hip_lib)
    dev = Device(hip_lib)
    a, w, _ = _inputs(m, n, k)
    want = (a.astype(np.float64) @ w.astype(np.float64).T).astype(np.int64)  # exact: |sums| < 2^53
    da, dw = dev.upload(a), dev.upload(w)
    out = dev.zeros((m, n), np.int32)
    print(f"case ragged raw m={m} n={n} k={k}", flush=True)
    assert L.sslm_hip_gemm_i32(da.ptr, dw.ptr, m, n, k, out.ptr) == 0
    assert np.array_equal(out.numpy(), want)


@pytest.mark.parametrize("m,n,k", [(1, 16, 16), (3, 48, 80), (16, 304, 144), (20, 64, 1552), (47, 528, 624), (64, 80, 4080),
                                   # 64 x 64 tiles: one row or column past a tile, and K a multiple of 128
                                   (65, 80, 48), (100, 208, 240), (203, 4880, 1552), (129, 64, 128), (192, 2064, 896),
                                   # larger tiles
                                   (512, 8192, 208), (300, 8176, 256), (512, 8192, 128)])
def test_ragged_requant_matches_oracle(m, n, k, hip_lib, oracle_lib):
    from oracle_bind import project_rows
    L = _lib(hip_lib)
    dev = Device(hip_lib)
    a, w, fold = _inputs(m, n, k)
    rows = np.unique(np.concatenate([np.arange(min(m, 3)), np.linspace(0, m - 1, 8).astype(int)]))
    codes_o, scales_o, st_o = project_rows(oracle_lib, a[rows], w, fold, IN_SCALE, SITE)
    da, dw, df = (dev.upload(x) for x in (a, w, fold))
    codes = dev.upload(np.full((m, n), 99, np.int8))
    me = dev.zeros((m, 2), np.int64)
    st = dev.upload(np.full((m,), 5, np.int32))
    print(f"case ragged requant m={m} n={n} k={k}", flush=True)
    assert L.sslm_hip_gemm_requant(da.ptr, dw.ptr, df.ptr, m, n, k, *IN_SCALE, *SITE, codes.ptr, me.ptr, st.ptr) == 0
    assert st.numpy()[rows].tolist() == st_o
    assert np.array_equal(codes.numpy()[rows], codes_o)
    assert [tuple(r) for r in me.numpy()[rows].tolist()] == scales_o


@pytest.mark.parametrize("off_a,off_w", [(4, 0), (0, 8), (12, 4)])
def test_ragged_operands_off_alignment(off_a, off_w, hip_lib):
    """Operands at any 4-byte address: past 64 rows they take the tiles that load through registers."""
    L = _lib(hip_lib)
    dev = Device(hip_lib)
    for m, n, k in [(65, 80, 48), (100, 208, 240), (300, 272, 1552)]:
        a, w, _ = _inputs(m, n, k)
        want = (a.astype(np.float64) @ w.astype(np.float64).T).astype(np.int64)
        da = dev.upload(np.concatenate([np.zeros(off_a, np.int8), a.ravel()]))
        dw = dev.upload(np.concatenate([np.zeros(off_w, np.int8), w.ravel()]))
        out = dev.zeros((m, n), np.int32)
        print(f"case ragged off alignment m={m} n={n} k={k} {off_a} {off_w}", flush=True)
        assert L.sslm_hip_gemm_i32(da.ptr + off_a, dw.ptr + off_w, m, n, k, out.ptr) == 0
        assert np.array_equal(out.numpy(), want)
