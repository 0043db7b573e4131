"""Decode of one to four sequences, where each funnel runs inside the GEMV that reads its codes: tokens
and KV against the C oracle over geometries that take each kernel instance, and refusals (a
pending token whose embedding is zero; at layer 1 a bias out of range, i-exp constants out of range in
one KV group's heads, a branch that dwarfs the residual stream) against the same sequences decoded
in a larger batch, whose row kernels are launches of their own."""
import struct

import numpy as np
import pytest

from oracle_bind import OracleModel
from superslm_amd.sslm import Model
from superslm_amd.sslm_artifact import ModelConfig, build_synthetic, with_weight_rows

pytestmark = pytest.mark.gpu

CURRENT_TOKEN_OFFSET = 72  # SSB3 blob: the pending token
BAD = 5


def _cfg(hidden, heads, kv, inter, bias=False, layers=2):
    return ModelConfig(hidden=hidden, layers=layers, heads=heads, kv_heads=kv, head_dim=hidden // heads, inter=inter,
                       vocab=512, context_cap=64, tie_embeddings=True, with_bias=bias)


SHAPES = {  # chunks per wave, tiles per block of gate|up, split of down
    "c2": _cfg(256, 4, 2, 4352, bias=True, layers=3),
    "c3": _cfg(1536, 12, 2, 4224, bias=True),
    "c4": _cfg(2048, 16, 2, 8960),
    "c7": _cfg(3584, 28, 4, 4224, bias=True),
    "wide_ffn": _cfg(896, 7, 1, 18944),
}
_MODELS = {}


def _model(name):
    if name not in _MODELS:
        _MODELS[name] = build_synthetic(SHAPES[name], seed=23)
    return _MODELS[name]


@pytest.mark.parametrize("shape", sorted(SHAPES))
@pytest.mark.parametrize("batch", [1, 2, 3, 4])
def test_chain_matches_oracle(shape, batch, hip_lib, oracle_lib):
    sm = _model(shape)
    L = sm.config.layers
    rng = np.random.default_rng(batch)
    prompts = [rng.integers(0, sm.config.vocab, size=3 + i) for i in range(batch)]
    om = OracleModel(oracle_lib, sm)
    want, kv = [], []
    for p in prompts:
        s = om.new_seq()
        assert s.prefill(p) == (0, len(p))
        toks = [s.decode_step(L) for _ in range(3)]
        assert all(st == 0 for st, _ in toks)
        want.append([t for _, t in toks])
        kv.append(s.kv)
    print(f"case chain {shape} batch={batch}", flush=True)
    model = Model(hip_lib, sm.to_array())
    pool = model.pool(batch)
    seqs = [pool.seq() for _ in prompts]
    for s, p in zip(seqs, prompts):
        assert s.prefill(p) == len(p)
    got = [model.decode_step(seqs, L) for _ in range(3)]
    assert [list(x) for x in zip(*got)] == want, "tokens differ"
    for i in range(batch):  # a sequence owns the block at the back of the pool's free list
        assert np.array_equal(pool.kv_block(batch - 1 - i), kv[i]), f"KV of sequence {i} differs"
    for s in seqs:
        s.release()
    pool.close()
    model.close()


def _bias_edit(m):
    m.biases["layer1.q_proj"] = (m.biases["layer1.q_proj"] * (1 << 34)).astype(np.int64)


def _scale_edit(**shifts):
    """Site constants of layer 0 and 1 (`l<layer>_<site>`) shifted by powers of two."""
    def edit(m):
        for name, shift in shifts.items():
            key = f"layer{name[1]}.{name[3:]}"
            sm, se = m.consts[key]
            m.consts[key] = (sm, se + shift)
    return edit


# layer 1 refuses in the attention (resolved and cleared by the context funnel inside the o GEMV), or in
# the residual after the o or down projection: a landed value past 2^31, or past int64
EDITS = {
    "bias": _bias_edit,
    "attn_high": _scale_edit(l1_softmax_khead1=40),
    "attn_low": _scale_edit(l1_softmax_khead1=-40),
    "o_wide": _scale_edit(l1_o_proj=40),
    "o_past_int64": _scale_edit(l0_mlp_residual=-40, l1_o_proj=40),
    "down_wide": _scale_edit(l1_down_proj=40),
    "down_past_int64": _scale_edit(l1_attn_residual=-40, l1_down_proj=40),
}


def _blobs(hip_lib, art, n, bad_at):
    """n saved sequences with a pending token each, sequence `bad_at`'s the zero-embedding one."""
    model = Model(hip_lib, art)
    pool = model.pool(1)
    out = []
    for i in range(n):
        s = pool.seq()
        b = bytearray(s.save())
        struct.pack_into("<i", b, CURRENT_TOKEN_OFFSET, BAD if i == bad_at else 20 + i)
        out.append(bytes(b))
        s.release()
    pool.close()
    return model, out


def _decode(model, blobs, budget, calls):
    pool = model.pool(len(blobs))
    seqs = [pool.restore(b) for b in blobs]
    got = []
    for _ in range(calls):
        st, toks = model.decode_step(seqs, budget, raw=True)
        got.append((st, toks, [s.save() for s in seqs]))
    for s in seqs:
        s.release()
    pool.close()
    return got


@pytest.mark.parametrize("kind,batch,bad_at", [("zero", 1, 0), ("zero", 3, 1), ("zero", 4, 3), ("bias", 1, -1), ("bias", 4, -1),
                                               ("clean", 4, -1)] +
                         [(k, b, -1) for k in EDITS if k != "bias" for b in (1, 3, 4)])
@pytest.mark.parametrize("budget", [3, 2, 1])
def test_chain_refusals_match_row_kernels(kind, batch, bad_at, budget, hip_lib):
    sm = build_synthetic(SHAPES["c2"], seed=23, edit=EDITS.get(kind))
    art = with_weight_rows(sm, "embed", {BAD: np.zeros(sm.config.hidden, np.int8)}) if kind == "zero" else sm.to_array()
    model, blobs = _blobs(hip_lib, art, 6, bad_at)
    print(f"case chain refusal {kind} batch={batch} budget={budget}", flush=True)
    few = _decode(model, blobs[:batch], budget, 3)
    again = _decode(model, blobs[:batch], budget, 3)  # in the same slots: nothing of a refusal is left behind
    many = _decode(model, blobs, budget, 3)
    assert few == again
    assert kind == "clean" or any(st != 0 for st, _, _ in few)
    for (st, toks, saved), (st6, toks6, saved6) in zip(few, many):
        if kind == "clean" or bad_at >= 0 or st != 0:
            assert st == st6
        if kind in EDITS:  # refused at layer 1, not before
            assert (st == 0) == (budget == 1 and saved is few[0][2])
        assert toks == toks6[:batch]
        assert saved == saved6[:batch], "sequence state differs"
    model.close()
