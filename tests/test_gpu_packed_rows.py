"""The packed decode GEMVs and LM head past 32 rows (up to four 16-token row groups in a block, two
row blocks past 64 tokens) against the C oracle: decode batches and prompts at the edges
of the row groups, over shapes that take each kernel -- K <= 2048 (four waves), K past 16 chunks
(eight waves, no second row block), and a split-K down projection (K > 4096)."""
import numpy as np
import pytest

from oracle_bind import OracleModel
from superslm_amd.sslm import Model
from superslm_amd.sslm_artifact import ModelConfig, build_synthetic

pytestmark = pytest.mark.gpu

SHAPES = {
    # gate|up and head over 2 chunks, down split over K = 4,352
    "split_down": ModelConfig(hidden=256, layers=2, heads=4, kv_heads=2, head_dim=64, inter=4352, vocab=1000,
                              context_cap=160, tie_embeddings=False, with_bias=True),
    # 17 chunks of 128: eight waves of four chunks
    "deep": ModelConfig(hidden=2176, layers=1, heads=17, kv_heads=1, head_dim=128, inter=320, vocab=528,
                        context_cap=160, tie_embeddings=True),
}
_ART = {}


def _model(name):
    if name not in _ART:
        _ART[name] = build_synthetic(SHAPES[name], seed=17)
    return _ART[name]


def _oracle(lib, sm, prompts, calls):
    om = OracleModel(lib, sm)
    seqs = [om.new_seq() for _ in prompts]
    for s, p in zip(seqs, prompts):
        assert s.prefill(p) == (0, len(p))
    toks = []
    for _ in range(calls):
        got = [s.decode_step(sm.config.layers) for s in seqs]
        assert all(st == 0 for st, _ in got)
        toks.append([t for _, t in got])
    return toks, [s.kv for s in seqs]


def _hip(lib, sm, prompts, calls):
    model = Model(lib, sm.to_array())
    pool = model.pool(len(prompts))
    seqs = [pool.seq() for _ in prompts]
    # a sequence owns the block at the back of the pool's free list
    blocks = list(range(len(prompts)))[::-1]
    for s, p in zip(seqs, prompts):
        assert s.prefill(p) == len(p)
    toks = [model.decode_step(seqs, sm.config.layers) for _ in range(calls)]
    kv = [pool.kv_block(b).copy() for b in blocks]
    for s in seqs:
        s.release()
    pool.close()
    model.close()
    return toks, kv


@pytest.mark.parametrize("shape", sorted(SHAPES))
@pytest.mark.parametrize("batch,length", [(33, 2), (48, 1), (64, 1), (65, 1), (127, 1), (128, 1), (1, 33), (1, 64), (1, 65),
                                          (1, 127), (2, 128), (1, 129)])
def test_packed_rows_match_oracle(shape, batch, length, hip_lib, oracle_lib):
    sm = _model(shape)
    rng = np.random.default_rng(batch * 1000 + length)
    prompts = [rng.integers(0, sm.config.vocab, size=length) for _ in range(batch)]
    want = _oracle(oracle_lib, sm, prompts, 3)
    print(f"case packed rows {shape} batch={batch} length={length}", flush=True)
    got = _hip(hip_lib, sm, prompts, 3)
    assert got[0] == want[0], "tokens differ"
    for i in range(batch):
        assert np.array_equal(got[1][i], want[1][i]), f"KV of sequence {i} differs"


@pytest.mark.parametrize("kv_heads,batch", [(2, 65), (2, 128), (4, 65), (4, 128)])
def test_fused_decode_rule_matches_oracle(kv_heads, batch, hip_lib, oracle_lib):
    """Past 64 sequences at a cap that takes the grouped decode attention: its blocks in one round of the
    CUs (two KV heads: the post-processing inside the attention) and in two (four: raw planes)."""
    sm = build_synthetic(ModelConfig(hidden=256, layers=2, heads=4, kv_heads=kv_heads, head_dim=64, inter=320, vocab=512,
                                     context_cap=1024, tie_embeddings=True, with_bias=True), seed=29)
    rng = np.random.default_rng(batch + kv_heads)
    prompts = [rng.integers(0, sm.config.vocab, size=1) for _ in range(batch)]
    want = _oracle(oracle_lib, sm, prompts, 3)
    print(f"case fused rule kv_heads={kv_heads} batch={batch}", flush=True)
    got = _hip(hip_lib, sm, prompts, 3)
    assert got[0] == want[0], "tokens differ"
    for i in range(batch):
        assert np.array_equal(got[1][i], want[1][i]), f"KV of sequence {i} differs"
