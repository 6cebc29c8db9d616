"""One token of each of several sessions over the fp32 cache, some past the
fused decode kernel's keys: the one-token kernels of long contexts with a
session axis (attn_wide.hip: scores with the RoPE and KV store, softmax, P.V)
against the oracle decoding each slot alone, bit for bit, at every head dim
and group they are built for."""
import numpy as np
import pytest

from dpuf_amd import model as M
from test_gpu_configs import WIDE, Pair, bits_equal, log, maxdiff

pytestmark = pytest.mark.gpu
FUSED = 4  # dpuf_amd_attn_path_count: the fused short-context decode kernel
LAYERS = 2


def _decode_sessions(eng, orc, nq, nkv, hd, max_seq, lens, steps):
    """Sessions of injected contexts (slot -> keys), decoded together; returns
    the attention launches counted per step as (wide, fused)."""
    shape = dict(hidden_size=256, intermediate_size=256, num_layers=LAYERS, num_q_heads=nq, num_kv_heads=nkv,
                 head_dim=hd, vocab_size=512, tie_word_embeddings=1)
    p = Pair(eng, orc, M.Model.build(shape, max_seq_len=max_seq, seed=501))
    rng = np.random.default_rng(502 + nq)
    for s, n in lens.items():
        p.set_slot(s)
        for layer in range(LAYERS):
            for kvh in range(nkv):
                p.set_kv(layer, kvh, 0, rng.standard_normal((n, hd), dtype=np.float32),
                         rng.standard_normal((n, hd), dtype=np.float32))
    slots = np.array(list(lens), np.int32)
    pos = np.array(list(lens.values()), np.int32)
    toks = rng.integers(0, 512, len(lens)).astype(np.int32)
    w0, f0 = eng.dpuf_amd_attn_path_count(WIDE), eng.dpuf_amd_attn_path_count(FUSED)
    for step in range(steps):
        log(f"sessions: groups of {nq // nkv}, head dim {hd}, positions {pos.tolist()}")
        lg = np.zeros((len(lens), 512), np.float32)
        got = np.full(len(lens), -1, np.int32)
        assert eng.dpuf_amd_engine_forward_slots(p.g, len(lens), M.ptr(slots), M.ptr(toks), M.ptr(pos), M.ptr(lg),
                                                 M.ptr(got)) == 0, eng.dpuf_amd_last_error()
        for i, s in enumerate(lens):
            assert orc.orc_engine_set_slot(p.o, s) == 0
            lo = np.zeros(512, np.float32)
            assert orc.orc_engine_forward(p.o, 1, M.ptr(toks[i:i + 1].copy()), int(pos[i]), None, 1, M.ptr(lo)) == 0
            assert bits_equal(lg[i], lo), (step, s, maxdiff(lg[i], lo))
        toks, pos = got.copy(), pos + np.int32(1)
    p.close()
    return ((eng.dpuf_amd_attn_path_count(WIDE) - w0) / (steps * LAYERS),
            (eng.dpuf_amd_attn_path_count(FUSED) - f0) / (steps * LAYERS))


@pytest.mark.parametrize("hd", [64, 128, 256])
@pytest.mark.parametrize("G", [2, 4])
def test_session_axis(eng, orc, G, hd):
    """Positions on each side of the 64-key chunks' borders and of the fused
    kernel's 192 keys, a first token, the last position of an odd max_seq."""
    lens = {6: 63, 1: 699, 0: 0, 5: 191, 2: 128, 7: 64, 3: 320}
    wide, fused = _decode_sessions(eng, orc, 2 * G, 2, hd, 701, lens, 2)
    assert (wide, fused) == (len(lens), 0)


def test_sessions_past_the_session_axis(eng, orc):
    """With a session past 8 192 keys the axis does not apply: the short
    sessions go through the fused kernel, the two others one by one."""
    wide, fused = _decode_sessions(eng, orc, 4, 2, 64, 8300, {4: 9, 0: 8250, 2: 150, 1: 300}, 2)
    assert wide <= 2 and fused == 1
