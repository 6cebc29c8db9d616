"""The matrix-instruction attention of several tokens (attn_tile.hip: scores,
softmax, P.V and the O-input prep) against the oracle, bit for bit: every head
dim and both caches, even groups that do and do not fill a 16-row tile, rows
resident in LDS and streamed, tiles whose last rows or keys are missing, and
scores rows that end inside a 16-byte piece."""
import numpy as np
import pytest

from dpuf_amd import abi
from dpuf_amd import model as M
from test_gpu_configs import Pair, bits_equal, log, maxdiff
from test_gpu_q8kv import Q8Pair

pytestmark = pytest.mark.gpu

# (query heads, KV heads, head dim, cached positions, tokens, max_seq)
CASES = [
    (4, 2, 64, 0, 2, 40),        # the smallest prompt
    (4, 2, 64, 3, 37, 40),       # ends at max_seq
    (8, 2, 128, 0, 33, 67),      # one row past a query tile; max_seq odd
    (8, 2, 128, 61, 6, 67),      # across the first chunk boundary, up to an odd max_seq
    (8, 2, 128, 955, 9, 970),    # resident rows, the longest (15 chunks of 64)
    (8, 2, 128, 958, 9, 970),    # streamed rows, the shortest (16 chunks)
    (8, 2, 128, 2042, 19, 2063), # streamed, 2061 keys
    (12, 2, 64, 70, 23, 96),     # groups of 6: 12 of 16 rows, 30 of 32
    (20, 2, 64, 30, 3, 64),      # groups of 10: one token per tile
    (32, 2, 128, 17, 3, 64),     # groups of 16
    (4, 2, 256, 120, 21, 150),   # chunks of 128 keys
    (4, 2, 256, 480, 40, 521),   # the same, streamed
]


@pytest.mark.parametrize("kv_type", [0, 1])
@pytest.mark.parametrize("nq,nkv,hd,ctx,n,max_seq", CASES)
def test_attention_of_several_tokens(eng, orc, nq, nkv, hd, ctx, n, max_seq, kv_type):
    shape = dict(hidden_size=256, intermediate_size=256, num_layers=2, num_q_heads=nq, num_kv_heads=nkv, head_dim=hd,
                 vocab_size=512, tie_word_embeddings=1)
    m = M.Model.build(shape, max_seq_len=max_seq, seed=401)
    cfg = abi.DpufModelConfig.from_buffer_copy(m.cfg.contents)
    cfg.kv_type = kv_type
    p = Q8Pair(eng, orc, m, cfg) if kv_type else Pair(eng, orc, m)
    rng = np.random.default_rng(402 + ctx)
    log(f"groups of {nq // nkv}, head dim {hd}, kv_type {kv_type}: {n} tokens after {ctx}")
    if ctx:
        for layer in range(2):
            for kvh in range(nkv):
                p.set_kv(layer, kvh, 0, rng.standard_normal((ctx, hd), dtype=np.float32),
                         rng.standard_normal((ctx, hd), dtype=np.float32))
    path = 5 if kv_type else 0
    c0 = eng.dpuf_amd_attn_path_count(path)
    lg, lo = p.forward(rng.integers(0, 512, n).astype(np.int32), ctx, only_last=0)
    assert eng.dpuf_amd_attn_path_count(path) - c0 == 2
    assert bits_equal(lg, lo), maxdiff(lg, lo)
    p.close()
