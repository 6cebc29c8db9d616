"""The attention of several tokens, the matrix-instruction kernels
(attn_tile.hip: scores, softmax, P.V and the O-input prep) and the split ones
that take few tokens over many keys, against the oracle, bit for bit: every
head dim and both caches, even groups that do and do not fill a 16-row tile,
rows resident in LDS and streamed, tiles whose last rows or keys are missing,
scores rows that end inside a 16-byte piece, and both sides of the rule that
chooses the kernels."""
import ctypes as C

import numpy as np
import pytest

from dpuf_amd import abi
from dpuf_amd import model as M
from test_gpu_configs import Pair, bits_equal, log, maxdiff
from test_gpu_q8kv import Q8Pair

pytestmark = pytest.mark.gpu

# (query heads, KV heads, head dim, cached positions, tokens, max_seq), and the
# routes over the fp32 and the int8 cache: R / S the matrix-instruction
# kernels with resident / streamed rows, P the split kernels (few tokens over
# many keys: one workgroup per CU at most of 256), M the softmax in memory
CASES = [
    (4, 2, 64, 0, 2, 40, "RR"),         # the smallest prompt
    (4, 2, 64, 3, 37, 40, "RR"),        # ends at max_seq
    (8, 2, 128, 0, 33, 67, "RR"),       # one row past a query tile; max_seq odd
    (8, 2, 128, 61, 6, 67, "RR"),       # across the first chunk boundary, up to an odd max_seq
    (8, 2, 128, 282, 6, 470, "RR"),     # the split kernels' range: int8 from 289 keys on
    (8, 2, 128, 283, 6, 470, "RP"),
    (8, 2, 128, 450, 6, 470, "RP"),     # fp32 from 457
    (8, 2, 128, 451, 6, 470, "PP"),
    (32, 8, 128, 600, 16, 620, "PP"),   # 256 split workgroups
    (32, 8, 128, 600, 17, 620, "RR"),   # 288
    (16, 8, 64, 735, 65, 810, "RR"),    # resident, the longest (25 chunks of 32 keys)
    (16, 8, 64, 736, 65, 810, "SS"),    # streamed, the shortest
    (32, 8, 128, 935, 25, 970, "RR"),   # resident, the longest (15 chunks of 64)
    (32, 8, 128, 936, 25, 970, "SS"),   # streamed, the shortest
    (32, 8, 128, 2038, 25, 2063, "SS"), # up to an odd max_seq
    (8, 2, 128, 955, 9, 970, "PP"),
    (8, 2, 128, 958, 9, 970, "PP"),
    (8, 2, 128, 2042, 19, 2063, "PP"),
    (12, 2, 64, 70, 23, 96, "RR"),      # groups of 6: 12 of 16 rows, 30 of 32
    (20, 2, 64, 30, 3, 64, "RR"),       # groups of 10: one token per tile
    (32, 2, 128, 17, 3, 64, "RR"),      # groups of 16
    (32, 2, 64, 1500, 4, 1510, "PM"),
    (4, 2, 256, 120, 21, 150, "RR"),    # chunks of 128 keys
    (4, 2, 256, 480, 40, 521, "RP"),    # five of them
    (16, 8, 256, 1007, 17, 1031, "RR"), # resident, the longest (8 chunks)
    (16, 8, 256, 1008, 17, 1031, "SS"), # streamed, the shortest
    (8, 2, 128, 7200, 2, 7240, "SS"),   # half a tile of rows, too long for the split kernels
]
# dpuf_amd_attn_path_count: the tile kernels, the split ones over the fp32
# cache, every int8 one, streamed rows, the softmax in memory
TILES, SPLIT, INT8, STREAMED, MEMORY = 0, 2, 5, 6, 7


@pytest.mark.parametrize("kv_type", [0, 1])
@pytest.mark.parametrize("nq,nkv,hd,ctx,n,max_seq,routes", CASES)
def test_attention_of_several_tokens(eng, orc, nq, nkv, hd, ctx, n, max_seq, routes, kv_type):
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
    paths = (TILES, SPLIT, INT8, STREAMED, MEMORY)
    c0 = [eng.dpuf_amd_attn_path_count(w) for w in paths]
    lg, lo = p.forward(rng.integers(0, 512, n).astype(np.int32), ctx, only_last=0)
    r = routes[kv_type]
    want = (r in "RS", r == "P" and not kv_type, kv_type, r == "S", r == "M")
    assert [eng.dpuf_amd_attn_path_count(w) - c for w, c in zip(paths, c0)] == [2 * int(w) for w in want]
    assert bits_equal(lg, lo), maxdiff(lg, lo)
    p.close()


class _Prep(C.Structure):
    _fields_ = [(f, C.c_void_p) for f in "qsmh"]


class _KvQ8(C.Structure):
    _fields_ = [(f, C.c_void_p) for f in ("kq", "vq", "ks", "vs")]


def _extreme(rng, kind, keys, hd):
    """[keys][hd] values whose products, sums or themselves leave the normal range."""
    scales = {"tiny": [1e-44, 1e-40, 1e-38, 1e-20, 1.0], "huge": [1.0, 1e20, 1e36, 1e38],
              "infinite": [1e-40, 1.0, 1e30]}[kind]
    with np.errstate(over="ignore"):
        x = (rng.standard_normal((keys, hd)) * rng.choice(scales, (keys, 1))).astype(np.float32)
    if kind == "infinite":
        at = rng.integers(0, keys, 6)
        x[at, rng.integers(0, hd, 6)] = [np.inf, -np.inf, np.inf, -np.inf, np.nan, np.inf]
    return x


# (the quantising store leaves finite scales of finite keys: no infinite int8 cache)
@pytest.mark.parametrize("kind,kv_type", [("tiny", 0), ("huge", 0), ("infinite", 0), ("tiny", 1), ("huge", 1)])
@pytest.mark.parametrize("nq,nkv,hd,ctx,n,max_seq,tiles", [
    (4, 2, 64, 80, 9, 96, 1), (8, 2, 128, 200, 7, 210, 1), (32, 8, 128, 1000, 25, 1030, 1), (8, 2, 256, 270, 5, 280, 1),
    (8, 2, 128, 1300, 7, 1310, 0)])
def test_attention_out_of_range_values(eng, orc, nq, nkv, hd, ctx, n, max_seq, tiles, kind, kv_type):
    """Keys and values that are denormal, that overflow the scores' and the
    outputs' chains, or that are infinite or NaN (the int8 cache: its scales):
    the fp32 matrix instructions' chains round, underflow and propagate them
    as the reference's fused multiply-adds do.  The launches alone, on device
    buffers, so that each attention output is compared: bit for bit, a NaN
    with a NaN."""
    rng = np.random.default_rng(403 + ctx)
    keys, G = ctx + n, nq // nkv
    q = rng.standard_normal((n, nq, hd)).astype(np.float32)
    kf, vf = (np.zeros((nkv, max_seq, hd), np.float32) for _ in range(2))
    for h in range(nkv):
        kf[h, :keys], vf[h, :keys] = _extreme(rng, kind, keys, hd), _extreme(rng, kind, keys, hd)
    if kv_type:
        kq, vq = (rng.integers(-127, 128, (nkv, max_seq, hd)).astype(np.int8) for _ in range(2))
        ks, vs = (np.abs(x[:, :, :hd // 32]).copy() for x in (kf, vf))
        host = [kq, vq, ks, vs]
    else:
        host = [kf, vf]
    log(f"out of range ({kind}): groups of {G}, head dim {hd}, kv_type {kv_type}, {n} tokens after {ctx}")
    P, I, F, Z = C.c_void_p, C.c_int32, C.c_float, C.c_size_t
    L = C.CDLL(eng._name)
    L.dpuf_hip_malloc.restype, L.dpuf_hip_malloc.argtypes = P, [Z]
    L.dpuf_hip_free.argtypes = [P]
    L.dpuf_hip_h2d.argtypes = L.dpuf_hip_d2h.argtypes = [P, P, Z, P]
    L.dpuf_hip_sync.argtypes = [P]
    L.dpuf_hip_attn_split.argtypes = [P, I, I, P, P, P, P, P, P, I, I, I, I, F, P, _Prep, P]
    L.dpuf_hip_attn_q8.argtypes = [P, I, I, P, _KvQ8, P, P, P, I, I, I, I, F, P, P, _Prep, P]
    bufs = []

    def dev(a):
        bufs.append(L.dpuf_hip_malloc(a.nbytes))
        assert bufs[-1]
        L.dpuf_hip_h2d(bufs[-1], M.ptr(a), a.nbytes, None)
        return bufs[-1]

    out = np.zeros((n, nq, hd), np.float32)
    scores = np.zeros(n * nq * (max_seq + 64), np.float32)  # a row of scores and 64 maxima per token and head
    dq, dout, dsc, dpos = dev(q), dev(out), dev(scores), dev(np.array([ctx], np.int32))
    dkv = [dev(a) for a in host]
    scale = float(np.float32(1.0 / np.sqrt(hd)))
    c0 = eng.dpuf_amd_attn_path_count(TILES)
    if kv_type:
        L.dpuf_hip_attn_q8(None, n, keys, dq, _KvQ8(*dkv), dout, dsc, dpos, nq, nkv, hd, max_seq, scale, None, None,
                           _Prep(), None)
    else:
        assert L.dpuf_hip_attn_split(None, n, keys, dq, dkv[0], dkv[1], dout, dsc, dpos, nq, nkv, hd, max_seq, scale,
                                     None, _Prep(), None) == 0
    assert eng.dpuf_amd_attn_path_count(TILES) - c0 == tiles
    L.dpuf_hip_d2h(M.ptr(out), dout, out.nbytes, None)
    assert L.dpuf_hip_sync(None) == 0
    for b in bufs:
        L.dpuf_hip_free(b)
    want = np.zeros_like(out)
    sc = [np.zeros(keys + 8, np.float32) for _ in range(2)]
    for m in range(n):
        for h in range(0, nq, 2):
            kv = [M.ptr(a[h // G]) for a in host]
            rows = [M.ptr(q[m, h]), M.ptr(q[m, h + 1]), M.ptr(sc[0]), M.ptr(sc[1]), M.ptr(want[m, h]),
                    M.ptr(want[m, h + 1])]
            if kv_type:
                orc.orc_attn_heads_q8(hd, ctx + m + 1, scale, kv[0], kv[2], kv[1], kv[3], *rows)
            else:
                orc.orc_attn_heads(hd, ctx + m + 1, scale, kv[0], kv[1], *rows)
    nan = np.isnan(want)
    log(f"  finite {np.isfinite(want).mean():.3f}, NaN {nan.mean():.3f}, |x| < 2^-126 {(np.abs(want) < 2.0**-126).mean():.3f}")
    assert np.isfinite(want).any()
    assert np.array_equal(np.isnan(out), nan)
    assert bits_equal(np.where(nan, 0, out), np.where(nan, 0, want))
