"""The work that programs have the token loop do, as timed cases.

Every case goes through the library's C entry points (ctypes, host buffers in
and out) as a serving program calls them: a resident engine, a KV cache that
already holds the conversation so far, then one call.

Three kinds of case:
  step   dpuf_engine_forward_batch of `rows` tokens at position `pos` of one
         slot (rows = 1: a decode step, more: a prompt or a chunk of one);
         returns the last row's logits.
  slots  dpuf_amd_engine_forward_slots: one next token for each of `sessions`
         slots whose contexts are spread from `pos` to `pos_hi`; returns every
         session's logits and greedy token.
  head   the final norm and LM head alone (an engine without layers, a hidden
         state in) over the full vocabulary, with the Zone-A early exit after
         `zone` tiles (0: without it); returns the logits.

Widths are the Qwen3-0.6B and Qwen3-8B shapes of dpuf_amd.model.  Most cases
run a block of four decoder layers of the 8B width (432 MB of weights, more
than the 256 MB Infinity Cache, so each layer's weights come from HBM as in
the whole model) under a 4 096-row vocabulary; two are whole models.

`plan` is "m12" (every matrix Mode 12, Q/K/V and gate/up sharing their sign
vectors, as the packer writes them) or "hybrid" (the had4p-hybrid plan: Modes
13 and 14, each matrix with signs of its own).  `kv` is "f32" or "q8".
`keep` > 0 prunes a prefill's down projection to that many 16-row tiles
(DPUF_PREFILL_KEEP_TILES).

Weights are N(0, 0.02) values quantised block by block to the packed formats,
cached K and V are N(0, 1), token ids uniform over the vocabulary.
"""
import ctypes as C
import math
import os

import numpy as np
import torch

from dpuf_amd import abi
from dpuf_amd import model as M

DEV = "cuda"
STD = 0.02
EPS = 1e-6
THETA = 1e6
DEADZONE = 0.005  # the engine's default SwiGLU dead zone
BLOCK_LAYERS = 4
BLOCK_VOCAB = 4096
ZONE_MARGIN = 0.8


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def _case(kind, **kw):
    c = dict(kind=kind, shape="8b", whole=False, plan="m12", kv="f32", rows=1, pos=0, keep=0, sessions=0, pos_hi=0,
             zone=0)
    c.update(kw)
    return c


def listed():
    return [
        # a chat reply of the small model, a few dozen tokens in: the smallest step
        _case("step", name="token_0p6b", shape="0.6b", whole=True, pos=75),
        # the same for the 8B shape: the framework's headline decode step
        _case("step", name="token_8b", whole=True, pos=50),
        # decode deep in a long document, at the widths of the 8B shape
        _case("step", name="token_long", pos=4095),
        # decode in a mid-length conversation with the int8 cache
        _case("step", name="token_q8", kv="q8", pos=1290),
        # decode with the had4p-hybrid weights, short context
        _case("step", name="token_hybrid", plan="hybrid", pos=130),
        # the headline prefill: a full 512-token call with 224 of 256 down tiles
        _case("step", name="prefill_512", rows=512, keep=224),
        # one user turn of a chat, appended to its history
        _case("step", name="turn_29", rows=29, pos=410),
        # the last 256-token chunk of a 4 096-token prompt, the CLI's chunk size
        _case("step", name="chunk_long", rows=256, pos=3840),
        # a paragraph-long turn on hybrid weights and the int8 cache
        _case("step", name="turn_hybrid_q8", plan="hybrid", kv="q8", rows=90, pos=700),
        # eight conversations of very different lengths served in one pass
        _case("slots", name="sessions_8", sessions=8, pos=60, pos_hi=2600),
        # four young conversations on hybrid weights
        _case("slots", name="sessions_4_hybrid", plan="hybrid", sessions=4, pos=20, pos_hi=180),
        # the LM head with the Zone-A early exit
        _case("head", name="head_zone", zone=1424),
    ]


# (query, key) pairs of the largest listed case, times its layers and heads: no drawn case has more
_PAIRS = 256 * 3968 * BLOCK_LAYERS * 32


def _log_int(rng, lo, hi):
    return min(hi, int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))


def draw(rng):
    kind = rng.choice(["token", "token", "prompt", "prompt", "prompt", "slots", "slots", "head"])
    if kind == "head":
        return _case("head", zone=0 if rng.random() < 0.3 else _log_int(rng, 256, 4096))
    small = rng.random() < 0.25
    opt = dict(shape="0.6b" if small else "8b", whole=small, plan="hybrid" if rng.random() < 0.3 else "m12",
               kv="q8" if rng.random() < 0.3 else "f32")
    if kind == "slots":
        lo = _log_int(rng, 8, 1000)
        return _case("slots", sessions=rng.randint(2, 8), pos=lo, pos_hi=_log_int(rng, lo, 3500), **opt)
    if kind == "token":
        return _case("step", pos=_log_int(rng, 1, 4095), **opt)
    rows = _log_int(rng, 2, 512)
    heads = 28 * 16 if small else BLOCK_LAYERS * 32
    top = min(4096 - rows, _PAIRS // (heads * rows) - rows)
    pos = 0 if top < 1 or rng.random() < 0.3 else _log_int(rng, 1, top)
    keep = 0 if small or rng.random() < 0.5 else 224
    return _case("step", rows=rows, pos=pos, keep=keep, **opt)


def _dims(case):
    d = dict(M.QWEN3_8B if case["shape"] == "8b" else M.QWEN3_0_6B)
    if case["kind"] == "head":
        d["num_layers"] = 0
    elif not case["whole"]:
        d["num_layers"], d["vocab_size"] = BLOCK_LAYERS, BLOCK_VOCAB
    return d


def _positions(case):
    """Context length of each session, spread over its logarithm."""
    n, lo, hi = case["sessions"], case["pos"], case["pos_hi"]
    return [int(round(lo * (hi / lo) ** (i / max(1, n - 1)))) for i in range(n)]


# ---------------------------------------------------------------------------
# weights
# ---------------------------------------------------------------------------

def _layer_mats(d):
    """(name, rows, cols, sign group) of a layer's matrices: matrices of one
    sign group share their sign vector under the Mode 12 plan."""
    H, I, hd = d["hidden_size"], d["intermediate_size"], d["head_dim"]
    qd, kvd = d["num_q_heads"] * hd, d["num_kv_heads"] * hd
    return [("w_q", qd, H, 0), ("w_k", kvd, H, 0), ("w_v", kvd, H, 0), ("w_o", H, qd, 1),
            ("w_gate", I, H, 2), ("w_up", I, H, 2), ("w_down", H, I, 3)]


def _mode(plan, layer, name):
    if plan == "m12":
        return 12
    six = name in ("w_down", "w_v", "w_k", "lm") or (name == "w_o" and layer % 2 == 0)
    return 14 if six else 13


class _Matrix:
    """One quantised matrix on the GPU: u, the codes [rows][cols], and its
    fp16 scales (Mode 12: s per 32 columns; Modes 13 / 14: d, m per 64)."""

    def __init__(self, gen, rows, cols, mode, signs):
        self.rows, self.cols, self.mode, self.signs = rows, cols, mode, signs
        w = torch.randn(rows, cols, generator=gen, device=DEV) * STD
        if mode == 12:
            w = w.view(rows, cols // 32, 32)
            self.s = (w.abs().amax(-1) / 7).half()
            u = torch.round(w / self.s.float().unsqueeze(-1)).clamp_(-8, 7) + 8
        else:
            top = 15 if mode == 13 else 63
            w = w.view(rows, cols // 64, 64)
            lo, hi = w.amin(-1), w.amax(-1)
            self.d, self.m = ((hi - lo) / top).half(), lo.half()
            u = torch.round((w - self.m.float().unsqueeze(-1)) / self.d.float().unsqueeze(-1)).clamp_(0, top)
        self.u = u.view(rows, cols).to(torch.uint8)

    def packed(self):
        """The .dpuf tiles (16-byte header, two 8-row groups, padded to 64
        bytes) as a host array, and the tile offsets."""
        t, nb = self.rows // 16, self.cols // 32
        u = self.u.view(t, 2, 8, nb, 4, 2, 4)  # tile, group, row, block, chunk, half, column
        q4 = ((u[:, :, :, :, :, 0] & 15) | ((u[:, :, :, :, :, 1] & 15) << 4)).permute(0, 1, 3, 4, 2, 5)
        if self.mode == 12:
            sc = self.s.view(t, 2, 8, nb).permute(0, 1, 3, 2).contiguous()
        else:
            sc = torch.stack([self.d.view(t, 2, 8, nb // 2), self.m.view(t, 2, 8, nb // 2)], 2)
            sc = sc.permute(0, 1, 4, 2, 3).contiguous()  # tile, group, 64-block, (d, m), row
        parts = [sc.view(t, 2, -1).view(torch.uint8), q4.reshape(t, 2, -1)]
        if self.mode == 14:
            hi = (u >> 4).view(t, 2, 4, 2, nb, 4, 2, 4)  # row = 2 * pair + parity
            hi = hi[:, :, 0] | hi[:, :, 1] << 2 | hi[:, :, 2] << 4 | hi[:, :, 3] << 6
            parts.append(hi.permute(0, 1, 3, 4, 5, 2, 6).reshape(t, 2, -1))
        body = torch.cat(parts, 2).view(t, -1)
        size = -(-(16 + body.shape[1]) // 64) * 64
        tiles = torch.zeros(t, size, dtype=torch.uint8, device=DEV)
        tiles[:, 4] = 16  # rows of the tile
        tiles[:, 16:16 + body.shape[1]] = body
        return tiles.cpu().numpy(), np.arange(t + 1, dtype=np.uint64) * np.uint64(size)

    def f64(self):
        """The rotated matrix in float64."""
        if self.mode == 12:
            return ((self.u.double() - 8).view(self.rows, -1, 32) * self.s.double().unsqueeze(-1)).view(self.rows, -1)
        return (self.u.double().view(self.rows, -1, 64) * self.d.double().unsqueeze(-1)
                + self.m.double().unsqueeze(-1)).view(self.rows, -1)


def _gen(seed, *what):
    g = torch.Generator(device=DEV)
    for w in what:
        seed = (seed * 1000003 + w + 1) % (1 << 61)
    g.manual_seed(seed)
    return g


def _norm(g, n):
    return 1 + 0.1 * torch.randn(n, generator=g, device=DEV)


def _signs(g, cols):
    return torch.randint(0, 256, (cols // 8,), generator=g, device=DEV, dtype=torch.uint8)


def _layer(case, d, seed, layer):
    """Matrices and norms of one layer."""
    g = _gen(seed, 1, layer)
    shared = {}
    mats = {}
    for name, rows, cols, grp in _layer_mats(d):
        key = grp if case["plan"] == "m12" else name
        if key not in shared:
            shared[key] = _signs(g, cols)
        mats[name] = _Matrix(g, rows, cols, _mode(case["plan"], layer, name), shared[key])
    norms = [_norm(g, d["hidden_size"]), _norm(g, d["head_dim"]), _norm(g, d["head_dim"]), _norm(g, d["hidden_size"])]
    return mats, norms


def _ends(case, d, seed):
    """Embedding matrix, LM head (the embedding itself when tied) and output norm."""
    g = _gen(seed, 2)
    V, H = d["vocab_size"], d["hidden_size"]
    # the layerless head engine reads no embedding row: its head serves as both
    if case["kind"] == "head" or d["tie_word_embeddings"]:
        tok = lm = _Matrix(g, V, H, _mode(case["plan"], 0, "tok"), _signs(g, H))
    else:
        tok = _Matrix(g, V, H, _mode(case["plan"], 0, "tok"), _signs(g, H))
        lm = _Matrix(g, V, H, _mode(case["plan"], 0, "lm"), _signs(g, H))
    return tok, lm, _norm(g, H)


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------

class _State:
    """A resident engine and one call's arguments."""

    def __init__(self, case, handle):
        self.case, self.h, self.lib = case, handle, abi.load_engine()

    def __del__(self):
        if self.h:
            self.lib.dpuf_engine_destroy(self.h)
            self.h = None


def _desc(mat, keep):
    tiles, offs = mat.packed()
    signs = mat.signs.cpu().numpy()
    keep += [tiles, offs, signs]
    w = abi.DpufWeightDesc()
    w.mode, w.rows, w.cols, w.n_tiles = mat.mode, mat.rows, mat.cols, mat.rows // 16
    w.tensor_base, w.tile_offsets, w.sign_bits = M.ptr(tiles), M.ptr(offs), M.ptr(signs)
    return w


def _floats(t, keep):
    a = t.cpu().numpy()
    keep.append(a)
    return M.ptr(a)


def _contexts(case):
    """(slot, context length) of every slot the call reads."""
    if case["kind"] == "slots":
        return list(enumerate(_positions(case)))
    return [(0, case["pos"])] if case["kind"] == "step" else []


def _cache(case, d, seed, slot, n):
    """Cached K and V of a slot, [layers][2][kv heads][n][head dim]."""
    return torch.randn(d["num_layers"], 2, d["num_kv_heads"], n, d["head_dim"], generator=_gen(seed, 3, slot),
                       device=DEV)


def _ids(case, d, seed):
    n = case["sessions"] if case["kind"] == "slots" else case["rows"]
    return torch.randint(0, d["vocab_size"], (n,), generator=_gen(seed, 4), device=DEV, dtype=torch.int32).cpu().numpy()


def _hidden(case, d, seed):
    return torch.randn(1, d["hidden_size"], generator=_gen(seed, 5), device=DEV)


def prepare(case, seed):
    lib = abi.load_engine()
    d = _dims(case)
    L = d["num_layers"]
    cfg = abi.DpufModelConfig()
    for k in ("hidden_size", "intermediate_size", "num_layers", "num_q_heads", "num_kv_heads", "head_dim",
              "vocab_size"):
        setattr(cfg, k, d[k])
    cfg.max_seq_len = 4352 if case["kind"] != "head" else 64
    cfg.has_qk_norm, cfg.rms_eps, cfg.rope_theta = 1, EPS, THETA
    cfg.kv_type = 1 if case["kv"] == "q8" else 0
    keep = []
    layers = (abi.DpufLayerWeights * max(1, L))()
    for l in range(L):
        mats, norms = _layer(case, d, seed, l)
        for name, mat in mats.items():
            setattr(layers[l], name, _desc(mat, keep))
        for name, n in zip(("attn_norm", "attn_q_norm", "attn_k_norm", "ffn_norm"), norms):
            setattr(layers[l], name, _floats(n, keep))
    tok, lm, out_norm = _ends(case, d, seed)
    wt = _desc(tok, keep)
    wl = wt if lm is tok else _desc(lm, keep)
    h = lib.dpuf_engine_create(C.byref(cfg), layers, C.byref(wt), C.byref(wl), _floats(out_norm, keep))
    if not h:
        raise RuntimeError("dpuf_engine_create: " + lib.dpuf_amd_last_error().decode())
    st = _State(case, h)
    V = d["vocab_size"]
    for slot, n in _contexts(case):
        if lib.dpuf_engine_set_slot(h, slot) != 0:
            raise RuntimeError("dpuf_engine_set_slot")
        if n == 0:
            continue
        kv = _cache(case, d, seed, slot, n).cpu().numpy()
        for l in range(L):
            for k in range(d["num_kv_heads"]):
                if lib.dpuf_amd_engine_set_kv(h, l, k, 0, n, M.ptr(kv[l, 0, k]), M.ptr(kv[l, 1, k])) != 0:
                    raise RuntimeError("dpuf_amd_engine_set_kv")
    lib.dpuf_engine_set_slot(h, 0)
    if case["kind"] == "slots":
        n = case["sessions"]
        st.slots = np.arange(n, dtype=np.int32)
        st.pos = np.array(_positions(case), dtype=np.int32)
        st.ids = _ids(case, d, seed)
        st.logits, st.tokens = np.zeros((n, V), np.float32), np.zeros(n, np.int32)
    elif case["kind"] == "head":
        st.x = _hidden(case, d, seed).cpu().numpy()
        st.logits = np.zeros(V, np.float32)
    else:
        st.ids = _ids(case, d, seed)
        st.logits = np.zeros(V, np.float32)
    return st


def _env(name, value):
    if value:
        os.environ[name] = str(value)
    else:
        os.environ.pop(name, None)


def run(st):
    c, lib = st.case, st.lib
    _env("DPUF_PREFILL_KEEP_TILES", c["keep"])
    _env("DPUF_EARLY_TILES", c["zone"])
    _env("DPUF_EARLY_MARGIN", ZONE_MARGIN if c["zone"] else 0)
    if c["kind"] == "slots":
        rc = lib.dpuf_amd_engine_forward_slots(st.h, c["sessions"], M.ptr(st.slots), M.ptr(st.ids), M.ptr(st.pos),
                                               M.ptr(st.logits), M.ptr(st.tokens))
        out = (st.logits, st.tokens)
    elif c["kind"] == "head":
        rc = lib.dpuf_engine_forward_batch_ex(st.h, 1, None, 0, M.ptr(st.x), None, None, None, None, 1,
                                              M.ptr(st.logits))
        out = st.logits
    elif c["rows"] == 1:
        rc = lib.dpuf_engine_forward_token(st.h, int(st.ids[0]), c["pos"], M.ptr(st.logits))
        out = st.logits
    else:
        rc = lib.dpuf_engine_forward_batch(st.h, c["rows"], M.ptr(st.ids), c["pos"], 1, M.ptr(st.logits))
        out = st.logits
    if rc != 0:
        raise RuntimeError(f"return code {rc}: " + lib.dpuf_amd_last_error().decode())
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def work(case):
    d = _dims(case)
    H, I, L, V, hd = d["hidden_size"], d["intermediate_size"], d["num_layers"], d["vocab_size"], d["head_dim"]
    qd, kvd = d["num_q_heads"] * hd, d["num_kv_heads"] * hd
    unit = {12: 144 / 256, 13: 144 / 256, 14: 208 / 256}  # bytes per weight
    rows = case["sessions"] if case["kind"] == "slots" else case["rows"]
    nbytes, flops = 0.0, 0.0
    for l in range(L):
        for name, r, c, _ in _layer_mats(d):
            if name == "w_down" and case["keep"] and rows > 1:
                r = min(r, case["keep"] * 16)
            nbytes += r * c * unit[_mode(case["plan"], l, name)]
            flops += 2.0 * rows * r * c
    lm_mode = _mode(case["plan"], 0, "tok" if d["tie_word_embeddings"] else "lm")
    lm_rows = rows if case["kind"] == "slots" else 1
    # the head: the zone's tiles are what every step needs, the rest only when the margin is not met
    head = case["zone"] * 16 or V
    nbytes += head * H * unit[lm_mode] + lm_rows * V * 4.0
    flops += 2.0 * lm_rows * head * H
    nbytes += rows * H * (4.0 if case["kind"] == "head" else unit[_mode(case["plan"], 0, "tok")])
    kv_row = 2 * kvd * (4.0 if case["kv"] == "f32" else 1.125)
    for _, n in _contexts(case):
        new = 1 if case["kind"] == "slots" else rows
        pairs = new * n + new * (new + 1) / 2
        nbytes += L * kv_row * (n + 2 * new)
        flops += 4.0 * L * qd * pairs
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # The framework's contract is the reference's fp32 operation order, bit
    # for bit: its tests compare bit patterns with the oracle, because any
    # reordered sum moves values across the int8 rounding of the next
    # activations (1 to 7 % of a logit after one step of a whole model) and
    # with them the greedy tokens.
    return "exact"


# ---------------------------------------------------------------------------
# the same mathematics in 64 bits
# ---------------------------------------------------------------------------

def _hadamard():
    h = torch.ones(1, 1, dtype=torch.float64, device=DEV)
    for _ in range(6):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)], 0)
    return h / 8


def _sign_vec(signs):
    bits = (signs.unsqueeze(1) >> torch.arange(8, device=DEV, dtype=torch.uint8)) & 1
    return 1 - 2 * bits.reshape(-1).double()


def _int8_blocks(x, floor):
    """x with every 32 values rounded to int8 multiples of their amax / 127."""
    b = x.view(*x.shape[:-1], -1, 32)
    amax = b.abs().amax(-1, keepdim=True)
    step = amax / 127
    q = torch.round(b / torch.where(amax > floor, step, torch.ones_like(step))) * step
    return torch.where(amax > floor, q, torch.zeros_like(q)).view(x.shape)


def _matmul(mat, x, keep=0):
    """W x of rows x: the activations rotated and rounded to int8 as the format says."""
    r = (x * _sign_vec(mat.signs)).view(x.shape[0], -1, 64) @ _hadamard()
    y = _int8_blocks(r.reshape(x.shape), 1e-4) @ mat.f64().t()
    if keep:
        y[:, keep * 16:] = 0
    return y


def _rms(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, pos):
    half = x.shape[-1] // 2
    freq = THETA ** (-torch.arange(half, device=DEV, dtype=torch.float64) / half)
    ang = pos.double().view(-1, 1, 1) * freq
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * ang.cos() - b * ang.sin(), b * ang.cos() + a * ang.sin()], -1)


def _attention(q, k, v, pos):
    """q [rows][heads][hd], k and v [kv heads][keys][hd]; row i sees keys up to pos[i]."""
    rows, nq, hd = q.shape
    group = nq // k.shape[0]
    mask = torch.arange(k.shape[1], device=DEV).view(1, -1) > pos.view(-1, 1)
    out = torch.empty_like(q)
    for h in range(nq):
        s = (q[:, h] @ k[h // group].t()) / math.sqrt(hd)
        out[:, h] = torch.softmax(s.masked_fill(mask, -math.inf), -1) @ v[h // group]
    return out.reshape(rows, nq * hd)


def exact(case, seed):
    d = _dims(case)
    tok, lm, out_norm = _ends(case, d, seed)
    if case["kind"] == "head":
        logits = _matmul(lm, _rms(_hidden(case, d, seed).double(), out_norm))[0]
        if case["zone"]:
            top = torch.topk(logits[:case["zone"] * 16], 2).values
            if float(top[0] - top[1]) >= ZONE_MARGIN:
                logits[case["zone"] * 16:] = -1e9
        return logits.cpu().numpy()
    ids = torch.from_numpy(_ids(case, d, seed)).long().to(DEV)
    rows, nq, nkv, hd = len(ids), d["num_q_heads"], d["num_kv_heads"], d["head_dim"]
    h = _embed_rows(tok, ids)
    ctx = _contexts(case)
    if case["kind"] == "slots":
        pos = torch.tensor(_positions(case), device=DEV)
        owner = [(s, n, slice(s, s + 1)) for s, n in ctx]
    else:
        pos = case["pos"] + torch.arange(rows, device=DEV)
        owner = [(0, case["pos"], slice(0, rows))]
    caches = [_cache(case, d, seed, s, n) for s, n, _ in owner]
    for l in range(d["num_layers"]):
        mats, norms = _layer(case, d, seed, l)
        x = _rms(h, norms[0])
        q = _rope(_rms(_matmul(mats["w_q"], x).view(rows, nq, hd), norms[1]), pos)
        k = _rope(_rms(_matmul(mats["w_k"], x).view(rows, nkv, hd), norms[2]), pos)
        v = _matmul(mats["w_v"], x).view(rows, nkv, hd)
        ao = torch.empty(rows, nq * hd, dtype=torch.float64, device=DEV)
        for (_, _, sl), cache in zip(owner, caches):
            kk = torch.cat([cache[l, 0].double(), k[sl].transpose(0, 1)], 1)
            vv = torch.cat([cache[l, 1].double(), v[sl].transpose(0, 1)], 1)
            if case["kv"] == "q8":
                kk, vv = _int8_blocks(kk, 1e-12), _int8_blocks(vv, 1e-12)
            ao[sl] = _attention(q[sl], kk, vv, pos[sl])
        h = h + _matmul(mats["w_o"], ao)
        x = _rms(h, norms[3])
        y = torch.nn.functional.silu(_matmul(mats["w_gate"], x)) * _matmul(mats["w_up"], x)
        y = torch.where(y.abs() >= DEADZONE, y, torch.zeros_like(y))
        h = h + _matmul(mats["w_down"], y, case["keep"] if rows > 1 and case["kind"] == "step" else 0)
    if case["kind"] == "step":
        return _matmul(lm, _rms(h[-1:], out_norm))[0].cpu().numpy()
    return _matmul(lm, _rms(h, out_norm)).cpu().numpy(), None


def _embed_rows(tok, ids):
    """Embedding rows: the stored rows rotated back."""
    sub = object.__new__(_Matrix)
    sub.rows, sub.cols, sub.mode, sub.u = len(ids), tok.cols, tok.mode, tok.u[ids]
    if tok.mode == 12:
        sub.s = tok.s[ids]
    else:
        sub.d, sub.m = tok.d[ids], tok.m[ids]
    return (sub.f64().view(len(ids), -1, 64) @ _hadamard()).reshape(len(ids), -1) * _sign_vec(tok.signs)
