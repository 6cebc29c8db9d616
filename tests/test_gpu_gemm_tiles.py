"""The tile shapes of the GEMM above 16 tokens (16 x 16, 16 x 32, 32 x 32 and
64 x 32 outputs per wave, chosen by the tiles per SIMD) against the oracle, bit
for bit, in every mode: sizes on each side of the rule, rows that end inside a
fragment, tokens that end inside a tile or leave a wave of a workgroup without
any, and K from one 64-block to several LDS stages with a partial last one."""
import numpy as np
import pytest

from dpuf_amd import model as M
from test_gpu_configs import Pair, bits_equal, log, maxdiff

pytestmark = pytest.mark.gpu

NAMES = {12: "hadamard4_packed", 13: "had4_asym", 14: "had6"}
# (rows, tokens): tiles per SIMD of a 256-CU device in the comment
SIZES = [
    (40, 17),      # < 1
    (4136, 40),    # < 1, the last fragment one group
    (4136, 250),   # 4.05: 16 x 32
    (5000, 270),   # 5.2: one token past a 16-token tile
    (6152, 250),   # 6.02: 32 x 32
    (8200, 289),   # 9.5: 64 x 32 in mode 13; a single token in the last workgroup
    (33000, 257),  # 34: 64 x 32 in mode 12
]


@pytest.mark.parametrize("mode", [12, 13, 14])
@pytest.mark.parametrize("cols", [64, 320, 1088])
@pytest.mark.parametrize("rows,m", SIZES)
def test_gemm_tiles(eng, orc, mode, cols, rows, m):
    if rows * m * cols > 5e9:
        cols = 192  # the oracle's time
    W = M.random_normal(rows * cols, 0.02, 7 + mode, f"t{rows}x{cols}").reshape(rows, cols)
    blob, d = M.pack_matrix(W, M.sign_bits(cols, 7, f"ts{rows}x{cols}"), mode=mode)
    x = np.random.default_rng(rows + cols + m).standard_normal((m, cols)).astype(np.float32)
    x[m - 1, :32] = 1e-6
    out_g = np.full((m, rows), np.nan, np.float32)
    out_o = np.full((m, rows), np.nan, np.float32)
    log(f"mode {mode} rows={rows} cols={cols} M={m}")
    getattr(eng, f"dpuf_matmul_qr_{NAMES[mode]}_f32")(m, rows, cols, d.n_tiles, M.ptr(x), d.tensor_base,
                                                      d.tile_offsets, d.sign_bits, M.ptr(out_g))
    if mode == 12:
        orc.orc_matmul_f32(m, rows, cols, d.n_tiles, M.ptr(x), d.tensor_base, d.tile_offsets, d.sign_bits,
                           M.ptr(out_o))
    else:
        orc.orc_matmul_asym_f32(int(mode == 14), m, rows, cols, d.n_tiles, M.ptr(x), d.tensor_base, d.tile_offsets,
                                d.sign_bits, M.ptr(out_o))
    assert np.isfinite(out_o).all()
    assert bits_equal(out_g, out_o), maxdiff(out_g, out_o)


@pytest.mark.parametrize("mode", [12, 13, 14])
@pytest.mark.parametrize("rows,m", [(40, 5), (4136, 12)] + SIZES)
def test_gemm_overflow(eng, orc, mode, rows, m):
    """Inputs whose partial sums pass the largest float: an output is infinite
    exactly where the reference's chain is (its infinities never come back into
    range, also where the full sum would), in every kernel above one token.
    The spread of a chain's end is 113 sqrt(blocks) times that of the inputs (32
    products with weights of 20 a block): a good part of the largest float, in
    modes 13 and 14 less, whose unsigned dots pass through larger sums."""
    cols = 192 if rows * m > 5e6 else 320
    W = M.random_normal(rows * cols, 20.0, 17 + mode, f"o{rows}x{cols}").reshape(rows, cols)
    blob, d = M.pack_matrix(W, M.sign_bits(cols, 7, f"os{rows}x{cols}"), mode=mode)
    sd = (0.7 if mode == 12 else 0.35) * 3.4e38 / (113 * np.sqrt(cols / 32))
    x = (np.random.default_rng(rows + cols + m).standard_normal((m, cols)) * sd).astype(np.float32)
    out_g = np.full((m, rows), np.nan, np.float32)
    out_o = np.full((m, rows), np.nan, np.float32)
    log(f"overflow: mode {mode} rows={rows} cols={cols} M={m}")
    getattr(eng, f"dpuf_matmul_qr_{NAMES[mode]}_f32")(m, rows, cols, d.n_tiles, M.ptr(x), d.tensor_base,
                                                      d.tile_offsets, d.sign_bits, M.ptr(out_g))
    if mode == 12:
        orc.orc_matmul_f32(m, rows, cols, d.n_tiles, M.ptr(x), d.tensor_base, d.tile_offsets, d.sign_bits,
                           M.ptr(out_o))
    else:
        orc.orc_matmul_asym_f32(int(mode == 14), m, rows, cols, d.n_tiles, M.ptr(x), d.tensor_base, d.tile_offsets,
                                d.sign_bits, M.ptr(out_o))
    bad = ~np.isfinite(out_o)
    assert 0.01 < bad.mean() < 0.99, bad.mean()
    nan = np.isnan(out_o)
    assert np.array_equal(np.isnan(out_g), nan)
    assert bits_equal(np.where(nan, 0, out_g), np.where(nan, 0, out_o)), (~np.isfinite(out_g)).sum() - bad.sum()


@pytest.mark.parametrize("n", [17, 29, 31, 32, 33, 70])
def test_gate_up_swiglu_tiles(eng, orc, n):
    """Gate, up, SwiGLU and the down input's prep in one launch (16 384 gate +
    up rows or more): tokens that fill its tile or end inside it, and 129
    64-column blocks, one past a multiple of the 8 XCDs.  Every row's residual
    of each layer and its logits."""
    shape = dict(hidden_size=256, intermediate_size=8256, num_layers=2, num_q_heads=4, num_kv_heads=2, head_dim=64,
                 vocab_size=512, tie_word_embeddings=1)
    p = Pair(eng, orc, M.Model.build(shape, max_seq_len=96, seed=411))
    p.capture(n)
    log(f"gate + up + SwiGLU: {n} tokens, 8 256 columns")
    lg, lo = p.forward(np.random.default_rng(412 + n).integers(0, 512, n).astype(np.int32), 0, only_last=0)
    cg, co = p.captured(n)
    assert bits_equal(cg, co), maxdiff(cg, co)
    assert bits_equal(lg, lo), maxdiff(lg, lo)
    p.close()
