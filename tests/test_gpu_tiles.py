"""The large-tile products at the edges of their tiles: rows, tokens and steps along K that leave remainders, every tile shape and
split that the plan picks, against the plain oracle."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import models
import nadosun_util as N
from folder_util import error, open_stage, run
from oracle.nadosun import NadosunOracle
from oracle.stage import StageOracle
from util import mesh

pytestmark = pytest.mark.gpu

# rms of a row's difference over the rms of all rows: the bound of the other bf16 comparisons with this oracle
BF16_LIMIT = 2e-2


@pytest.mark.parametrize("width,ff,tokens", [
    (136, 130, 128),        # one tile of rows and a few rows more, one of tokens
    (136, 1090, 129),       # a row of tokens past the tile; down projection of 34 steps, whole or in slices of 17
    (320, 1160, 191),       # 38 steps: two left behind whole rounds of the stages
    (256, 4100, 383),       # down projection in several slices, the last one shorter
    (128, 28800, 250),      # enough tiles of 256 x 128 to fill the chip
    (128, 28800, 300),      # 256 x 192: the second tile of tokens mostly empty
    (128, 28804, 385),      # one token in the last tile, four rows in the last block
])
def test_products_of_many_tokens(tmp_path, width, ff, tokens):
    """A feed-forward of `ff` behind attention over `tokens` tokens: products of (rows, K) = (ff, width) and (width, ff)."""
    cfg = N.config(64, width, 8, [N.attention(2, 1, 64, 50, ff=ff)])
    w = N.random_weights(cfg, 3)
    folder = N.write_folder(str(tmp_path / "model"), cfg, w)
    t = N.prompt(cfg, tokens, 9)
    want = NadosunOracle(cfg, w).forward(t)[-100:]
    plain = open_stage(folder, "bf16", n_ctx=512, batch=512, tuning={"tile_copies": 0})
    st = open_stage(folder, "bf16", n_ctx=512, batch=512)
    got = run(st, t, [tokens], last=100)
    # the same tiles over weights in plain rows: the same products in the same order
    assert np.array_equal(run(plain, t, [tokens], last=100), got)
    plain.close()
    rows = run(st, t, [tokens], last=100, linear_tile_min_tokens=1 << 20)      # the weight-streaming kernel on the same inputs
    st.close()
    assert np.isfinite(got).all()
    assert error(got, want) < BF16_LIMIT, (width, ff, tokens, error(got, want))
    # the two add the same products of the same bf16 values in another order (1e-6); a result next to a rounding point of the next
    # product's bf16 input moves by 2^-8 of itself there: a small share of what the oracle's bound allows for all inputs
    assert error(got, rows) < BF16_LIMIT / 2, (width, ff, tokens, error(got, rows))


def kquant(n_embd, n_head, n_kv, n_ff):
    return dict(arch="llama", n_layer=1, n_embd=n_embd, n_head=n_head, n_head_kv=n_kv, head_dim=128, n_ff=n_ff, n_vocab=256, eps=1e-5, rope=1e4)


@pytest.mark.parametrize("shape,tokens", [
    ((512, 4, 1, 768), 129),        # matrices of one launch that end inside a tile of 256 rows; slices along K; a token past the tile
    ((512, 4, 1, 768), 143),        # the last block of 16 tokens one short
    ((256, 2, 1, 28672), 140),      # 256 x 192, most of it empty
    ((256, 2, 1, 14336), 256),      # 256 x 128
    ((256, 2, 1, 28672), 256),      # 256 x 256
    ((1024, 8, 2, 2816), 385),      # down projection of 88 steps in slices; three query heads' worth of rows in the last tile
])
def test_kquant_products_of_many_tokens(tmp_path, shape, tokens):
    """A chunk through one layer over f16 copies, against the oracle and against the GEMM that forms the same weights as it goes."""
    m = mesh()
    cfg = kquant(*shape)
    path = str(tmp_path / "model.gguf")
    tensors = models.write_model(path, cfg, [0], seed=7)
    x = np.random.Generator(np.random.PCG64(tokens)).standard_normal((tokens, cfg["n_embd"])).astype(np.float32)
    want = StageOracle(cfg, tensors, 0, 1, 512, blas=True).forward(x, np.arange(tokens))
    got = {}
    for copies in (0, 1):
        st = m.Stage(path, 0, 1, n_ctx=512, n_batch_max=512, tuning={"tile_copies": copies})
        ses = st.session()
        got[copies] = ses.decode(x, np.arange(tokens)).view(np.float32).reshape(want.shape)
        assert ses.f16_saturations() == 0
        ses.close()
        st.close()
    norm = np.linalg.norm(want)
    # f16 activations over one layer: 11 bits in the inputs of four products (the bound of the other f16 paths)
    assert np.linalg.norm(got[1] - want) / norm < 3e-3, (shape, tokens)
    # the same f16 weights and inputs summed in another order: what a rounding point of the next input next to a sum can move
    assert np.linalg.norm(got[1] - got[0]) / norm < 1e-3, (shape, tokens)


@pytest.mark.parametrize("n_embd,ff,tokens", [
    (256, 256, 17),         # one round of four steps along K; every expert in a tile of at most 32 pairs
    (512, 256, 65),
    (256, 512, 150),        # an expert past one tile of 128
    (512, 768, 301),        # remainders of one to four groups of 32 pairs
])
def test_expert_products_over_ragged_loads(tmp_path, n_embd, ff, tokens):
    """A chunk through two expert layers (q4_K and q6_K down projections) whose experts get from a few pairs to most tokens: the
    expert tiles against the oracle and against the 16-pair integer kernel."""
    m = mesh()
    cfg = dict(arch="qwen3moe", n_layer=2, n_embd=n_embd, n_head=4, n_head_kv=2, head_dim=128, n_ff=0, n_vocab=256, eps=1e-6, rope=1e6,
               n_expert=24, n_expert_used=3, n_ff_exp=ff, qk_norm=True)
    path = str(tmp_path / "model.gguf")
    tensors = models.write_model(path, cfg, [0, 1], seed=5, router="zipf")
    x = models.zipf_hidden_state(np.random.Generator(np.random.PCG64(tokens)), tokens, n_embd)
    orc = StageOracle(cfg, tensors, 0, 2, 512, blas=True)
    want = orc.forward(x, np.arange(tokens)) - x
    got, ids = {}, {}
    for tiles in (0, 1):
        st = m.Stage(path, 0, 2, n_ctx=512, n_batch_max=512)
        ses = st.session(moe_gemm=tiles, moe_gemm_min_pairs=1)
        got[tiles] = ses.decode(x, np.arange(tokens)).view(np.float32).reshape(want.shape) - x
        ids[tiles] = np.sort(ses.moe_last_ids(tokens), axis=1)
        assert ses.f16_saturations() == 0
        ses.close()
        st.close()
    # a token whose routing a rounding point moved is another computation: at most a few near ties, not compared
    same = (ids[0] == np.sort(np.stack(orc.last_expert_ids), axis=1)).all(axis=1) & (ids[0] == ids[1]).all(axis=1)
    assert same.mean() > 0.97
    norm = np.linalg.norm(want[same])
    # f16 activations: 11 bits in the inputs of the four products of each layer, and once more through the second layer
    assert np.linalg.norm((got[1] - want)[same]) / norm < 6e-3
    assert np.linalg.norm((got[1] - got[0])[same]) / norm < 6e-3


@pytest.mark.parametrize("shape,tokens", [
    ((256, 2, 1, 256), 17),         # four steps along K: one for each group of waves; padding columns
    ((512, 4, 1, 768), 32),         # the full 32-column tile; 12 steps
    ((512, 4, 1, 2816), 33),        # 44 steps in slices of eleven, six and five of them for a slice's two groups
    ((1024, 8, 2, 2816), 64),       # the full 64-column tile
    ((256, 2, 1, 33024), 47),       # more row blocks than compute units: K in one piece
])
def test_kquant_products_of_few_tokens(tmp_path, shape, tokens):
    """A chunk of 17 to 64 tokens through one layer, against the oracle and against the 128-column tile."""
    m = mesh()
    cfg = kquant(*shape)
    path = str(tmp_path / "model.gguf")
    tensors = models.write_model(path, cfg, [0], seed=11)
    x = np.random.Generator(np.random.PCG64(tokens)).standard_normal((tokens, cfg["n_embd"])).astype(np.float32)
    want = StageOracle(cfg, tensors, 0, 1, 128, blas=True).forward(x, np.arange(tokens))
    st = m.Stage(path, 0, 1, n_ctx=128, n_batch_max=128)
    got = {}
    for narrow in (0, 1):
        ses = st.session(gemm_narrow=narrow)
        got[narrow] = ses.decode(x, np.arange(tokens)).view(np.float32).reshape(want.shape)
        assert ses.f16_saturations() == 0
        ses.close()
    st.close()
    norm = np.linalg.norm(want)
    # f16 activations over one layer: 11 bits in the inputs of four products
    assert np.linalg.norm(got[1] - want) / norm < 3e-3, (shape, tokens)
    # the same weights and inputs, sums along K met in another order
    assert np.linalg.norm(got[1] - got[0]) / norm < 1e-3, (shape, tokens)


@pytest.mark.parametrize("shape,tokens", [
    ((256, 2, 1, 256), 17),         # four steps along K, one per group; two columns' worth past the first block
    ((768, 6, 2, 2816), 32),        # twelve steps; all columns
    ((512, 4, 1, 33024), 23),       # more row blocks than compute units: two groups
    ((512, 4, 1, 768), 5),          # one block of 16 columns
])
def test_gate_up_of_a_decode_batch(tmp_path, shape, tokens):
    """A batch of single steps through two layers with gate / up on the register-formed tile, the norm before it handed over, against
    the oracle and against the f16 skinny GEMM."""
    m = mesh()
    cfg = dict(kquant(*shape), n_layer=2)
    path = str(tmp_path / "model.gguf")
    tensors = models.write_model(path, cfg, [0, 1], seed=13)
    x = np.random.Generator(np.random.PCG64(tokens)).standard_normal((tokens, cfg["n_embd"])).astype(np.float32)
    pos, seq = np.zeros(tokens, np.int32), np.arange(tokens, dtype=np.int32)
    want = StageOracle(cfg, tensors, 0, 2, 64, n_seq_max=tokens, blas=True).forward(x, pos, seq=seq)
    st = m.Stage(path, 0, 2, n_ctx=64, n_seq_max=tokens, n_batch_max=32)
    got = {}
    for least in (1, 33):
        ses = st.session(reg_min_tokens=least, reg_min_blocks=1)
        got[least] = ses.decode(x, pos, seq=seq).view(np.float32).reshape(want.shape)
        assert ses.f16_saturations() == 0
        ses.close()
    st.close()
    norm = np.linalg.norm(want)
    # f16 activations over two layers: 11 bits in the inputs of eight products
    assert np.linalg.norm(got[1] - want) / norm < 4e-3, (shape, tokens)
    # the same inputs and weights of one rounding each, formed in two ways and summed in two orders
    assert np.linalg.norm(got[1] - got[33]) / norm < 2e-3, (shape, tokens)
