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


# What a case is for is which kernel it reaches: tile (of 64-row by 64-token waves) and slices along K.  test_dispatch.py holds the
# launches of the built library against it.  Steps are of 32 elements of K (padded to 64), the tiles keep 5 (2 x 2), 4 (4 x 2) or 3 of them in LDS.
#   (width, ff, tokens), tile and slices of the product up (K = width), and down (K = ff)
BF16_CASES = [
    # one tile of tokens, two of rows with a few rows in the second; six steps each: one behind a whole round
    ((136, 130, 128), (2, 2, 1), (2, 2, 1)),
    ((136, 1090, 129), (2, 2, 1), (2, 2, 4)),       # a token past the tile; down 36 steps: four slices of nine, four behind a round
    ((320, 1160, 191), (2, 2, 1), (2, 2, 4)),       # ten steps, no remainder; down 38: slices of 10, 10, 10 and 8
    ((256, 4100, 383), (2, 2, 1), (2, 2, 8)),       # eight steps: three behind a round; down 130: slices of 17, the last of 11
    ((64, 8196, 385), (4, 2, 1), (2, 2, 8)),        # two steps, fewer than the stages; down 258: slices of 33, the last of 27
    ((128, 28800, 250), (4, 2, 1), (2, 2, 8)),      # four steps; enough tiles of 256 x 128 to fill the chip; down 900: slices of 113, the last of 109
    ((128, 28800, 300), (4, 3, 1), (2, 2, 8)),      # 256 x 192: the second tile of tokens mostly empty; four steps: one behind a round
    ((64, 28804, 300), (4, 3, 1), (2, 2, 8)),       # two steps, four rows in the last block; down 902: slices of 113, the last of 111
    ((192, 28800, 300), (4, 3, 1), (2, 2, 8)),      # six steps: whole rounds
    ((128, 28804, 385), (4, 4, 1), (2, 2, 8)),      # one token in the last tile
    ((64, 28800, 385), (4, 4, 1), (2, 2, 8)),       # two steps
    # slices in a number that is no power of two: five of 41 steps, the last of 40; three of 44, the last of 42; seven of 41, the last of 36
    ((1032, 6500, 385), (2, 2, 1), (2, 2, 5)),
    ((2100, 4100, 385), (2, 2, 1), (2, 2, 3)),
    ((1032, 9000, 400), (4, 2, 1), (2, 2, 7)),
]


@pytest.mark.parametrize("width,ff,tokens", [c[0] for c in BF16_CASES])
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


#   (width, heads, kv heads, ff), tokens, tile and slices of q/k/v, o, gate/up and down
KQUANT_MANY_CASES = [
    ((512, 4, 1, 768), 129, (2, 2, 1), (2, 2, 1), (2, 2, 1), (2, 2, 1)),        # a token past the tile; 16 and 24 steps
    ((512, 4, 1, 768), 143, (2, 2, 1), (2, 2, 1), (2, 2, 1), (2, 2, 1)),        # the last block of 16 tokens one short
    ((256, 2, 1, 28672), 140, (2, 2, 1), (2, 2, 1), (4, 3, 1), (2, 2, 8)),      # 256 x 192, most of it empty
    ((256, 2, 1, 14336), 256, (2, 2, 1), (2, 2, 1), (4, 2, 1), (2, 2, 8)),      # 256 x 128
    ((256, 2, 1, 28672), 256, (2, 2, 1), (2, 2, 1), (4, 4, 1), (2, 2, 8)),      # 256 x 256
    # down projection of 88 steps in slices of eleven; three query heads' worth of rows in the last tile
    ((1024, 8, 2, 2816), 385, (2, 2, 1), (2, 2, 1), (2, 2, 1), (2, 2, 8)),
    # every product in slices: rotation and append behind q/k/v, SwiGLU behind the slices of the pair; the tile of tokens full but for one, and whole
    ((2048, 16, 4, 2048), 129, (2, 2, 4), (2, 2, 8), (2, 2, 4), (2, 2, 8)),
    ((2048, 16, 4, 2048), 200, (2, 2, 4), (2, 2, 4), (2, 2, 4), (2, 2, 4)),
    ((2304, 2, 1, 2304), 129, (2, 2, 8), (2, 2, 1), (4, 3, 8), (2, 2, 4)),      # the sliced pair on 256 x 192: nine steps a slice
    ((3328, 2, 1, 768), 700, (2, 2, 8), (2, 2, 1), (4, 2, 4), (2, 2, 1)),       # ... on 256 x 128: 26 steps a slice
    # q/k/v on tiles of 256 rows of which one holds k's last rows and v's first: in slices, on 256 x 128 and 256 x 192; in one piece
    ((4096, 12, 3, 256), 129, (4, 2, 8), (2, 2, 4), (2, 2, 8), (2, 2, 1)),
    ((2560, 30, 5, 256), 129, (4, 3, 8), (2, 2, 4), (2, 2, 8), (2, 2, 1)),
    ((256, 22, 11, 256), 700, (4, 2, 1), (2, 2, 8), (2, 2, 1), (2, 2, 1)),
    # slices that are no power of two: five of 42 steps, the last of 40; three of 67, the last of 66
    ((2304, 2, 1, 6656), 129, (2, 2, 8), (2, 2, 1), (2, 2, 1), (2, 2, 5)),
    ((2816, 2, 1, 6400), 257, (2, 2, 8), (2, 2, 1), (4, 3, 2), (2, 2, 3)),
    # waves with both, one and none of their two halves of 32 tokens: a whole half and a token past it, behind a whole wave and in front of empty ones
    ((512, 4, 1, 768), 160, (2, 2, 1), (2, 2, 1), (2, 2, 1), (2, 2, 1)),
    ((512, 4, 1, 768), 161, (2, 2, 1), (2, 2, 1), (2, 2, 1), (2, 2, 1)),
    ((2048, 16, 4, 2048), 288, (2, 2, 2), (2, 2, 4), (2, 2, 2), (2, 2, 4)),
    ((256, 2, 1, 28672), 289, (2, 2, 1), (2, 2, 1), (4, 3, 1), (2, 2, 8)),
    ((256, 2, 1, 28672), 417, (2, 2, 1), (2, 2, 1), (4, 4, 1), (2, 2, 8)),
]


@pytest.mark.parametrize("shape,tokens", [c[:2] for c in KQUANT_MANY_CASES])
def test_kquant_products_of_many_tokens(tmp_path, shape, tokens):
    """A chunk through one layer over f16 copies, against the oracle and against the GEMM that forms the same weights as it goes."""
    m = mesh()
    cfg = kquant(*shape)
    path = str(tmp_path / "model.gguf")
    tensors = models.write_model(path, cfg, [0], seed=7)
    x = np.random.Generator(np.random.PCG64(tokens)).standard_normal((tokens, cfg["n_embd"])).astype(np.float32)
    want = StageOracle(cfg, tensors, 0, 1, 768, blas=True).forward(x, np.arange(tokens))
    got = {}
    for copies in (0, 1):
        st = m.Stage(path, 0, 1, n_ctx=768, n_batch_max=768, tuning={"tile_copies": copies})
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


# (width, heads, kv heads, ff), tokens, slices of the product down without copies
MANY_SLICES_CASES = [
    ((2816, 2, 1, 4096), 300, 3),           # slices of 22, 22 and 20 steps of 64 on the 128-row tile
    ((5120, 2, 1, 7680), 40, 6),            # of 20 on the register-formed tile
    ((5120, 2, 1, 7936), 64, 6),            # 21, the last of 19
]


@pytest.mark.parametrize("shape,tokens", [c[:2] for c in MANY_SLICES_CASES])
def test_slices_in_any_number(tmp_path, shape, tokens):
    m = mesh()
    cfg = kquant(*shape)
    path = str(tmp_path / "model.gguf")
    tensors = models.write_model(path, cfg, [0], seed=7, fast=True)
    x = np.random.Generator(np.random.PCG64(tokens)).standard_normal((tokens, cfg["n_embd"])).astype(np.float32)
    want = StageOracle(cfg, tensors, 0, 1, 512, blas=True).forward(x, np.arange(tokens))
    st = m.Stage(path, 0, 1, n_ctx=512, n_batch_max=512, tuning={"tile_copies": 0})
    got = []
    for split in (1, 0):
        ses = st.session(gemm_splitk=split)
        got.append(ses.decode(x, np.arange(tokens)).view(np.float32).reshape(want.shape))
        ses.close()
    st.close()
    # (the bounds of the products above)
    assert np.linalg.norm(got[0] - want) < 3e-3 * np.linalg.norm(want), np.linalg.norm(got[0] - want) / np.linalg.norm(want)
    assert np.linalg.norm(got[0] - got[1]) < 1e-3 * np.linalg.norm(want)


# (width, heads, kv heads, ff), tokens, whether v of another type goes with q and k
TYPES_CASES = [
    ((2048, 16, 4, 512), 65, True),         # four slices of K; a token past the narrow tiles
    ((2048, 16, 4, 512), 256, True),        # whole tiles of tokens
    ((2048, 16, 4, 512), 300, False),       # four slices of q and k, two with v
    ((512, 4, 1, 768), 65, True),           # not split
    ((512, 4, 1, 768), 129, True),
    ((256, 44, 11, 256), 700, True),        # 55 + 11 row blocks by six of tokens
    ((256, 80, 8, 256), 700, False),        # q and k on the 256-row tile
]


@pytest.mark.parametrize("arch", ["llama", "qwen2"])
@pytest.mark.parametrize("swap", [False, True])
@pytest.mark.parametrize("shape,tokens,rides", TYPES_CASES)
def test_projections_of_two_types(tmp_path, monkeypatch, shape, tokens, rides, swap, arch):
    """q and k of q4_K and v of q6_K, or the other way round, in one launch and in three, against the oracle."""
    m = mesh()
    cfg = dict(kquant(*shape), arch=arch, bias=arch == "qwen2")
    path = str(tmp_path / "model.gguf")
    if swap:
        monkeypatch.setattr(models, "q4km_type", lambda name, *a: models.Q4_K if name == "attn_v" else models.Q6_K)
    tensors = models.write_model(path, cfg, [0], seed=7, fast=True)
    assert tensors["blk.0.attn_v.weight"][0] != tensors["blk.0.attn_q.weight"][0]
    x = np.random.Generator(np.random.PCG64(tokens)).standard_normal((tokens, cfg["n_embd"])).astype(np.float32)
    want = StageOracle(cfg, tensors, 0, 1, 768, blas=True).forward(x, np.arange(tokens))
    st = m.Stage(path, 0, 1, n_ctx=768, n_batch_max=768, tuning={"tile_copies": 0})
    got = []
    for fused in (1, 0):
        ses = st.session(gemm_fused=fused)
        got.append(ses.decode(x, np.arange(tokens)).view(np.float32).reshape(want.shape))
        ses.close()
    st.close()
    # the bounds of the products above: f16 inputs of four products; the same weights and inputs summed in another order
    assert np.linalg.norm(got[0] - want) < 3e-3 * np.linalg.norm(want), np.linalg.norm(got[0] - want) / np.linalg.norm(want)
    assert np.linalg.norm(got[0] - got[1]) < 1e-3 * np.linalg.norm(want)


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


@pytest.mark.parametrize("n_embd,tokens", [(512, 65), (1024, 515), (512, 770), (2048, 514)])
def test_router_of_a_chunk_over_tokens_a_workgroup(tmp_path, n_embd, tokens):
    """Two, three or four tokens a workgroup of the router, with one or two left over, and expert rows that its eight waves do not
    share evenly; the gathered rows in quarters."""
    m = mesh()
    cfg = dict(arch="qwen3moe", n_layer=1, n_embd=n_embd, n_head=4, n_head_kv=2, head_dim=128, n_ff=0, n_vocab=256, eps=1e-6, rope=1e6,
               n_expert=27, n_expert_used=3, n_ff_exp=256, qk_norm=True)
    path = str(tmp_path / "model.gguf")
    tensors = models.write_model(path, cfg, [0], seed=6, router="zipf")
    x = models.zipf_hidden_state(np.random.Generator(np.random.PCG64(tokens)), tokens, n_embd)
    orc = StageOracle(cfg, tensors, 0, 1, 1024, blas=True)
    want = orc.forward(x, np.arange(tokens)) - x
    st = m.Stage(path, 0, 1, n_ctx=1024, n_batch_max=1024)
    ses = st.session(moe_gemm_min_pairs=1)
    got = ses.decode(x, np.arange(tokens)).view(np.float32).reshape(want.shape) - x
    same = (np.sort(ses.moe_last_ids(tokens), axis=1) == np.sort(np.stack(orc.last_expert_ids), axis=1)).all(axis=1)
    ses.close()
    st.close()
    assert same.mean() > 0.97           # (near ties, as above)
    # f16 activations: 11 bits in the inputs of the layer's products
    assert np.linalg.norm((got - want)[same]) / np.linalg.norm(want[same]) < 3e-3


# width, experts, tokens, whether gate and up are of q6_K; whether the expert launch reads the router's rows by its slots, not a gathered copy
EXPERT_ROWS_CASES = [
    (512, 24, 33, False, True),
    (1024, 24, 130, True, True),            # a large expert: a tile of 128 pairs and one behind it
    (2048, 40, 301, False, True),
    (2048, 40, 77, True, True),
    (512, 120, 200, False, False),          # many short expert rows: their router writes none
    (512, 120, 257, False, True),
    (4096, 24, 33, False, False),
    (256, 24, 33, False, False),
]


def expert_config(n_embd, n_expert, n_layer=1):
    return dict(arch="qwen3moe", n_layer=n_layer, n_embd=n_embd, n_head=4, n_head_kv=2, head_dim=128, n_ff=0, n_vocab=256, eps=1e-6, rope=1e6,
                n_expert=n_expert, n_expert_used=3, n_ff_exp=256, qk_norm=True)


@pytest.mark.parametrize("n_embd,n_expert,tokens,q6,rows", EXPERT_ROWS_CASES)
def test_expert_products_over_rows_by_slot(tmp_path, monkeypatch, n_embd, n_expert, tokens, q6, rows):
    m = mesh()
    cfg = expert_config(n_embd, n_expert)
    path = str(tmp_path / "model.gguf")
    if q6:
        plain = models.q4km_type
        monkeypatch.setattr(models, "q4km_type", lambda name, *a: models.Q6_K if name in ("ffn_gate_exps", "ffn_up_exps") else plain(name, *a))
    tensors = models.write_model(path, cfg, [0], seed=6, router="zipf", fast=True)
    assert tensors["blk.0.ffn_gate_exps.weight"][0] == (models.Q6_K if q6 else models.Q4_K)
    x = models.zipf_hidden_state(np.random.Generator(np.random.PCG64(tokens)), tokens, n_embd)
    orc = StageOracle(cfg, tensors, 0, 1, 512, blas=True)
    want = orc.forward(x, np.arange(tokens)) - x
    st = m.Stage(path, 0, 1, n_ctx=512, n_batch_max=512)
    ses = st.session(moe_gemm_min_pairs=1)
    for _ in range(2):                      # (rows and slots of another routing lie in the buffers the second time)
        got = ses.decode(x, np.arange(tokens)).view(np.float32).reshape(want.shape) - x
        same = (np.sort(ses.moe_last_ids(tokens), axis=1) == np.sort(np.stack(orc.last_expert_ids), axis=1)).all(axis=1)
        assert same.mean() > 0.97           # (near ties, as above)
        # f16 activations: 11 bits in the inputs of the layer's products
        assert np.linalg.norm((got - want)[same]) / np.linalg.norm(want[same]) < 3e-3
        ses.decode(np.ascontiguousarray(x[::-1]), np.arange(tokens))
    assert ses.f16_saturations() == 0
    ses.close()
    st.close()


def test_clamped_rows_count_once_a_slot(tmp_path):
    """Values past the range of f16 in the normalised rows: counted by pairs of neighbours, for every expert of the token."""
    m = mesh()
    n_embd, tokens = 512, 40
    cfg = expert_config(n_embd, 24)
    path = str(tmp_path / "model.gguf")
    kvs, tensors = models.build_tensors(cfg, [0], seed=6, fast=True)
    g = np.ones(n_embd, np.float32)
    g[[6, 7, 100, 301]] = 1e5
    blank = ("ffn_gate_exps", "ffn_up_exps", "ffn_down_exps", "attn_output")       # (nothing else that could be clamped, and rows as they come in)
    tensors = [(n, t, d, g.view(np.uint8) if "ffn_norm" in n else np.zeros_like(data) if any(b in n for b in blank) else data) for n, t, d, data in tensors]
    models.G.write_gguf(path, kvs, tensors)
    x = np.random.Generator(np.random.PCG64(3)).standard_normal((tokens, n_embd)).astype(np.float32)
    y = x * (1 / np.sqrt((x.astype(np.float64) ** 2).mean(axis=1, keepdims=True) + 1e-6)) * g
    assert np.abs(np.abs(y) / 65504 - 1).min() > 1e-4
    pairs = int((np.abs(y) > 65504).reshape(tokens, -1, 2).any(axis=2).sum())
    assert pairs
    st = m.Stage(path, 0, 1, n_ctx=512, n_batch_max=512)
    ses = st.session(moe_gemm_min_pairs=1)
    ses.decode(x, np.arange(tokens))
    assert ses.f16_saturations() == pairs * cfg["n_expert_used"]
    ses.close()
    st.close()


#   shape as above, tokens, (32-column groups, groups of waves, slices) of gate/up and down
KQUANT_FEW_CASES = [
    ((256, 2, 1, 256), 17, (1, 4, 1), (1, 4, 1)),       # four steps along K: one for each group of waves; padding columns
    ((512, 4, 1, 768), 32, (1, 4, 1), (1, 4, 1)),       # the full 32-column tile; 12 steps
    ((512, 4, 1, 2816), 33, (2, 4, 1), (2, 2, 4)),      # 44 steps in slices of eleven, six and five of them for a slice's two groups
    ((1024, 8, 2, 2816), 64, (2, 2, 2), (2, 2, 4)),     # the full 64-column tile; the pair in slices
    # more row blocks than compute units: two groups of waves, K in one piece (512 blocks and more: the 256-row tile takes those)
    ((256, 2, 1, 20480), 20, (1, 2, 1), (1, 2, 16)),
    ((256, 2, 1, 20480), 47, (2, 2, 1), (2, 2, 16)),
    ((512, 4, 1, 32512), 33, (2, 2, 1), (2, 2, 16)),
]


@pytest.mark.parametrize("shape,tokens", [c[:2] for c in KQUANT_FEW_CASES])
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


#   shape as above, tokens, groups of waves of gate/up
DECODE_BATCH_CASES = [
    ((256, 2, 1, 256), 17, 4),          # four steps along K, one per group; two columns' worth past the first block
    ((768, 6, 2, 2816), 32, 4),         # twelve steps; all columns
    ((512, 4, 1, 33024), 23, 2),        # more row blocks than compute units: two groups
    ((512, 4, 1, 768), 5, 4),           # one block of 16 columns
]


@pytest.mark.parametrize("shape,tokens", [c[:2] for c in DECODE_BATCH_CASES])
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


# super-blocks of 256 along K per wave of the f16 skinny GEMM: rounds of two, one left over, waves with one more than others, fewer
# super-blocks than waves
@pytest.mark.parametrize("width,ff", [(256, 256), (512, 1280), (768, 3840), (1280, 5376), (2048, 6400)])
def test_batches_of_decode_steps_along_k(tmp_path, width, ff):
    """Every product of two layers (q6_K v and down projections in the first) for 4 to 32 decode steps, at K of `width` and `ff`."""
    m = mesh()
    cfg = dict(arch="llama", n_layer=2, n_embd=width, n_head=width // 128, n_head_kv=width // 256, head_dim=128, n_ff=ff, n_vocab=256, eps=1e-5, rope=1e4)
    path = os.path.join(str(tmp_path), "model.gguf")
    tensors = models.write_model(path, cfg, [0, 1], seed=4)
    st = m.Stage(path, 0, 2, n_ctx=16, n_seq_max=32, n_batch_max=32)
    ses = st.session()
    orc = StageOracle(cfg, tensors, 0, 2, 16, n_seq_max=32)
    rng = np.random.Generator(np.random.PCG64(5))
    done = np.zeros(32, np.int32)
    for T in (4, 11, 16, 17, 32):
        x = rng.standard_normal((T, width)).astype(np.float32)
        pos, seq = done[:T].copy(), list(range(T))
        done[:T] += 1
        got = ses.decode(x, pos, seq=seq).view(np.float32).reshape(T, width).astype(np.float64)
        want = orc.forward(x, pos, seq=seq).astype(np.float64)
        # activations rounded to f16 in front of every product (2^-12 root mean square, seven products and the attention): 4 * 2^-12 * sqrt(8)
        assert np.linalg.norm(got - want) <= 2.8e-3 * np.linalg.norm(want), (T, np.linalg.norm(got - want) / np.linalg.norm(want))
    ses.close()
    st.close()


# super-blocks of a wave of the launches behind a norm: one; two; two or three; one, and none for some waves
@pytest.mark.parametrize("width", [2048, 4096, 5120, 1280])
def test_norms_handed_over_to_short_walks(tmp_path, width):
    """The partial sums of a norm that reach a launch behind its weights, where its walk is too short to cover them: against norm launches
    of their own, and the same bits call after call."""
    m = mesh()
    cfg = dict(arch="llama", n_layer=3, n_embd=width, n_head=width // 128, n_head_kv=width // 256, head_dim=128, n_ff=1280, n_vocab=256, eps=1e-5, rope=1e4)
    path = os.path.join(str(tmp_path), "model.gguf")
    models.write_model(path, cfg, [0, 1, 2], seed=4)
    st = m.Stage(path, 0, 3, n_ctx=16, n_seq_max=32, n_batch_max=32)
    ses = [st.session(skinny_norm_fused=on) for on in (1, 0)]
    rng = np.random.Generator(np.random.PCG64(5))
    for T in (4, 16, 17, 32):
        x = rng.standard_normal((T, width)).astype(np.float32) * (10.0 ** rng.uniform(-2, 2, (T, 1))).astype(np.float32)
        pos, seq = np.zeros(T, np.int32), list(range(T))
        outs = [s.decode(x, pos, seq=seq).view(np.float32).reshape(T, width).astype(np.float64) for s in ses]
        for _ in range(8):
            assert np.array_equal(ses[0].decode(x, pos, seq=seq).view(np.float32).reshape(T, width), outs[0]), (width, T)
        # a norm of its own rounds scaled rows to f16, the hand-over rows before their scale (2^-12 of themselves each, root mean
        # square): six products behind one; 4 * 2^-12 * sqrt(2 * 6)
        worst = np.max(np.linalg.norm(outs[0] - outs[1], axis=1) / np.linalg.norm(outs[1], axis=1))
        assert worst <= 3.4e-3, (width, T, worst)
    for s in ses:
        s.close()
    st.close()


# width, ff, tokens, and of the down projection's launch: tile-rows a workgroup, slices along K, workgroups a slice
STEP_SLICE_CASES = [
    ((2048, 4352), 17, (3, 4, 43)),         # slices of 5, 5, 5 and 2 super-blocks for eight waves, two rows in the last group; one column past a block
    ((5376, 8704), 24, (4, 3, 84)),         # 12, 12 and 10
    ((5120, 8704), 32, (5, 4, 64)),         # 9, 9, 9 and 7; every column
]


# the same of one block of columns, whose walks have to be longer to be cut: 27 super-blocks a slice, three or four a wave; a part of the block and all of it
STEP_SLICE_FEW_CASES = [((5120, 27648), 5, (5, 4, 64)), ((5120, 27648), 16, (5, 4, 64))]


@pytest.mark.parametrize("shape,tokens", [c[:2] for c in STEP_SLICE_CASES + STEP_SLICE_FEW_CASES])
def test_down_projections_of_decode_steps_in_slices(tmp_path, shape, tokens):
    """Two layers (q4_K down projection, whose sums write the next norm's rows, then q6_K) against the oracle and against whole launches."""
    m = mesh()
    width, ff = shape
    cfg = dict(kquant(width, 2, 1, ff), n_layer=2)
    path = os.path.join(str(tmp_path), "model.gguf")
    tensors = models.write_model(path, cfg, [0, 1], seed=4, fast=True)
    assert [tensors["blk.%d.ffn_down.weight" % i][0] for i in (0, 1)] == [models.Q4_K, models.Q6_K]
    st = m.Stage(path, 0, 2, n_ctx=16, n_seq_max=32, n_batch_max=32)
    ses = [st.session(gemm_splitk=on) for on in (1, 0)]
    orc = StageOracle(cfg, tensors, 0, 2, 16, n_seq_max=32, blas=True)
    rng = np.random.Generator(np.random.PCG64(5))
    for step in range(2):
        x = rng.standard_normal((tokens, width)).astype(np.float32)
        pos, seq = [step] * tokens, list(range(tokens))
        got, whole = [s.decode(x, pos, seq=seq).view(np.float32).reshape(tokens, width).astype(np.float64) for s in ses]
        want = orc.forward(x, pos, seq=seq).astype(np.float64)
        # activations rounded to f16 in front of every product (2^-12 root mean square, eight products): 4 * 2^-12 * sqrt(8)
        assert np.linalg.norm(got - want) <= 2.8e-3 * np.linalg.norm(want), (tokens, np.linalg.norm(got - want) / np.linalg.norm(want))
        # the same products in another order; behind it a norm of its own rounds scaled rows to f16, the hand-over rows before their scale
        assert np.linalg.norm(got - whole) <= 2e-3 * np.linalg.norm(whole), tokens
    for s in ses:
        s.close()
    st.close()


# rows of one and two groups of eight a thread, whole and with idle threads; token counts of every tile that splits
@pytest.mark.parametrize("width,heads", [(768, 6), (2048, 16), (4096, 32), (5120, 40)])
def test_norms_ride_with_the_sums_of_slices(tmp_path, width, heads):
    """Chunks whose output and down projections are split: the next norm's rows from the launch that adds the slices against a norm launch of
    their own, and against the oracle."""
    m = mesh()
    cfg = dict(arch="llama", n_layer=3, n_embd=width, n_head=heads, n_head_kv=2, head_dim=128, n_ff=1280, n_vocab=256, eps=1e-5, rope=1e4)
    path = os.path.join(str(tmp_path), "model.gguf")
    tensors = models.write_model(path, cfg, [0, 1, 2], seed=4)
    st = m.Stage(path, 0, 3, n_ctx=256, n_seq_max=1, n_batch_max=256)
    rng = np.random.Generator(np.random.PCG64(5))
    for T in (17, 33, 70, 130, 200):
        x = rng.standard_normal((T, width)).astype(np.float32)
        x[:, 3] *= 20.0
        out = []
        for rides in (1, 0):
            ses = st.session(gemm_norm_rides=rides)
            out.append(ses.decode(x, np.arange(T)).view(np.float32).reshape(T, width).astype(np.float64))
            ses.close()
        want = StageOracle(cfg, tensors, 0, 3, 256, blas=True).forward(x, np.arange(T)).astype(np.float64)
        size = np.linalg.norm(want)
        # the two norms add a row's squares in another order (2^-24 of the scale), which moves a value of f16 where it sits next to a
        # rounding point: fewer than one in 2^10, by 2^-11 of itself
        assert np.linalg.norm(out[0] - out[1]) <= 2.0 ** -11 * size, (width, T, np.linalg.norm(out[0] - out[1]) / size)
        # f16 inputs of seven products a layer and weights rounded once (2^-12 root mean square each): 4 * 2^-12 * sqrt(3 * 10)
        assert np.linalg.norm(out[0] - want) <= 5.4e-3 * size, (width, T, np.linalg.norm(out[0] - want) / size)
    st.close()
