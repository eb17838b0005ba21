"""Expert products of decode steps on the f16 matrix cores (expert_step): every count of waves along K, items of 1 to 8 pairs, experts
with several items, both weight types on both sides, against the oracle and against the mat-vec kernel's 16-bit fixed point."""
import numpy as np
import pytest

import gguf_util as G
import models
from oracle.stage import StageOracle
from util import mesh

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


# 512: two super-blocks along K; 1024: four; 2048: eight; feed-forward rows of one, three and five
@pytest.mark.parametrize("n_embd,ff", [(512, 256), (1024, 768), (2048, 1280)])
@pytest.mark.parametrize("gate", [models.Q4_K, models.Q6_K])
def test_expert_products_of_decode_steps(tmp_path, n_embd, ff, gate):
    m = mesh()
    NE = 24
    cfg = dict(arch="qwen3moe", n_layer=2, n_embd=n_embd, n_head=4, n_head_kv=2, head_dim=128, n_ff=0, n_vocab=256, eps=1e-6, rope=1e6,
               n_expert=NE, n_expert_used=4, n_ff_exp=ff, qk_norm=True)
    kvs, tl = models.build_tensors(cfg, [0, 1], seed=7, router="zipf")
    rng = np.random.Generator(np.random.PCG64(n_embd + gate))
    tl = [(n, gate, d, models.random_tensor(rng, gate, ff * NE, n_embd)) if "gate_exps" in n or "up_exps" in n else (n, t, d, x) for n, t, d, x in tl]
    assert {t for n, t, _, _ in tl if "down_exps" in n} == {models.Q4_K, models.Q6_K}
    path = str(tmp_path / "model.gguf")
    G.write_gguf(path, kvs, tl)
    st = m.Stage(path, 0, 2, n_ctx=16, n_seq_max=32, n_batch_max=32)
    tensors = {n: (t, d, x) for n, t, d, x in tl}
    for T in (1, 2, 7, 16, 17, 32):
        x = models.zipf_hidden_state(np.random.Generator(np.random.PCG64(T)), T, n_embd)
        pos, seq = np.zeros(T, np.int32), np.arange(T, dtype=np.int32)
        orc = StageOracle(cfg, tensors, 0, 2, 16, n_seq_max=32, blas=True)
        want = orc.forward(x, pos, seq=seq) - x
        got, ids = [], []
        for least in (1, 33):
            ses = st.session(moe_step_min_tokens=least, moe_gemm=0)
            got.append(ses.decode(x, pos, seq=seq).view(np.float32).reshape(x.shape) - x)
            ids.append(np.sort(ses.moe_last_ids(T), axis=1))
            assert ses.f16_saturations() == 0
            ses.close()
        same = (ids[0] == np.sort(np.stack(orc.last_expert_ids), axis=1)).all(axis=1) & (ids[0] == ids[1]).all(axis=1)
        assert same.mean() > 0.9            # (a near tie of the routing that a last bit moved is another computation)
        norm = np.linalg.norm(want[same])
        # 16-bit fixed point per 32 elements on the mat-vec side: about 2e-5 a product, four products.  From 17 tokens on the second
        # layer's attention rounds its inputs to f16: of two inputs 3e-5 apart one in 16 rounds to the next value, 4.9e-4 off, 1.2e-4 in
        # the mean square; twice that
        assert np.linalg.norm((got[0] - got[1])[same]) / norm < (1e-4 if T <= 16 else 2.5e-4), T
        assert np.linalg.norm((got[0] - want)[same]) / norm < (2e-4 if T <= 16 else 3e-3), T
    st.close()


def scaled(tensors, factors):
    """The tensors with the f32 vectors or the block factors of those whose name ends so multiplied: by one number, or block by block."""
    out = []
    for n, t, d, x in tensors:
        for end, f in factors.items():
            if not n.endswith(end):
                continue
            if t == models.F32:
                x = (x.view(np.float32) * np.float32(f)).view(np.uint8)
                continue
            block, at = {models.Q4_K: (144, (0, 2)), models.Q6_K: (210, (208,))}[t]
            x = x.copy().reshape(-1, block)
            for i in at:
                h = np.ascontiguousarray(x[:, i:i + 2]).view(np.float16)[:, 0].astype(np.float32) * np.resize(np.float32(f), len(x))
                x[:, i:i + 2] = h.astype(np.float16).view(np.uint8).reshape(-1, 2)
            x = x.reshape(-1)
        out.append((n, t, d, x))
    return out


def blocks_of_rows(n_rows, row_len, of_row):
    """of_row(row) for every block of a matrix of that many rows."""
    return np.repeat([of_row(r) for r in range(n_rows)], row_len // 256).astype(np.float32)


# Exponents of factors: on the normalised rows (router weights take it back), on the down projection, and between the SwiGLU outputs that
# meet its first super-block and the others, which its factors take back.  Outputs of about 2^24, 2^34 (rows beyond 65504), 2^-15 and
# 2^-23, and outputs of one row 2^16 apart.
@pytest.mark.parametrize("rows,down,first", [(0, 0, 0), (13, 0, 0), (18, 0, 0), (-6, 10, 0), (-10, 20, 0), (0, 6, 16)])
def test_activations_of_any_size_keep_their_precision(tmp_path, rows, down, first):
    m = mesh()
    NE, FF, E = 24, 512, 512
    cfg = dict(arch="qwen3moe", n_layer=2, n_embd=E, n_head=4, n_head_kv=2, head_dim=128, n_ff=0, n_vocab=256, eps=1e-6, rope=1e6, n_expert=NE,
               n_expert_used=4, n_ff_exp=FF, qk_norm=True)
    kvs, tl = models.build_tensors(cfg, [0, 1], seed=3)
    factors = {"ffn_norm.weight": 2.0 ** rows, "gate_inp.weight": 2.0 ** -rows, "down_exps.weight": 2.0 ** down}
    if first:
        # up's rows 0 to 255 larger, down's first super-block smaller by as much
        factors["up_exps.weight"] = blocks_of_rows(NE * FF, E, lambda r: 2.0 ** (first // 2) if r % FF < 256 else 2.0 ** (-first // 2))
        factors["down_exps.weight"] = np.resize(np.float32([2.0 ** (down - first // 2), 2.0 ** (down + first // 2)]), NE * E * FF // 256)
    tl = scaled(tl, factors)
    path = str(tmp_path / "model.gguf")
    G.write_gguf(path, kvs, tl)
    st = m.Stage(path, 0, 2, n_ctx=16, n_seq_max=8, n_batch_max=16)
    for T in (1, 5):
        x = np.random.Generator(np.random.PCG64(T)).standard_normal((T, E)).astype(np.float32)
        pos, seq = np.zeros(T, np.int32), np.arange(T, dtype=np.int32)
        orc = StageOracle(cfg, {n: (t, d, v) for n, t, d, v in tl}, 0, 2, 16, n_seq_max=8)
        want = orc.forward(x, pos, seq=seq) - x
        got = []
        for least in (1, 33):           # this kernel, and the mat-vec form with a scale per 32 values
            ses = st.session(moe_step_min_tokens=least)
            got.append(ses.decode(x, pos, seq=seq).view(np.float32).reshape(x.shape) - x)
            assert (np.sort(ses.moe_last_ids(T), axis=1) == np.sort(np.stack(orc.last_expert_ids), axis=1)).all()
            assert ses.f16_saturations() == 0
            ses.close()
        # Either way the attention of the layers rounds queries, keys and values to f16: 2^-12 at most of each value, a third to a half of
        # it in the mean square, 1.4e-4 for two of them one after another; the products add 2e-5 to it.
        errors = [np.linalg.norm(g - want) / np.linalg.norm(want) for g in got]
        assert errors[0] < 2e-4 and errors[0] < 1.5 * errors[1], (T, errors)
    st.close()
