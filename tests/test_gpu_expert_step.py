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


def test_swiglu_beyond_f16_is_kept_and_beyond_its_range_counted(tmp_path):
    """Outputs of 1e5 to 2^22 stay exact to their 22 bits (f16 alone ends at 65504)."""
    m = mesh()
    cfg = dict(arch="qwen3moe", n_layer=1, n_embd=512, n_head=4, n_head_kv=2, head_dim=128, n_ff=0, n_vocab=256, eps=1e-6, rope=1e6, n_expert=24,
               n_expert_used=4, n_ff_exp=256, qk_norm=True)
    for gain, clamps in ((400.0, False), (20000.0, True)):
        kvs, tl = models.build_tensors(cfg, [0], seed=3)
        tl = [(n, t, d, (x.view(np.float32) * gain).view(np.uint8)) if n.endswith("ffn_norm.weight") else (n, t, d, x) for n, t, d, x in tl]
        tl = [(n, t, d, (x.view(np.float32) / gain).view(np.uint8)) if n.endswith("gate_inp.weight") else (n, t, d, x) for n, t, d, x in tl]
        path = str(tmp_path / "model.gguf")
        G.write_gguf(path, kvs, tl)
        st = m.Stage(path, 0, 1, n_ctx=16, n_seq_max=8, n_batch_max=16)
        x = np.random.Generator(np.random.PCG64(1)).standard_normal((5, 512)).astype(np.float32)
        pos, seq = np.zeros(5, np.int32), np.arange(5, dtype=np.int32)
        ses = st.session()
        got = ses.decode(x, pos, seq=seq).view(np.float32).reshape(x.shape)
        assert np.isfinite(got).all()
        assert (ses.f16_saturations() > 0) == clamps
        if not clamps:
            want = StageOracle(cfg, {n: (t, d, v) for n, t, d, v in tl}, 0, 1, 16, n_seq_max=8).forward(x, pos, seq=seq)
            assert np.linalg.norm(got - want) / np.linalg.norm(want) < 2e-4
        ses.close()
        st.close()
