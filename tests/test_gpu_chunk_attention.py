"""Attention of prompt chunks at the edges of its steps: 64 keys a wave, 128 a workgroup of two key groups, over cached positions
that end anywhere in a step, for the head sizes and query heads per KV head that choose its launches."""
import os

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import models
import oracle
from oracle.stage import StageOracle
from util import mesh

pytestmark = pytest.mark.gpu

CHUNKS = [(0, 17), (0, 64), (0, 65), (1, 127), (0, 129), (63, 40), (64, 64), (127, 33), (128, 192), (300, 97), (190, 257)]
# f16 queries, probabilities and activations of one layer's products (2^-12 of themselves, root mean square, ten roundings on the
# way through the layer, weights of the large tile rounded once more): 4 * 2^-12 * sqrt(12)
TOL = 3.4e-3


# four heads a workgroup; one head and four query tiles; head_dim 64 with two heads and two query tiles; five waves; eight heads
@pytest.mark.parametrize("name", ["tiny-kv3", "tiny-mha", "tiny-llama", "tiny-g5", "tiny-g8"])
def test_chunks_end_anywhere_in_a_step(tmp_path, name):
    m, cfg = mesh(), models.CONFIGS[name]
    path = os.path.join(str(tmp_path), name + ".gguf")
    tensors = models.write_model(path, cfg, [0], seed=6)
    st = m.Stage(path, 0, 1, n_ctx=512, n_seq_max=len(CHUNKS), n_batch_max=320)
    E, HK, D = cfg["n_embd"], cfg["n_head_kv"], cfg["head_dim"]
    rng = np.random.Generator(np.random.PCG64(8))
    ses = st.session()
    orc = StageOracle(cfg, tensors, 0, 1, 512, n_seq_max=len(CHUNKS), blas=True)
    for i, (past, T) in enumerate(CHUNKS):
        if past:
            k, v = (rng.standard_normal((past, HK, D)).astype(np.float16).view(np.uint16) for _ in "kv")
            ses.kv_write(0, i, 0, k, v)
            orc.k[0, i, :, :past], orc.v[0, i, :, :past] = k.transpose(1, 0, 2), v.transpose(1, 0, 2)
        x = rng.standard_normal((T, E)).astype(np.float32)
        pos, seq = np.arange(past, past + T), np.full(T, i, np.int32)
        got = ses.decode(x, pos, seq=seq).view(np.float32).reshape(T, E).astype(np.float64)
        want = orc.forward(x, pos, seq=seq).astype(np.float64)
        worst = np.max(np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1))
        assert np.linalg.norm(got - want) <= TOL * np.linalg.norm(want) and worst <= 2 * TOL, (name, past, T, worst)
    ses.close()
    st.close()


# one and two key groups: walks of 320 keys and the next, walks that are split (533 and 900 keys in two and three), and short ones
@pytest.mark.parametrize("name", ["tiny-kv3", "tiny-mha"])
def test_walks_of_one_and_two_key_groups(tmp_path, name):
    m, cfg = mesh(), models.CONFIGS[name]
    path = os.path.join(str(tmp_path), name + ".gguf")
    tensors = models.write_model(path, cfg, [0], seed=6)
    chunks = [(0, 319), (0, 320), (0, 321), (280, 40), (281, 40), (500, 33), (870, 30), (0, 20)]
    st = m.Stage(path, 0, 1, n_ctx=1024, n_seq_max=len(chunks), n_batch_max=336)
    E, HK, D = cfg["n_embd"], cfg["n_head_kv"], cfg["head_dim"]
    rng = np.random.Generator(np.random.PCG64(18))
    ses = st.session()
    orc = StageOracle(cfg, tensors, 0, 1, 1024, n_seq_max=len(chunks), blas=True)
    for i, (past, T) in enumerate(chunks):
        if past:
            k, v = (rng.standard_normal((past, HK, D)).astype(np.float16).view(np.uint16) for _ in "kv")
            ses.kv_write(0, i, 0, k, v)
            orc.k[0, i, :, :past], orc.v[0, i, :, :past] = k.transpose(1, 0, 2), v.transpose(1, 0, 2)
        x = rng.standard_normal((T, E)).astype(np.float32)
        pos, seq = np.arange(past, past + T), np.full(T, i, np.int32)
        got = ses.decode(x, pos, seq=seq).view(np.float32).reshape(T, E).astype(np.float64)
        want = orc.forward(x, pos, seq=seq).astype(np.float64)
        worst = np.max(np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1))
        assert np.linalg.norm(got - want) <= TOL * np.linalg.norm(want) and worst <= 2 * TOL, (name, past, T, worst)
    ses.close()
    st.close()


def half(x):
    return x.view(np.float16).astype(np.float32)


# heads per KV head, KV heads and the shape of the workgroup: four and five waves, six of six heads and of three heads and two query tiles,
# one head and four query tiles, eight
QUANT = {"four": (4, 3), "five": (5, 2), "six": (6, 2), "three": (3, 2), "one": (1, 4), "eight": (8, 32)}


@pytest.mark.parametrize("kv_types", [(oracle.Q8_0, oracle.Q4_0), (oracle.Q4_0, oracle.Q4_0)])
@pytest.mark.parametrize("shape", sorted(QUANT))
def test_chunks_over_quantised_rows(tmp_path, shape, kv_types):
    """Chunks whose workgroups decode the cache rows themselves, at the edges of their steps, one and two key groups, against the oracle over
    the rows that the device's cache holds."""
    group, n_kv = QUANT[shape]
    # (eight waves a workgroup from 256 workgroups of 32 queries on)
    chunks = [(0, 225), (100, 230)] if shape == "eight" else [(0, 17), (0, 65), (63, 40), (64, 64), (127, 33), (0, 127), (300, 97), (190, 150)]
    m = mesh()
    cfg = dict(arch="llama", n_layer=1, n_embd=512, n_head=group * n_kv, n_head_kv=n_kv, head_dim=128, n_ff=512, n_vocab=256, eps=1e-5, rope=1e4)
    path = os.path.join(str(tmp_path), "model.gguf")
    tensors = models.write_model(path, cfg, [0], seed=6)
    st = m.Stage(path, 0, 1, n_ctx=512, n_seq_max=len(chunks), n_batch_max=256, kv_types=kv_types)
    rng = np.random.Generator(np.random.PCG64(28))
    ses = st.session(chunk_kv16=0)
    orc = StageOracle(cfg, tensors, 0, 1, 512, n_seq_max=len(chunks), blas=True, kv_types=kv_types)
    for i, (past, T) in enumerate(chunks):
        if past:
            k, v = (rng.standard_normal((past, n_kv, 128)).astype(np.float16).view(np.uint16) for _ in "kv")
            ses.kv_write(0, i, 0, k, v)
            orc.k[0, i, :, :past], orc.v[0, i, :, :past] = (half(r).transpose(1, 0, 2) for r in ses.kv_read(0, i, 0, past))
        x = rng.standard_normal((T, 512)).astype(np.float32)
        pos, seq = np.arange(past, past + T), np.full(T, i, np.int32)
        got = ses.decode(x, pos, seq=seq).view(np.float32).reshape(T, 512).astype(np.float64)
        rows = tuple(half(r) for r in ses.kv_read(0, i, past, T))
        want = orc.forward(x, pos, seq=seq, kv_rows={0: rows}).astype(np.float64)
        worst = np.max(np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1))
        # (kv_read rounds a row's values to f16, as the kernel that multiplies them does)
        assert np.linalg.norm(got - want) <= TOL * np.linalg.norm(want) and worst <= 2 * TOL, (shape, past, T, worst)
    ses.close()
    st.close()


@pytest.mark.parametrize("kv_types", [(oracle.F16, oracle.F16), (oracle.Q8_0, oracle.Q4_0)])
@pytest.mark.parametrize("name", ["tiny-llama", "tiny-odd", "tiny-kv3", "tiny-qwen3"])     # head_dim 64 and 128, 8, 7, 18 and 16 vectors, both modes, norms
def test_rotated_rows_of_a_long_chunk(tmp_path, name, kv_types):
    """A chunk whose head vectors share a token's sines against the same tokens in pieces of one vector a wave."""
    m, cfg = mesh(), models.CONFIGS[name]
    path = os.path.join(str(tmp_path), name + ".gguf")
    models.write_model(path, cfg, [0], seed=7)
    T = 193
    st = m.Stage(path, 0, 1, n_ctx=256, n_seq_max=2, n_batch_max=256, kv_types=kv_types)
    ses = st.session(gemv_rope=0)
    x = np.random.Generator(np.random.PCG64(3)).standard_normal((T, cfg["n_embd"])).astype(np.float32)
    ses.decode(x, np.arange(T), seq=np.zeros(T, np.int32))
    for t in range(0, T, 97):
        n = min(97, T - t)
        ses.decode(x[t:t + n], np.arange(t, t + n), seq=np.ones(n, np.int32))
    for kind, whole, parts in zip("kv", ses.kv_read(0, 0, 0, T), ses.kv_read(0, 1, 0, T)):
        a, b = (r.view(np.float16).astype(np.float64) for r in (whole, parts))
        # the projections may be summed in another order and the rows are rounded once: 2^-11 of f16 rows; quantised ones move by a
        # step of 1 / 127 or 1 / 8 of the block's largest value (2 to 3 deviations) in the few places next to a rounding point
        tol = 2.0 ** -11 if kv_types[0] == oracle.F16 else 2.0 ** -7 if kind == "k" else 2.0 ** -4
        assert np.linalg.norm(a - b) / np.linalg.norm(b) <= tol, (name, kv_types, kind)
    ses.close()
    st.close()
