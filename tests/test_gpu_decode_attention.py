"""Decode attention over the session's cache rows at the edges of its key blocks (32 keys a wave, 128 a workgroup), both head
sizes, every cache tier, alone and split, against a float64 softmax over the rows as the cache holds them."""
import os

import numpy as np
import pytest

torch = pytest.importorskip("torch")

import models
import oracle
from util import mesh

pytestmark = pytest.mark.gpu

TIERS = [(oracle.F16, oracle.F16), (oracle.Q8_0, oracle.Q4_0), (oracle.Q4_0, oracle.Q4_0)]
KEYS = [1, 2, 31, 32, 33, 64, 95, 127, 128, 129, 160, 255, 257, 384, 513]
# Q and the probabilities are rounded to f16 (2^-12 of themselves, root mean square), a quantised row's product with its block
# scale once more: independent errors of three roundings on weights that sum to one stay below 2^-11 of the result; four times that
TOL = 4 * 2.0 ** -11


@pytest.mark.parametrize("kv_types", TIERS)
@pytest.mark.parametrize("name", ["tiny-llama", "tiny-g5", "tiny-g8"])      # head_dim 64; 128 with groups of 5 and 8
def test_key_block_edges(tmp_path, name, kv_types):
    m, cfg = mesh(), models.CONFIGS[name]
    path = os.path.join(str(tmp_path), name + ".gguf")
    models.write_model(path, cfg, [0], seed=3)
    st = m.Stage(path, 0, 1, n_ctx=max(KEYS), n_seq_max=len(KEYS), n_batch_max=32, kv_types=kv_types)
    H, HK, D = cfg["n_head"], cfg["n_head_kv"], cfg["head_dim"]
    rng = np.random.Generator(np.random.PCG64(9))
    ses = st.session()
    for i, n in enumerate(KEYS):
        # (every other sequence's rows past its keys hold large values: a key block reaches past the last key)
        rows = max(KEYS)
        k, v = rng.standard_normal((rows, HK, D)), rng.standard_normal((rows, HK, D))
        k[n:] *= 50.0 * (i % 2)
        v[n:] *= 1000.0 * (i % 2)
        ses.kv_write(0, i, 0, k.astype(np.float16).view(np.uint16), v.astype(np.float16).view(np.uint16))
    q = rng.standard_normal((len(KEYS), H, D)).astype(np.float32) * 1.5
    qd = torch.from_numpy(q).cuda()
    for batch in ([[i] for i in range(len(KEYS))] + [list(range(len(KEYS)))]):
        part = qd[batch].contiguous()
        out = torch.full_like(part, float("nan"))
        torch.cuda.synchronize()
        ses.attn_dev(0, part.data_ptr(), [KEYS[i] - 1 for i in batch], out.data_ptr(), seq=batch)
        ses.synchronize()
        got = out.cpu().numpy().astype(np.float64)
        for j, i in enumerate(batch):
            kd, vd = (r.view(np.float16).astype(np.float64).repeat(H // HK, axis=1) for r in ses.kv_read(0, i, 0, KEYS[i]))
            s = np.einsum("hd,nhd->hn", q[i].astype(np.float64), kd) / np.sqrt(D)
            p = np.exp(s - s.max(1, keepdims=True))
            want = np.einsum("hn,nhd->hd", p / p.sum(1, keepdims=True), vd)
            rel = np.linalg.norm(got[j] - want) / np.linalg.norm(want)
            assert rel <= TOL, (name, kv_types, KEYS[i], len(batch), rel)
    ses.close()
    st.close()


@pytest.mark.parametrize("splits", [1, 2, 3])
@pytest.mark.parametrize("name", ["tiny-llama", "tiny-g5"])
def test_walks_of_more_than_one_block_a_wave(tmp_path, name, splits):
    """f16 rows beyond 128 keys a split come as whole rows of K (of one block a wave as shares of rows)."""
    m, cfg = mesh(), models.CONFIGS[name]
    path = os.path.join(str(tmp_path), name + ".gguf")
    models.write_model(path, cfg, [0], seed=4)
    H, HK, D = cfg["n_head"], cfg["n_head_kv"], cfg["head_dim"]
    keys = [128 * splits + 1, 128 * splits + 31, 1, 256 * splits, 256 * splits + 1, 33, 129]
    st = m.Stage(path, 0, 1, n_ctx=max(keys), n_seq_max=len(keys), n_batch_max=32, kv_types=TIERS[0])
    rng = np.random.Generator(np.random.PCG64(10))
    ses = st.session(attn_split_target=splits * HK * len(keys))
    for i, n in enumerate(keys):
        k, v = rng.standard_normal((max(keys), HK, D)), rng.standard_normal((max(keys), HK, D))
        k[n:], v[n:] = 50.0, 1000.0
        ses.kv_write(0, i, 0, k.astype(np.float16).view(np.uint16), v.astype(np.float16).view(np.uint16))
    q = rng.standard_normal((len(keys), H, D)).astype(np.float32) * 1.5
    qd = torch.from_numpy(q).cuda()
    out = torch.full_like(qd, float("nan"))
    torch.cuda.synchronize()
    ses.attn_dev(0, qd.data_ptr(), [n - 1 for n in keys], out.data_ptr(), seq=list(range(len(keys))))
    ses.synchronize()
    got = out.cpu().numpy().astype(np.float64)
    for i, n in enumerate(keys):
        kd, vd = (r.view(np.float16).astype(np.float64).repeat(H // HK, axis=1) for r in ses.kv_read(0, i, 0, n))
        s = np.einsum("hd,nhd->hn", q[i].astype(np.float64), kd) / np.sqrt(D)
        p = np.exp(s - s.max(1, keepdims=True))
        want = np.einsum("hn,nhd->hd", p / p.sum(1, keepdims=True), vd)
        rel = np.linalg.norm(got[i] - want) / np.linalg.norm(want)
        assert rel <= TOL, (name, splits, n, rel)
    ses.close()
    st.close()


@pytest.mark.parametrize("kv_types", TIERS)
@pytest.mark.parametrize("tokens,lines", [(1, (384,)), (40, (512,)), (60, (1024, 1536, 1920))])
def test_lengths_where_walks_begin_to_be_split(tmp_path, kv_types, tokens, lines):
    """Two KV heads: 2, 80 and 120 (token, head) pairs, for which a launch of one workgroup a CU would have 64, 3 and 2 splits."""
    m, name = mesh(), "tiny-llama"
    cfg = models.CONFIGS[name]
    path = os.path.join(str(tmp_path), name + ".gguf")
    models.write_model(path, cfg, [0], seed=5)
    H, HK, D = cfg["n_head"], cfg["n_head_kv"], cfg["head_dim"]
    assert HK == 2
    longest = max(lines) + 1
    st = m.Stage(path, 0, 1, n_ctx=longest, n_seq_max=2, n_batch_max=64, kv_types=kv_types)
    rng = np.random.Generator(np.random.PCG64(11))
    ses = st.session()
    for i in range(2):
        k, v = (rng.standard_normal((longest, HK, D)).astype(np.float16) for _ in range(2))
        ses.kv_write(0, i, 0, k.view(np.uint16), v.view(np.uint16))
    rows = [[r.view(np.float16).astype(np.float64).repeat(H // HK, axis=1) for r in ses.kv_read(0, i, 0, longest)] for i in range(2)]
    q = rng.standard_normal((tokens, H, D)).astype(np.float32) * 1.5
    qd = torch.from_numpy(q).cuda()
    for line in lines:
        for most in (line, line + 1):
            keys = [most] + [int(n) for n in rng.integers(1, most + 1, tokens - 1)]
            out = torch.full_like(qd, float("nan"))
            torch.cuda.synchronize()
            ses.attn_dev(0, qd.data_ptr(), [n - 1 for n in keys], out.data_ptr(), seq=[i % 2 for i in range(tokens)])
            ses.synchronize()
            got = out.cpu().numpy().astype(np.float64)
            for i, n in enumerate(keys):
                kd, vd = (r[:n] for r in rows[i % 2])
                s = np.einsum("hd,nhd->hn", q[i].astype(np.float64), kd) / np.sqrt(D)
                p = np.exp(s - s.max(1, keepdims=True))
                want = np.einsum("hn,nhd->hd", p / p.sum(1, keepdims=True), vd)
                rel = np.linalg.norm(got[i] - want) / np.linalg.norm(want)
                assert rel <= TOL, (kv_types, tokens, most, n, rel)
    ses.close()
    st.close()
