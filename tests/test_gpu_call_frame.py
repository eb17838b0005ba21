"""What stands around the layers of a call: the caller's f32 rows read and written where they lie (16-byte aligned device
memory) or through copies (anything else), positions as launch arguments (up to 32 tokens) or through pinned slots, logits of
one row straight to host memory.  Every way is the same arithmetic, so outputs are compared bit for bit."""
import os

import numpy as np
import pytest

import models
from util import mesh

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def open_stage(tmp_path, name, lb, le, n_batch):
    m = mesh()
    cfg = models.CONFIGS[name]
    path = os.path.join(str(tmp_path), name + ".gguf")
    models.write_model(path, cfg, range(cfg["n_layer"]), seed=5, with_embd=True, with_output=True)
    st = m.Stage(path, lb, le, n_ctx=128, n_seq_max=40, n_batch_max=n_batch)
    os.unlink(path)
    return cfg, st


def dev_call(st, x, pos, seq, shift=0, out="other", graphs=0):
    """The call over device memory, `shift` floats off its start; out: other memory, the input's own, one row further on."""
    ses = st.session(graphs=graphs)
    T, E = x.shape
    buf = torch.empty(shift + (T + 1) * E, dtype=torch.float32, device="cuda")
    d_in = buf[shift:shift + T * E]
    d_in.copy_(torch.from_numpy(x).reshape(-1))
    d_out = dict(other=torch.empty(shift + T * E, dtype=torch.float32, device="cuda")[shift:], same=d_in, overlap=buf[shift + E:shift + (T + 1) * E])[out]
    torch.cuda.synchronize()
    ses.decode_dev(d_in.data_ptr(), pos, d_out.data_ptr(), T * E * 4, seq=seq)
    ses.synchronize()
    y = d_out.cpu().numpy().reshape(T, E).copy()
    if out == "other":
        assert np.array_equal(d_in.cpu().numpy().reshape(T, E), x)
    ses.close()
    return y


# 1, 3: mat-vecs; 4, 16: one block of columns; 32, 33: launch arguments and slots, two blocks of columns and the large tile
@pytest.mark.parametrize("tokens", [1, 3, 4, 16, 32, 33])
@pytest.mark.parametrize("name", ["tiny-llama", "tiny-moe"])
@pytest.mark.parametrize("layers", [1, 2])
def test_rows_in_place_equal_rows_copied(tmp_path, name, layers, tokens):
    cfg, st = open_stage(tmp_path, name, 0, layers, 64)
    rng = np.random.Generator(np.random.PCG64(tokens))
    x = rng.standard_normal((tokens, cfg["n_embd"])).astype(np.float32)
    for pos, seq in ((np.zeros(tokens, np.int32), np.arange(tokens, dtype=np.int32)), (np.arange(tokens, dtype=np.int32), np.full(tokens, 39, np.int32))):
        copied = dev_call(st, x, pos, seq, shift=1)
        for kw in (dict(), dict(out="same"), dict(out="overlap"), dict(graphs=1), dict(shift=4)):
            assert np.array_equal(dev_call(st, x, pos, seq, **kw), copied), kw
        ses = st.session()
        assert np.array_equal(ses.decode(x, pos, seq=seq).view(np.float32).reshape(x.shape), copied)
        ses.close()
    st.close()


@pytest.mark.parametrize("where", ["input", "output", "both"])
def test_rows_in_pinned_host_memory_take_copies(tmp_path, where):
    """An aligned pointer that a copy accepts, and no memory of the device: what the rows are read from or written to in place."""
    cfg, st = open_stage(tmp_path, "tiny-llama", 0, 2, 64)
    for T in (1, 16, 33):
        x = np.random.Generator(np.random.PCG64(T)).standard_normal((T, cfg["n_embd"])).astype(np.float32)
        pos, seq = np.zeros(T, np.int32), np.arange(T, dtype=np.int32)
        want = dev_call(st, x, pos, seq)
        d_in = torch.empty(x.shape, dtype=torch.float32, pin_memory=True) if where != "output" else torch.empty(x.shape, dtype=torch.float32, device="cuda")
        d_out = torch.zeros(x.shape, dtype=torch.float32, pin_memory=True) if where != "input" else torch.zeros(x.shape, dtype=torch.float32, device="cuda")
        assert d_in.data_ptr() % 16 == 0 and d_out.data_ptr() % 16 == 0
        d_in.copy_(torch.from_numpy(x))
        torch.cuda.synchronize()
        ses = st.session()
        ses.decode_dev(d_in.data_ptr(), pos, d_out.data_ptr(), x.nbytes, seq=seq)
        ses.synchronize()
        assert np.array_equal(d_out.cpu().numpy(), want)
        ses.close()
    st.close()


def test_calls_queued_without_a_wait_keep_their_own_positions(tmp_path):
    cfg, st = open_stage(tmp_path, "tiny-llama", 0, 2, 64)
    E = cfg["n_embd"]
    rng = np.random.Generator(np.random.PCG64(3))
    x = torch.from_numpy(rng.standard_normal((100, E)).astype(np.float32)).cuda()
    outs = []
    for wait in (True, False):
        ses = st.session()
        out = torch.empty_like(x)
        at = 0
        torch.cuda.synchronize()
        for step in range(40):
            n = (1, 2, 5)[step % 3]                      # (a copy per slot would go round the ring five times)
            if at + n > 100:
                break
            ses.decode_dev(x[at:].data_ptr(), np.full(n, step, np.int32), out[at:].data_ptr(), n * E * 4, seq=np.arange(n, dtype=np.int32))
            if wait:
                ses.synchronize()
            at += n
        ses.synchronize()
        outs.append(out[:at].cpu().numpy())
        ses.close()
    assert np.array_equal(outs[0], outs[1])
    st.close()


def test_one_row_of_logits_equals_its_row_among_several(tmp_path):
    cfg, st = open_stage(tmp_path, "tiny-llama", 0, models.CONFIGS["tiny-llama"]["n_layer"], 64)
    ids = np.arange(5, dtype=np.int32)
    pos = np.zeros(5, np.int32)
    m = mesh()
    rows = []
    for want in (None, np.array([0, 0, 1, 0, 0], np.uint8)):
        ses = st.session()
        rows.append(ses.decode(ids, pos, seq=np.arange(5, dtype=np.int32), in_fmt=m.TOKENS, out_fmt=m.LOGITS, want=want).view(np.float32).reshape(-1, cfg["n_vocab"]))
        ses.close()
    np.testing.assert_allclose(rows[1][0], rows[0][2], rtol=0, atol=1e-5 * np.abs(rows[0]).max())     # (one column or five to a pass over the weights)
    st.close()
