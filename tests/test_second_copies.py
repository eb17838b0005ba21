"""Second copies of the weights (tile_copies) where memory is short: a stage opens without them, and allocations that find no
other room get theirs."""
import os
import sys
import threading
import time

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import models
import nadosun_util as N
from hip_host_util import call
from util import mesh

CFG = dict(arch="llama", n_layer=2, n_embd=512, n_head=4, n_head_kv=2, head_dim=128, n_ff=1536, n_vocab=256, eps=1e-5, rope=1e4)
TOKENS = 200


def write(kind, path):
    if kind == "gguf":
        path = os.path.join(path, "model.gguf")
        models.write_model(path, CFG, [0, 1], seed=3)
        return path
    cfg = N.config(64, 512, 8, [N.attention(4, 2, 128, 50, ff=1536)] * 2)
    return N.write_folder(os.path.join(path, "model"), cfg, N.random_weights(cfg, 3))


def open_stage(path, **kw):
    return mesh().Stage(path, 0, 2, n_ctx=512, n_batch_max=256, **kw)


def uses_copies(host, session):
    """Whether a prefill call of the session runs over the copies."""
    m = mesh()
    host.launches()
    if session.stage.info.n_vocab == 64:
        session.seq_reset(0)
        session.decode(np.zeros(TOKENS, np.int32), np.arange(TOKENS), in_fmt=m.TOKENS)
    else:
        session.decode(np.zeros((TOKENS, 512), np.float32), np.arange(TOKENS))
    names = [n for n, _, _ in host.launches()]
    tiles = [n for n in names if n.startswith(("gemm_f16_kernel", "linear_tile_kernel"))]
    if session.stage.info.n_vocab == 64:
        assert tiles
        return all(n.startswith("linear_tile_kernel<0,0") or n.startswith("linear_tile_kernel<1,0") for n in tiles)
    return bool(tiles)


def held(host, path, **kw):
    """Bytes of a stage, and of a session."""
    before = host.used
    st = open_stage(path, **kw)
    stage = host.used - before
    ses = st.session()
    session = host.used - before - stage
    ses.close()
    st.close()
    assert host.used == before
    return stage, session


def short_at_open(host, path, left):
    plain, session = held(host, path, tuning={"tile_copies": 0})
    copies = held(host, path)[0] - plain
    assert copies > 0
    # room for the copies by the rule when it is asked; then another process leaves `left` of what they need
    host.memory(plain + 20 * copies)
    host.take_after_info(int((20 - left) * copies))
    st = open_stage(path)
    assert host.used == plain, "nothing of the copies is kept"
    host.others(0)
    host.memory(plain + session)
    ses = st.session()
    out = uses_copies(host, ses)
    ses.close()
    st.close()
    return out, host.used


@pytest.mark.parametrize("kind", ["gguf", "folder"])
@pytest.mark.parametrize("left", [0.01, 0.6, 2])
def test_a_stage_opens_without_the_copies_that_find_no_room(tmp_path, kind, left):
    """Memory that was free when the rule was asked and is not when the copies are made (0.01: not for the first, 0.6: not for the
    last; 2: for all of them, but no longer within the rule)."""
    assert call(short_at_open, path=write(kind, str(tmp_path)), left=left) == [False, 0]


def with_room(host, path):
    st = open_stage(path)
    ses = st.session()
    return uses_copies(host, ses)


@pytest.mark.parametrize("kind", ["gguf", "folder"])
def test_a_stage_with_room_keeps_them(tmp_path, kind):
    assert call(with_room, path=write(kind, str(tmp_path))) is True


def sessions_that_need_the_room(host, path):
    plain, session = held(host, path, tuning={"tile_copies": 0})
    copies = held(host, path)[0] - plain
    n = int(np.ceil(8 * copies / session)) + 1
    # as much as n sessions of a stage without copies take, of which the copies are less than an eighth
    host.memory(plain + n * session)
    st = open_stage(path)
    assert host.used == plain + copies
    first = st.session()
    out = [uses_copies(host, first)]
    more = [st.session() for _ in range(n - 1)]
    assert host.used == plain + n * session
    out += [uses_copies(host, first), uses_copies(host, more[-1])]
    for s in more + [first]:
        s.close()
    st.close()
    # the next stage opens with copies again
    st = open_stage(path)
    ses = st.session()
    out += [uses_copies(host, ses)]
    ses.close()
    st.close()
    return out, host.used


@pytest.mark.parametrize("kind", ["gguf", "folder"])
def test_sessions_get_the_room_that_the_copies_hold(tmp_path, kind):
    assert call(sessions_that_need_the_room, path=write(kind, str(tmp_path))) == [[True, False, False, True], 0]


def stages_and_weights_that_need_the_room(host, path):
    m = mesh()
    plain, session = held(host, path, tuning={"tile_copies": 0})
    copies = held(host, path)[0] - plain
    host.memory(plain + 10 * copies)
    a = open_stage(path)
    b = open_stage(path, tuning={"tile_copies": 0})
    # what is left and one byte of what a's copies hold, in rows of 256 f32
    rows = (10 * copies - plain) // 1024 - (copies // 2) // 1024
    data = np.zeros((rows, 256), np.float32)
    w = m.Weight(m.F32, data, rows, 256)
    assert host.used == 2 * plain + rows * 1024
    too_much = None
    try:
        m.Weight(m.F32, data, rows, 256)
    except m.MeshError as e:
        too_much = e.code
    w.close()
    ses = a.session()
    out = uses_copies(host, ses)            # (and no error of the refused one left for a launch)
    for x in (ses, a, b):
        x.close()
    return [too_much, out, host.used]


def test_other_stages_and_weights_get_it_too(tmp_path):
    m = mesh()
    assert call(stages_and_weights_that_need_the_room, path=write("gguf", str(tmp_path))) == [m.ERR_NOMEM, False, 0]


def graphs_and_copies(host, path):
    plain, session = held(host, path, tuning={"tile_copies": 0})
    host.memory(plain + 12 * session)
    # calls of 24 tokens over the copies, captured
    st = open_stage(path, tuning={"skinny_f16": 0, "tile_min_tokens": 1, "gemm_min_tokens": 17, "skinny_min_tokens": 100000, "graphs": 1})
    ses = st.session()
    pos, seq = np.zeros(24, np.int32), np.zeros(24, np.int32)
    names, replays = [], []

    def step():
        host.launches()
        ses.decode(np.zeros((24, 512), np.float32), pos, seq=seq)
        names.append(any(n.startswith("gemm_f16_kernel") for n, _, _ in host.launches()))
        replays.append(ses.graph_replays)

    for _ in range(3):
        step()
    more = [st.session()]
    while True:
        try:
            more.append(st.session())
        except Exception:
            break
    for _ in range(3):
        step()
    return names, replays


def test_a_captured_call_over_the_copies_is_not_replayed_without_them(tmp_path):
    """The first call runs, the second is captured and replayed, later ones are replays; behind the copies' end it starts anew."""
    names, replays = call(graphs_and_copies, path=write("gguf", str(tmp_path)))
    assert names == [True, True, False, False, False, False]
    assert replays == [0, 1, 2, 2, 3, 4]


def threads_and_copies(host, path):
    plain, session = held(host, path, tuning={"tile_copies": 0})
    copies = held(host, path)[0] - plain
    n = int(np.ceil(8 * copies / session)) + 4
    host.memory(plain + n * session)
    st = open_stage(path)
    ses = [st.session() for _ in range(3)]
    stop, calls, errors = threading.Event(), [0, 0, 0], []

    def work(i):
        try:
            while not stop.is_set():
                ses[i].decode(np.zeros((TOKENS, 512), np.float32), np.arange(TOKENS))
                calls[i] += 1
        except Exception as e:
            errors.append(str(e))

    ts = [threading.Thread(target=work, args=(i,), daemon=True) for i in range(3)]
    for t in ts:
        t.start()

    def wait(since):
        end = time.monotonic() + 20
        while min(c - a for c, a in zip(calls, since)) < 20 and not errors and time.monotonic() < end:
            time.sleep(0.001)

    wait([0, 0, 0])
    more = [st.session() for _ in range(n - 3)]         # waits for its turn among the calls, and gets the copies' room
    at = list(calls)
    wait(at)
    stop.set()
    for t in ts:
        t.join()
    assert min(c - a for c, a in zip(calls, at)) >= 20
    return errors, uses_copies(host, ses[0]), len(more) == n - 3 and host.used == plain + n * session


def test_calls_on_other_threads_go_on(tmp_path):
    assert call(threads_and_copies, path=write("gguf", str(tmp_path))) == [[], False, True]


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["gguf", "folder"])
def test_a_session_goes_on_after_its_stage_gave_the_copies_back(tmp_path, kind):
    """A session too large for any GPU is refused as ever; the copies are gone then, and the other session's next call, queued with
    launches over the copies still under way, gives what a stage without copies gives."""
    torch = pytest.importorskip("torch")
    m = mesh()
    path = write(kind, str(tmp_path))
    rng = np.random.Generator(np.random.PCG64(8))
    if kind == "gguf":
        x, fmt = rng.standard_normal((TOKENS, 512)).astype(np.float32), m.F32
    else:
        x, fmt = rng.integers(0, 64, TOKENS).astype(np.int32), m.TOKENS

    def run(ses):
        if kind == "folder":
            ses.seq_reset(0)
        return ses.decode(x, np.arange(TOKENS), in_fmt=fmt).view(np.float32)

    plain = open_stage(path, tuning={"tile_copies": 0})
    ses = plain.session()
    without = run(ses)
    ses.close()
    plain.close()
    st = open_stage(path)
    huge = mesh().Stage(path, 0, 2, n_ctx=1 << 30, n_seq_max=64, n_batch_max=16)
    ses = st.session()
    with_copies = run(ses)
    if kind == "gguf":
        xd, out = torch.from_numpy(x).cuda(), torch.empty(TOKENS, 512, device="cuda")
        torch.cuda.synchronize()
        for _ in range(20):
            ses.decode_dev(xd.data_ptr(), np.arange(TOKENS), out.data_ptr(), out.numel() * 4)
    with pytest.raises(m.MeshError) as e:
        huge.session()
    assert e.value.code == m.ERR_NOMEM
    huge.close()
    if kind == "gguf":
        ses.synchronize()
        assert np.array_equal(out.cpu().numpy().reshape(-1), with_copies)
    assert np.array_equal(run(ses), without)
    ses.close()
    st.close()
