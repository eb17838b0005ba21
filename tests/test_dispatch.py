"""Which kernels the calls of test_gpu_tiles.py and test_gpu_fullsize.py reach, as the built library launches them (host memory, no GPU)."""
import os
import sys
import tempfile

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import models
import nadosun_util as N
import nutavik_util as U
import test_gpu_nutavik as nutavik
import test_gpu_tiles as tiles
from hip_host_util import call
from util import mesh

Q4_K, Q6_K = 12, 14
ROWS, SWIGLU, PARTIAL = 0, 1, 2                     # gemm_f16_kernel's first argument
DENSE, SPLIT, NORM = 0, 1, 3                        # gemm_reg_kernel's third


def products(host):
    return [(n, g) for n, g, _ in host.launches() if n.startswith(("gemm_", "linear_")) and "epilogue" not in n]


def kquant_products(host, cfg, layers, tokens, decode=False, tuning=None, options=None):
    m = mesh()
    host.memory(1 << 37)
    n_seq = tokens if decode else 1
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "model.gguf")
        models.write_model(path, cfg, layers, seed=1, fast=True)
        st = m.Stage(path, layers[0], layers[-1] + 1, n_ctx=max(tokens, 64), n_seq_max=n_seq, n_batch_max=max(tokens, 32 if decode else 512), tuning=tuning)
    ses = st.session(**(options or {}))
    host.launches()
    pos, seq = (np.zeros(tokens, np.int32), np.arange(tokens)) if decode else (np.arange(tokens), None)
    ses.decode(np.zeros((tokens, cfg["n_embd"]), np.float32), pos, seq=seq)
    return products(host)


def bf16_products(host, width, ff, tokens, copies):
    m = mesh()
    host.memory(1 << 37)
    cfg = N.config(64, width, 8, [N.attention(2, 1, 64, 50, ff=ff)])
    with tempfile.TemporaryDirectory() as d:
        st = m.Stage(N.write_folder(d, cfg, N.random_weights(cfg, 3)), 0, -1, n_ctx=512, n_seq_max=4, n_batch_max=512, tuning={"tile_copies": copies})
    ses = st.session()
    host.launches()
    ses.decode(np.zeros(tokens, np.int32), np.arange(tokens), in_fmt=m.TOKENS)
    return products(host)


@pytest.mark.parametrize("copies", [0, 1])
@pytest.mark.parametrize("case,up,down", tiles.BF16_CASES)
def test_products_of_many_tokens(case, up, down, copies):
    width, ff, tokens = case
    got = call(bf16_products, width=width, ff=ff, tokens=tokens, copies=copies)
    big = [(n, g) for n, g in got if n.startswith("linear_tile_kernel")]
    # the feed-forward's: the one of most rows, and what follows it
    at = max(range(len(big)), key=lambda i: big[i][1][0] * int(big[i][0][:-1].split(",")[2])) if ff > 200 else 2
    for (name, grid), (wm, wt, slices), rows in zip(big[at:at + 2], (up, down), (ff, width)):
        assert name == "linear_tile_kernel<0,%d,%d,%d>" % (0 if copies else 1, wm, wt)
        assert grid[:2] == [-(-rows // (64 * wm)) * -(-tokens // (64 * wt)), slices]


@pytest.mark.parametrize("case", tiles.KQUANT_MANY_CASES)
def test_kquant_products_of_many_tokens(case):
    (width, heads, kv, ff), tokens, *plans = case
    got = call(kquant_products, cfg=tiles.kquant(*case[0]), layers=[0], tokens=tokens)
    assert len(got) == 4
    for i, ((name, grid), (wm, wt, slices), rows) in enumerate(zip(got, plans, ((heads + 2 * kv) * 128, width, 2 * ff, width))):
        out = PARTIAL if slices > 1 else SWIGLU if i == 2 else ROWS
        assert name == "gemm_f16_kernel<%d,%d,%d>" % (out, wm, wt), i
        assert grid[:2] == [-(-rows // (64 * wm)) * -(-tokens // (64 * wt)), slices], i


@pytest.mark.parametrize("case", tiles.KQUANT_FEW_CASES)
def test_kquant_products_of_few_tokens(case):
    (width, heads, kv, ff), tokens, gate_up, down = case
    got = call(kquant_products, cfg=tiles.kquant(*case[0]), layers=[0], tokens=tokens)[-2:]
    for (name, grid), (columns, groups, slices), type_, rows in zip(got, (gate_up, down), (Q4_K, Q6_K), (2 * ff, width)):
        assert name == "gemm_reg_kernel<%d,%d,%d,%d>" % (type_, columns, SPLIT if slices > 1 else DENSE, groups)
        assert grid == [rows // 128, 1, slices]
    # (the other side of the test's comparison)
    other = call(kquant_products, cfg=tiles.kquant(*case[0]), layers=[0], tokens=tokens, options={"gemm_narrow": 0})[-2:]
    assert [n.split("<")[0] for n, _ in other] == ["gemm_kq_kernel"] * 2


@pytest.mark.parametrize("case", tiles.DECODE_BATCH_CASES)
def test_gate_up_of_a_decode_batch(case):
    (width, heads, kv, ff), tokens, groups = case
    cfg = dict(tiles.kquant(*case[0]), n_layer=2)
    got = call(kquant_products, cfg=cfg, layers=[0, 1], tokens=tokens, decode=True, options={"reg_min_tokens": 1, "reg_min_blocks": 1})
    assert [g for n, g in got if n == "gemm_reg_kernel<%d,1,%d,%d>" % (Q4_K, NORM, groups)] == [[ff // 64, 1, 1]] * 2
    other = call(kquant_products, cfg=cfg, layers=[0, 1], tokens=tokens, decode=True, options={"reg_min_tokens": 33, "reg_min_blocks": 1})
    assert not any(n.startswith("gemm_reg") for n, _ in other)


@pytest.mark.parametrize("n_embd,n_expert,tokens,q6,rows", tiles.EXPERT_ROWS_CASES)
def test_expert_products_over_rows_by_slot(n_embd, n_expert, tokens, q6, rows):
    names = [n for n, _ in call(kquant_products, cfg=tiles.expert_config(n_embd, n_expert), layers=[0], tokens=tokens, options={"moe_gemm_min_pairs": 1})]
    assert [n for n in names if n.startswith("gemm_expert")] == ["gemm_expert_kernel<%d,%d>" % (Q4_K, 4 if rows else 2), "gemm_expert_kernel<%d,2>" % Q6_K], names


@pytest.mark.parametrize("shape,tokens,slices", tiles.MANY_SLICES_CASES)
def test_slices_in_any_number(shape, tokens, slices):
    name, grid = call(kquant_products, cfg=tiles.kquant(*shape), layers=[0], tokens=tokens, tuning={"tile_copies": 0})[-1]
    assert name.startswith("gemm_reg_kernel<%d," % Q6_K if tokens <= 64 else "gemm_kq_kernel<%d," % Q6_K), name
    assert grid == [shape[0] // 128, -(-tokens // 128), slices]


@pytest.mark.parametrize("shape,tokens,rides", tiles.TYPES_CASES)
def test_projections_of_two_types(shape, tokens, rides):
    names = [n for n, _ in call(kquant_products, cfg=tiles.kquant(*shape), layers=[0], tokens=tokens, tuning={"tile_copies": 0})]
    assert any(n.startswith("gemm_kq_types_kernel<%d,%d," % (Q4_K, Q6_K)) for n in names) == rides, names
    # (a call of few tokens, which the narrow tiles take)
    names = [n for n, _ in call(kquant_products, cfg=tiles.kquant(*shape), layers=[0], tokens=64, tuning={"tile_copies": 0})]
    assert not any("types" in n for n in names)


@pytest.mark.parametrize("case", tiles.STEP_SLICE_CASES)
def test_down_projections_of_decode_steps_in_slices(case):
    (width, ff), tokens, (rows, slices, groups) = case
    cfg = dict(tiles.kquant(width, 2, 1, ff), n_layer=2)
    sliced = lambda **kw: [c for c in call(kquant_products, cfg=cfg, layers=[0, 1], decode=True, **kw) if c[0].startswith("gemm_skinny_slice")]
    assert sliced(tokens=tokens) == [["gemm_skinny_slice_kernel<%d,%d,2>" % (t, rows), [slices, groups, 1]] for t in (Q4_K, Q6_K)]
    assert sliced(tokens=16) == []                                         # (16 columns: longer walks only)
    assert sliced(tokens=tokens, options={"gemm_splitk": 0}) == []


@pytest.mark.parametrize("case", tiles.STEP_SLICE_FEW_CASES)
def test_down_projections_of_few_decode_steps_in_slices(case):
    (width, ff), tokens, (rows, slices, groups) = case
    cfg = dict(tiles.kquant(width, 2, 1, ff), n_layer=2)
    sliced = lambda **kw: [c for c in call(kquant_products, cfg=cfg, layers=[0, 1], decode=True, **kw) if c[0].startswith("gemm_skinny_slice")]
    assert sliced(tokens=tokens) == [["gemm_skinny_slice_kernel<%d,%d,1>" % (t, rows), [slices, groups, 1]] for t in (Q4_K, Q6_K)]
    assert sliced(tokens=tokens, options={"gemm_splitk": 0}) == []
    # (walks of 22 tiles)
    assert call(kquant_products, cfg=tiles.kquant(width, 2, 1, 22528), layers=[0], decode=True, tokens=tokens)[-1][0].startswith("gemm_skinny_kernel")


@pytest.mark.parametrize("name,layers,tokens", [("llama3-8b", [3], 2048), ("qwen2.5-32b", [7], 1664)])
def test_prefill_of_the_full_sizes(name, layers, tokens):
    """Over the copies the large tile of gemm_f16.hip; without them the 256-row tile, or with gemm_big=0 the 128 x 128 one."""
    cfg = models.CONFIGS[name]
    kernels = [{n.split("<")[0] for n, _ in call(kquant_products, cfg=cfg, layers=layers, tokens=tokens, tuning=t, options=o)}
               for t, o in ((None, None), ({"tile_copies": 0}, None), ({"tile_copies": 0}, {"gemm_big": 0}))]
    assert kernels[0] == {"gemm_f16_kernel"}
    assert "gemm_big_kernel" in kernels[1] and kernels[1] <= {"gemm_big_kernel", "gemm_kq_kernel"}
    assert kernels[2] == {"gemm_kq_kernel"}


def state_launches(host, cfg, lens, products=False):
    m = mesh()
    host.memory(1 << 37)
    with tempfile.TemporaryDirectory() as d:
        st = m.Stage(N.write_folder(d, cfg, U.random_weights(cfg, 3)), 0, -1, n_ctx=512, n_seq_max=len(lens), n_batch_max=2048)
    ses = st.session()
    host.launches()
    ses.decode(np.zeros(sum(lens), np.int32), np.concatenate([np.arange(n) for n in lens]), seq=np.repeat(np.arange(len(lens)), lens), in_fmt=m.TOKENS)
    return [c for c in host.launches() if c[0].startswith(("state_scan", "gated_step") + (("linear_step",) if products else ()))]


@pytest.mark.parametrize("layers", nutavik.STEP_SLICE_LAYERS)
def test_single_steps_of_states_in_slices(layers):
    """Slices of 32 value columns whose heads the output product norms (input kind 7); one workgroup a head where the gates don't lie on 16 bytes."""
    for slot, l in enumerate(layers):
        x = l["mixer"]
        # the gate stands behind q, k and v
        kv = x.get("kv_heads", x["heads"])
        sliced = (2 * kv * x["dim"] + x["heads"] * x["vdim"]) % 4 == 0
        got = call(state_launches, cfg=U.config(50, 72, [l]), lens=[1], products=True)
        (name, grid, _), = [c for c in got if c[0].startswith("gated_step")]
        assert grid == [x["heads"], 1, x["vdim"] // 32 if sliced else 1], (slot, name, grid)
        assert any(n.startswith("linear_step_kernel<") and n.split("<")[1].split(",")[2] == "7" for n, _, _ in got) == sliced, got


PLAIN, PIPED, SHORT = 0, 1, 2                       # state_scan_kernel's third argument


@pytest.mark.parametrize("name,lens", nutavik.SHORT_CALLS + [("wide-states", [33, 8])])
def test_scans_of_states(name, lens):
    """Of every width of states: pipelined up to a workgroup a CU where there is a second chunk; beyond two, four waves for sequences of up to three."""
    cfg = U.CONFIGS[name] if isinstance(name, str) else name
    got = call(state_launches, cfg=cfg, lens=lens)
    assert len(got) == len(cfg["layers"])
    for (name, grid, threads), l in zip(got, cfg["layers"]):
        x = l["mixer"]
        workgroups = [x["heads"], -(-x["vdim"] // 16), len(lens)]
        n = np.prod(workgroups)
        mode = PIPED if n <= 256 and max(lens) > 32 else SHORT if n > 512 and max(lens) <= 96 else PLAIN
        assert name == "state_scan_kernel<%d,%d,%d>" % (l["type"] == "delta", -(-x["dim"] // 64), mode)
        assert grid == workgroups and threads == (256 if mode == SHORT else 384)


# KV heads, cache types, tokens, keys of the longest walk; key splits of the f32 kernel (a workgroup a CU, 64 keys a split at least; two for quantised rows from
# 64 (token, head) pairs on) and of the matrix-core one (a merge only where it pays)
ATTENTION_SPLITS = [
    (2, (1, 1), 1, 100, 2, 1), (2, (1, 1), 1, 384, 6, 1), (2, (1, 1), 1, 385, 7, 7), (8, (1, 1), 16, 1500, 2, 1), (8, (1, 1), 16, 1537, 2, 2),
    (8, (8, 2), 16, 1500, 4, 2), (8, (8, 2), 8, 300, 5, 1), (2, (8, 2), 4, 200, 4, 1),
]


def attention_launches(host, n_kv, kv_types, tokens, keys, matrix_cores, least=1):
    m = mesh()
    host.memory(1 << 37)
    cfg = dict(arch="llama", n_layer=1, n_embd=512, n_head=2 * n_kv, n_head_kv=n_kv, head_dim=64, n_ff=512, n_vocab=256, eps=1e-5, rope=1e4)
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "model.gguf")
        models.write_model(path, cfg, [0], seed=1, fast=True)
        st = m.Stage(path, 0, 1, n_ctx=keys, n_seq_max=tokens, n_batch_max=32, kv_types=kv_types)
    ses = st.session(attn_mma_min_tokens=least)
    host.launches()
    rows = np.zeros((tokens, 2 * n_kv, 64), np.float32)
    ses.attn_dev(0, rows.ctypes.data, [keys - 1] * tokens, rows.ctypes.data, seq=np.arange(tokens), matrix_cores=matrix_cores)
    direct = [(n, g) for n, g, _ in host.launches() if n.startswith("attn_") and "combine" not in n]
    ses.decode(np.zeros((tokens, 512), np.float32), [keys - 1] * tokens, seq=np.arange(tokens))
    return direct + [(n, g) for n, g, _ in host.launches() if n.startswith("attn_") and "combine" not in n]


@pytest.mark.parametrize("case", ATTENTION_SPLITS)
@pytest.mark.parametrize("matrix_cores", [0, 1])
def test_key_splits_go_by_the_kernel_that_is_launched(case, matrix_cores):
    """Of the entry point that names its kernel, whatever the session's switch says, and of the layers, which go by the switch."""
    n_kv, kv_types, tokens, keys, *splits = case
    for least in (1, 1 << 20):
        direct, layer = call(attention_launches, n_kv=n_kv, kv_types=kv_types, tokens=tokens, keys=keys, matrix_cores=matrix_cores, least=least)
        assert direct[0].startswith("attn_mma_kernel" if matrix_cores else "attn_kernel") and direct[1][0] == splits[matrix_cores]
        assert layer[0].startswith("attn_mma_kernel" if least == 1 else "attn_kernel") and layer[1][0] == splits[1 if least == 1 else 0]


def graph_walks(host, folder, tokens, keys):
    """Attention kernel of the launches that the last of each run of three calls made, one run for each length: none where a graph ran."""
    m = mesh()
    host.memory(1 << 37)
    with tempfile.TemporaryDirectory() as d:
        if folder:
            st = m.Stage(N.write_folder(d, c := N.config(64, 256, 512, [N.attention(2, 1, 64, 400, ff=128)]), N.random_weights(c, 3)), 0, -1, n_ctx=512, n_seq_max=tokens, n_batch_max=16)
        else:
            path = os.path.join(d, "model.gguf")
            models.write_model(path, models.CONFIGS["tiny-llama"], [0], seed=1, fast=True)
            st = m.Stage(path, 0, 1, n_ctx=512, n_seq_max=tokens, n_batch_max=16)
    ses = st.session(graphs=1)
    out = []
    for n in keys:
        pos, seq = [n - 1] * tokens, np.arange(tokens)
        first = None
        for _ in range(3):
            host.launches()
            if folder:
                ses.decode(np.zeros(tokens, np.int32), pos, seq=seq, in_fmt=m.TOKENS)
            else:
                ses.decode(np.zeros((tokens, 256), np.float32), pos, seq=seq)
            got = [k for k, _, _ in host.launches() if k.startswith("attn_mma")]
            first = got if first is None else first
        assert got == []
        out.append(first)
    return out


@pytest.mark.parametrize("folder", [False, True])
def test_a_replayed_graph_has_the_kernel_of_the_length(folder):
    """At most 128 keys (one block of 32 for each of four waves) and more of them, both unsplit, are graphs of their own."""
    got = call(graph_walks, folder=folder, tokens=2, keys=[100, 128, 129, 300, 100])
    assert got == [["attn_mma_kernel<64,1,1,0>"], [], ["attn_mma_kernel<64,1,1,1>"], [], []]


def routers(host, n_embd, n_expert, tokens):
    m = mesh()
    host.memory(1 << 37)
    cfg = dict(arch="qwen3moe", n_layer=1, n_embd=n_embd, n_head=4, n_head_kv=2, head_dim=128, n_ff=0, n_vocab=256, eps=1e-6, rope=1e6,
               n_expert=n_expert, n_expert_used=2, n_ff_exp=256, qk_norm=True)
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "model.gguf")
        models.write_model(path, cfg, [0], seed=1, fast=True)
        st = m.Stage(path, 0, 1, n_ctx=2048, n_seq_max=1, n_batch_max=2048)
    ses = st.session()
    out = []
    for T in tokens:
        host.launches()
        ses.decode(np.zeros((T, n_embd), np.float32), np.arange(T))
        out += [(n, g[0]) for n, g, _ in host.launches() if n.startswith("moe_router")]
    return out


@pytest.mark.parametrize("n_embd,n_expert,whole", [(512, 95, False), (512, 96, True), (1024, 95, False), (1024, 512, True), (2048, 512, False)])
def test_router_of_many_short_expert_rows(n_embd, n_expert, whole):
    """Many experts over a small hidden size: a token a workgroup while every token has a CU of its own."""
    v = n_embd // 256
    got = call(routers, n_embd=n_embd, n_expert=n_expert, tokens=[65, 256, 257, 600, 1000])
    small = [["moe_router_fused_kernel<%d,1024>" % v, 65], ["moe_router_fused_kernel<%d,1024>" % v, 256]]
    chunk = [["moe_router_chunk_kernel<%d,2>" % v, 33], ["moe_router_chunk_kernel<%d,2>" % v, 128]]
    assert got[:2] == (small if whole else chunk)
    assert got[2:] == [["moe_router_chunk_kernel<%d,2>" % v, 129], ["moe_router_chunk_kernel<%d,3>" % v, 200], ["moe_router_chunk_kernel<%d,4>" % v, 250]]
