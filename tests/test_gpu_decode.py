"""Paged decode on the GPU vs the float64 oracle (layers/attention.py:71-74).

Every case runs the full decode step -- store_kvcache of the new token, then
paged decode over context_lens tokens -- and the oracle replays the same step
from the cache contents taken before the store.
"""
import numpy as np
import pytest
import torch

from nano_qwen_amd import kernels
from oracle.inputs import make_decode_case
from tests.parity import (TOL_BF16, TOL_FP8, assert_close, decode_reference, f64, full_decode_check,
                          snapshot_decode)

pytestmark = pytest.mark.gpu


def run_step(case):
    kernels.store_kvcache(case["k_new"], case["v_new"], case["k_cache"], case["v_cache"],
                          case["slot_mapping"], case["k_scale"], case["v_scale"])
    out = kernels.paged_decode(case["q"].unsqueeze(1), case["k_cache"], case["v_cache"],
                               case["context_lens"], case["block_tables"], case["scale"],
                               case["k_scale"], case["v_scale"])
    torch.cuda.synchronize()
    return out


def check(case, seq_ids, tol, all_rows=False):
    """The float64 oracle on ``seq_ids`` (end to end from the pre-store
    cache); with ``all_rows`` also every row of the batch against the float32
    device reference."""
    print(f"[decode] {case['name']} B={case['batch']} Hq={case['hq']} Hkv={case['hkv']} "
          f"kv={case['k_cache'].dtype} seqs={list(seq_ids)[:8]}", flush=True)
    snapshot_decode(case, seq_ids)
    out = run_step(case)
    assert out.shape == (case["batch"], 1, case["hq"], case["d"])
    ref = decode_reference(case, seq_ids)
    res = assert_close(f64(out[list(seq_ids), 0]), ref, **tol, what=case["name"])
    if all_rows:
        mx, mn = full_decode_check(case, out, tol)
        print(f"[decode] {case['name']} all {case['batch']} rows: max-abs {mx:.2e} mean-abs {mn:.2e}", flush=True)
    case["_out"] = out
    return res


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_decode_cfg1_shape(cuda, dtype):
    case = make_decode_case("cfg1", seed=0, device=cuda, dtype=dtype)
    check(case, range(case["batch"]), TOL_BF16)


@pytest.mark.parametrize("split", [128, 512, 4096])
@pytest.mark.parametrize("seed", [0, 1])
def test_decode_cfg2_small_splits(cuda, split, seed, monkeypatch):
    monkeypatch.setenv("NQ_DECODE_SPLIT_TOKENS", str(split))
    case = make_decode_case("cfg2", seed=seed, device=cuda, batch=6, ctx=(1, 1300))
    check(case, range(6), TOL_BF16)


@pytest.mark.parametrize("G", [1, 2, 8, 16])
def test_decode_group_sizes(cuda, G):
    case = make_decode_case("cfg2", seed=3, device=cuda, batch=3, ctx=(200, 700), hq=2 * G, hkv=2)
    check(case, range(3), TOL_BF16)


def _with_lengths(case, lens, cuda):
    """The case rebuilt over a fresh pool for the given context lengths, each
    sequence's blocks a random permutation of the pool, table entries past
    the context stale or out of range (never read)."""
    n_seq = len(lens)
    bs = case["block_size"]
    pool = case["num_blocks"]
    need = int(sum((int(c) + bs - 1) // bs for c in lens))
    perm = torch.randperm(max(pool, need + 2), generator=torch.Generator().manual_seed(1))
    case["k_cache"] = torch.randn(len(perm), bs, 8, 128, device=cuda).mul_(0.5).to(torch.bfloat16)
    case["v_cache"] = torch.randn(len(perm), bs, 8, 128, device=cuda).mul_(0.5).to(torch.bfloat16)
    W = int(max((int(c) + bs - 1) // bs for c in lens)) + 2
    bt = torch.full((n_seq, W), -1, dtype=torch.int32)
    off = 0
    for b, c in enumerate(lens.tolist()):
        n = (c + bs - 1) // bs
        bt[b, :n] = perm[off:off + n].to(torch.int32)
        off += n
    bt[:, -1] = 10 ** 6         # stale / out-of-range entries past ctx are never read
    slot = [int(bt[b, (c - 1) // bs]) * bs + (c - 1) % bs for b, c in enumerate(lens.tolist())]
    case.update(block_tables=bt.to(cuda), context_lens=lens.to(cuda),
                slot_mapping=torch.tensor(slot, dtype=torch.int32, device=cuda), num_blocks=len(perm))
    return case


def test_decode_edge_lengths(cuda):
    # lengths at and around block / step / split boundaries, plus ctx = 1
    case = make_decode_case("cfg2", seed=4, device=cuda, batch=10, ctx=(1, 1))
    lens = torch.tensor([1, 2, 31, 32, 33, 255, 256, 257, 512, 513], dtype=torch.int32)
    check(_with_lengths(case, lens, cuda), range(10), TOL_BF16)


def test_decode_many_splits_merge(cuda, monkeypatch):
    """128-token splits: rows of 1, 16, 17, 32, 33 and 40 splits, so the
    merge takes its splits in one, two and three chunks of 16, and short rows
    in the same launch have every later split empty."""
    monkeypatch.setenv("NQ_DECODE_SPLIT_TOKENS", "128")
    case = make_decode_case("cfg2", seed=8, device=cuda, batch=8, ctx=(1, 1))
    lens = torch.tensor([1, 100, 2048, 2049, 4096, 4097, 5000, 300], dtype=torch.int32)
    check(_with_lengths(case, lens, cuda), range(8), TOL_BF16)


@pytest.mark.parametrize("d", [128, 256])
@pytest.mark.parametrize("streamk", ["0", "1"])
def test_decode_merge_groups(cuda, d, streamk, monkeypatch):
    """Few sequences with hundreds of pieces per head: the merge's 8 thread
    groups take 8 pieces each per round (64 in all), so rows of 1, 2, 8, 9,
    64, 65 and 71 splits (stream-K at head_dim 256: 32-token ranges) end
    inside, at and past a group's chunk and the round."""
    monkeypatch.setenv("NQ_DECODE_SPLIT_TOKENS", "128")
    monkeypatch.setenv("NQ_DECODE_STREAMK", streamk)
    case = make_decode_case("cfg2", seed=21, device=cuda, batch=8, ctx=(1, 1), hq=4096 // d, hkv=1024 // d, d=d)
    lens = torch.tensor([0, 128, 129, 1024, 1025, 8192, 8193, 9000], dtype=torch.int32)
    case = _with_lengths(case, lens, cuda)
    for name in ("k_cache", "v_cache"):
        case[name] = case[name].view(-1, 256, 1024 // d, d)
    case["slot_mapping"][0] = -1
    check(case, range(1, 8), TOL_BF16)
    assert torch.all(case["_out"][0] == 0)


def test_decode_ctx1_returns_new_value(cuda):
    case = make_decode_case("cfg2", seed=5, device=cuda, batch=4, ctx=(1, 1))
    out = run_step(case)
    G = case["hq"] // case["hkv"]
    want = case["v_new"].repeat_interleave(G, dim=1)
    assert torch.equal(out[:, 0], want), "softmax over a single key must return that value exactly"


def test_decode_zero_context_rows(cuda):
    case = make_decode_case("cfg2", seed=6, device=cuda, batch=5, ctx=(300, 900))
    ctx = case["context_lens"].clone()
    ctx[1] = 0
    ctx[3] = 0
    case["context_lens"] = ctx
    slot = case["slot_mapping"].clone()
    slot[1] = -1
    slot[3] = -1
    case["slot_mapping"] = slot
    snapshot_decode(case, [0, 2, 4])
    out = run_step(case)
    assert torch.all(out[1] == 0) and torch.all(out[3] == 0)
    ref = decode_reference(case, [0, 2, 4])
    assert_close(f64(out[[0, 2, 4], 0]), ref, **TOL_BF16, what="zero-ctx batch")


def test_decode_block_permutation_bit_identical(cuda):
    case = make_decode_case("cfg2", seed=7, device=cuda, batch=4, ctx=(500, 1500))
    out1 = run_step(case)
    nb = case["k_cache"].shape[0]
    perm = torch.randperm(nb, generator=torch.Generator().manual_seed(3)).to(cuda)
    inv = torch.argsort(perm)
    k2, v2 = case["k_cache"][perm].contiguous(), case["v_cache"][perm].contiguous()
    bt = case["block_tables"].long()
    bt2 = torch.where(bt >= 0, inv[bt.clamp(min=0)], -1).to(torch.int32)
    out2 = kernels.paged_decode(case["q"].unsqueeze(1), k2, v2, case["context_lens"], bt2, case["scale"])
    torch.cuda.synchronize()
    assert torch.equal(out1, out2)


def test_decode_hip_graph_replay(cuda):
    """Capture store + decode once, replay with new metadata in the static
    buffers, as the reference's graph decode does (engine/model_runner.py:319-336)."""
    mk = lambda seed: make_decode_case("cfg2", seed=seed, device=cuda, batch=8, ctx=(100, 2000), min_pool=200)
    case = mk(8)
    W = 11                                   # static table width > any ceil(2000/256)
    static_bt = torch.zeros(8, W, dtype=torch.int32, device=cuda)
    static_ctx = torch.zeros(8, dtype=torch.int32, device=cuda)
    static_slot = torch.full((8,), -1, dtype=torch.int32, device=cuda)
    static_q = torch.zeros_like(case["q"])
    static_k = torch.zeros_like(case["k_new"])
    static_v = torch.zeros_like(case["v_new"])
    out = torch.zeros(8, 1, case["hq"], 128, dtype=case["q"].dtype, device=cuda)

    def step():
        kernels.store_kvcache(static_k, static_v, case["k_cache"], case["v_cache"], static_slot)
        kernels.paged_decode(static_q.unsqueeze(1), case["k_cache"], case["v_cache"], static_ctx,
                             static_bt, case["scale"], out=out)

    step()  # warm-up: the split-K workspace is allocated outside the capture
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        step()
    for rep, seed in enumerate([8, 9, 10, 11]):
        c = mk(seed)
        assert c["num_blocks"] == case["num_blocks"]
        c["k_cache"], c["v_cache"] = case["k_cache"], case["v_cache"]   # one persistent pool
        snapshot_decode(c, list(range(8)))
        static_bt.fill_(-1)
        static_bt[:, :c["block_tables"].shape[1]] = c["block_tables"]
        static_ctx.copy_(c["context_lens"])
        static_slot.copy_(c["slot_mapping"])
        static_q.copy_(c["q"])
        static_k.copy_(c["k_new"])
        static_v.copy_(c["v_new"])
        g.replay()
        torch.cuda.synchronize()
        ref = decode_reference(c, list(range(8)))
        assert_close(f64(out[:, 0]), ref, **TOL_BF16, what=f"graph replay {rep}")
        # an eager decode of the same state agrees bit for bit
        eager = kernels.paged_decode(static_q.unsqueeze(1), case["k_cache"], case["v_cache"], static_ctx,
                                     static_bt, case["scale"])
        torch.cuda.synchronize()
        assert torch.equal(eager, out)


@pytest.mark.slow
def test_decode_cfg2_full(cuda):
    case = make_decode_case("cfg2", seed=0, device=cuda)
    seqs = np.random.default_rng(0).choice(case["batch"], 12, replace=False).tolist()
    check(case, seqs, TOL_BF16, all_rows=True)


@pytest.mark.slow
def test_decode_cfg4_full_split_k(cuda):
    case = make_decode_case("cfg4", seed=0, device=cuda)
    check(case, [0, 5], TOL_BF16, all_rows=True)


@pytest.mark.slow
def test_decode_cfg5_full_fp8(cuda):
    """Every row of cfg5 against the float32 reference over the fp8 codes
    dequantized in float32, and against the reference the configuration
    names: attention computed in float32 over K/V dequantized to bf16."""
    from oracle import sdpa_path
    case = make_decode_case("cfg5", seed=0, device=cuda)
    seqs = np.random.default_rng(1).choice(case["batch"], 10, replace=False).tolist()
    check(case, seqs, TOL_FP8, all_rows=True)
    out = case["_out"].squeeze(1).float()
    # the cache now holds the stored new tokens: dequantize code x scale to
    # bf16, then attention in float32 over the bf16 pools
    kb = (case["k_cache"].float() * case["k_scale"].view(1, 1, -1, 1)).to(torch.bfloat16)
    vb = (case["v_cache"].float() * case["v_scale"].view(1, 1, -1, 1)).to(torch.bfloat16)
    ref = sdpa_path.paged_decode(case["q"], kb, vb, case["block_tables"], case["context_lens"].cpu(), case["scale"])
    err = (out - ref).abs()
    mx, mn = float(err.max()), float(err.mean())
    print(f"[decode] cfg5 all {case['batch']} rows vs bf16-dequantized: max-abs {mx:.2e} mean-abs {mn:.2e}",
          flush=True)
    assert mx <= TOL_FP8["max_abs"] and mn <= TOL_FP8["mean_abs"], (mx, mn)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_decode_fp8_small(cuda, dtype):
    case = make_decode_case("cfg5", seed=2, device=cuda, batch=6, ctx=(1, 1500), dtype=dtype)
    check(case, range(6), TOL_FP8)


def test_decode_fp8_vs_bf16_dequantized_reference(cuda):
    """The target's stated fp8 reference: attention in fp32 over K/V
    dequantized to bf16 (code value * scale, rounded to bf16)."""
    from oracle import paged as P
    from tests.parity import subpool
    case = make_decode_case("cfg5", seed=3, device=cuda, batch=4, ctx=(600, 2000))
    out = run_step(case)
    k = (case["k_cache"].float() * case["k_scale"].view(1, 1, -1, 1)).to(torch.bfloat16)
    v = (case["v_cache"].float() * case["v_scale"].view(1, 1, -1, 1)).to(torch.bfloat16)
    ids = list(range(4))
    ks, vs, table, _ = subpool(k, v, case["block_tables"], case["context_lens"].cpu(), ids)
    ref = P.paged_decode(f64(case["q"]).astype(np.float32), f64(ks).astype(np.float32),
                         f64(vs).astype(np.float32), table, case["context_lens"].cpu().numpy(), case["scale"])
    assert_close(f64(out[ids, 0]), ref, **TOL_FP8, what="fp8 vs bf16-dequantized fp32 reference")


@pytest.mark.parametrize("kv", ["same", "fp8"])
@pytest.mark.parametrize("split", [0, 512])
def test_decode_head_dim_256(cuda, kv, split, monkeypatch):
    """head_dim 256, the reference model's own full-attention layers
    (models/qwen3_5.py:69-72 with the transformers default), one- and
    multi-split plans, 16-bit and fp8 caches."""
    if split:
        monkeypatch.setenv("NQ_DECODE_SPLIT_TOKENS", str(split))
    name = "cfg5" if kv == "fp8" else "cfg2"
    case = make_decode_case(name, seed=7 + split, device=cuda, batch=6, ctx=(1, 1500), d=256, hq=16, hkv=2)
    check(case, range(6), TOL_FP8 if kv == "fp8" else TOL_BF16)


def test_decode_head_dim_256_f16_groups(cuda):
    case = make_decode_case("cfg2", seed=9, device=cuda, batch=4, ctx=(300, 900), d=256, hq=8, hkv=8,
                            dtype=torch.float16)
    check(case, range(4), TOL_BF16)


def test_decode_graph_survives_workspace_growth(cuda):
    """A graph captured with a small split-K workspace keeps replaying
    correctly after an eager decode on the same stream has grown that
    stream's workspace with a bigger plan (the old buffer stays alive), and
    its replays match the eager result bit for bit."""
    mk = lambda seed: make_decode_case("cfg2", seed=seed, device=cuda, batch=4, ctx=(700, 2000), min_pool=80)
    case = mk(12)
    W = 8
    static_bt = torch.full((4, W), -1, dtype=torch.int32, device=cuda)
    static_bt[:, :case["block_tables"].shape[1]] = case["block_tables"]
    static_ctx = case["context_lens"].clone()
    out = torch.zeros(4, 1, case["hq"], 128, dtype=case["q"].dtype, device=cuda)
    step = lambda: kernels.paged_decode(case["q"].unsqueeze(1), case["k_cache"], case["v_cache"], static_ctx,
                                        static_bt, case["scale"], out=out)
    assert kernels.decode_plan(4, case["hq"], case["hkv"], W, 256, case["k_cache"].dtype)[0] > 1
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        step()                                   # allocates this stream's workspace
        side.synchronize()
        key = kernels._key(cuda)
        captured_ws = kernels._workspaces[key].data_ptr()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=side):   # the capture reuses that workspace
            step()
        assert kernels._workspaces[key].data_ptr() == captured_ws
        eager = step().clone()
        side.synchronize()
        # an eager decode on the same stream with a plan that needs far more
        # workspace: the shim replaces the buffer and keeps the old one alive
        big = make_decode_case("cfg4", seed=13, device=cuda, batch=8, ctx=(30000, 32768))
        kernels.paged_decode(big["q"].unsqueeze(1), big["k_cache"], big["v_cache"], big["context_lens"],
                             big["block_tables"], big["scale"])
        side.synchronize()
        assert kernels._workspaces[key].data_ptr() != captured_ws, "the big plan must have grown the workspace"
        assert any(t.data_ptr() == captured_ws for t in kernels._retired)
        del big
        torch.cuda.empty_cache()
        junk = torch.full((1 << 26,), 7, dtype=torch.int32, device=cuda)   # reuse of freed memory would show
        for rep in range(3):
            out.zero_()
            g.replay()
            side.synchronize()
            assert torch.equal(out, eager), f"replay {rep} after the workspace grew"
        del junk
    torch.cuda.synchronize()
    snapshot_decode(case, list(range(4)))
    ref = decode_reference(dict(case, slot_mapping=torch.full((4,), -1, dtype=torch.int32, device=cuda)),
                           list(range(4)))
    assert_close(f64(out[:, 0]), ref, **TOL_BF16, what="replay after growth vs oracle")


def test_release_workspaces_then_decode_again(cuda):
    """Dropping the per-stream buffers (no graph holds them here) leaves the
    next decode to allocate a fresh workspace, with the same result."""
    case = make_decode_case("cfg4", seed=1, device=cuda, batch=2, ctx=(5000, 9000))
    out1 = run_step(case)
    assert kernels.release_workspaces(cuda) >= 1
    out2 = kernels.paged_decode(case["q"].unsqueeze(1), case["k_cache"], case["v_cache"], case["context_lens"],
                                case["block_tables"], case["scale"])
    torch.cuda.synchronize()
    assert torch.equal(out1, out2)
