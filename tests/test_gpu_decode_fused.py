"""The one-launch decode of small batches (paged_decode_fused_kernel): four
waves share a split's steps, and the last workgroup of a (sequence, kv head)
merges its splits.

Every row against the float32 device reference (oracle/sdpa_path) and a few
against the float64 oracle; the counters are zero again after every launch.
"""
import ctypes

import pytest
import torch

from nano_qwen_amd import kernels
from oracle.inputs import make_decode_case
from tests.parity import TOL_BF16, TOL_FP8, assert_close, decode_reference, f64, full_decode_check, snapshot_decode

pytestmark = pytest.mark.gpu


def _fused(case):
    config = (ctypes.c_int64 * 4)()
    kernels.check(kernels.lib().nq_decode_config(
        case["batch"], case["hq"], case["hkv"], case["d"], case["block_tables"].shape[1], case["block_size"],
        kernels.dtype_code(case["k_cache"].dtype), config), "config")
    return config[0] > 0


def _step(case, gate=None):
    out = kernels.paged_decode(case["q"].unsqueeze(1), case["k_cache"], case["v_cache"], case["context_lens"],
                               case["block_tables"], case["scale"], case["k_scale"], case["v_scale"], gate=gate,
                               k=case["k_new"], v=case["v_new"], slot_mapping=case["slot_mapping"])
    torch.cuda.synchronize()
    assert kernels._key(case["q"].device) in kernels._decode_counters    # without a slot: two launches
    for pool in kernels._counter_pools.values():
        assert int(pool.count_nonzero()) == 0
    return out


def _set_lengths(case, lens):
    """Shorter contexts within the case's tables (the first row is a padded one)."""
    bs = case["block_size"]
    for b, n in enumerate(lens):
        assert n <= int((case["block_tables"][b] >= 0).sum()) * bs
        case["context_lens"][b] = n
        case["slot_mapping"][b] = -1 if n == 0 else int(case["block_tables"][b, (n - 1) // bs]) * bs + (n - 1) % bs


@pytest.mark.parametrize("kw", [
    dict(hq=32, hkv=8), dict(hq=8, hkv=2), dict(hq=4, hkv=4), dict(hq=16, hkv=1), dict(hq=24, hkv=2),
    dict(hq=32, hkv=8, dtype=torch.float16), dict(hq=32, hkv=8, kv="fp8"), dict(hq=3, hkv=1, kv="fp8"),
    dict(hq=16, hkv=4, d=256), dict(hq=16, hkv=1, d=256), dict(hq=16, hkv=2, d=256, kv="fp8"),
], ids=str)
@pytest.mark.parametrize("longest", [40, 500, 3000])
def test_fused_decode(cuda, kw, longest):
    """Rows that end inside, at and past a step, a wave's turn, a split and the
    table, down to 0 and 1 tokens, with the new token's store; with the gate
    the output is torch's gate of the ungated one."""
    lens = {40: [0, 1, 32, 33], 500: [0, 31, 127, 129, 256, 500], 3000: [0, 513, 1025, 3000]}[longest]
    if kw.get("d", 128) == 128 and kw.get("kv") != "fp8":    # what 16-bit rows take in one launch
        longest = min(longest, 16384 // kw["hkv"] - 100)
        lens = [longest] if longest > 500 else lens
    case = make_decode_case("cfg2", seed=len(lens), device=cuda, batch=len(lens), ctx=(longest, longest), **kw)
    if len(lens) > 1:
        _set_lengths(case, lens)
    assert _fused(case)
    tol = TOL_FP8 if kw.get("kv") == "fp8" else TOL_BF16
    rows = [r for r in range(len(lens)) if int(case["context_lens"][r]) > 0]
    snapshot_decode(case, rows)
    out = _step(case)
    full_decode_check(case, out, tol)
    assert_close(f64(out[rows, 0]), decode_reference(case, rows), **tol, what="fused decode")
    assert torch.equal(_step(case), out)
    gate = torch.randn(out.shape, generator=torch.Generator(device=cuda).manual_seed(1), device=cuda).to(out.dtype)
    got, want = _step(case, gate), out * torch.sigmoid(gate)
    off = (got.view(torch.int16).int() - want.view(torch.int16).int()).abs()
    assert int(off.max()) <= 1 and float((off > 0).float().mean()) <= 2e-3


def test_fused_decode_first_call_in_a_capture(cuda):
    """A stream whose first decode is a captured one takes a zeroed slot (or the
    two-launch path); replays on new lengths equal the eager result."""
    case = make_decode_case("cfg2", seed=3, device=cuda, batch=2, ctx=(700, 700), hq=8, hkv=2)
    assert _fused(case)
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    q = case["q"].unsqueeze(1)
    args = (q, case["k_cache"], case["v_cache"], case["context_lens"], case["block_tables"], case["scale"])
    kernels.paged_decode(*args)    # loads the kernels
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        out = kernels.paged_decode(*args)
    for lens in ([700, 1], [129, 512], [33, 699]):
        case["context_lens"].copy_(torch.tensor(lens, dtype=torch.int32))
        want = kernels.paged_decode(*args)
        for _ in range(3):
            out.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, want)


def test_fused_decode_streams_have_their_own_counters(cuda):
    case = make_decode_case("cfg2", seed=4, device=cuda, batch=2, ctx=(700, 700), hq=8, hkv=2)
    args = (case["q"].unsqueeze(1), case["k_cache"], case["v_cache"], case["context_lens"], case["block_tables"],
            case["scale"])
    want = kernels.paged_decode(*args)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    outs = []
    for _ in range(20):
        for s in streams:
            with torch.cuda.stream(s):
                outs.append(kernels.paged_decode(*args))
    torch.cuda.synchronize()
    assert all(torch.equal(o, want) for o in outs)
    slots = [kernels._decode_counters[(0, s.cuda_stream)].data_ptr() for s in streams]
    assert slots[0] != slots[1]


def _capture_two(device):
    """Two graphs on torch's own capture stream, as two runners capture, of
    three decodes each: (arguments, graphs, outputs, eager results)."""
    cases = [make_decode_case("cfg2", seed=s, device=device, batch=2, ctx=(700, 700), hq=8, hkv=2) for s in (5, 6)]
    assert all(map(_fused, cases))
    args = [(c["q"].unsqueeze(1), c["k_cache"], c["v_cache"], c["context_lens"], c["block_tables"], c["scale"])
            for c in cases]
    want = [kernels.paged_decode(*a) for a in args]
    torch.cuda.synchronize()
    graphs, outs, slots = [], [], []
    for a in args:
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            outs.append([kernels.paged_decode(*a) for _ in range(3)])
            slots.append(kernels._capture_counters[kernels._key(device)][1])
        graphs.append(graph)
    return args, graphs, outs, want, slots


def _replay(graph, got, want):
    for o in got:
        o.zero_()
    graph.replay()
    torch.cuda.synchronize()
    assert all(torch.equal(o, want) for o in got)


def test_fused_decode_captures_have_their_own_counters(cuda):
    """Spoiled counters of anything else -- every slot of the pool but the graph's
    own, as overlapping replays leave them -- do not reach a graph's replays."""
    args, graphs, outs, want, slots = _capture_two(cuda)
    pool = kernels._counter_pools[0]
    eager = kernels._decode_counters[kernels._key(cuda)]
    assert len({t.data_ptr() for t in (*slots, eager)}) == 3
    for _ in range(3):
        for graph, got, w, slot in zip(graphs, outs, want, slots):
            pool.fill_(7)
            slot.zero_()
            _replay(graph, got, w)
            assert not slot.any()
    pool.zero_()
    for _ in range(3):
        for graph, got, w in zip(graphs, outs, want):
            _replay(graph, got, w)
            assert torch.equal(kernels.paged_decode(*args[0]), want[0])
    assert not pool.any()


def test_fused_decode_counters_of_a_larger_decode(cuda):
    """A capture whose second decode is larger takes counters for it, too."""
    small, large = (make_decode_case("cfg2", seed=s, device=cuda, batch=b, ctx=(400, 400), hq=8, hkv=2)
                    for s, b in ((7, 1), (8, 200)))
    args = [(c["q"].unsqueeze(1), c["k_cache"], c["v_cache"], c["context_lens"], c["block_tables"], c["scale"])
            for c in (small, large)]
    assert _fused(small) and _fused(large)
    want = [kernels.paged_decode(*a) for a in args]
    graph = torch.cuda.CUDAGraph()
    key = []
    with torch.cuda.graph(graph):
        outs = []
        for i in (0, 1, 0):
            outs.append(kernels.paged_decode(*args[i]))
            key.append(kernels._capture_counters[kernels._key(cuda)][1])
    assert key[0].numel() * 4 == 4096 and key[1].numel() * 4 == 28 << 10 and key[2] is key[1]
    for _ in range(3):
        for o in outs:
            o.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(o, want[i]) for o, i in zip(outs, (0, 1, 0)))
    assert not kernels._counter_pools[0].any()


def test_fused_decode_spoiled_counters_do_not_last(cuda, monkeypatch):
    """Captures that find no room in the pool share a slot: what an overlap leaves in it (here
    in every slot but the eager stream's) ends with the next replay."""
    kernels.release_workspaces()
    with torch.inference_mode():    # a pool made there is used outside, too
        kernels._take_counter_slot(kernels._key(cuda), 0, 4096, False)
    monkeypatch.setitem(kernels._counter_bytes_taken, (0, 1), kernels._COUNTER_HALF_BYTES)
    args, graphs, outs, want, slots = _capture_two(cuda)
    assert slots[0].data_ptr() == slots[1].data_ptr()
    pool = kernels._counter_pools[0]
    eager = kernels._decode_counters[kernels._key(cuda)]
    for _ in range(3):
        for graph, got, w in zip(graphs, outs, want):
            with torch.inference_mode():
                pool.fill_(7)
                eager.zero_()
            _replay(graph, got, w)
            assert torch.equal(kernels.paged_decode(*args[0]), want[0])
    kernels.release_workspaces()
    torch.cuda.synchronize()


def test_released_counters_outlive_their_streams_work(cuda):
    """The pool is made on one stream and used on others: released while another
    stream's decode is still to run, its memory is not handed out before that."""
    case = make_decode_case("cfg2", seed=9, device=cuda, batch=2, ctx=(700, 700), hq=8, hkv=2)
    args = (case["q"].unsqueeze(1), case["k_cache"], case["v_cache"], case["context_lens"], case["block_tables"],
            case["scale"])
    want = kernels.paged_decode(*args)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        kernels.paged_decode(*args)
        torch.cuda.synchronize()
        pool = kernels._counter_pools[0]
        where, shape = pool.data_ptr(), pool.shape
        torch.cuda._sleep(1_000_000_000)
        out = kernels.paged_decode(*args)
    del pool
    kernels.release_workspaces()
    taken = [torch.full(shape, 3, dtype=torch.int32, device=cuda) for _ in range(100)]
    assert not side.query()    # still to run
    assert all(t.data_ptr() != where for t in taken)
    torch.cuda.synchronize()
    assert torch.equal(out, want)
