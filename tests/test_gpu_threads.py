"""Host threads that share a stream: calls of several launches over the stream's
buffers (prefill ranges and their merge, GDN segments, split-K decode) give
what they give one after another."""
import threading

import pytest
import torch

from nano_qwen_amd import kernels
from oracle.inputs import make_decode_case, make_prefill_case
from tests.test_prefill_ranges import would_cut

pytestmark = pytest.mark.gpu


def _prefill(device, i):
    c = make_prefill_case("cfg3", seed=i, device=device, nseq=2, lq=(90, 300), prefix_blocks=(3, 8))
    assert would_cut(2, c["q"].shape[0], c["max_seqlen_q"], c["max_seqlen_k"], c["hq"], c["hkv"], c["d"],
                     c["k_cache"].dtype)
    kernels.store_kvcache(c["k_new"], c["v_new"], c["k_cache"], c["v_cache"], c["slot_mapping"])
    return lambda: kernels.varlen_prefill(c["q"], c["k_cache"], c["v_cache"], c["cu_seqlens_q"], c["cu_seqlens_k"],
                                          c["max_seqlen_q"], c["max_seqlen_k"], c["scale"],
                                          block_table=c["block_tables"])


def _gdn(device, i):
    g = torch.Generator(device=device).manual_seed(i)
    n = 900 + 200 * i
    rand = lambda *s: torch.randn(*s, generator=g, device=device)
    x = [rand(n, 4, 128).bfloat16() for _ in range(3)]
    a, b = rand(n, 4).bfloat16(), rand(n, 4).bfloat16()
    A_log, dt = rand(4), rand(4)
    cu = torch.tensor([0, n], dtype=torch.int32, device=device)
    idx = torch.zeros(1, dtype=torch.int32, device=device)
    assert kernels.lib().nq_gdn_prefill_workspace_bytes(1, n, 4) > 0

    def call():
        state = torch.zeros(1, 4, 128, 128, device=device)
        out = kernels.gdn_prefill(*x, a, b, A_log, dt, cu, state, idx)
        return torch.cat([out.float().flatten(), state.flatten()])
    return call


def _decode(device, i):
    c = make_decode_case("cfg2", seed=i, device=device, batch=2 + i, ctx=(3000, 5000), hq=32, hkv=8)
    plan = kernels.decode_plan(2 + i, 32, 8, c["block_tables"].shape[1], c["block_size"], c["k_cache"].dtype)
    assert plan[0] > 1
    return lambda: kernels.paged_decode(c["q"].unsqueeze(1), c["k_cache"], c["v_cache"], c["context_lens"],
                                        c["block_tables"], c["scale"])


@pytest.mark.parametrize("make", [_prefill, _gdn, _decode])
def test_threads_on_one_stream(cuda, make):
    calls = [make(cuda, i) for i in range(4)]
    want = [call() for call in calls]
    torch.cuda.synchronize()
    start, fails = threading.Barrier(4), []

    def body(i):
        start.wait()
        outs = [calls[i]() for _ in range(25)]
        torch.cuda.synchronize()
        if not all(torch.equal(o, want[i]) for o in outs):
            fails.append(i)
    threads = [threading.Thread(target=body, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not fails
