"""C entry points that a caller may use in place of the ones the shim calls:
the same results, and their own argument checks."""
import pytest
import torch

from nano_qwen_amd import kernels
from nano_qwen_amd.kernels import check, dtype_code, lib, ptr, stream_of
from oracle.inputs import make_decode_case, make_prefill_case

pytestmark = pytest.mark.gpu


def _decode_args(c, out, ns, st, ws):
    q = c["q"]
    return (ptr(q), q.stride(0), q.stride(1), ptr(c["k_cache"]), ptr(c["v_cache"]), ptr(c["block_tables"]),
            c["block_tables"].stride(0), c["block_tables"].shape[1], ptr(c["context_lens"])), (
            ptr(out), out.stride(0), out.stride(1), c["batch"], c["hq"], c["hkv"], c["d"], c["block_size"],
            c["num_blocks"], c["scale"], ns, st, ptr(ws), ws.numel(), dtype_code(q.dtype),
            dtype_code(c["k_cache"].dtype), None, None)


def test_decode_entries(cuda):
    """nq_paged_decode_fused with a caller's plan and counters, and
    nq_paged_decode_gated, against the shim."""
    c = make_decode_case("cfg2", seed=1, device=cuda, batch=3, ctx=(200, 700), hq=8, hkv=2)
    gate = torch.randn_like(c["q"])
    shim = lambda **kw: kernels.paged_decode(c["q"].unsqueeze(1), c["k_cache"], c["v_cache"], c["context_lens"],
                                             c["block_tables"], c["scale"], **kw)[:, 0]
    want, gated = shim(), shim(gate=gate)
    ws = torch.empty(1 << 22, dtype=torch.uint8, device=cuda)
    counters = torch.zeros(3 * 2 * 64 + 64, dtype=torch.uint8, device=cuda)
    out = torch.empty_like(c["q"])
    for st in (128, 256):
        ns = -(-c["block_tables"].shape[1] * c["block_size"] // st)
        head, tail = _decode_args(c, out, ns, st, ws)

        def fused(g, cnt, nbytes):
            gs = (None, 0, 0) if g is None else (ptr(g), g.stride(0), g.stride(1))
            return lib().nq_paged_decode_fused(*head, None, 0, None, 0, None, -1, *tail, *gs, cnt, nbytes,
                                               stream_of(out))
        check(fused(None, ptr(counters), 3 * 2 * 64), "fused")
        assert float((out.float() - want.float()).abs().max()) <= 2e-2
        if st == 128:
            assert torch.equal(out, want)    # the shim's own plan
        check(fused(gate, ptr(counters), 3 * 2 * 64), "fused, gated")
        assert float((out.float() - gated.float()).abs().max()) <= 2e-2
        assert not counters.any()
        assert fused(None, ptr(counters), 3 * 2 * 64 - 1) == -1
        assert fused(None, ptr(counters) + 4, 3 * 2 * 64) == -1
        assert fused(None, None, 3 * 2 * 64) == -1
        check(lib().nq_paged_decode_gated(*head, *tail, ptr(gate), gate.stride(0), gate.stride(1), stream_of(out)),
              "gated")
        assert float((out.float() - gated.float()).abs().max()) <= 2e-2


def test_prefill_gated_entry(cuda):
    """nq_varlen_prefill_gated runs whole items: the shim's result for a batch
    that runs so, bit for bit."""
    c = make_prefill_case("cfg3", seed=2, device=cuda, nseq=3, lq=(20, 300), prefix_blocks=(0, 0))
    q, k, v = c["q"], c["k_new"], c["v_new"]
    assert lib().nq_prefill_split_workspace_bytes(3, q.shape[0], c["max_seqlen_q"], c["max_seqlen_k"], c["hq"],
                                                  c["hkv"], c["d"]) == 0
    gate = torch.randn_like(q)
    want = kernels.varlen_prefill(q, k, v, c["cu_seqlens_q"], c["cu_seqlens_k"], c["max_seqlen_q"],
                                  c["max_seqlen_k"], c["scale"], gate=gate)
    out, ws = torch.empty_like(q), kernels.prefill_workspace(cuda)
    check(lib().nq_varlen_prefill_gated(
        ptr(q), q.stride(0), q.stride(1), ptr(k), ptr(v), k.stride(0), ptr(c["cu_seqlens_q"]), ptr(c["cu_seqlens_k"]),
        c["max_seqlen_q"], c["max_seqlen_k"], None, 0, 0, 0, ptr(out), out.stride(0), out.stride(1), 3, c["hq"],
        c["hkv"], c["d"], 0, c["scale"], 1, dtype_code(q.dtype), dtype_code(k.dtype), None, None, ptr(ws),
        ws.numel() * 4, ptr(gate), gate.stride(0), gate.stride(1), q.shape[0], stream_of(q)), "gated")
    assert torch.equal(out, want)
