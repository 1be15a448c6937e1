"""Prefill work distribution on the GPU: kv-head slots shared by several XCDs,
and launches cut into equal key ranges whose partial outputs are merged.

Every output row against the float32 device reference (oracle/sdpa_path), a
few rows against the float64 oracle.
"""
import pytest
import torch

from nano_qwen_amd import kernels
from oracle.inputs import make_prefill_case
from tests.parity import TOL_BF16, TOL_FP8, assert_close, f64
from tests.test_gpu_prefill import check, run_step
from tests.test_prefill_ranges import would_cut

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("hq,hkv,d", [(4, 1, 128), (16, 1, 128), (8, 2, 128), (16, 4, 128), (4, 4, 128), (16, 4, 256),
                                      (4, 2, 256), (4, 1, 256)])
def test_prefill_shared_slots(cuda, hq, hkv, d):
    """1, 2 or 4 kv-head slots: 8, 4 or 2 XCDs take a slot's query tiles in
    turn, so lengths of one row, of fewer tiles than XCDs, of whole and of
    one-over tile counts leave some of them with none, one and several."""
    for prefix in ((0, 0), (1, 2)):
        case = make_prefill_case("cfg3", seed=hq + hkv, device=cuda, nseq=7, lq=(1, 700), prefix_blocks=prefix, hq=hq,
                                 hkv=hkv, d=d)
        check(case, range(7), TOL_BF16, rows_per_seq=6, all_rows=True)


@pytest.mark.parametrize("hkv,d", [(4, 128), (2, 128), (1, 128), (4, 256), (2, 256)])
@pytest.mark.parametrize("lq", [1, 32, 33, 64, 257])
def test_prefill_whole_groups(cuda, hkv, d, lq):
    """8 groups or more of equal lengths, or of less than two query tiles per
    XCD of a slot, stay whole: one tile, one over, and more tiles than that.  A
    batch that shares its slots (one sequence shorter) gives the same bits for
    the sequences they have in common."""
    case = make_prefill_case("cfg3", seed=lq, device=cuda, nseq=8, lq=(lq, lq), prefix_blocks=(0, 0), hq=4 * hkv,
                             hkv=hkv, d=d)
    check(case, range(8), TOL_BF16, rows_per_seq=6, all_rows=True)
    out = run_step(case)
    n = 7 * lq
    cu = case["cu_seqlens_q"].clone()
    cu[8] = n + (lq + 1) // 2
    q, k, v = (case[x][:int(cu[8])] for x in ("q", "k_new", "v_new"))
    other = kernels.varlen_prefill(q, k, v, cu, cu, lq, lq, case["scale"])
    assert torch.equal(other[:n], out[:n])


@pytest.mark.parametrize("hkv,d", [(4, 128), (2, 128), (4, 256)])
@pytest.mark.parametrize("kv", ["same", "fp8"])
def test_prefill_ranges_whole_groups(cuda, hkv, d, kv):
    """Ranges over 8 groups or more of one query tile each, behind prefixes of different lengths."""
    case = make_prefill_case("cfg3", seed=9, device=cuda, nseq=8, lq=(1, 20), prefix_blocks=(2, 9), hq=4 * hkv, hkv=hkv,
                             d=d, kv=kv)
    assert _ranges(case)
    check(case, range(8), TOL_FP8 if kv == "fp8" else TOL_BF16, rows_per_seq=8, all_rows=True)


def _ranges(case):
    """Whether the library cuts the case's launch (as tests/test_prefill_ranges.py asks it)."""
    kv = case["k_cache"].dtype if case["block_tables"] is not None else case["k_new"].dtype
    return would_cut(case["nseq"], case["q"].shape[0], case["max_seqlen_q"], case["max_seqlen_k"], case["hq"],
                     case["hkv"], case["d"], kv)


@pytest.mark.parametrize("kw", [
    dict(nseq=1, lq=(1111, 1111), prefix_blocks=(0, 0)),                 # packed, cuts at any tile
    dict(nseq=3, lq=(1, 900), prefix_blocks=(0, 0), hq=8, hkv=2),        # packed, shared slots
    dict(nseq=1, lq=(1, 1), prefix_blocks=(31, 31)),                     # one row, one item per kv head
    dict(nseq=4, lq=(20, 300), prefix_blocks=(9, 20)),                   # paged, half without a prefix
    dict(nseq=4, lq=(20, 300), prefix_blocks=(9, 20), dtype=torch.float16, hq=64),
    dict(nseq=3, lq=(33, 200), prefix_blocks=(7, 24), kv="fp8"),
    dict(nseq=2, lq=(64, 700), prefix_blocks=(0, 6), hq=16, hkv=4, d=256),
    dict(nseq=2, lq=(64, 300), prefix_blocks=(4, 9), hq=16, hkv=2, d=256, kv="fp8"),
    dict(nseq=2, lq=(64, 500), prefix_blocks=(2, 3), hq=12, hkv=3),      # slots that do not divide 8
], ids=str)
def test_prefill_ranges(cuda, kw):
    tol = TOL_FP8 if kw.get("kv") == "fp8" else TOL_BF16
    case = make_prefill_case("cfg3", seed=3, device=cuda, **kw)
    assert _ranges(case)
    check(case, range(kw["nseq"]), tol, rows_per_seq=8, all_rows=True)


def test_prefill_ranges_gate_and_reuse(cuda):
    """Gated = the eager gate of the ungated output (at most one ulp on 0.1% of
    elements, as for whole items); a smaller launch that reuses the partial
    buffer of a larger one does not see its pieces; a repeat is bit-identical."""
    big = make_prefill_case("cfg3", seed=5, device=cuda, nseq=4, lq=(100, 300), prefix_blocks=(9, 20))
    small = make_prefill_case("cfg3", seed=6, device=cuda, nseq=1, lq=(90, 90), prefix_blocks=(3, 3))
    assert _ranges(big) and _ranges(small)
    first = run_step(small)
    out = run_step(big)
    assert torch.equal(run_step(small), first)
    assert torch.equal(run_step(big), out)
    gate = torch.randn(out.shape, generator=torch.Generator(device=cuda).manual_seed(1), device=cuda).to(out.dtype)
    got = kernels.varlen_prefill(big["q"], big["k_cache"], big["v_cache"], big["cu_seqlens_q"], big["cu_seqlens_k"],
                                 big["max_seqlen_q"], big["max_seqlen_k"], big["scale"],
                                 block_table=big["block_tables"], gate=gate)
    want = out * torch.sigmoid(gate)
    off = (got.view(torch.int16).int() - want.view(torch.int16).int()).abs()
    assert int(off.max()) <= 1 and float((off > 0).float().mean()) <= 1e-3


@pytest.mark.parametrize("lq,d", [(1, 128), (40, 128), (1, 256), (40, 256)])
def test_prefill_ranges_invisible_front(cuda, lq, d):
    """The first half of the table missing: an item's first pieces hold no
    visible key, more of them than the merge reads at once.  The visible keys
    all score -196 (log2), so a row is the mean of the values it sees."""
    case = make_prefill_case("cfg3", seed=7, device=cuda, nseq=1, lq=(lq, lq), prefix_blocks=(31, 31), hq=8, hkv=2, d=d)
    assert _ranges(case)
    hidden = 16 * case["block_size"]
    case["q"].fill_(1.0)
    case["k_cache"].fill_(-196.0 / (case["scale"] * d * 1.4427))
    case["block_tables"][0, :16] = -1
    out = kernels.varlen_prefill(case["q"], case["k_cache"], case["v_cache"], case["cu_seqlens_q"], case["cu_seqlens_k"],
                                 case["max_seqlen_q"], case["max_seqlen_k"], case["scale"],
                                 block_table=case["block_tables"])
    v = case["v_cache"][case["block_tables"][0, 16:].long()].flatten(0, 1)[:case["lk"][0] - hidden].double()
    upto = torch.arange(v.shape[0] - lq, v.shape[0], device=cuda)
    want = (v.cumsum(0)[upto] / (upto + 1).view(-1, 1, 1)).repeat_interleave(4, 1)
    assert_close(f64(out), f64(want), **TOL_BF16, what="visible half")


@pytest.mark.parametrize("d", [128, 256])
def test_prefill_ranges_nan_key(cuda, d):
    """A NaN key reaches its heads' rows whichever piece holds it, beside pieces without visible keys too."""
    case = make_prefill_case("cfg3", seed=8, device=cuda, nseq=1, lq=(20, 20), prefix_blocks=(31, 31), hq=8, hkv=2, d=d)
    assert _ranges(case)
    case["block_tables"][0, 4:8] = -1
    for t in (3, 2300, 7700):
        k = case["k_cache"].clone()
        k[case["block_tables"][0, t // 256], t % 256, 1, 9] = float("nan")
        out = kernels.varlen_prefill(case["q"], k, case["v_cache"], case["cu_seqlens_q"], case["cu_seqlens_k"],
                                     case["max_seqlen_q"], case["max_seqlen_k"], case["scale"],
                                     block_table=case["block_tables"])
        assert out[:, 4:].isnan().all() and not out[:, :4].isnan().any()
