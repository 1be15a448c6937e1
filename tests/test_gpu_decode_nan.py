"""Pieces of a context whose scores are NaN, or give no key any weight: a NaN
in a query or a cached key reaches the output at every context length, and a
row all of whose later pieces are without weight is still written."""
import pytest
import torch

from nano_qwen_amd import kernels
from oracle.inputs import make_decode_case
from tests.parity import TOL_BF16, TOL_FP8, assert_close, f64

pytestmark = pytest.mark.gpu

SCHEDULES = {"own": {}, "split-K": {"NQ_DECODE_SPLIT_TOKENS": "128", "NQ_DECODE_STREAMK": "0"},
             "stream-K": {"NQ_DECODE_SPLIT_TOKENS": "128", "NQ_DECODE_STREAMK": "1"}}


@pytest.fixture(params=list(SCHEDULES))
def schedule(request, monkeypatch):
    for name, value in SCHEDULES[request.param].items():
        monkeypatch.setenv(name, value)


def _case(device, ctx, batch, **kw):
    case = make_decode_case("cfg2", seed=ctx, device=device, batch=batch, ctx=(ctx, ctx), **kw)
    kernels.store_kvcache(case["k_new"], case["v_new"], case["k_cache"], case["v_cache"], case["slot_mapping"],
                          case["k_scale"], case["v_scale"])
    return case


def _decode(case):
    out = torch.full_like(case["q"], 7.0).unsqueeze(1)    # a row that is not written shows
    kernels.paged_decode(case["q"].unsqueeze(1), case["k_cache"], case["v_cache"], case["context_lens"],
                         case["block_tables"], case["scale"], case["k_scale"], case["v_scale"], out=out)
    torch.cuda.synchronize()
    return out[:, 0]


def _slot(case, row, t):
    bs = case["block_size"]
    return int(case["block_tables"][row, t // bs]), t % bs


@pytest.mark.parametrize("d", [128, 256])
@pytest.mark.parametrize("ctx", [100, 300, 500, 2000, 9000])
def test_nan_key_reaches_the_output(cuda, schedule, ctx, d):
    """One NaN in one cached key of row 0, kv head 1: NaN in that row's heads of
    that kv head, whichever piece holds the key; every other output is as without it."""
    hq, hkv = (16, 4) if d == 256 else (8, 2)
    case = _case(cuda, ctx, 2, hq=hq, hkv=hkv, d=d)
    G = hq // hkv
    clean = _decode(case)
    assert not clean.isnan().any()
    for t in (0, 130, 299, ctx - 1):
        if t >= ctx:
            continue
        block, off = _slot(case, 0, t)
        value = case["k_cache"][block, off, 1, 5].clone()
        case["k_cache"][block, off, 1, 5] = float("nan")
        out = _decode(case)
        case["k_cache"][block, off, 1, 5] = value
        assert out[0, G:2 * G].isnan().all(), f"key {t}"
        out[0, G:2 * G] = clean[0, G:2 * G]
        assert torch.equal(out, clean)


@pytest.mark.parametrize("kw", [dict(hq=8, hkv=2), dict(hq=16, hkv=4, d=256), dict(hq=8, hkv=2, kv="fp8"),
                                dict(hq=32, hkv=8, kv="fp8")], ids=str)
@pytest.mark.parametrize("ctx", [100, 300, 2000])
def test_nan_query_reaches_the_output(cuda, schedule, ctx, kw):
    """A NaN in one query: every score of that head is NaN, in every piece."""
    case = _case(cuda, ctx, 2, **kw)
    clean = _decode(case)
    case["q"][1, 3, 17] = float("nan")
    out = _decode(case)
    assert out[1, 3].isnan().all()
    out[1, 3] = clean[1, 3]
    assert torch.equal(out, clean)


@pytest.mark.parametrize("kw", [dict(hq=8, hkv=2), dict(hq=16, hkv=4, d=256), dict(hq=8, hkv=2, kv="fp8")], ids=str)
@pytest.mark.parametrize("ctx,seen", [(129, 128), (300, 128), (500, 256), (2000, 128), (2000, 1024)])
def test_rows_whose_later_pieces_have_no_weight(cuda, schedule, ctx, seen, kw):
    """Table entries past ``seen`` tokens missing: the pieces there hold tokens
    but no visible key.  The row is the attention over the first ``seen``."""
    case = _case(cuda, ctx, 2, bs=128, **kw)
    short = dict(case, context_lens=torch.full_like(case["context_lens"], seen))
    want = _decode(short)
    case["block_tables"][:, seen // case["block_size"]:] = -1
    out = _decode(case)
    tol = TOL_FP8 if kw.get("kv") == "fp8" else TOL_BF16
    assert_close(f64(out), f64(want), **tol, what="visible part")
    case["block_tables"][:] = -1    # and without any visible key: zeros
    assert not _decode(case).any()
