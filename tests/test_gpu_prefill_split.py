"""Prefill work distribution on the GPU: kv-head slots shared by several XCDs.

Every output row against the float32 device reference (oracle/sdpa_path), a
few rows against the float64 oracle.
"""
import pytest
import torch

from oracle.inputs import make_prefill_case
from tests.parity import TOL_BF16, TOL_FP8
from tests.test_gpu_prefill import check

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
