"""Row groups (tokens x splits) around multiples of eight with several head
groups: the workgroup order puts whole eights on the XCDs and the rest in linear
order, and every (token, split, head group) must be computed exactly once."""
import pytest
import torch

import dsa_amd
from dsa_amd import Tuning
from _parity import check
from oracle import dsa_oracle as O
from test_gpu_parity import _random_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")
    torch.cuda.init()


@pytest.mark.parametrize("tokens", [1, 7, 8, 9, 15, 17])
@pytest.mark.parametrize("heads,config", [
    (48, Tuning(16, 64, 1, kv_waves=4, mfma=16, pv_cols=128)),
    (80, Tuning(16, 64, 3, kv_waves=4, mfma=16, pv_cols=128, fused_merge=True)),
    (96, Tuning(32, 32, 5, kv_waves=2, stages=4, mfma=16, pv_cols=128)),
    (128, Tuning(64, 32, 1, kv_waves=2, stages=4, mfma=16, pv_cols=128)),
    (256, Tuning(128, 32, 1, stages=4, mfma=16, pv_cols=128))], ids=str)
def test_every_group_once(tokens, heads, config):
    data = _random_case(tokens * heads, tokens, 1, heads, 500, 320)
    out = dsa_amd.forward(*data, config=config)
    check(f"groups {tokens}x{heads}", *out, O.reference(*(t.cpu() for t in data)))
