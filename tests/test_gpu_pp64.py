"""The 64-head ping-pong kernel (two streams of tiles, one per wave group)
against the CPU oracle at the parity bounds.

Its schedule turns on the number of 32-slot tiles a workgroup is left with
after the masked slots are compacted away -- 1 (the second stream is empty),
odd, even, and around the four ring stages -- and its epilogue adds the two
streams' sums, each under its own reference max.
"""
import pytest
import torch

import dsa_amd
from dsa_amd import Tuning
from _parity import OUT_TOL, STAT_RTOL
from oracle import dsa_oracle as O
from test_gpu_parity import _masked_rows, _random_case, _run_and_check

pytestmark = pytest.mark.gpu


def _plan(split=1):
    return Tuning(64, 32, split, kv_waves=2, stages=4, mfma=16, pv_cols=128)


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")
    torch.cuda.init()


@pytest.mark.parametrize("B,SQ,H,L,K,split", [
    (1, 1, 64, 1, 1, 1), (1, 3, 64, 5, 33, 1), (2, 2, 64, 300, 64, 1), (1, 2, 128, 300, 65, 1),
    (1, 2, 192, 999, 97, 1), (3, 1, 64, 999, 128, 1), (1, 2, 64, 999, 129, 1), (1, 2, 128, 4000, 161, 2),
    (2, 3, 64, 4000, 1000, 3), (1, 9, 64, 9000, 2048, 1), (1, 2, 64, 9000, 2047, 8), (1, 1, 128, 20000, 4096, 2)])
def test_edge_shapes(B, SQ, H, L, K, split):
    _run_and_check(f"pp64-{B}x{SQ}x{H}x{L}x{K}-s{split}", _random_case(B * 1000 + K + split, B, SQ, H, L, K),
                   config=_plan(split))


@pytest.mark.parametrize("split", [1, 3])
def test_masked_rows(split):
    """Rows with 1, 31, 32, 33, 64, ... valid slots among 2048 (max gated per
    query over the heads: one score alone can sit near zero)."""
    B, SQ, H, L, K = 1, 12, 64, 6000, 2048
    g = torch.Generator().manual_seed(170 + split)
    q, kv, qr, kr = (torch.randn(s, generator=g).bfloat16()
                     for s in ((B, SQ, H, 512), (B, L, 1, 512), (B, SQ, H, 64), (B, L, 1, 64)))
    ids = _masked_rows(190 + split, SQ, L, K).view(B, SQ, 1, K).contiguous()
    got = dsa_amd.forward(*(t.cuda() for t in (q, kv, qr, kr, ids)), config=_plan(split))
    ref = O.reference(q, kv, qr, kr, ids)
    acc, am = O.accuracy(got[0].cpu(), ref[0]), O.accuracy(got[1].cpu(), ref[1])
    assert acc["finite"] and acc["max_row_normalized"] <= OUT_TOL
    assert am["max_row_normalized"] <= STAT_RTOL and O.rel_error(got[2].cpu(), ref[2]) <= STAT_RTOL


@pytest.mark.parametrize("hot", [40, 1, 2047, 1000])
def test_late_maximum_takes_the_second_pass(hot):
    """One slot, in a tile of either stream, beats every other score by more
    than 2^64: the stream that holds it recomputes, the other's sum fades."""
    B, SQ, H, L, K = 1, 2, 64, 4096, 2048
    g = torch.Generator().manual_seed(hot)
    q = torch.randn(B, SQ, H, 512, generator=g).bfloat16()
    q[..., 0] = 40.0
    kv = torch.randn(B, L, 1, 512, generator=g).bfloat16()
    qr, kr = torch.randn(B, SQ, H, 64, generator=g).bfloat16(), torch.randn(B, L, 1, 64, generator=g).bfloat16()
    ids = torch.stack([torch.randperm(L - 1, generator=g)[:K] for _ in range(SQ)]).view(B, SQ, 1, K).int()
    kv[0, L - 1, 0, 0] = 60.0  # score +100, about 144 in log2 units
    ids[..., hot] = L - 1
    _run_and_check(f"pp64-hot{hot}", tuple(t.cuda() for t in (q, kv, qr, kr, ids)), config=_plan())


def test_no_valid_slot_gives_nan():
    data = list(_random_case(3, 1, 2, 64, 500, 100))
    data[4][0, 1] = -1
    out = dsa_amd.forward(*data, config=_plan())[0]
    assert torch.isfinite(out[0, 0].float()).all() and torch.isnan(out[0, 1].float()).all()


def test_paged_equals_contiguous_and_repeats():
    q, kv, qr, kr, ids = _random_case(21, 2, 5, 64, 1024, 700)
    table = torch.randperm(2 * 1024 // 16, device="cuda").int().view(2, -1)
    pool, rope = torch.empty_like(kv).view(-1, 16, 1, 512), torch.empty_like(kr).view(-1, 16, 1, 64)
    pool[table.view(-1).long()] = kv.view(-1, 16, 1, 512)
    rope[table.view(-1).long()] = kr.view(-1, 16, 1, 64)
    want = dsa_amd.forward(q, kv, qr, kr, ids, config=_plan(), scale=0.1)
    for _ in range(3):
        got = dsa_amd.forward(q, pool, qr, rope, ids, config=_plan(), scale=0.1, block_table=table)
        for a, b in zip(got, want):
            assert torch.equal(a, b)
