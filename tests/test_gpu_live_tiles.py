"""Rows whose tail is masked: for chunks (32 queries of a sequence or more) the
kernels run only the tiles up to the last valid slot of their range, so a padded
row must give the bits of the same row with its tail cut off (a call of one
query, which runs every tile), and a masked slot in the middle must still be
skipped."""
import pytest
import torch

import dsa_amd
from dsa_amd import Tuning
from _parity import OUT_TOL, STAT_RTOL
from oracle import dsa_oracle as O

pytestmark = pytest.mark.gpu

PLANS = [Tuning(16, 64, 1, kv_waves=4, mfma=16, pv_cols=128), Tuning(32, 64, 1, kv_waves=4, mfma=16, pv_cols=128),
         Tuning(16, 32, 1, kv_waves=2, stages=4, mfma=16, pv_cols=128),
         Tuning(32, 32, 1, kv_waves=2, stages=4, mfma=16, pv_cols=128),
         Tuning(16, 64, 1, kv_waves=4, mfma=16), Tuning(32, 64, 1, kv_waves=2, mfma=16), Tuning(64, 64, 1, mfma=16),
         Tuning(64, 64, 1, kv_waves=2), Tuning(128, 32, 1, stages=4)]


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")
    torch.cuda.init()


def _case(seed, counts, K=1024, L=3000, H=128):
    g = torch.Generator().manual_seed(seed)
    SQ = len(counts)
    q, kv, qr, kr = (torch.randn(s, generator=g).bfloat16()
                     for s in ((1, SQ, H, 512), (1, L, 1, 512), (1, SQ, H, 64), (1, L, 1, 64)))
    ids = torch.full((1, SQ, 1, K), -1, dtype=torch.int32)
    for s, n in enumerate(counts):
        ids[0, s, 0, :n] = torch.randint(0, L, (n,), generator=g, dtype=torch.int32)
        ids[0, s, 0, 1:n:7] = L + 9  # masked slots in between
    return q, kv, qr, kr, ids


COUNTS = [1, 2, 31, 32, 33, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 513, 1023, 1024] + [300 + 7 * i for i in range(16)]


@pytest.mark.parametrize("plan", PLANS, ids=str)
def test_padded_rows(plan):
    data = _case(plan.bm + plan.bn, COUNTS)
    dev = tuple(t.cuda() for t in data)
    got = dsa_amd.forward(*dev, config=plan)
    ref = O.reference(*data)
    acc = O.accuracy(got[0].cpu(), ref[0])
    assert acc["finite"] and acc["max_row_normalized"] <= OUT_TOL
    assert O.rel_error(got[2].cpu(), ref[2]) <= STAT_RTOL
    for s in (0, 4, 7, 13):  # cut behind the last valid slot's tile: the same bits
        cut = -(-COUNTS[s] // plan.bn) * plan.bn
        one = dsa_amd.forward(dev[0][:, s:s + 1].contiguous(), dev[1], dev[2][:, s:s + 1].contiguous(), dev[3],
                              dev[4][:, s:s + 1, :, :cut].contiguous(), config=plan)
        for a, b in zip((got[0][:, s:s + 1], got[1][:, :, s:s + 1], got[2][:, :, s:s + 1]), one):
            assert torch.equal(a, b), (s, COUNTS[s])


def test_fp8_rows_padded():
    q, kv, qr, kr, ids = (t.cuda() for t in _case(9, COUNTS, H=64))
    rows = dsa_amd.quantize_kv_fp8(kv, kr)
    deq, rope = O.dequant_fp8_rows(rows)
    for plan in (Tuning(16, 64, 2, kv_waves=4, mfma=16), Tuning(32, 64, 1, kv_waves=2, mfma=16), Tuning(64, 64, 3, mfma=16)):
        got = dsa_amd.forward(q, rows, qr, None, ids, config=plan)
        want = dsa_amd.forward(q, deq.cuda(), qr, rope.cuda(), ids, config=plan)
        for a, b in zip(got, want):
            assert torch.equal(a, b)


@pytest.mark.parametrize("plan", [Tuning(16, 64, 4, kv_waves=4, mfma=16, pv_cols=128),
                                  Tuning(16, 64, 4, kv_waves=4, mfma=16, pv_cols=128, fused_merge=True),
                                  Tuning(32, 32, 8, kv_waves=2, stages=4, mfma=16, pv_cols=128),
                                  Tuning(64, 64, 3, mfma=16), Tuning(64, 64, 2, kv_waves=2)], ids=str)
def test_split_ranges_without_a_valid_slot(plan):
    data = _case(plan.split, [1, 30, 70, 130, 300, 600, 1024, 5] * 4)
    out, mx, sm = (t.cpu() for t in dsa_amd.forward(*(t.cuda() for t in data), config=plan))
    ref = O.reference(*data)
    acc = O.accuracy(out, ref[0])
    assert acc["finite"] and acc["max_row_normalized"] <= OUT_TOL
    # The max of a row with one valid slot is a single score, 576 products of
    # unit variance over 24 summed in fp32: an absolute error of some 1e-6
    # however near to zero the score lies, so it is gated against the largest
    # max of its query's heads, not element by element.
    assert O.accuracy(mx, ref[1])["max_row_normalized"] <= STAT_RTOL
    assert O.rel_error(sm, ref[2]) <= STAT_RTOL


@pytest.mark.parametrize("plan", PLANS[:7], ids=str)
def test_last_slot_decides_nothing_but_the_tiles_run(plan):
    """A range looks for its last valid slot only where its last slot is masked:
    rows that end in a valid slot behind masked ones, in an index past the cache,
    or (paged) in a slot of an unbacked block give the bits of the same row with
    the masked slots written as -1 and of a call of one query, which looks at none."""
    K, L, bs = 384, 960, 16
    q, kv, qr, kr, ids = (t.cuda() for t in _case(3, [K] * 32, K=K, L=L))
    ids[0, 0, 0, 5:K - 1] = -1           # one valid slot at either end
    ids[0, 1, 0, 70:] = L                # past the cache
    ids[0, 2, 0, 33:] = -2 ** 31
    ids[0, 3, 0, :-2] = -1               # the last but one
    ids[0, 3, 0, -1] = 2 ** 31 - 1
    ids[0, 4, 0, K - 40:] = 17           # of an unbacked block, below
    table = torch.randperm(L // bs, generator=torch.Generator().manual_seed(1)).int().cuda()[None]
    pool, rpool = torch.empty_like(kv).view(L // bs, bs, 1, 512), torch.empty_like(kr).view(L // bs, bs, 1, 64)
    pool[table[0].long()], rpool[table[0].long()] = kv.view(L // bs, bs, 1, 512), kr.view(L // bs, bs, 1, 64)
    table[0, 1] = -1
    seen = torch.where((ids < 0) | (ids >= L) | (ids // bs == 1), -1, ids)
    got = dsa_amd.forward(q, pool, qr, rpool, ids, config=plan, block_table=table)
    want = dsa_amd.forward(q, kv, qr, kr, seen, config=plan)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    for s in range(6):
        one = dsa_amd.forward(q[:, s:s + 1].contiguous(), kv, qr[:, s:s + 1].contiguous(), kr,
                              seen[:, s:s + 1].contiguous(), config=plan)
        for a, b in zip((got[0][:, s:s + 1], got[1][:, :, s:s + 1], got[2][:, :, s:s + 1]), one):
            assert torch.equal(a, b), s
