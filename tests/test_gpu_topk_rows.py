"""The top-k selection over rows held in registers, at the row lengths where its
layout changes (a wave's 64-entry steps come in fours, 16 waves; 8 to 64 keys
per thread; the lengths that hand over to the segmented and the memory path),
bit for bit against the oracle, with ties, NaNs and selections past the rows
that are assembled in LDS."""
import pytest
import torch

import dsa_amd
from oracle import dsa_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")
    torch.cuda.init()


def _check(logits, lengths, k, tag):
    """Also without the segmented kernels, which few rows above 32768 would take."""
    want = O.indexer_topk_ref(logits, lengths, k)
    few_long = logits.shape[0] * logits.shape[1] <= 32 and logits.shape[2] > 32768
    for segmented in (True, False) if few_long else (True,):
        got = dsa_amd.indexer_topk(logits.cuda(), lengths.cuda(), k, segmented=segmented)
        assert torch.equal(got.cpu(), want), (tag, segmented)


@pytest.mark.parametrize("L", [2, 63, 64, 65, 4095, 4096, 4097, 8192, 8193, 16384, 16385, 32768, 32769, 65536, 65537])
@pytest.mark.parametrize("ties", [False, True])
def test_row_lengths(L, ties):
    g = torch.Generator().manual_seed(L)
    logits = torch.randn(1, 6, L, generator=g)
    if ties:
        logits = (logits * 3).round()
    lengths = torch.tensor([[L, max(1, L - 1), max(1, L // 2 + 1), max(1, L // 3), 1, 0]], dtype=torch.int32)
    for k in sorted({1, max(1, L // 2 - 1), min(L, 2048), min(L - 1, 4096), min(L - 1, 4097), L - 1}):
        _check(logits, lengths, k, (L, ties, k))


@pytest.mark.parametrize("L", [5000, 20000, 40000])
def test_infinities_and_nans(L):
    """-inf, +inf and NaNs of either sign order by their bits, the NaN with every
    bit set (the key of an absent slot) included."""
    g = torch.Generator().manual_seed(L)
    bits = torch.randn(1, 4, L, generator=g).view(torch.int32).clone()
    bits[..., ::5] = 0x7F800000
    bits[..., 1::5] = -0x00800000          # -inf
    bits[..., 2::7] = 0x7FC00001
    bits[..., 3::7] = -1                   # every bit set
    bits[0, 3] = -1
    lengths = torch.tensor([[L, L - 77, L // 2, L - 3]], dtype=torch.int32)
    for k in (100, L // 2 - 1, L - 100):
        _check(bits.view(torch.float32), lengths, k, (L, k))


def test_many_rows_of_every_length():
    L, rows = 9000, 700
    g = torch.Generator().manual_seed(1)
    logits = torch.randn(1, rows, L, generator=g).abs().sqrt()
    lengths = torch.randint(0, L + 1, (1, rows), generator=g, dtype=torch.int32)
    _check(logits, lengths, 512, "many")


@pytest.mark.parametrize("L", [16384, 16385, 20000, 32768])
@pytest.mark.parametrize("rows", [3, 40])
def test_rows_of_zeros(L, rows):
    """Logits that a relu has clipped: half of a row in one first-digit bin, the
    threshold above it, in it, and among its ties."""
    g = torch.Generator().manual_seed(L + rows)
    logits = torch.randn(1, rows, L, generator=g).clamp(min=0)
    lengths = torch.randint(L // 2, L + 1, (1, rows), generator=g, dtype=torch.int32)
    lengths[0, 0] = L
    for k in (64, L // 4, L // 2 + L // 4):
        _check(logits, lengths, k, (L, rows, k))
