"""The fp8 cache row kernels against the same arithmetic as tensor code.

``quantize_kv_fp8`` writes GPU tensors with one kernel; its bytes must equal
those of the tensor code (run on the same GPU tensors) for every bf16 block
maximum, zeros, infinities and NaNs included, at row counts around a wave's
pair of rows and the grid's reach, and for strided and misaligned views.
"""
import pytest
import torch

import dsa_amd
from dsa_amd import kvcache

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no ROCm GPU")
    torch.cuda.init()


def _tensor_code(monkeypatch, *args, **kw):
    with monkeypatch.context() as m:
        m.setattr(kvcache, "_plain_gpu_pair", lambda *_: False)
        return dsa_amd.quantize_kv_fp8(*args, **kw)


def _launched(monkeypatch, *args, **kw):
    """The call's rows, with the kernel shown to be what wrote them."""
    calls = []
    inner = kvcache._quantize_gpu
    with monkeypatch.context() as m:
        m.setattr(kvcache, "_quantize_gpu", lambda *a: calls.append(1) or inner(*a))
        rows = dsa_amd.quantize_kv_fp8(*args, **kw)
    assert calls
    return rows


@pytest.mark.parametrize("pow2", [True, False])
def test_every_block_maximum(monkeypatch, pow2):
    """One block per bf16 bit pattern (as its first value), the rest of the
    block fractions of it and the other sign."""
    g = torch.Generator().manual_seed(7)
    head = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    frac = torch.rand(65536, 127, generator=g) * 2 - 1
    body = (head.float()[:, None] * frac).bfloat16()
    kv = torch.cat([head[:, None], body], 1).reshape(-1, 512).cuda()
    kr = torch.randn(kv.shape[0], 64, generator=g).bfloat16().cuda()
    assert torch.equal(_launched(monkeypatch, kv, kr, pow2_scales=pow2),
                       _tensor_code(monkeypatch, kv, kr, pow2_scales=pow2))


@pytest.mark.parametrize("pow2", [True, False])
@pytest.mark.parametrize("rows", [1, 2, 3, 7, 8, 9, 32767, 32769, 65537])
def test_row_counts(monkeypatch, rows, pow2):
    g = torch.Generator().manual_seed(rows)
    kv = (torch.randn(rows, 1, 512, generator=g) * torch.rand(rows, 1, 1, generator=g) * 9).bfloat16()
    kr = torch.randn(rows, 1, 64, generator=g).bfloat16()
    kv[rows // 2, 0, 128:256] = 0
    out = _launched(monkeypatch, kv.cuda(), kr.cuda(), pow2_scales=pow2)
    assert out.shape == (rows, 1, 656)
    assert torch.equal(out, _tensor_code(monkeypatch, kv.cuda(), kr.cuda(), pow2_scales=pow2))
    if pow2:  # and the CPU's (which rounds amax / 448 itself, not a product with 1 / 448)
        assert torch.equal(out.cpu(), dsa_amd.quantize_kv_fp8(kv, kr))


def test_views(monkeypatch):
    g = torch.Generator().manual_seed(3)
    both = torch.randn(6, 577 + 3, generator=g).bfloat16().cuda()
    cases = [(both[:, 1:513], both[:, 513:577]),                       # strided and misaligned
             (both[::2, :512], both[::2, 512:576]),                    # every other row
             (both.reshape(-1)[1:513], both.reshape(-1)[601:665])]     # contiguous, 2-byte aligned
    for kv, kr in cases:
        assert torch.equal(_launched(monkeypatch, kv, kr), _tensor_code(monkeypatch, kv, kr))


def test_empty_and_mixed_devices():
    kv, kr = torch.empty(0, 512, dtype=torch.bfloat16), torch.empty(0, 64, dtype=torch.bfloat16)
    assert dsa_amd.quantize_kv_fp8(kv.cuda(), kr.cuda()).shape == (0, 656)
    with pytest.raises(RuntimeError):
        dsa_amd.quantize_kv_fp8(torch.zeros(2, 512).bfloat16().cuda(), torch.zeros(2, 64).bfloat16())
