"""The fp8 cache row kernels against the same arithmetic as tensor code.

``quantize_kv_fp8`` writes GPU tensors with one kernel; its bytes must equal
those of the tensor code (run on the same GPU tensors) for every bf16 block
maximum, zeros, infinities and NaNs included, at row counts around a wave's
pair of rows and the grid's reach, and for strided and misaligned views.
"""
import weakref

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


def test_function_modes_see_the_operations(monkeypatch):
    """A torch_function mode sees every operation of the row writer, as of any
    tensor code; a default device is no such observer."""
    from torch.overrides import TorchFunctionMode

    seen = []

    class Watch(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(getattr(func, "__name__", str(func)))
            return func(*args, **(kwargs or {}))

    g = torch.Generator().manual_seed(13)
    kv, kr = torch.randn(5, 512, generator=g).bfloat16().cuda(), torch.randn(5, 64, generator=g).bfloat16().cuda()
    want = _launched(monkeypatch, kv, kr)
    with Watch():
        rows = dsa_amd.quantize_kv_fp8(kv, kr)
    assert torch.equal(rows, want) and {"float", "where", "frexp", "cat"} <= set(seen)
    with torch.device("cpu"):
        assert torch.equal(_launched(monkeypatch, kv, kr), want)


def test_rows_without_the_library(monkeypatch, tmp_path):
    """A package whose library is not built writes the rows as tensor code."""
    from dsa_amd import _lib

    g = torch.Generator().manual_seed(12)
    kv, kr = torch.randn(5, 512, generator=g).bfloat16().cuda(), torch.randn(5, 64, generator=g).bfloat16().cuda()
    want = _launched(monkeypatch, kv, kr)
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", tmp_path / "missing.so")
    assert torch.equal(dsa_amd.quantize_kv_fp8(kv, kr), want)


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


# ------------------------------------------------- the cache expanded to bf16

def _expanding_case(batch, queries, heads, length, topk, block, seed):
    """A call that expands its cache; returns (args, block table, contiguous
    rows, the slots' validity through the table)."""
    g = torch.Generator().manual_seed(seed)
    rows = kvcache.quantize_kv_fp8((torch.randn(batch, length, 1, 512, generator=g) * 2).bfloat16(),
                                   torch.randn(batch, length, 1, 64, generator=g).bfloat16(), pow2_scales=seed % 2 == 0)
    q = torch.randn(batch, queries, heads, 512, generator=g).bfloat16()
    qr = torch.randn(batch, queries, heads, 64, generator=g).bfloat16()
    ids = torch.randint(0, length, (batch, queries, 1, topk), generator=g, dtype=torch.int32)
    u = torch.rand(ids.shape, generator=g)
    ids[u < 0.1] = -1
    ids[u > 0.97] = length + 5
    table = pool = None
    if block:
        per = length // block
        blocks = batch * per + 3
        table = torch.randperm(blocks, generator=g)[:batch * per].view(batch, per).int()
        pool = torch.randint(0, 120, (blocks, block, 1, 656), generator=g, dtype=torch.uint8)
        pool[table.reshape(-1).long()] = rows.reshape(batch * per, block, 1, 656)
        table[:, 0] = torch.tensor([-1, blocks, 2 ** 31 - 1])[:batch]  # unbacked: slots of block 0 are masked
        table[:, -1] = -7
    ids[..., 0] = min(length - 1, max(block, 1) + 1)  # one backed slot in every row
    return q, qr, ids, rows, table, pool


@pytest.mark.parametrize("shape,block", [((1, 257, 128, 1024, 257), 0), ((2, 130, 16, 96, 64), 16),
                                         ((3, 90, 48, 333, 40), 0), ((1, 300, 64, 192, 2048), 64),
                                         ((3, 100, 32, 128, 300), 8)])
def test_expanded_call_equals_bf16_call(shape, block):
    from dsa_amd import api
    from oracle import dsa_oracle as O

    batch, queries, heads, length, topk = shape
    assert api.expands_rows(shape)
    q, qr, ids, rows, table, pool = _expanding_case(*shape, block, seed=heads)
    kv, rope = O.dequant_fp8_rows(rows)
    seen = ids.clone()
    if block:  # the slots of unbacked blocks, masked by hand
        entry = table.long()[torch.arange(batch)[:, None, None, None],
                             (ids.long().clamp(0, length - 1) // block)]
        seen[(entry < 0) | (entry >= pool.shape[0])] = -1
    args = (q.cuda(), (rows if table is None else pool).cuda(), qr.cuda(), None, ids.cuda())
    (got, launches) = dsa_amd.forward(*args, block_table=None if table is None else table.cuda(),
                                      return_kernels=True)
    assert launches[0].name == "expand_rows"
    want = dsa_amd.forward(q.cuda(), kv.cuda(), qr.cuda(), rope.cuda(), seen.cuda())
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_call_without_room_runs_on_the_rows(monkeypatch):
    from dsa_amd import api

    shape = (1, 257, 16, 512, 64)
    q, qr, ids, rows, _, _ = _expanding_case(*shape, 0, seed=4)
    args = (q.cuda(), rows.cuda(), qr.cuda(), None, ids.cuda())
    want = dsa_amd.forward(*args, config=dsa_amd.plan_call(shape, None, 256, kv_fp8=True)[0])
    monkeypatch.setattr(api, "_expanded_cache", lambda *_: None)
    got, launches = dsa_amd.forward(*args, return_kernels=True)
    assert all(l.name != "expand_rows" for l in launches)
    for a, b in zip(got, want):
        assert torch.equal(a, b)


class _BudgetTorch:
    """``torch`` whose ``empty``/``empty_like``/``zeros`` raise OutOfMemoryError
    beyond ``budget`` live bytes (an idealised card; the tensors are real)."""

    def __init__(self, budget):
        self.budget, self.live, self.peak = budget, 0, 0

    def __getattr__(self, name):
        attr = getattr(torch, name)
        if name not in ("empty", "empty_like", "zeros"):
            return attr

        def allocate(*args, **kwargs):
            t = attr(*args, **kwargs)
            size = t.numel() * t.element_size()
            if self.live + size > self.budget:
                del t
                raise torch.OutOfMemoryError("beyond the test's budget")
            self.live += size
            self.peak = max(self.peak, self.live)
            weakref.finalize(t, self._free, size)
            return t
        return allocate

    def _free(self, size):
        self.live -= size


@pytest.mark.parametrize("shape,value_dim", [((1, 300, 96, 1024, 4096), 0),     # the bf16 plan splits too
                                             ((1, 300, 96, 1024, 4096), 128),   # ... merge and projection in one
                                             ((1, 257, 128, 1024, 257), 128)])  # no split, projected afterwards
def test_expansion_never_takes_a_buffer_the_call_needs(monkeypatch, shape, value_dim):
    """With any memory from what the call needs on the fp8 rows upwards it
    succeeds: expanded where everything fits beside the cache, else on the rows."""
    from dsa_amd import api

    q, qr, ids, rows, _, _ = _expanding_case(*shape, 0, seed=6)
    args = (q.cuda(), rows.cuda(), qr.cuda(), None, ids.cuda())
    kw = {"w_uv": torch.randn(shape[2], value_dim, 512).bfloat16().cuda() * 0.04} if value_dim else {}

    def run(budget, room=True, **more):
        api._arrivals.clear()
        spy = _BudgetTorch(budget)
        with monkeypatch.context() as m:
            m.setattr(api, "torch", spy)
            if not room:
                m.setattr(api, "_expanded_cache", lambda *_: None)
            out, launches = dsa_amd.forward(*args, return_kernels=True, **kw, **more)
        return out, launches[0].name == "expand_rows", spy.peak

    on_rows, expanded, need = run(1 << 40, room=False)
    assert not expanded
    as_bf16, expanded, full = run(1 << 40)
    assert expanded and full >= need
    cache = shape[0] * shape[3] * 1152
    for budget in (need, need + cache // 2, need + cache - 1, full - 1, full):
        out, expanded, _ = run(budget)
        assert expanded == (budget >= full), (budget, need, full)
        for a, b in zip(out, as_bf16 if expanded else on_rows):
            assert torch.equal(a, b)


def test_call_without_room_keeps_the_allocators_cache():
    """Where the copy cannot be had, torch's allocator is not asked for it: it
    would wait for the device and give every cached block back first."""
    shape = (1, 512, 16, 65536, 2048)  # a copy of 72 MiB
    q, qr, ids, rows, _, _ = _expanding_case(*shape, 0, seed=2)
    args = (q.cuda(), rows.cuda(), qr.cuda(), None, ids.cuda())
    want = dsa_amd.forward(*args, config=dsa_amd.plan_call(shape, None, 256, kv_fp8=True)[0])
    got, launches = dsa_amd.forward(*args, return_kernels=True)
    assert launches[0].name == "expand_rows"
    del got
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    kept = torch.empty(16 << 20, device="cuda", dtype=torch.uint8)
    del kept  # a cached block
    room = 40 << 20  # the call's own buffers and no copy
    total = torch.cuda.mem_get_info()[1]
    before = torch.cuda.get_per_process_memory_fraction()
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + room) / total)
    try:
        retries = torch.cuda.memory_stats()["num_alloc_retries"]
        for _ in range(2):
            got, launches = dsa_amd.forward(*args, return_kernels=True)
            assert launches[0].name != "expand_rows"
            for a, b in zip(got, want):
                assert torch.equal(a, b)
            del got
        assert torch.cuda.memory_stats()["num_alloc_retries"] == retries
    finally:
        torch.cuda.set_per_process_memory_fraction(before)


@pytest.mark.parametrize("shape", [(1, 300, 128, 1024, 512),    # neither plan fuses its merge
                                   (1, 257, 16, 1024, 4096)])   # both do, one counter a token
def test_expansion_does_not_depend_on_arrivals(shape):
    """The caller's own counters change nothing but whose counters are used."""
    q, qr, ids, rows, _, _ = _expanding_case(*shape, 0, seed=8)
    args = (q.cuda(), rows.cuda(), qr.cuda(), None, ids.cuda())
    want, launches = dsa_amd.forward(*args, return_kernels=True)
    own = torch.zeros(shape[0] * shape[1] * shape[2] // 16, device="cuda", dtype=torch.int32)
    got, with_own = dsa_amd.forward(*args, return_kernels=True, arrivals=own)
    assert with_own == launches and launches[0].name == "expand_rows"
    torch.cuda.synchronize()
    assert not own.any()
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_counters_of_the_fp8_plans_size_are_taken():
    """Enough counters for the plan on the fp8 rows (32 heads a workgroup), too
    few for the bf16 plan (16 heads): such a call runs on the fp8 rows."""
    shape = (1, 256, 32, 1024, 4096)
    on_rows, as_bf16 = dsa_amd.plan_call(shape, kv_fp8=True)[0], dsa_amd.plan_call(shape)[0]
    assert on_rows.fused_merge and as_bf16.fused_merge and on_rows.bm > as_bf16.bm
    q, qr, ids, rows, _, _ = _expanding_case(*shape, 0, seed=10)
    args = (q.cuda(), rows.cuda(), qr.cuda(), None, ids.cuda())
    want = dsa_amd.forward(*args, config=on_rows)
    own = torch.zeros(shape[0] * shape[1] * shape[2] // on_rows.bm, device="cuda", dtype=torch.int32)
    got, launches = dsa_amd.forward(*args, return_kernels=True, arrivals=own)
    assert launches[0].name != "expand_rows"
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    with pytest.raises(ValueError, match="counters"):
        dsa_amd.forward(*args, arrivals=own[1:])
