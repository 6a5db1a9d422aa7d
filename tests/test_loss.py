"""Chunked readout + cross-entropy (dabsn_amd.loss) against F.cross_entropy.

Mirrors the reference's tests/test_loss_chunking.py cases (forward, gradients for several
chunk budgets, ignore_index, the single-chunk path, the from-logits variant, the ``off``
switch) on this package's device path: the row kernels run as HIP on the GPU, and on the
CPU through the test-only oracle kernels, which checks the chunking, masking and gradient
assembly of loss.py itself. fp32 throughout (the HIP kernels take fp32/bf16): loss relative
1e-5 and gradients normwise 1e-5 against fp64 torch on the same fp32 values; bf16 logits
relative 1e-2 against the fp32 loss of the same bf16 hidden/weight.
"""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from dabsn_amd import loss as L
from helpers import rel_err
from oracle import torch_backend


@pytest.fixture(scope="module", autouse=True)
def _oracle_cpu_kernels():
    torch_backend.register()


def _case(seed, B, T, H, V, bias=True, dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    hidden = torch.randn(B, T, H, generator=g).to(dtype)
    weight = (torch.randn(V, H, generator=g) / H ** 0.5).to(dtype)
    b = torch.randn(V, generator=g).to(dtype) if bias else None
    targets = torch.randint(0, V, (B, T), generator=g)
    return hidden, weight, b, targets


def _naive(hidden, weight, bias, targets, ignore_index=-100):
    """fp64 F.linear + F.cross_entropy on the same values, with gradients."""
    leaves = [None if x is None else x.detach().double().requires_grad_(True)
              for x in (hidden, weight, bias)]
    logits = F.linear(leaves[0], leaves[1], leaves[2])
    loss = F.cross_entropy(logits.reshape(-1, logits.shape[-1]), targets.reshape(-1),
                           ignore_index=ignore_index)
    loss.backward()
    return loss.detach(), [None if x is None else x.grad for x in leaves]


def _run(hidden, weight, bias, targets, device, **kw):
    leaves = [None if x is None else x.detach().to(device).requires_grad_(True)
              for x in (hidden, weight, bias)]
    loss = L.chunked_linear_cross_entropy(leaves[0], leaves[1], leaves[2], targets.to(device), **kw)
    loss.backward()
    return loss.detach().cpu(), [None if x is None else x.grad.cpu() for x in leaves]


def _check(got, want, tol=1e-5):
    loss, grads = got
    ref_loss, ref_grads = want
    assert abs(float(loss) - float(ref_loss)) <= tol * abs(float(ref_loss))
    for a, b in zip(grads, ref_grads):
        assert (a is None) == (b is None)
        if a is not None:
            assert rel_err(a, b) <= tol


DEVICES = ["cpu", pytest.param("cuda", marks=pytest.mark.gpu)]


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("budget", [1, 7 * 50, 10_000])
def test_loss_and_gradients_match_cross_entropy_for_any_chunking(device, budget):
    """reference test_loss_chunking.py:45-65 (budgets 1 row, 7 rows, everything)."""
    h, w, b, t = _case(1, 3, 5, 7, 50)
    _check(_run(h, w, b, t, device, chunk_budget=budget), _naive(h, w, b, t))


@pytest.mark.parametrize("device", DEVICES)
def test_ignore_index_masks_positions(device):
    """reference test_loss_chunking.py:68-89."""
    h, w, b, t = _case(2, 2, 8, 6, 30)
    t[:, ::2] = -100
    _check(_run(h, w, b, t, device, chunk_budget=1, ignore_index=-100),
           _naive(h, w, b, t, ignore_index=-100))


@pytest.mark.parametrize("device", DEVICES)
def test_no_bias_and_single_chunk(device):
    h, w, _, t = _case(3, 2, 4, 5, 16, bias=False)
    _check(_run(h, w, None, t, device, chunk_budget=1 << 30), _naive(h, w, None, t))


@pytest.mark.parametrize("device", DEVICES)
def test_from_logits_variant_matches(device):
    """reference test_loss_chunking.py:108-117, with its gradient."""
    g = torch.Generator().manual_seed(4)
    logits = torch.randn(37, 60, generator=g)
    t = torch.randint(0, 60, (37,), generator=g)
    x = logits.detach().to(device).clone().requires_grad_(True)
    got = L.chunked_cross_entropy_from_logits(x, t.to(device), chunk_budget=1)
    got.backward()
    xl = logits.detach().double().requires_grad_(True)
    ref = F.cross_entropy(xl, t)
    ref.backward()
    assert abs(float(got.detach()) - float(ref.detach())) <= 1e-5 * float(ref.detach())
    assert rel_err(x.grad.cpu(), xl.grad) <= 1e-5


def test_off_switch_uses_full_cross_entropy(monkeypatch):
    """reference test_loss_chunking.py:120-131."""
    monkeypatch.setenv("DABSN_LOSS_CHUNK_SCORES", "off")
    h, w, b, t = _case(5, 2, 6, 8, 40)
    got = L.chunked_linear_cross_entropy(h, w, b, t)
    assert abs(float(got) - float(_naive(h, w, b, t)[0])) <= 1e-5 * float(got)


@pytest.mark.gpu
def test_readout_size_loss_on_device_bf16(cuda_device):
    """Vocabulary 32000 at bf16 with several chunks: against the fp32 loss and gradients of
    the same bf16 hidden and weight."""
    h, w, b, t = _case(6, 2, 512, 256, 32000, dtype=torch.bfloat16)
    leaves = [x.to(cuda_device).requires_grad_(True) for x in (h, w, b)]
    loss = L.chunked_linear_cross_entropy(*leaves, t.to(cuda_device), chunk_budget=1 << 22)
    loss.backward()
    ref = [x.float().to(cuda_device).requires_grad_(True) for x in (h, w, b)]
    want = F.cross_entropy(F.linear(*ref).reshape(-1, 32000), t.to(cuda_device).reshape(-1))
    want.backward()
    assert loss.dtype == torch.float32
    assert abs(float(loss.detach()) - float(want.detach())) <= 1e-2 * float(want.detach())
    for a, r in zip(leaves, ref):
        assert rel_err(a.grad.float().cpu(), r.grad.cpu()) <= 2e-2


@pytest.mark.gpu
def test_out_of_range_target_is_reported(cuda_device):
    x = torch.randn(3, 10, device=cuda_device)
    with pytest.raises(RuntimeError, match="outside"):
        L.chunked_cross_entropy_from_logits(x, torch.tensor([1, 10, 2], device=cuda_device))


@pytest.mark.gpu
@pytest.mark.parametrize("rows,V", [(1, 1), (15, 7), (16, 8), (17, 2047), (33, 2048), (16, 2056),
                                    (40, 257)])
def test_split_gradient_planes_hold_the_fp32_gradient(cuda_device, rows, V):
    """The three bf16 planes of the readout's gradient sum to the fp32 gradient bit for bit
    (bf16 logits, ignored rows, an infinite logit's NaN row), and the bias partials to its
    column sums: rows fp32 additions of terms below 1, so rows * 2^-24 each."""
    from dabsn_amd import _lib
    from dabsn_amd.kernels import ops

    g = torch.Generator().manual_seed(rows * 10007 + V)
    x = (torch.randn(rows, V, generator=g) * 4).to(torch.bfloat16)
    if rows == 40:
        x[3, 5] = float("inf")
    t = torch.randint(0, V, (rows,), generator=g)
    t[::5] = -100
    x, t = x.to(cuda_device), t.to(cuda_device)
    lse, _ = ops.ce_rows(x, t, -100)
    scale = torch.tensor([0.37], device=cuda_device)
    want = ops.ce_rows_backward(x, t, -100, lse, scale)
    lib, ldp = _lib.load(), -(-V // 8) * 8
    planes = torch.zeros(3, rows, ldp, device=cuda_device, dtype=torch.bfloat16)
    part = torch.empty(lib.dabsn_hip_ce_split_parts(rows), V, device=cuda_device)
    word = torch.zeros(1, device=cuda_device, dtype=torch.int32)
    p = lambda v: v.data_ptr()  # noqa: E731
    assert lib.dabsn_hip_ce_split(rows, V, p(x), V, p(t), -100, p(lse), p(scale), p(planes),
                                  rows * ldp, ldp, p(part), p(word), None) == 0
    torch.cuda.synchronize()
    d = planes.double().sum(0)[:, :V]
    assert torch.equal(torch.nan_to_num(d, 7.0, 8.0, 9.0),
                       torch.nan_to_num(want.double(), 7.0, 8.0, 9.0))
    if rows != 40:  # there the NaN row leaves no finite column sum
        err = (part.double().sum(0) - want.double().sum(0)).abs().max()
        assert float(err) <= rows * 2.0 ** -24


@pytest.mark.gpu
def test_split_gradient_planes_below_their_exact_range(cuda_device):
    """Gradients of words whose logits lie up to 100 below the largest: the planes hold every
    bit of a value of at least 2^-110 and all but what lies below bf16's smallest subnormal,
    2^-133, of a smaller one."""
    from dabsn_amd import _lib
    from dabsn_amd.kernels import ops

    rows, V = 5, 808
    x = (-torch.arange(V, dtype=torch.float32) / 8).repeat(rows, 1)
    x = x.to(torch.bfloat16).to(cuda_device)
    t = torch.zeros(rows, dtype=torch.int64, device=cuda_device)
    lse, _ = ops.ce_rows(x, t, -100)
    scale = torch.tensor([0.37], device=cuda_device)
    want = ops.ce_rows_backward(x, t, -100, lse, scale).double()
    lib = _lib.load()
    planes = torch.zeros(3, rows, V, device=cuda_device, dtype=torch.bfloat16)
    word = torch.zeros(1, device=cuda_device, dtype=torch.int32)
    p = lambda v: v.data_ptr()  # noqa: E731
    assert lib.dabsn_hip_ce_split(rows, V, p(x), V, p(t), -100, p(lse), p(scale), p(planes),
                                  rows * V, V, None, p(word), None) == 0
    torch.cuda.synchronize()
    err = (planes.double().sum(0) - want).abs()
    exact = want.abs() >= 2.0 ** -110
    assert bool(exact.any()) and bool((~exact & (want != 0)).any())
    assert float(err[exact].max()) == 0 and float(err.max()) <= 2.0 ** -133


@pytest.mark.gpu
@pytest.mark.parametrize("N,V,H,budget,bias", [(1, 5, 3, None, True), (70, 33, 48, 16 * 33, True),
                                               (64, 129, 96, 16 * 129, False),
                                               (300, 1000, 200, 40 * 1000, True),
                                               (513, 4099, 73, 1 << 18, True)])
def test_bf16_readout_gradients_match_fp64(cuda_device, N, V, H, budget, bias):
    """One chunk, several chunks in a group, several groups with a shorter last one, odd
    vocabularies and widths: gradients against fp64 on the same bf16 values. The logits are
    rounded to bf16 (2^-9 of values up to about 5 standard deviations, an error of some
    1e-2 in a softmax weight, random over a row's terms) and the gradients once more
    (2^-9), so 1e-2 in the norm."""
    h, w, b, t = _case(N + V, 1, N, H, V, bias=bias, dtype=torch.bfloat16)
    t[:, ::7] = -100
    leaves = [None if x is None else x.to(cuda_device).requires_grad_(True) for x in (h, w, b)]
    loss = L.chunked_linear_cross_entropy(*leaves, t.to(cuda_device), chunk_budget=budget)
    loss.backward()
    ref_loss, ref = _naive(h, w, b, t)
    if t.ne(-100).any():
        assert abs(float(loss.detach()) - float(ref_loss)) <= 1e-2 * abs(float(ref_loss))
        for a, r in zip(leaves, ref):
            assert (a is None) == (r is None)
            if a is not None:
                assert a.grad.dtype == torch.bfloat16
                err = (a.grad.double().cpu() - r).norm() / r.norm()
                assert float(err) <= 1e-2
    else:  # every row ignored
        assert all(a is None or float(a.grad.float().abs().max()) == 0 for a in leaves)


def test_the_split_products_run_where_they_pay():
    """Small vocabularies, small weights and small calls keep the fp32 products."""
    for n, v, h in [(16384, 60, 64), (16384, 60, 2048), (16384, 400, 2048), (16384, 1024, 1024),
                    (8192, 2048, 256), (16384, 1300, 800), (256, 32000, 64), (300, 5001, 77), (0, 32000, 2048)]:
        assert not L._split_pays(n, v, h)
    for n, v, h in [(8192, 32000, 2048), (256, 32000, 2048), (6250, 32000, 64), (16384, 12000, 1024)]:
        assert L._split_pays(n, v, h)


@pytest.mark.gpu
@pytest.mark.parametrize("N,V,H,chunk,bias", [(1, 5, 3, 1, True), (70, 33, 48, 16, True),
                                              (64, 129, 96, 16, False), (300, 1000, 200, 40, True),
                                              (513, 4099, 73, 63, True), (40, 70, 6, 40, True)])
def test_split_products_match_the_fp32_ones(cuda_device, N, V, H, chunk, bias):
    """Both routes of the bf16 readout's backward at sizes of either: one chunk, chunks in a
    group, groups with a shorter last one, odd vocabularies and widths. Both products sum the
    same exact terms in fp32 (some 1e-6 apart) and round once to bf16: a value near the middle
    of two bf16 values rounds to either, 2^-8 of itself, so 2^-8 of the value."""
    from dabsn_amd.kernels import ops

    h, w, b, t = _case(N + V, 1, N, H, V, bias=bias, dtype=torch.bfloat16)
    h, t = h.reshape(N, H).to(cuda_device), t.reshape(N).to(cuda_device)
    w, b = w.to(cuda_device), None if b is None else b.to(cuda_device)
    t[::7] = -100
    lse, _ = ops.ce_rows(torch.nn.functional.linear(h, w, b), t, -100)
    scale = torch.tensor([0.37], device=cuda_device)
    gh, gw, gb = ops.linear_ce_backward_bf16(h, w, b, t, lse, scale, chunk, -100)
    d = torch.cat([ops.ce_rows_backward(torch.nn.functional.linear(h[s:s + chunk], w, b),
                                        t[s:s + chunk], -100, lse[s:s + chunk], scale)
                   for s in range(0, N, chunk)]).double()
    for got, want in ((gh, d @ w.double()), (gw, d.t() @ h.double())):
        err = (got.double() - want).abs()
        assert bool((err <= 2.0 ** -8 * want.abs() + 1e-6 * want.abs().max()).all())
        assert float(err.norm()) <= 2.0 ** -8 * float(want.norm())
    assert gb.numel() == (V if bias else 0)
    if bias:
        assert float((gb.double() - d.sum(0)).abs().max()) <= N * 2.0 ** -24


@pytest.mark.gpu
def test_split_products_bound_their_memory(cuda_device):
    """One chunk of many rows against few words: the products' copies (18 H bytes a row, 1.2 GB
    for these rows at once) stay within 512 MB beside the gradients (151 MB), the planes and
    logits (8 V bytes a row of a group) and the partials."""
    from dabsn_amd.kernels import ops

    N, V, H = 16384, 1024, 4096
    h = torch.randn(N, H, device=cuda_device).to(torch.bfloat16)
    w = torch.randn(V, H, device=cuda_device).to(torch.bfloat16)
    t = torch.randint(0, V, (N,), device=cuda_device)
    lse, scale = torch.zeros(N, device=cuda_device), torch.tensor([1e-9], device=cuda_device)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    base = torch.cuda.memory_allocated()
    ops.linear_ce_backward_bf16(h, w, None, t, lse, scale, N, -100)
    torch.cuda.synchronize()
    assert torch.cuda.max_memory_allocated() - base <= (512 << 20) + (192 << 20)


@pytest.mark.gpu
@pytest.mark.parametrize("N,V,H", [(50, 100, 64), (1500, 2048, 1024)])
def test_bf16_readout_backward_inside_autocast_keeps_fp32_products(cuda_device, N, V, H):
    """The gradients of a backward call inside a bf16 autocast region are those of one outside."""
    h, w, b, t = _case(N, 1, N, H, V, dtype=torch.bfloat16)
    grads = []
    for inside in (False, True):
        leaves = [x.to(cuda_device).requires_grad_(True) for x in (h, w, b)]
        with torch.autocast("cuda", torch.bfloat16, enabled=inside):
            L.chunked_linear_cross_entropy(*leaves, t.to(cuda_device)).backward()
        grads.append([x.grad for x in leaves])
    assert all(torch.equal(x, y) for x, y in zip(*grads))


@pytest.mark.gpu
def test_bf16_readout_reports_a_bad_target_in_any_chunk(cuda_device):
    h, w, b, t = _case(9, 1, 40, 16, 30, dtype=torch.bfloat16)
    t[0, 3] = 30
    with pytest.raises(RuntimeError, match="outside"):
        L.chunked_linear_cross_entropy(h.to(cuda_device), w.to(cuda_device), b.to(cuda_device),
                                       t.to(cuda_device), chunk_budget=8 * 30)
