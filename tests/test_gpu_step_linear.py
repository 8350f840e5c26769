"""The block step's projections with what is folded into them
(block_step_linear, block_step_row_parts) against float64 torch, at the edges
of the 16 x 16 tiles, the 32-deep K slices and the K parts."""

from __future__ import annotations

import ctypes

import pytest
import torch

from spikegpt_myelin_amd import _lib

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)
# A sum of K fp32 products in another order: K 2^-24 of the sum of magnitudes
# bounds it; its square root is typical.
RTOL = 2e-6


def _rand(*shape, seed):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(DEV)


def _run(mode, xs, ws, outs, parts=1, extra=None):
    a = _lib.StepLinearArgs()
    for j, (x, w) in enumerate(zip(xs, ws)):
        a.x[j], a.w[j] = x.data_ptr(), w.data_ptr()
    for j, o in enumerate(outs):
        a.out[j] = o.data_ptr()
    a.batch, a.k, a.n0 = xs[0].shape[0], xs[0].shape[1], ws[0].shape[0]
    a.n1 = ws[1].shape[0] if mode == _lib.STEP_LINEAR_KEY_REC else 0
    for name, t in (extra or {}).items():
        setattr(a, name, t.data_ptr())
    lib = _lib.load()
    _lib.check(lib.block_step_linear(mode, ctypes.byref(a), parts,
                                     torch.cuda.current_stream().cuda_stream), "linear")
    torch.cuda.synchronize()


def _close(got, want):
    err = (got.double() - want).norm() / want.norm()
    assert float(err) < RTOL, f"{float(err):.2e}"


@pytest.mark.parametrize("B,K,N", [(1, 4, 1), (1, 128, 128), (15, 36, 20), (16, 768, 768),
                                   (17, 100, 33), (64, 768, 768), (130, 512, 96),
                                   (256, 256, 640)])
def test_plain_and_key_receptance(B, K, N):
    print(f"step linear B={B} K={K} N={N}", flush=True)
    x0, x1 = _rand(B, K, seed=1), _rand(B, K, seed=2)
    w0, w1 = _rand(4 * N, K, seed=3), _rand(N, K, seed=4)
    out = torch.full((B, N), 7.0, device=DEV)
    _run(_lib.STEP_LINEAR_PLAIN, [x1], [w1], [out])
    _close(out, x1.double() @ w1.double().t())
    key, rec = torch.empty(B, 4 * N, device=DEV), torch.empty(B, N, device=DEV)
    _run(_lib.STEP_LINEAR_KEY_REC, [x0, x1], [w0, w1], [key, rec])
    _close(key, torch.relu(x0.double() @ w0.double().t()).square())
    # (Another tile may split K over its waves differently: not bit for bit.)
    _close(rec, x1.double() @ w1.double().t())


@pytest.mark.parametrize("B,K,N,parts", [(1, 3072, 768, 4), (3, 100, 40, 2), (18, 2052, 68, 3),
                                         (64, 40, 16, 4)])
def test_parts_add_up(B, K, N, parts):
    # (64, 40, 16, 4): two K slices for four parts, so two parts are empty.
    print(f"step linear parts B={B} K={K} N={N} parts={parts}", flush=True)
    x, w = _rand(B, K, seed=5), _rand(N, K, seed=6)
    out = torch.full((parts, B, N), float("nan"), device=DEV)
    _run(_lib.STEP_LINEAR_PLAIN, [x], [w], [out], parts)
    want = x.double() @ w.double().t()
    _close(out.sum(0), want)
    # The row kernel adds them in order: residual + sum, without a LIF.
    res, mem, mem_out = _rand(B, N, seed=7), _rand(B, N, seed=8), torch.empty(B, N, device=DEV)
    got = res.clone()
    r = _lib.StepRowArgs()
    r.batch, r.channels, r.residual, r.add = B, N, got.data_ptr(), out.data_ptr()
    r.membrane_in, r.membrane_out, r.ln_eps = mem.data_ptr(), mem_out.data_ptr(), 1e-5
    lib = _lib.load()
    _lib.check(lib.block_step_row_parts(1, ctypes.byref(r), parts,
                                        torch.cuda.current_stream().cuda_stream), "row")
    torch.cuda.synchronize()
    total = out[0].clone()
    for p in range(1, parts):
        total += out[p]
    assert torch.equal(got, res + total) and torch.equal(mem_out, mem)
    assert 1 <= lib.block_step_linear_parts(B, K, N) <= 4


@pytest.mark.parametrize("B,C", [(1, 4), (2, 36), (16, 128), (33, 260)])
def test_kvr_equals_products_then_wkv_kernel(B, C):
    print(f"step kvr B={B} C={C}", flush=True)
    xs = [_rand(B, C, seed=10 + j) for j in range(3)]
    ws = [_rand(C, C, seed=20 + j) / C ** 0.5 for j in range(3)]
    td, tf = _rand(C, seed=30), _rand(C, seed=31)
    num, den, ls = _rand(B, C, seed=32), _rand(B, C, seed=33).abs() + 0.5, _rand(B, C, seed=34)
    state = [t.clone() for t in (num, den, ls)]
    out = torch.empty(B, C, device=DEV)
    names = ("num", "den", "ls")
    extra = {"time_decay": td, "time_first": tf}
    extra.update({f"{n}_in": t for n, t in zip(names, state)})
    extra.update({f"{n}_out": t for n, t in zip(names, state)})  # in place
    _run(_lib.STEP_LINEAR_KVR, xs, ws, [out], extra=extra)
    k, v, r = (x.double() @ w.double().t() for x, w in zip(xs, ws))
    n64, d64, l64 = num.double(), den.double(), ls.double()
    top = torch.maximum(l64, tf.double() + k)
    e1, e2 = torch.exp(l64 - top), torch.exp(tf.double() + k - top)
    want = torch.sigmoid(r) * (e1 * n64 + e2 * v) / (e1 * d64 + e2)
    dec = l64 - torch.exp(td.double())
    top = torch.maximum(dec, k)
    e1, e2 = torch.exp(dec - top), torch.exp(k - top)
    for got, ref in zip((out, *state), (want, e1 * n64 + e2 * v, e1 * d64 + e2, top)):
        _close(got, ref)


@pytest.mark.parametrize("B,K,C", [(1, 4, 4), (31, 60, 36), (33, 64, 512), (130, 772, 516),
                                   (256, 768, 768)])
def test_tiled_products(B, K, C):
    # THREE, and KEY_REC beyond 256 tiles: the edges of 32 x 32 tiles and of
    # 64-deep slabs.
    print(f"step gemm B={B} K={K} C={C}", flush=True)
    xs = [_rand(B, K, seed=40 + j) for j in range(3)]
    ws = [_rand(C, K, seed=50 + j) for j in range(3)]
    outs = [torch.full((B, C), 3.0, device=DEV) for _ in range(3)]
    _run(_lib.STEP_LINEAR_THREE, xs, ws, outs)
    for x, w, o in zip(xs, ws, outs):
        _close(o, x.double() @ w.double().t())
    if ((B + 15) // 16) * ((C + 15) // 16) > 256:
        wk = _rand(4 * C, K, seed=60)
        key, rec = torch.empty(B, 4 * C, device=DEV), torch.empty(B, C, device=DEV)
        _run(_lib.STEP_LINEAR_KEY_REC, xs[:2], [wk, ws[1]], [key, rec])
        _close(key, torch.relu(xs[0].double() @ wk.double().t()).square())
        assert torch.equal(rec, outs[1])


@pytest.mark.parametrize("B,K,N", [(1, 252, 5), (2, 260, 37), (3, 512, 40), (4, 772, 33),
                                   (1, 1024, 7), (2, 1028, 8), (4, 1032, 6), (3, 3072, 96),
                                   (1, 4096, 9), (2, 4356, 10)])
def test_few_rows(B, K, N):
    # One wave per dot product: the ends of 256-column pieces, of four of them,
    # and of the four waves' shares of a long K; rows and columns past the end.
    test_plain_and_key_receptance(B, K, N)


@pytest.mark.parametrize("B,C", [(1, 260), (2, 252), (3, 256), (4, 772), (4, 1028), (4, 128)])
def test_few_rows_kvr(B, C):
    test_kvr_equals_products_then_wkv_kernel(B, C)


def test_argument_errors():
    lib = _lib.load()
    a = _lib.StepLinearArgs()
    a.batch, a.k, a.n0 = 1, 6, 1
    assert lib.block_step_linear(0, ctypes.byref(a), 1, None) == 1
    a.k = 8
    assert lib.block_step_linear(0, ctypes.byref(a), 1, None) == 1  # null pointers
    assert lib.block_step_linear(1, ctypes.byref(a), 2, None) == 1  # parts: PLAIN only
    assert lib.block_step_linear(7, ctypes.byref(a), 1, None) == 1
