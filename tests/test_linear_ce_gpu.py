"""Fused linear-cross-entropy HIP kernels vs the float64 oracle, mirroring the
reference's tests/tritium/test_cross_entropy.py (dtypes, vocab sizes, row
counts, autograd, 3-D hidden) plus ignore_index, int32/int64 targets, ragged
and odd sizes, the multi-chunk backward and the W = 0 closed form.
Tolerance: north-star max-abs 2e-2 for 16-bit inputs (loss, dhidden,
dweight), 1e-4 for fp32; the reference's own loss test uses rtol 2e-2,
atol 2e-3 (tests/tritium/test_cross_entropy.py:73)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import helion_amd as tritium
import oracle
from _helpers import DTYPES, np32, randn

pytestmark = pytest.mark.gpu

ATOL = {torch.float32: 1e-4, torch.float16: 2e-2, torch.bfloat16: 2e-2}


def _inputs(n, d, v, dtype, seed=0, ignore_frac=0.0, tdtype=torch.int64, wscale=0.02):
    g = torch.Generator().manual_seed(seed)
    h = torch.randn((n, d), generator=g).to(dtype)
    w = (torch.randn((v, d), generator=g) * wscale).to(dtype)
    t = torch.randint(0, v, (n,), generator=g)
    k = int(round(n * ignore_frac))
    if k:
        t[torch.randperm(n, generator=g)[:k]] = -100
    return h.cuda(), w.cuda(), t.to(tdtype).cuda()


def _close(got, want, atol, what):
    got = np32(got).reshape(np.shape(want))
    err = float(np.max(np.abs(got - np.asarray(want, dtype=np.float64)))) if got.size else 0.0
    scale = float(np.max(np.abs(want))) if np.size(want) else 0.0
    assert err <= atol, f"{what}: max|err| {err:.3e} > {atol} (max|ref| {scale:.3e})"
    return err


def _run(n, d, v, dtype, seed=0, ignore_frac=0.0, tdtype=torch.int64, chunk_rows=0,
         wscale=0.02, backward=None):
    h, w, t = _inputs(n, d, v, dtype, seed, ignore_frac, tdtype, wscale)
    loss, lse = tritium.linear_ce._linear_cross_entropy_forward(h, w, t)
    ref_loss, ref_lse = oracle.linear_ce.forward(np32(h), np32(w), np32(t))
    tol = ATOL[dtype]
    _close(loss, ref_loss, tol, "loss")
    _close(lse, ref_lse, tol, "lse")
    g = torch.tensor(1.0, device="cuda")
    backward = backward or tritium.linear_ce._backward
    dh, dw = backward(g, h, w, t, lse, True, True, -100, chunk_rows)
    edh, edw = oracle.linear_ce.backward(1.0, np32(h), np32(w), np32(t), ref_lse)
    _close(dh, edh, tol, "dhidden")
    _close(dw, edw, tol, "dweight")
    # a scale-aware check: the gradients are small numbers, 2e-2 alone would pass zeros
    for got, want, name in ((dh, edh, "dhidden"), (dw, edw, "dweight")):
        ref = np.asarray(want, dtype=np.float64)
        rel = np.linalg.norm(np32(got).astype(np.float64) - ref) / max(np.linalg.norm(ref), 1e-30)
        assert rel < (2e-2 if dtype != torch.float32 else 1e-4), f"{name}: relative L2 {rel:.3e}"


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("vocab", [128, 1000, 1024])
@pytest.mark.parametrize("n_rows", [1, 16, 128])
def test_linear_ce_forward_backward(dtype, vocab, n_rows):
    _run(n_rows, 64, vocab, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
def test_linear_ce_ragged_and_ignore_index(dtype):
    _run(300, 96, 777, dtype, seed=3, ignore_frac=0.1)
    _run(129, 256, 2049, dtype, seed=4, ignore_frac=0.01, tdtype=torch.int32)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_linear_ce_multi_chunk_backward(dtype):
    # five vocab chunks of 256 rows: dhidden accumulates across chunks in fp32
    _run(200, 128, 1200, dtype, seed=5, ignore_frac=0.05, chunk_rows=256)


@pytest.mark.parametrize("need", [(True, False), (False, True)])
def test_linear_ce_backward_one_gradient(need):
    # tritium_linear_ce_bwd with only dhidden or only dweight requested (the
    # other pointer NULL), over several chunks
    h, w, t = _inputs(150, 64, 700, torch.bfloat16, seed=12, ignore_frac=0.05)
    loss, lse = tritium.linear_ce._linear_cross_entropy_forward(h, w, t)
    ref_loss, ref_lse = oracle.linear_ce.forward(np32(h), np32(w), np32(t))
    edh, edw = oracle.linear_ce.backward(1.0, np32(h), np32(w), np32(t), ref_lse)
    dh, dw = tritium.linear_ce._backward(torch.tensor(1.0, device="cuda"), h, w, t, lse,
                                         need[0], need[1], -100, 256)
    assert (dh is None) != need[0] and (dw is None) != need[1]
    if need[0]:
        _close(dh, edh, 2e-2, "dhidden")
    else:
        _close(dw, edw, 2e-2, "dweight")


def test_linear_ce_odd_hidden_size_is_padded():
    _run(40, 37, 300, torch.bfloat16, seed=6)
    _run(40, 37, 300, torch.float32, seed=6)


def test_linear_ce_autograd_3d_and_needs_input_grad():
    h, w, t = _inputs(2 * 33, 64, 500, torch.bfloat16, seed=7, ignore_frac=0.05)
    h3 = h.view(2, 33, 64).clone().requires_grad_(True)
    t2 = t.view(2, 33)
    wg = w.clone().requires_grad_(True)
    loss = tritium.linear_cross_entropy(h3, wg, t2)
    loss.backward(torch.tensor(0.5, device="cuda"))
    ref_loss, ref_lse = oracle.linear_ce.forward(np32(h), np32(w), np32(t))
    edh, edw = oracle.linear_ce.backward(0.5, np32(h), np32(w), np32(t), ref_lse)
    _close(loss, ref_loss, 2e-2, "loss")
    assert h3.grad.shape == (2, 33, 64)
    _close(h3.grad.view(-1, 64), edh, 2e-2, "dhidden")
    _close(wg.grad, edw, 2e-2, "dweight")
    # only the weight needs a gradient
    loss = tritium.linear_cross_entropy(h3.detach(), wg, t2)
    wg.grad = None
    loss.backward()
    _close(wg.grad, edw / 0.5, 2e-2, "dweight only")


def test_linear_ce_zero_weight_closed_form():
    # W = 0: loss = ln V, dH = 0, dW = (1/V - onehot)^T h / N_valid
    n, d, v = 64, 32, 100
    h, _, t = _inputs(n, d, v, torch.float32, seed=8, ignore_frac=0.25)
    w = torch.zeros((v, d), device="cuda")
    loss, lse = tritium.linear_ce._linear_cross_entropy_forward(h, w, t)
    assert abs(float(loss) - np.log(v)) < 1e-5
    dh, dw = tritium.linear_ce._backward(torch.tensor(1.0, device="cuda"), h, w, t, lse, True,
                                         True, -100)
    valid = np32(t) != -100
    onehot = np.zeros((n, v))
    onehot[np.nonzero(valid)[0], np32(t)[valid].astype(int)] = 1.0
    expect = ((1.0 / v - onehot) * valid[:, None]).T @ np32(h).astype(np.float64) / valid.sum()
    assert float(torch.abs(dh).max()) == 0.0
    _close(dw, expect, 1e-6, "dweight closed form")


def test_linear_ce_all_ignored_is_nan_with_zero_grads():
    h, w, t = _inputs(8, 32, 50, torch.float32, seed=9)
    t = torch.full_like(t, -100)
    loss, lse = tritium.linear_ce._linear_cross_entropy_forward(h, w, t)
    assert torch.isnan(loss)
    dh, dw = tritium.linear_ce._backward(torch.tensor(1.0, device="cuda"), h, w, t, lse, True,
                                         True, -100)
    assert float(dh.abs().max()) == 0.0 and float(dw.abs().max()) == 0.0


def test_linear_ce_matches_torch_library_routine():
    import torch.nn.functional as F

    h, w, t = _inputs(96, 128, 3000, torch.bfloat16, seed=10, ignore_frac=0.02)
    loss = tritium.linear_cross_entropy(h, w, t)
    ref = F.cross_entropy(F.linear(h.float(), w.float()), t, ignore_index=-100)
    torch.testing.assert_close(loss, ref, rtol=2e-2, atol=2e-3)


def test_linear_ce_deterministic():
    h, w, t = _inputs(256, 128, 2000, torch.bfloat16, seed=11)
    hs = h.clone().requires_grad_(True)
    ws = w.clone().requires_grad_(True)
    out = []
    for _ in range(2):
        hs.grad = ws.grad = None
        tritium.linear_cross_entropy(hs, ws, t).backward()
        out.append((hs.grad.clone(), ws.grad.clone()))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])


def test_linear_ce_empty_rows():
    h = torch.empty((0, 64), device="cuda", dtype=torch.bfloat16)
    w = torch.randn((10, 64), device="cuda").bfloat16()
    t = torch.empty((0,), device="cuda", dtype=torch.int64)
    assert float(tritium.linear_cross_entropy(h, w, t)) == 0.0


# ------------------------------------------------- MFMA backward edge cases
# The 16-bit backward (tritium_linear_ce_bwd) recomputes the logits per vocabulary
# chunk and runs dW = G^T H and dH = G W on the GEMM core with MN-contiguous
# operands (transposing LDS reads): tile edges in every dimension, vocab sizes
# that are not a multiple of 8 (the last granule of a G row is padding), token
# counts that leave a partial K tile, and one to several chunks.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,d,v,ignore_frac,tdtype,chunk", [
    (1, 32, 128, 0.0, torch.int64, 0),
    (130, 64, 1001, 0.1, torch.int32, 0),     # vocab not a multiple of 8
    (257, 128, 2049, 0.05, torch.int64, 0),   # past the 256-token and 256-vocab tile edges
    (64, 40, 300, 0.0, torch.int64, 0),       # hidden_size padded to 48
    (300, 264, 1537, 0.02, torch.int64, 512), # 3 chunks, the last one 513 rows
    (513, 96, 640, 0.0, torch.int32, 256),    # K tiles of 64 tokens plus a partial one
    (300, 264, 5000, 0.02, torch.int64, 0),   # dH split over K (4 fp32 partials, summed in order)
    (2100, 64, 600, 0.01, torch.int64, 0),    # dW split over the tokens (2 partials)
    (300, 64, 6000, 0.0, torch.int32, 2560),  # 3 chunks with dH split in 2
])
def test_linear_ce_mfma_backward_edges(dtype, n, d, v, ignore_frac, tdtype, chunk):
    print(f"[lce bwd] {dtype} n={n} d={d} v={v} chunk={chunk}", flush=True)
    _run(n, d, v, dtype, seed=20, ignore_frac=ignore_frac, tdtype=tdtype, chunk_rows=chunk)


def _row_errors(got, want):
    """Relative error of every row (2-norm over the row's, at least the mean row's)."""
    norm = want.norm(dim=1)
    return (got.float() - want).norm(dim=1) / norm.clamp(min=float(norm.mean()))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,d,v,chunk", [
    (2100, 768, 50257, 0),      # dW: 591 tiles, 512 in two rounds and ragged rows over 2 token ranges
    (8300, 2048, 20001, 0),     # dW and dH (264 tiles, 8 of them over the vocabulary)
    (8300, 2048, 20001, 16384), # the same, dH summed over two chunks of unlike length
])
def test_linear_ce_backward_whole_rounds_and_split_rest(dtype, n, d, v, chunk):
    # grids with a badly filled last round: the rows of whole rounds in one product, the
    # others split over the reduction; every row against fp32 products.  G and the result
    # are rounded to 16 bits (2^-8 of a value at most, in bf16): 2^-8 for each, and as much
    # for the sums.  The loss is scaled by 2^14, as training in fp16 does: the entries of G
    # (1 / (v n) = 1e-8 here) would be subnormal in fp16
    print(f"[lce bwd] {dtype} n={n} d={d} v={v} chunk={chunk}", flush=True)
    h, w, t = _inputs(n, d, v, dtype, seed=30, ignore_frac=0.01)
    _, lse = tritium.linear_ce._linear_cross_entropy_forward(h, w, t)
    dh, dw = tritium.linear_ce._backward(torch.tensor(2.0 ** 14, device="cuda"), h, w, t, lse,
                                         True, True, -100, chunk)
    hf, wf = h.float(), w.float()
    keep = t != -100
    g = torch.softmax(hf @ wf.t(), 1)
    g[keep.nonzero()[:, 0], t[keep]] -= 1.0
    g *= (2.0 ** 14 * keep / keep.sum())[:, None]
    for got, want, name in ((dw, g.t() @ hf, "dweight"), (dh, g @ wf, "dhidden")):
        err = _row_errors(got, want)
        assert float(err.max()) < 3 * 2.0 ** -8, f"{name} row {int(err.argmax())}: {float(err.max()):.3e}"


@pytest.mark.parametrize("n,d,v,chunk", [
    (300, 64, 6200, 3072),   # dH over 3 ranges; the last chunk (56 rows) fills one of them
    (300, 64, 10400, 5120),  # 5 ranges; the last chunk (160 rows) three
])
def test_linear_ce_backward_last_chunk_with_fewer_ranges(n, d, v, chunk):
    _run(n, d, v, torch.bfloat16, seed=31, ignore_frac=0.02, chunk_rows=chunk)


def test_linear_ce_confident_targets():
    # targets at each row's arg-max with large logits: p(target) is close to 1 and the
    # target entry of G is a small difference p - 1
    n, d, v = 128, 64, 777
    h, w, _ = _inputs(n, d, v, torch.bfloat16, seed=21, wscale=1.5)
    t = (h.float() @ w.float().t()).argmax(dim=1)
    loss, lse = tritium.linear_ce._linear_cross_entropy_forward(h, w, t)
    ref_loss, ref_lse = oracle.linear_ce.forward(np32(h), np32(w), np32(t))
    assert float(loss) < 0.5  # most rows have p(target) near 1
    dh, dw = tritium.linear_ce._backward(torch.tensor(1.0, device="cuda"), h, w, t, lse, True,
                                         True, -100)
    edh, edw = oracle.linear_ce.backward(1.0, np32(h), np32(w), np32(t), ref_lse)
    for got, want, name in ((dh, edh, "dhidden"), (dw, edw, "dweight")):
        ref = np.asarray(want, dtype=np.float64)
        rel = np.linalg.norm(np32(got).astype(np.float64) - ref) / max(np.linalg.norm(ref), 1e-30)
        assert rel < 2e-2, f"{name}: relative L2 {rel:.3e}"


def test_linear_ce_chunking_only_changes_dhidden_rounding():
    # one chunk vs four: dweight's rows are the same products (bitwise; 512 tokens are never
    # split, the test below is of more), dhidden differs only by the fp32 accumulation
    # across chunks before its one rounding
    h, w, t = _inputs(512, 256, 1024, torch.bfloat16, seed=22, ignore_frac=0.03)
    loss, lse = tritium.linear_ce._linear_cross_entropy_forward(h, w, t)
    g = torch.tensor(0.75, device="cuda")
    dh1, dw1 = tritium.linear_ce._backward(g, h, w, t, lse, True, True, -100, 1024)
    dh4, dw4 = tritium.linear_ce._backward(g, h, w, t, lse, True, True, -100, 256)
    assert torch.equal(dw1, dw4)
    x, y = dh4.double(), dh1.double()
    assert float((x - y).norm() / y.norm()) < 5e-3


def test_linear_ce_chunking_does_not_change_split_dweight_rows():
    # tokens enough to split (8300), chunks of two rounds of tiles and more: rows past the
    # whole rounds of the vocabulary's tiles are split over the tokens, the same rows in the
    # same ranges however the vocabulary is cut (one chunk; two with the boundary inside the
    # split rows or at their start)
    h, w, t = _inputs(8300, 2048, 20001, torch.bfloat16, seed=32, ignore_frac=0.03)
    _, lse = tritium.linear_ce._linear_cross_entropy_forward(h, w, t)
    g = torch.tensor(0.75, device="cuda")
    dh1, dw1 = tritium.linear_ce._backward(g, h, w, t, lse, True, True, -100, 0)
    for chunk in (18432, 17408, 16384):
        dh, dw = tritium.linear_ce._backward(g, h, w, t, lse, True, True, -100, chunk)
        assert torch.equal(dw, dw1), chunk
        assert float((dh.double() - dh1.double()).norm() / dh1.double().norm()) < 5e-3, chunk


def test_linear_ce_autograd_keeps_no_logit_buffer_and_retain_graph():
    h, w, t = _inputs(200, 64, 900, torch.bfloat16, seed=23, ignore_frac=0.1)
    hs, ws = h.clone().requires_grad_(True), w.clone().requires_grad_(True)
    loss = tritium.linear_cross_entropy(hs, ws, t) * 3.0
    # what the forward keeps for the backward: the inputs and the fp32 lse only
    saved = loss.grad_fn.next_functions[0][0].saved_tensors
    assert [tuple(x.shape) for x in saved] == [(200, 64), (900, 64), (200,), (200,)]
    loss.backward(retain_graph=True)
    g1 = (hs.grad.clone(), ws.grad.clone())
    loss.backward()
    for first, total in zip(g1, (hs.grad, ws.grad)):
        assert torch.equal(total, 2 * first)
    import torch.nn.functional as F
    hr, wr = h.float().requires_grad_(True), w.float().requires_grad_(True)
    (F.cross_entropy(hr @ wr.t(), t, ignore_index=-100) * 3.0).backward()

    def rel(a, b):
        a, b = a.double(), b.double()
        return float((a - b).norm() / b.norm())

    assert rel(g1[0], hr.grad) < 2e-2 and rel(g1[1], wr.grad) < 2e-2
