"""Attention HIP kernels (MFMA and SIMT) vs the float64 oracle,
mirroring the reference's tests/tritium/test_attention.py (head dims, GQA,
non-causal, KV-cache decode, autograd) plus the module's strided layout, ragged
lengths, q_len != kv_len and head_dim 128.  Tolerance: bf16/fp16 max-abs 2e-2
(+2e-2 relative, as tests/_utils.py:14-17), fp32 1e-5."""

from __future__ import annotations

import importlib
import numpy as np
import pytest
import torch

import helion_amd as tritium
import oracle
from _helpers import DTYPES, assert_close, np32, randn

pytestmark = pytest.mark.gpu

ATOL = {torch.float32: 1e-5, torch.float16: 2e-2, torch.bfloat16: 2e-2}


def _check(dtype, b, h, hkv, tq, tkv, d, causal, seed=0, grads=True, layout="bhtd"):
    def make(n, t, s):
        if layout == "bthd":  # what helion.Attention passes: view(b, s, n, d).transpose(1, 2)
            return randn((b, t, n, d), dtype, s).transpose(1, 2)
        return randn((b, n, t, d), dtype, s)

    q, k, v = make(h, tq, seed), make(hkv, tkv, seed + 1), make(hkv, tkv, seed + 2)
    do = randn((b, h, tq, d), dtype, seed + 3)
    qs, ks, vs = (t.detach().requires_grad_(grads) for t in (q, k, v))
    o = tritium.attention(qs, ks, vs, is_causal=causal)
    eo, lse = oracle.attention.forward(np32(q), np32(k), np32(v), causal)
    tol = ATOL[dtype]
    assert_close(o, eo, tol, tol, "o")
    if not grads:
        return
    o.backward(do)
    edq, edk, edv = oracle.attention.backward(np32(do), np32(q), np32(k), np32(v), lse, causal)
    assert_close(qs.grad, edq, tol, tol, "dq")
    assert_close(ks.grad, edk, tol, tol, "dk")
    assert_close(vs.grad, edv, tol, tol, "dv")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("head_dim", [16, 32, 64, 128])
@pytest.mark.parametrize(("batch", "n_heads", "seq"), [(1, 4, 64), (2, 8, 128)])
def test_attention_forward_backward(dtype, head_dim, batch, n_heads, seq):
    _check(dtype, batch, n_heads, n_heads, seq, seq, head_dim, True)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("causal", [True, False])
def test_attention_head_dim_256(dtype, causal):
    # the MFMA path at head_dim 256 (forward kernel with one wavefront per SIMD,
    # dQ kernel, dV and dK as two passes): several tiles, GQA, ragged lengths
    _check(dtype, 2, 4, 4, 192, 192, 256, causal, seed=21)
    _check(dtype, 1, 4, 2, 77, 130, 256, causal, seed=22)
    _check(dtype, 1, 2, 2, 130, 70, 256, causal, seed=23, layout="bthd")


@pytest.mark.parametrize("dtype", DTYPES)
def test_attention_grouped_query(dtype):
    _check(dtype, 2, 8, 2, 128, 128, 64, True, seed=4)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("causal", [False, True])
def test_attention_ragged_and_unequal_lengths(dtype, causal):
    _check(dtype, 1, 2, 2, 77, 77, 64, causal, seed=7)
    _check(dtype, 1, 2, 1, 50, 200, 128, causal, seed=8)
    _check(dtype, 1, 2, 2, 200, 50, 32, causal, seed=9)


@pytest.mark.parametrize("dtype", DTYPES)
def test_attention_non_causal(dtype):
    _check(dtype, 1, 4, 4, 64, 64, 32, False, seed=10)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_attention_module_layout_strided(dtype):
    # the reference's strided-dq bug (attention.py:625-629 vs 645) must not recur
    _check(dtype, 2, 4, 4, 96, 96, 64, True, seed=11, layout="bthd")
    _check(dtype, 2, 4, 2, 130, 130, 128, True, seed=12, layout="bthd")


@pytest.mark.parametrize("dtype", DTYPES)
def test_attention_kv_cache_single_query(dtype):
    b, h, kv_len, d = 2, 4, 64, 32
    cache_k = randn((b, h, 80, d), dtype, 1)
    cache_v = randn((b, h, 80, d), dtype, 2)
    k, v = cache_k[:, :, :kv_len], cache_v[:, :, :kv_len]  # strided cache slices
    q = k[:, :, -1:, :].contiguous()
    o = tritium.attention(q, k, v, is_causal=False)
    eo, _ = oracle.attention.forward(np32(q), np32(k), np32(v), False)
    tol = 1e-4 if dtype == torch.float32 else 2e-2
    assert_close(o, eo, tol, tol)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize(("b", "h", "hkv", "kv_len"),
                         [(1, 4, 4, 1), (2, 8, 4, 7), (1, 6, 2, 300), (2, 16, 4, 5000),
                          (1, 8, 1, 2500), (3, 32, 32, 1030)])
def test_attention_decode_split_kv(dtype, head_dim, b, h, hkv, kv_len):
    # q_len 1 against strided cache slices takes the split-KV decode kernels (groups of 1,
    # 2, 3 (padded to 4), 4 and 8 query heads per kv head); o and lse against the oracle
    print(f"[decode] {dtype} d={head_dim} b={b} h={h} hkv={hkv} L={kv_len}", flush=True)
    cache_k = randn((b, hkv, kv_len + 40, head_dim), dtype, 3)
    cache_v = randn((b, hkv, kv_len + 40, head_dim), dtype, 4)
    k, v = cache_k[:, :, :kv_len], cache_v[:, :, :kv_len]
    q = randn((b, 1, h, head_dim), dtype, 5).transpose(1, 2)  # the module's layout
    o = tritium.attention(q, k, v, is_causal=False)
    eo, e_lse = oracle.attention.forward(np32(q), np32(k), np32(v), False)
    assert_close(o, eo, 2e-2, 2e-2, "o")
    from helion_amd.attention import _attention_forward
    _, lse = _attention_forward(q, k, v, False)
    assert_close(lse, e_lse, 1e-4, 1e-4, "lse")


def test_attention_decode_grads_through_general_backward():
    # the decode forward's (o, lse) feed the general backward kernels
    b, h, hkv, kv_len, d = 2, 8, 2, 333, 128
    q = randn((b, h, 1, d), torch.bfloat16, 7).requires_grad_(True)
    k = randn((b, hkv, kv_len, d), torch.bfloat16, 8).requires_grad_(True)
    v = randn((b, hkv, kv_len, d), torch.bfloat16, 9).requires_grad_(True)
    do = randn((b, h, 1, d), torch.bfloat16, 10)
    tritium.attention(q, k, v, is_causal=False).backward(do)
    eo, lse = oracle.attention.forward(np32(q), np32(k), np32(v), False)
    edq, edk, edv = oracle.attention.backward(np32(do), np32(q), np32(k), np32(v), lse, False)
    assert_close(q.grad, edq, 2e-2, 2e-2, "dq")
    assert_close(k.grad, edk, 2e-2, 2e-2, "dk")
    assert_close(v.grad, edv, 2e-2, 2e-2, "dv")


def test_attention_decode_workspace_cache_is_bounded():
    # one workspace per (device, stream), only the most recent few streams keep theirs;
    # each stream's decode still matches the oracle
    att = importlib.import_module("helion_amd.attention")
    b, h, hkv, kv_len, d = 1, 4, 2, 700, 64
    q = randn((b, h, 1, d), torch.bfloat16, 11)
    k = randn((b, hkv, kv_len, d), torch.bfloat16, 12)
    v = randn((b, hkv, kv_len, d), torch.bfloat16, 13)
    eo, _ = oracle.attention.forward(np32(q), np32(k), np32(v), False)
    streams = [torch.cuda.Stream() for _ in range(att._DECODE_WS_KEEP + 3)]
    for st in streams:
        st.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(st):
            o = tritium.attention(q, k, v, is_causal=False)
        torch.cuda.current_stream().wait_stream(st)
        assert_close(o, eo, 2e-2, 2e-2, "o")
        assert len(att._DECODE_WS) <= att._DECODE_WS_KEEP
    keys = list(att._DECODE_WS)
    assert keys[-1][1] == streams[-1].cuda_stream


def test_attention_large_head_bf16_t1024():
    _check(torch.bfloat16, 1, 2, 2, 1024, 1024, 128, True, seed=13)


@pytest.mark.parametrize("causal", [False, True])
def test_attention_gqa_many_tiles_ragged(causal):
    # several kv and query workgroups per head, GQA group of 4, length not a tile multiple
    _check(torch.bfloat16, 1, 8, 2, 700, 700, 128, causal, seed=14)
    _check(torch.float16, 2, 4, 1, 333, 333, 64, causal, seed=15)


# head_dim 128 backward: dK/dV store dS and dQ is formed from it (the default
# where the workspace fits), or the dQ kernel recomputes S and dP (workspace
# limit 0).  Both against the oracle: ragged tiles, Tq < Tkv and Tq > Tkv
# (the causal mask is top-left), GQA, a single row.
DS_SHAPES = [(1, 2, 2, 77, 77), (1, 2, 1, 50, 200), (1, 2, 1, 200, 50), (2, 4, 2, 333, 333),
             (1, 2, 2, 64, 64), (1, 1, 1, 1, 1), (1, 2, 2, 129, 127), (1, 4, 4, 384, 384)]


@pytest.mark.parametrize("head_dim", [128])
@pytest.mark.parametrize("stored", [True, False])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize(("b", "h", "hkv", "tq", "tkv"), DS_SHAPES)
def test_attention_backward_stored_and_recomputed_ds(monkeypatch, stored, causal, b, h, hkv, tq,
                                                     tkv, head_dim):
    A = importlib.import_module("helion_amd.attention")
    if not stored:
        monkeypatch.setattr(A, "DS_WORKSPACE_MAX_BYTES", 0)
    _check(torch.bfloat16, b, h, hkv, tq, tkv, head_dim, causal, seed=31 + tq + tkv)


@pytest.mark.parametrize("head_dim", [64, 128])
def test_attention_longest_first_order(head_dim):
    # causal grids whose (batch, head) count is a multiple of the 8 XCDs take their
    # tiles longest first across each XCD's slices (at head_dim 128 the dQ-from-dS
    # kernel in groups of four slices: 6 per XCD here, a group of 4 and one of 2);
    # the order must not change the results.  GQA: dK/dV over 24 kv slices.
    _check(torch.bfloat16, 2, 24, 24, 512, 512, head_dim, True, seed=41)
    _check(torch.bfloat16, 2, 24, 12, 512, 512, head_dim, True, seed=42)


def test_attention_persistent_dkdv_pairs():
    # head_dim 128 grids with >= 2 kv tiles per compute unit and (batch, kv head)s in
    # multiples of the 8 XCDs run the persistent dK/dV kernel, which deals the kv-tile
    # pairs (t, n - 1 - t) of each head round-robin: 4 kv tiles per head (2 pairs), then 5
    # (an odd count: the middle tile is a work unit of its own) and GQA over 128 kv heads
    _check(torch.bfloat16, 4, 32, 32, 512, 512, 128, True, seed=51)
    _check(torch.bfloat16, 4, 32, 32, 640, 640, 128, True, seed=52)
    _check(torch.bfloat16, 8, 32, 16, 512, 512, 128, True, seed=53)


def test_attention_stored_ds_deterministic_fp16():
    q = randn((2, 4, 300, 128), torch.float16, 1).requires_grad_(True)
    k = randn((2, 2, 300, 128), torch.float16, 2).requires_grad_(True)
    v = randn((2, 2, 300, 128), torch.float16, 3).requires_grad_(True)
    grads = []
    for _ in range(2):
        q.grad = k.grad = v.grad = None
        tritium.attention(q, k, v).sum().backward()
        grads.append((q.grad.clone(), k.grad.clone(), v.grad.clone()))
    for a, b in zip(*grads):
        assert torch.equal(a, b)


def test_attention_invariants():
    # T = 1 -> o = v; causal row 0 -> o[0] = v[0]; uniform v rows -> o = v
    q = randn((1, 2, 1, 64), torch.bfloat16, 1)
    k = randn((1, 2, 1, 64), torch.bfloat16, 2)
    v = randn((1, 2, 1, 64), torch.bfloat16, 3)
    assert torch.equal(tritium.attention(q, k, v), v)
    q = randn((1, 2, 130, 64), torch.bfloat16, 4)
    k = randn((1, 2, 130, 64), torch.bfloat16, 5)
    v = randn((1, 2, 1, 64), torch.bfloat16, 6).expand(1, 2, 130, 64).contiguous()
    o = tritium.attention(q, k, v)
    assert_close(o, np32(v), 1e-2, 1e-2)
    v2 = randn((1, 2, 130, 64), torch.bfloat16, 7)
    o2 = tritium.attention(q, k, v2)
    assert torch.equal(o2[:, :, 0], v2[:, :, 0])


def test_attention_deterministic():
    q = randn((1, 4, 256, 64), torch.bfloat16, 1).requires_grad_(True)
    k = randn((1, 4, 256, 64), torch.bfloat16, 2).requires_grad_(True)
    v = randn((1, 4, 256, 64), torch.bfloat16, 3).requires_grad_(True)
    grads = []
    for _ in range(2):
        q.grad = k.grad = v.grad = None
        tritium.attention(q, k, v).sum().backward()
        grads.append((q.grad.clone(), k.grad.clone(), v.grad.clone()))
    for a, b in zip(*grads):
        assert torch.equal(a, b)


def _check_heads(dtype, b, h, hkv, t, d, causal, heads, seed, grads=False):
    """Run the full (b, h, t, d) problem, check the listed (batch, kv head)
    slices -- with every query head of each kv head's group -- against the
    oracle (the problem is independent per (batch, kv head))."""
    group = h // hkv
    q, k, v = randn((b, h, t, d), dtype, seed), randn((b, hkv, t, d), dtype, seed + 1), \
        randn((b, hkv, t, d), dtype, seed + 2)
    do = randn((b, h, t, d), dtype, seed + 3)
    qs, ks, vs = (x.detach().requires_grad_(grads) for x in (q, k, v))
    o = tritium.attention(qs, ks, vs, is_causal=causal)
    if grads:
        o.backward(do)
    tol = ATOL[dtype]
    for bi, kh in heads:
        hq = slice(kh * group, (kh + 1) * group)
        sel = lambda x, hs: np32(x[bi:bi + 1, hs])  # noqa: E731
        eo, lse = oracle.attention.forward(sel(q, hq), sel(k, slice(kh, kh + 1)),
                                           sel(v, slice(kh, kh + 1)), causal)
        assert_close(o[bi:bi + 1, hq], eo, tol, tol, f"o[{bi},{kh}]")
        if grads:
            edq, edk, edv = oracle.attention.backward(
                sel(do, hq), sel(q, hq), sel(k, slice(kh, kh + 1)), sel(v, slice(kh, kh + 1)),
                lse, causal)
            assert_close(qs.grad[bi:bi + 1, hq], edq, tol, tol, f"dq[{bi},{kh}]")
            assert_close(ks.grad[bi:bi + 1, kh:kh + 1], edk, tol, tol, f"dk[{bi},{kh}]")
            assert_close(vs.grad[bi:bi + 1, kh:kh + 1], edv, tol, tol, f"dv[{bi},{kh}]")


# head_dim 128 problems with at least 4 workgroups of (256-row query tile
# pairs) per CU take the 8-wavefront ping-pong forward and dQ kernels; these
# grids (1024 workgroups) reach them on a 256-CU part, with one and with an
# odd number of query tiles, ragged lengths, GQA and the non-causal mask.
def test_attention_pingpong_grid():
    _check_heads(torch.bfloat16, 4, 256, 256, 256, 128, True,
                 [(0, 0), (1, 77), (3, 255)], seed=21, grads=True)
    _check_heads(torch.float16, 2, 256, 64, 731, 128, True, [(0, 0), (1, 63)], seed=22,
                 grads=True)
    _check_heads(torch.bfloat16, 2, 256, 256, 600, 128, False, [(0, 5), (1, 250)], seed=23)


# fp32 at head_dim 64 and 128 runs the fp32 matrix kernels: 64-row tiles (128
# query rows a workgroup in the head_dim 128 forward) swept by two wavefronts a
# row block, or four (head_dim 64, small grids).  Edges: rows and keys just over and
# under 32, 64 and 128, a half without keys, Tq != Tkv under the top-left mask, GQA,
# strided module views.  (Rows that see few others -- here a single key, or a single
# query in dK/dV -- and, further down, rows that are not 16-byte aligned take the SIMT
# kernels.)
# Tolerance 1e-5: fp32 sums of at most 300 terms of order 1.
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize(("b", "h", "hkv", "tq", "tkv", "layout"), [
    (1, 1, 1, 1, 1, "bhtd"), (1, 2, 2, 31, 33, "bhtd"), (2, 2, 1, 65, 63, "bthd"),
    (1, 4, 2, 129, 127, "bthd"), (1, 2, 2, 1, 300, "bhtd"), (1, 2, 1, 300, 20, "bhtd"),
    (4, 4, 2, 192, 192, "bthd"), (2, 8, 8, 257, 257, "bhtd")])
def test_attention_fp32_matrix_kernels(b, h, hkv, tq, tkv, layout, causal, head_dim):
    _check(torch.float32, b, h, hkv, tq, tkv, head_dim, causal, seed=61, layout=layout)


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_attention_fp32_few_rows(causal, head_dim):
    # rows that see few others take the SIMT kernels, each of forward, dQ and dK/dV by its
    # own count: both sides of every line (13 keys forward; 16 or 18 keys or queries
    # backward; one query of 16 keys in 512 heads), GQA, and keys past the last query's
    # block (zero gradients, no block computed)
    for h, hkv, tq, tkv in ((4, 2, 5, 200), (4, 4, 1, 200), (4, 1, 13, 13), (4, 4, 14, 14),
                            (4, 2, 16, 40), (4, 2, 17, 17), (4, 4, 18, 40), (4, 1, 19, 19),
                            (4, 2, 300, 13), (4, 4, 300, 17), (2, 2, 300, 19), (2, 2, 40, 300)):
        _check(torch.float32, 1, h, hkv, tq, tkv, head_dim, causal, seed=76)
    _check(torch.float32, 64, 8, 8, 1, 16, head_dim, causal, seed=77)


@pytest.mark.parametrize("causal", [False, True])
def test_attention_fp32_large_grid(causal):
    # 640 row tiles: two wavefronts a row block at head_dim 64 (four below 257 or 513)
    _check_heads(torch.float32, 8, 16, 16, 300, 64, causal, [(0, 0), (5, 3), (7, 15)], seed=75,
                 grads=True)


@pytest.mark.parametrize("head_dim", [64, 128])
def test_attention_fp32_hidden_rows_that_are_not_finite(head_dim):
    # keys and queries that the mask hides share 32-row blocks with visible ones and are
    # multiplied by zero weights there: what they hold must not reach the result.  Rows
    # that see no infinity or NaN equal the oracle on clean inputs
    x = [randn((1, 2, 100, head_dim), torch.float32, 140 + i) for i in range(4)]  # q, k, v, do
    eo, lse = oracle.attention.forward(*(np32(t) for t in x[:3]), True)
    edq, edk, edv = oracle.attention.backward(np32(x[3]), *(np32(t) for t in x[:3]), lse, True)

    def run(q, k, v, do):
        q, k, v = (t.detach().requires_grad_(True) for t in (q, k, v))
        o = tritium.attention(q, k, v)
        o.backward(do)
        return o, q.grad, k.grad, v.grad

    # a cache longer than the queries, its unwritten rows NaN: no query sees them
    k, v = (torch.cat([t, torch.full_like(t[:, :, :28], float("nan"))], 2) for t in x[1:3])
    o, dq, dk, dv = run(x[0], k, v, x[3])
    for got, want, name in ((o, eo, "o"), (dq, edq, "dq"), (dk[:, :, :100], edk, "dk"),
                            (dv[:, :, :100], edv, "dv")):
        assert_close(got, want, 1e-5, 1e-5, name)
    assert not dk[:, :, 100:].any() and not dv[:, :, 100:].any()
    # an infinite value and a NaN key: the rows before them
    k, v = x[1].clone(), x[2].clone()
    v[0, 0, 50, 3], k[0, 1, 52, 0] = float("inf"), float("nan")
    o, dq, _, _ = run(x[0], k, v, x[3])
    assert torch.isinf(o[0, 0, 50:, 3]).all() and torch.isnan(o[0, 1, 52:]).all()
    assert_close(o[:, :, :50], eo[:, :, :50], 1e-5, 1e-5, "o")
    assert_close(dq[:, :, :50], edq[:, :, :50], 1e-5, 1e-5, "dq")
    # a NaN gradient and an infinite query: the keys after them
    q, do = x[0].clone(), x[3].clone()
    do[0, :, 20], q[0, :, 80] = float("nan"), float("inf")
    _, _, dk, dv = run(q, x[1], x[2], do)
    assert torch.isnan(dv[0, :, :21]).all() and torch.isnan(dk[0, :, :81]).any(-1).all()
    assert_close(dk[:, :, 81:], edk[:, :, 81:], 1e-5, 1e-5, "dk")
    assert_close(dv[:, :, 81:], edv[:, :, 81:], 1e-5, 1e-5, "dv")
    do = x[3].clone()
    do[0, :, 42, 1] = float("inf")
    _, _, dk, dv = run(*x[:3], do)
    assert torch.isinf(dv[0, :, :43, 1]).all()
    assert_close(dk[:, :, 43:], edk[:, :, 43:], 1e-5, 1e-5, "dk")
    assert_close(dv[:, :, 43:], edv[:, :, 43:], 1e-5, 1e-5, "dv")
    # no mask, a last block that is not full: an infinite last value is an infinite output
    v = x[2].clone()
    v[0, 0, 99, 5] = float("inf")
    o = tritium.attention(x[0], x[1], v, is_causal=False)
    assert torch.isinf(o[0, 0, :, 5]).all() and torch.isfinite(o[0, 1]).all()


@pytest.mark.parametrize("head_dim", [64, 128])
def test_attention_fp32_values_near_the_largest(head_dim):
    # key 130 scores 5.4 above the keys before it: a weight of e^5.4 = 221 would take a
    # value of 2e36 past the largest float32, 3.4e38, which the running sum itself stays
    # below (at most 160 weights of 1, 3.2e38).  Every value is the same, so the output is
    # that value, within the roundings of a sum of 160 terms
    q = torch.zeros((1, 1, 64, head_dim), device="cuda")
    k = torch.zeros((1, 1, 160, head_dim), device="cuda")
    q[..., 0] = 1.0
    k[:, :, 130, 0] = 5.4 * head_dim ** 0.5
    v = torch.full((1, 1, 160, head_dim), 2e36, device="cuda")
    o = tritium.attention(q, k, v, is_causal=False)
    assert_close(o / 2e36, np.ones(o.shape), 160 * 2.0 ** -24, 0.0)


def test_attention_fp32_unaligned_rows():
    x = [randn((1, 2, 70, 67), torch.float32, 71 + i)[..., 1:65] for i in range(3)]
    o = tritium.attention(*x)
    eo, _ = oracle.attention.forward(*(np32(t) for t in x), True)
    assert_close(o, eo, 1e-5, 1e-5)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize(("b", "h", "hkv", "kv_len"), [
    (1, 3, 3, 1024), (1, 4, 2, 511), (2, 3, 3, 513), (9, 12, 12, 300),
    (2, 12, 3, 65), (1, 8, 1, 700), (1, 12, 4, 1025), (2, 16, 4, 4100), (40, 32, 8, 96)])
def test_attention_decode_routes(dtype, head_dim, b, h, hkv, kv_len):
    # one or two heads per kv head and up to 64 K elements of keys: one launch of 16
    # wavefronts; groups of 3 and more: the matrix-core kernel, whole and ragged 32-key tiles
    k, v = (randn((b, hkv, kv_len + 5, head_dim), dtype, 80 + i)[:, :, :kv_len] for i in range(2))
    q = randn((b, h, 1, head_dim), dtype, 82)
    o = tritium.attention(q, k, v, is_causal=False)
    eo, e_lse = oracle.attention.forward(np32(q), np32(k), np32(v), False)
    assert_close(o, eo, 2e-2, 2e-2, "o")
    from helion_amd.attention import _attention_forward
    _, lse = _attention_forward(q, k, v, False)
    assert_close(lse, e_lse, 1e-4, 1e-4, "lse")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize(("b", "h", "hkv", "kv_len"), [
    (65, 24, 8, 32), (65, 32, 8, 33), (65, 24, 8, 256), (65, 32, 8, 257), (2, 12, 4, 12),
    (2, 16, 4, 13), (33, 12, 4, 600), (33, 24, 4, 600), (257, 6, 2, 300)])
def test_attention_decode_groups_on_large_and_small_grids(dtype, head_dim, b, h, hkv, kv_len):
    # groups of 3, 4 and 6: short caches at head_dim 128 on the vector kernel (up to 32 or 256
    # keys where the kv heads fill the chip, 12 in fp16 else), chunks that fit the chip at once
    k, v = (randn((b, hkv, kv_len, head_dim), dtype, 80 + i) for i in range(2))
    q = randn((b, h, 1, head_dim), dtype, 82)
    o = tritium.attention(q, k, v, is_causal=False)
    eo, _ = oracle.attention.forward(np32(q), np32(k), np32(v), False)
    assert_close(o, eo, 2e-2, 2e-2, "o")


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize(("b", "h", "hkv", "kv_len"), [
    (128, 4, 2, 300), (129, 4, 2, 300), (257, 1, 1, 511)])
def test_attention_decode_one_launch_up_to_one_workgroup_a_unit(head_dim, b, h, hkv, kv_len):
    k, v = (randn((b, hkv, kv_len, head_dim), torch.bfloat16, 80 + i) for i in range(2))
    q = randn((b, h, 1, head_dim), torch.bfloat16, 82)
    o = tritium.attention(q, k, v, is_causal=False)
    eo, _ = oracle.attention.forward(np32(q), np32(k), np32(v), False)
    assert_close(o, eo, 2e-2, 2e-2, "o")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("e", [12, 20, 30, 36])
def test_attention_decode_small_weights(dtype, head_dim, e):
    # key 0 takes almost the whole weight and its value is zero: the output is made of
    # weights near 2^-e alone, which keep their fp32 precision in the groups' matrix kernel.
    # Bound: the rounding to 16 bits (2^-8 or 2^-11 of the value, 2^-25 where fp16 is
    # subnormal), and 2^-17 for the exponent of a weight formed in fp32 (scores up to 64)
    q, k = torch.zeros((1, 8, 1, head_dim)), torch.zeros((1, 2, 512, head_dim))
    q[..., 0], k[:, :, 0, 0] = 8.0, e * float(np.log(2.0)) * head_dim ** 0.5 / 8.0
    q[..., 1:9] = randn((1, 8, 1, 8), seed=93, device="cpu")
    k[:, :, 1:, 1:9] = randn((1, 2, 511, 8), seed=94, device="cpu", scale=0.3)
    v = randn((1, 2, 512, head_dim), seed=95, device="cpu").abs() * 40 * 2.0 ** min(e, 8)
    v[:, :, 0] = 0
    q, k, v = (t.to(dtype).cuda() for t in (q, k, v))
    o = tritium.attention(q, k, v, is_causal=False)
    eo, _ = oracle.attention.forward(np32(q), np32(k), np32(v), False)
    half_ulp = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert_close(o, eo, half_ulp + 2.0 ** -17, 2.0 ** -25 if dtype == torch.float16 else 0.0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("kv_len", [200, 517, 5000])
def test_attention_decode_every_score_minus_infinity(dtype, kv_len):
    # the same answer whatever the heads per kv head (vector and matrix kernels, one chunk
    # and several): an lse of NaN, an output of zero
    from helion_amd.attention import _attention_forward
    for hkv in (4, 2, 1):
        q = torch.ones((1, 4, 1, 64), dtype=dtype, device="cuda")
        k, v = (randn((1, hkv, kv_len, 64), dtype, 96 + i) for i in range(2))
        k[..., 0] = float("-inf")
        o, lse = _attention_forward(q, k, v, False)
        assert torch.isnan(lse).all() and not o.any(), hkv


def test_attention_decode_infinite_value():
    # an infinite value is an infinite output in its column, not a NaN (the split weights'
    # lower terms multiply it by zero or by a negative number)
    q, k = randn((1, 8, 1, 128), torch.bfloat16, 90), randn((1, 2, 3000, 128), torch.bfloat16, 91)
    v = randn((1, 2, 3000, 128), torch.bfloat16, 92)
    v[0, 1, 1234, 7] = float("inf")
    o = tritium.attention(q, k, v, is_causal=False)
    assert torch.isinf(o[0, 4:, 0, 7]).all()
    o[0, 4:, 0, 7] = 0
    v[0, 1, 1234, 7] = 0
    eo, _ = oracle.attention.forward(np32(q), np32(k), np32(v), False)
    eo[0, 4:, 0, 7] = 0
    assert_close(o, eo, 2e-2, 2e-2)


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_attention_forward_split_and_whole_tiles(head_dim, causal):
    # small grids take 64-row query tiles whose two wavefronts a row block sweep alternate
    # 32-key halves (a half without keys, without visible keys, ragged), at head_dim 128 from
    # two K/V tiles on; large ones 128-row tiles
    for tq, tkv in ((1, 31), (33, 33), (64, 96), (65, 97), (130, 64), (300, 40), (95, 128)):
        _check(torch.float16, 1, 4, 2, tq, tkv, head_dim, causal, seed=100, grads=False)
    _check(torch.bfloat16, 2, 3, 3, 257, 257, head_dim, causal, seed=101, layout="bthd")
    _check_heads(torch.bfloat16, 8, 32, 8, 301, head_dim, causal, [(0, 0), (7, 7)], seed=102)


@pytest.mark.parametrize("causal", [False, True])
def test_attention_backward_split_and_whole_tiles(causal):
    # small grids of more than one 128-row tile take 64-row workgroup tiles, two wavefronts a
    # row block on alternate 32-row halves of the tiles they sweep (a half out of range, masked
    # out, ragged); dQ and dK/dV decide separately, so one may split and the other not
    for tq, tkv in ((129, 31), (129, 129), (161, 300), (300, 161), (192, 256), (130, 1), (33, 700)):
        _check(torch.float16, 1, 4, 2, tq, tkv, 64, causal, seed=120)
    _check(torch.bfloat16, 2, 3, 3, 417, 417, 64, causal, seed=121, layout="bthd")
    _check(torch.bfloat16, 4, 32, 1, 140, 280, 64, causal, seed=122)  # no mask: dQ whole, dK/dV split
    _check_heads(torch.bfloat16, 5, 20, 20, 300, 64, causal, [(0, 0), (4, 19)], seed=123,
                 grads=True)  # whole tiles


@pytest.mark.parametrize("stored", [True, False])
@pytest.mark.parametrize("causal", [False, True])
def test_attention_split_pairs(monkeypatch, causal, stored):
    # head_dim 128, small grids: 64 kv rows a workgroup, two wavefront pairs a row block on
    # alternate halves of every query tile (a half out of range, masked out, ragged), with
    # and without the stored dS; (33, 33), a single step over one key tile, stays whole
    if not stored:
        monkeypatch.setattr(importlib.import_module("helion_amd.attention"), "DS_WORKSPACE_MAX_BYTES", 0)
    for tq, tkv in ((1, 129), (31, 200), (33, 33), (129, 129), (161, 300), (300, 161), (192, 256)):
        _check(torch.float16, 1, 4, 2, tq, tkv, 128, causal, seed=130)
    _check(torch.bfloat16, 2, 3, 3, 417, 417, 128, causal, seed=131, layout="bthd")
    _check_heads(torch.bfloat16, 5, 20, 20, 300, 128, causal, [(0, 0), (4, 19)], seed=132,
                 grads=True)  # 300 whole tiles: neither split nor persistent


@pytest.mark.parametrize("head_dim", [64, 128])
def test_attention_split_lines_at_unequal_lengths(head_dim):
    # where few keys meet many queries (or the reverse) under the causal mask the tiles are
    # alike (or see none), and whole tiles are taken up to smaller grids: shapes on either
    # side, in the forward, dQ and dK/dV
    for b, h, tq, tkv in ((1, 24, 1030, 70), (1, 8, 1030, 70), (1, 16, 64, 2100), (1, 4, 100, 2100),
                          (1, 6, 600, 2100), (1, 12, 1300, 1000), (2, 16, 63, 63), (1, 4, 200, 33)):
        _check(torch.bfloat16, b, h, h, tq, tkv, head_dim, True, seed=140)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_attention_order_over_uneven_slices(dtype):
    # causal grids whose slices do not divide over the 8 XCDs take their tiles rank by
    # rank over all slices: block counts that are and are not multiples of 8, GQA
    _check(dtype, 1, 12, 12, 260, 260, 64, True, seed=110)
    _check(dtype, 3, 4, 2, 520, 520, 128, True, seed=111)
    _check(dtype, 1, 20, 4, 390, 450, 64, True, seed=112)
