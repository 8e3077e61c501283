"""Attention over bf16 rows (tq_dense_attention) against fp64 softmax attention:
tile and split edges, every mask form, strided operands, position bounds, continued splits, and
the routes of the chunked path and the dense-buffer merge onto it."""

import math

import pytest
import torch

from turboquant.runtime import attention as A
from turboquant.runtime import kernels as K
from turboquant.runtime.packed_qmse_cache import PackedMSELayer
from turboquant.runtime.synthetic import kv_bf16

pytestmark = pytest.mark.gpu

D = 128
SCALE = 1.0 / math.sqrt(D)
#: fp32 logits (128 exact products, error <= 128 * 2^-24 * sum |q k| / sqrt(D)), weights and sums:
#: with |logits| below ~10 the weights are within 1e-6, the normalised output within 1e-5 of its maximum
TOL32 = 1e-5


def randn(shape, seed, dtype=torch.float32):
    return torch.randn(shape, generator=torch.Generator(device="cuda").manual_seed(seed), device="cuda").to(dtype)


def oracle(q, k, v, add):
    """fp64 attention; add [B or 1, Q or 1, Sq or 1, n] additive (or None); rows without tokens are 0."""
    g = q.shape[1] // k.shape[1]
    lg = q.double() @ k.double().repeat_interleave(g, 1).transpose(-1, -2) * SCALE
    if add is not None:
        lg = lg + add.double()
    m = lg.amax(-1, keepdim=True)
    p = torch.exp(lg - torch.where(torch.isfinite(m), m, torch.zeros_like(m)))
    return (p @ v.double().repeat_interleave(g, 1)) / p.sum(-1, keepdim=True).clamp(min=1e-30)


def check(got, ref, dtype):
    tol = TOL32 if dtype == torch.float32 else 2 ** -8  # bf16 output: half an ulp of the largest value
    assert got.dtype == dtype and got.shape == ref.shape
    assert torch.isfinite(got).all()
    assert (got.double() - ref).abs().max() <= tol * ref.abs().max()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("B,Hkv,g,Sq,n,mask,splits", [
    (1, 1, 1, 1, 1, None, 1), (2, 2, 4, 1, 31, "bool", 1), (1, 2, 5, 3, 32, "f32", 1), (2, 1, 16, 2, 33, "lowest", 2),
    (1, 2, 4, 9, 1000, "bool", 7), (2, 2, 7, 9, 129, "heads", 3), (1, 1, 4, 33, 4097, None, 64),
    (1, 2, 2, 100, 257, "row", 9),
])
def test_dense_attention_matches_fp64(cuda, dtype, B, Hkv, g, Sq, n, mask, splits):
    q = randn((B, Sq, Hkv * g, D), 1, dtype).transpose(1, 2)  # strided over heads and tokens
    buf = randn((B, Hkv, n + 5, 2 * D), 2, torch.bfloat16)
    k, v = buf[:, :, 2:n + 2, :D], buf[:, :, 3:n + 3, D:]
    add = m = None
    if mask in ("bool", "heads"):
        m = randn((B, Hkv * g if mask == "heads" else 1, Sq, n + 3), 3)[..., 3:] > -0.5  # odd byte offsets
        m[0, 0, 0] = False  # a row with nothing attended
        add = torch.zeros(m.shape, device="cuda").masked_fill(~m, float("-inf"))
    elif mask == "f32":
        m = add = randn((B, 1, Sq, n), 3)
    elif mask == "row":
        m = add = randn((1, 1, 1, n), 3)
    elif mask == "lowest":  # finite masks of the type's lowest value: a row of them is an even average
        add = torch.zeros((B, 1, Sq, n), device="cuda")
        add[:, :, :, ::3] = torch.finfo(torch.float32).min
        add[1] = torch.finfo(torch.float32).min
        m = add
    got = K.DenseAttention(q, Hkv, splits).add(k, v, n, 0, splits, SCALE, mask=m, out=dtype)
    ref = oracle(q, k, v, add)
    if mask == "lowest":
        ref[1] = v[1].double().mean(1).repeat_interleave(g, 0)[:, None]
    check(got, ref, dtype)


@pytest.mark.parametrize("Sq,n", [(1, 1), (1, 40), (40, 70)])
def test_an_infinite_value_stays_infinite(cuda, Sq, n):
    """A weight of few bits (1 for a single token, 1 / n for equal keys) has zero lower terms."""
    q, k = randn((1, 4, Sq, D), 1, torch.bfloat16), torch.zeros((1, 1, n, D), dtype=torch.bfloat16, device="cuda")
    v = randn((1, 1, n, D), 2, torch.bfloat16)
    v[0, 0, n // 2, 5] = float("inf")
    v[0, 0, n - 1, 7] = float("-inf")
    out = K.DenseAttention(q, 1, 1).add(k, v, n, 0, 1, SCALE, out=torch.float32)
    assert (out[..., 5] == float("inf")).all() and (out[..., 7] == float("-inf")).all()
    rest = [d for d in range(D) if d not in (5, 7)]
    check(out[..., rest], oracle(q, k, v[..., rest], None), torch.float32)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("Sq", [1, 12, 40])  # one, two and four waves per workgroup
@pytest.mark.parametrize("form", ["key", "few bits", "query"])
def test_infinite_products_keep_their_sign(cuda, dtype, Sq, form):
    """Logits of -inf leave their token out, whatever terms an fp32 query is held in (a query element of
    few bits has zero lower terms, an infinity no others); +inf makes NaN of its row and no other."""
    n, tok = 70, 37
    q, k, v = randn((1, 4, Sq, D), 1, dtype), randn((1, 1, n, D), 2, torch.bfloat16), randn((1, 1, n, D), 3, torch.bfloat16)
    add = torch.zeros(1, 1, 1, n, device="cuda")
    if form == "query":  # head 1: -inf for every token
        k[..., 7] = -1.0 - k[..., 7].abs()
        q[0, 1, :, 7] = float("inf")
        out = K.DenseAttention(q, 1, 1).add(k, v, n, 0, 1, SCALE, out=torch.float32)
        assert (out[0, 1] == 0).all()  # nothing attended
        q[0, 1, :, 7] = float("-inf")
        assert K.DenseAttention(q, 1, 1).add(k, v, n, 0, 1, SCALE, out=torch.float32)[0, 1].isnan().all()
    else:
        k[0, 0, tok, 9] = float("-inf")
        q[..., 9] = 1.5 if form == "few bits" else q[..., 9].abs() + 0.1
        q[0, 1, :, 9] *= -1
        add[..., tok] = float("-inf")
        out = K.DenseAttention(q, 1, 1).add(k, v, n, 0, 1, SCALE, out=torch.float32)
        assert out[0, 1].isnan().all()
    heads = [0, 2, 3]
    k = k.masked_fill(k.isinf(), 0.0)
    q = q.masked_fill(q.isinf(), 0.0)
    check(out[:, heads], oracle(q[:, heads], k, v, add), torch.float32)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("Sq", [1, 12, 40])  # one, two and four waves per workgroup
@pytest.mark.parametrize("tok", [3, 140, 299])  # in the first, the second and the last range
def test_an_infinite_value_in_continued_partials(cuda, dtype, Sq, tok):
    """The second walk of a range starts from the partials it was given, whole or already infinite."""
    n = 300
    q, k, v = randn((1, 4, Sq, D), 1, dtype), randn((1, 1, n, D), 2, torch.bfloat16), randn((1, 1, n, D), 3, torch.bfloat16)
    v[0, 0, tok, 5], v[0, 0, tok, 7] = float("inf"), float("-inf")
    att = K.DenseAttention(q, 1, 2)
    for a, b in ((0, 128), (128, 200), (200, n)):
        out = att.add(k[:, :, a:b], v[:, :, a:b], b - a, 0, 2, SCALE, accumulate=a > 0,
                      out=torch.float32 if b == n else None)
    assert (out[..., 5] == float("inf")).all() and (out[..., 7] == float("-inf")).all()
    rest = [d for d in range(D) if d not in (5, 7)]
    check(out[..., rest], oracle(q, k, v[..., rest], None), torch.float32)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("Sq", [1, 12, 40])  # one, two and four waves per workgroup
@pytest.mark.parametrize("form", ["mask", "bounds", "far below", "faint"])
def test_values_of_unattended_tokens_add_nothing(cuda, dtype, Sq, form):
    """A weight of 0 (masked, out of bounds, 2^-x that underflows) leaves out a value of the type's
    largest magnitude; a faint one (2^-120) adds its product, beside an infinity elsewhere in the tile."""
    n, tok = 70, 37
    q, k = randn((1, 4, Sq, D), 1, dtype), torch.zeros((1, 1, n, D), dtype=torch.bfloat16, device="cuda")
    v = randn((1, 1, n, D), 2, torch.bfloat16)
    v[0, 0, tok, 6], v[0, 0, tok, 9] = torch.finfo(torch.bfloat16).max, -torch.finfo(torch.bfloat16).max
    v[0, 0, tok + 1, 5] = float("inf")
    add, kw = torch.zeros(1, 1, 1, n, device="cuda"), {}
    if form == "mask":
        add[..., tok] = float("-inf")
        kw["mask"] = add == 0
    elif form == "bounds":
        add[..., :tok + 1] = float("-inf")
        kw["starts"] = torch.tensor([tok + 1], dtype=torch.int32, device="cuda")
        kw["ends"] = torch.tensor([n], dtype=torch.int32, device="cuda")
    else:
        q[..., 0] = 16.0
        k[0, 0, tok, 0] = -200.0 if form == "far below" else -58.75  # logits of -283 and -83.1
    out = K.DenseAttention(q, 1, 1).add(k, v, n, 0, 1, SCALE, out=torch.float32, **kw)
    assert (out[..., 5] == float("inf")).all()
    rest = [d for d in range(D) if d != 5]
    ref = oracle(q, k, v[..., rest], add)
    # a logit of 83 is rounded at 2^-24 of it, twice: 1e-5 of a faint weight, 2e-5 with exp2's own error;
    # and a weight's third term ends at 2^-133, the last bit of bf16
    err = (out[..., rest].double() - ref).abs().amax((0, 1, 2))
    scale = ref.abs().amax((0, 1, 2))
    if form == "faint":
        last = 2.0 ** -133 * v[..., rest].abs().double().amax((0, 1, 2)) / (n - 1)
        assert (err <= 4e-5 * scale.clamp(min=1.0) + last).all()
    else:
        assert (err <= TOL32 * scale.clamp(min=1.0)).all()


@pytest.mark.parametrize("Sq", [1, 20])
def test_position_bounds_continued_partials_and_another_part(cuda, Sq):
    B, Hkv, g, n = 3, 2, 4, 300
    q, k, v = (randn(s, 5 + i, torch.bfloat16) for i, s in
               enumerate([(B, Hkv * g, Sq, D), (B, Hkv, n, D), (B, Hkv, n, D)]))
    starts = torch.tensor([0, 150, 90], dtype=torch.int32, device="cuda")
    ends = torch.tensor([400, 333, 90], dtype=torch.int32, device="cuda")  # the last row attends to nothing
    pos = torch.arange(n, device="cuda") + 100
    ok = (pos >= starts[:, None]) & (pos < ends[:, None])
    add = torch.zeros(B, 1, 1, n, device="cuda").masked_fill(~ok[:, None, None], float("-inf"))
    att = K.DenseAttention(q, Hkv, 4)
    for a, b in ((0, 128), (128, 131), (131, n)):  # the same splits over three ranges, one almost empty
        got = att.add(k[:, :, a:b], v[:, :, a:], b - a, 0, 4, SCALE, starts=starts, ends=ends, pos0=100 + a,
                      accumulate=a > 0, out=torch.float32 if b == n else None)
    check(got, oracle(q, k, v, add), torch.float32)
    # the first 100 tokens as another part, the rest as partials
    lg = (q.float() @ k[:, :, :100].float().repeat_interleave(g, 1).transpose(-1, -2)) * SCALE
    prev = torch.softmax(lg, -1) @ v[:, :, :100].float().repeat_interleave(g, 1)
    got = K.DenseAttention(q, Hkv, 2).add(k[:, :, 100:], v[:, :, 100:], n - 100, 0, 2, SCALE, out=torch.float32, prev=prev,
                                          prev_lse=torch.logsumexp(lg, -1))
    check(got, oracle(q, k, v, None), torch.float32)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_chunked_native_route_agrees_with_torch_operations(cuda, dtype, monkeypatch):
    """Packed history in several segments, a dense buffer and new tokens under a mask wider than the
    tokens, against the torch operations of the same function (taken when autograd is on)."""
    B, Hq, Hkv, N, nd, Sq = 2, 8, 2, 1500, 7, 5
    layer = PackedMSELayer(bits=3, quantize_decode=False)
    layer.initialize_from_dense(kv_bf16((B, Hkv, N, D), seed=1), kv_bf16((B, Hkv, N, D), seed=2))
    layer._lazy_update = True
    layer.update(kv_bf16((B, Hkv, nd, D), seed=3), kv_bf16((B, Hkv, nd, D), seed=4))
    nk, nv = kv_bf16((B, Hkv, 3, D), seed=5), kv_bf16((B, Hkv, 3, D), seed=6)
    q = randn((B, Hq, Sq, D), 7, dtype)
    mask = randn((B, 1, Sq, N + nd + 9), 8) > -1.0
    monkeypatch.setattr(A, "_ROW_BYTES", 700 * B * Hkv * D * 4)
    kw = dict(new_key=nk, new_value=nv, n_kv_groups=Hq // Hkv, attention_mask=mask, chunk_size=64)
    native = A._native_chunked
    calls = []
    monkeypatch.setattr(A, "_native_chunked", lambda *a: calls.append(1) or native(*a))
    got = A.chunked_turboquant_attention(q, layer, **kw)
    assert calls
    qg = q.clone().requires_grad_()
    ref = A.chunked_turboquant_attention(qg, layer, **kw)
    assert len(calls) == 1 and ref.requires_grad
    check(got, ref.detach().double(), dtype)


def test_calls_beyond_the_grid_take_torch_operations(cuda, monkeypatch):
    """65536 KV heads of a batch, then both routes with the limit lowered."""
    B, Hkv, n = 8192, 8, 2
    q, k, v = (randn((B, Hkv, s, D), i, torch.bfloat16) for i, s in enumerate((1, n, n)))
    got = A.chunked_turboquant_attention(q, PackedMSELayer(bits=3), new_key=k, new_value=v)
    check(got, oracle(q, k, v, None), torch.bfloat16)
    del q, k, v

    layer = PackedMSELayer(bits=3, quantize_decode=False)
    layer.initialize_from_dense(kv_bf16((2, 2, 300, D), seed=1), kv_bf16((2, 2, 300, D), seed=2))
    layer._lazy_update = True
    layer.update(kv_bf16((2, 2, 5, D), seed=3), kv_bf16((2, 2, 5, D), seed=4))
    q = randn((2, 8, 1, D), 7, torch.bfloat16)
    calls, add = [], K.DenseAttention.add
    monkeypatch.setattr(K.DenseAttention, "add", lambda *a, **kw: calls.append(1) or add(*a, **kw))
    for route in (lambda: A.fused_attention(q, layer, 4),
                  lambda: A.chunked_turboquant_attention(q, layer, n_kv_groups=4)):
        calls.clear()
        native = route()
        assert calls
        calls.clear()
        with monkeypatch.context() as m:
            m.setattr(K.DenseAttention, "MAX_BLOCKS", 3)
            ref = route()
        assert not calls
        check(native, ref.double(), torch.bfloat16)
