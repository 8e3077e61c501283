"""Prefill encoder (bf16 products, fp32 chains where a bound leaves the result open) against the CPU
oracle, bit for bit, where its bounds are put to the test: outputs exactly on a boundary by the
hundred per vector, vectors whose squares under- or overflow, zeros, infinities and NaN among
ordinary ones, sizes off the tiles, every width and group size."""

import numpy as np
import pytest
import torch

from oracle import oracle as O
from turboquant.runtime import kernels as K
from turboquant.runtime.params import layer_codecs, split_codecs
from turboquant.runtime.synthetic import kv_bf16

pytestmark = pytest.mark.gpu

D = 128


def u16(t):
    return t.contiguous().view(torch.int16).cpu().numpy().view(np.uint16)


def hard_rows(tokens: int, seed: int) -> torch.Tensor:
    """[1, 2, tokens, D]: mostly ordinary vectors; every fifth is one of the hard kinds."""
    g = torch.Generator().manual_seed(seed)
    x = kv_bf16((1, 2, tokens, D), seed=seed, device="cpu").float()
    kinds = torch.zeros(9, D)
    kinds[1, :4] = torch.tensor([3.0, -3.0, 3.0, 3.0])      # four equal magnitudes: u = 1/2 or 0 exactly
    kinds[2] = 0.25 * torch.randint(0, 2, (D,), generator=g) - 0.125
    kinds[3] = 1e-21 * torch.randn(D, generator=g)          # squares underflow to subnormals
    kinds[4] = 1e-30 * torch.randn(D, generator=g)          # squares vanish
    kinds[5] = 1e17 * torch.randn(D, generator=g)
    kinds[6] = 1e25 * torch.randn(D, generator=g)           # squares overflow
    kinds[7, 5], kinds[7, 9] = float("inf"), 1.0
    kinds[8] = torch.randn(D, generator=g)
    kinds[8, 70] = float("nan")
    i = torch.arange(tokens)
    hard = i % 5 == 0
    x[:, :, hard] = kinds[(i[hard] // 5) % 9]
    return x.to(torch.bfloat16).cuda()


def buffers(x, rb, sb):
    B, H, T, _ = x.shape
    mk = lambda *s, dt=torch.uint8: torch.zeros(B, H, T + 3, *s, dtype=dt, device="cuda")  # noqa: E731
    return mk(rb), mk(dt=torch.float16), mk(sb), mk(dt=torch.float16)


def compare(x, got, ref, T):
    for name, a, b in zip(("codes", "norms", "signs", "rnorms"), got, ref):
        a = a[:, :, 2:2 + T]
        a = u16(a).reshape(-1) if a.dtype == torch.float16 else a.cpu().numpy().reshape(b.shape)
        if b.dtype == np.uint16:  # NaN payloads are not part of the format
            nan = lambda v: (v & 0x7FFF) > 0x7C00  # noqa: E731
            assert np.array_equal(nan(a), nan(b)), name
            a, b = np.where(nan(a), 0, a), np.where(nan(b), 0, b)
        assert np.array_equal(a, b), f"{name}: {(a != b).sum()} of {b.size} differ"


# one, two and four vectors per workgroup, a tile per workgroup, one pass, one and two tiles per wave
@pytest.mark.parametrize("T", [1, 128, 129, 257, 521, 12 * 1024 + 5, 17 * 1024 + 5, 25 * 1024 + 5])
@pytest.mark.parametrize("rotation", ["haar", "permutation"])
@pytest.mark.parametrize("bits,prod", [(1, False), (2, False), (3, False), (4, False), (1, True), (2, True), (3, True)])
def test_plain_prefill_encoder_on_hard_rows(cuda, bits, prod, rotation, T):
    """A permutation matrix as the rotation puts z = u on the boundaries below exactly."""
    x = hard_rows(T, 3 * bits + prod)
    lc = layer_codecs(D, bits + 1 if prod else bits, 0, prod, cuda)
    c = lc.key if prod else lc.value
    R, C, Bd = c.rotation, c.centers, c.boundaries
    if rotation == "permutation":
        R = torch.eye(D, device=cuda)[torch.randperm(D, generator=torch.Generator().manual_seed(bits)).to(cuda)].contiguous()
        n = (1 << bits) - 1
        Bd = (torch.arange(n, device=cuda) - n // 2) * 0.125  # 0, +-1/8, ...: u = 0 is a boundary
        C = torch.cat((Bd - 0.0625, Bd[-1:] + 0.0625))
    codec = K.CodecParams(bits=bits, rotation=R, centers=C.contiguous(), boundaries=Bd.contiguous())
    kc, kn, ks, kr = buffers(x, K.row_bytes(D, bits), D // 8)
    h = [t.cpu().numpy() for t in (R, C, Bd)]
    rows = u16(x).reshape(-1, D)
    if prod:
        K.quantize_prod(x, codec, lc.qjl, kc, kn, ks, kr, offset=2)
        ref = O.encode_prod(rows, bits, h[0], h[1], h[2], lc.qjl.cpu().numpy())
        compare(x, (kc, kn, ks, kr), ref, T)
    else:
        K.quantize_mse(x, codec, kc, kn, offset=2)
        compare(x, (kc, kn), O.encode_mse(rows, bits, h[0], h[2]), T)


# a tile per workgroup, and one and two tiles per wave (on 256 CUs)
@pytest.mark.parametrize("T", [521, 8192 + 19, 12 * 1024 + 19, 25 * 1024 + 19])
@pytest.mark.parametrize("d,bits,extra,qjl", [(3, 4, 1, True), (4, 4, 4, False), (8, 3, 4, True), (13, 2, 3, False),
                                              (33, 1, 1, False), (40, 2, 2, True), (60, 4, 3, True)])
def test_group_prefill_encoder_on_hard_rows(cuda, d, bits, extra, qjl, T):
    """Both groups of a split, the outlier group up to 8 bits (7 with the sketch)."""
    outl = np.sort(np.random.default_rng(d).choice(D, d, replace=False))
    sc = split_codecs(np.setdiff1d(np.arange(D), outl), outl, bits, extra, 0, qjl, cuda)
    x = hard_rows(T, d)
    for g in (sc.key_normal, sc.key_outlier, sc.value_normal, sc.value_outlier):
        kc, kn, ks, kr = buffers(x, K.row_bytes(g.dim, g.bits), K.row_bytes(g.dim, 1))
        rows = u16(x).reshape(-1, D)[:, g.channels]
        h = [t.cpu().numpy() for t in (g.rotation, g.centers, g.boundaries)]
        if g.qjl is not None:
            K.quantize_group(x, g, kc, kn, ks, kr, offset=2)
            ref = O.encode_prod(rows, g.bits, h[0], h[1], h[2], g.qjl.cpu().numpy())
            # a norm beyond fp16: 0 * inf outside the group makes the residual norm NaN, stored as 1
            ref[3][ref[1] == 0x7C00] = 0x3C00
            compare(x, (kc, kn, ks, kr), ref, T)
        else:
            K.quantize_group(x, g, kc, kn, offset=2)
            compare(x, (kc, kn), O.encode_mse(rows, g.bits, h[0], h[2]), T)
        for t in (kc, ks) if g.qjl is not None else (kc,):
            assert int(t[:, :, :2].count_nonzero()) == 0 and int(t[:, :, T + 2:].count_nonzero()) == 0


# one and two tiles per wave
@pytest.mark.parametrize("scale,T", [(1e-30, 17 * 1024 + 5), (1e-37, 25 * 1024 + 5), (float("inf"), 17 * 1024 + 5)])
@pytest.mark.parametrize("group", [False, True])
def test_prefill_encoder_with_matrices_outside_the_bounds_range(cuda, scale, group, T):
    """Matrices whose rows' squares vanish (1e-30), whose second bf16 terms are lost (1e-37), or that
    hold an infinity, which makes NaN of a zero vector's products too: the chains decide all of it."""
    x = hard_rows(T, 5)
    sc = split_codecs(np.setdiff1d(np.arange(D), [3, 40, 41, 90]), np.array([3, 40, 41, 90]), 4, 1, 0, True, cuda)
    lc = layer_codecs(D, 4, 0, True, cuda)
    val, key, S = (sc.value_normal, sc.key_normal, sc.key_normal.qjl) if group else (lc.value, lc.key, lc.qjl)

    def bad(m):
        m = m.clone() if scale == float("inf") else m * scale
        if scale == float("inf"):
            m[5, 7] = scale
        return m

    def space(m, c):
        return None if m is None else torch.from_numpy(K.group_matrix(m.cpu().numpy(), c.channels)).to(cuda)

    rows = u16(x).reshape(-1, D)
    rows = rows[:, val.channels] if group else rows
    by = 1.0 if scale == float("inf") else scale
    for c, R, Bd, Sq in ((val, bad(val.rotation), val.boundaries * by, None), (key, key.rotation, key.boundaries, bad(S))):
        kc, kn, ks, kr = buffers(x, K.row_bytes(rows.shape[1], c.bits), K.row_bytes(rows.shape[1], 1))
        if group:
            codec = K.GroupCodec(c.channels, c.bits, R, c.centers, Bd, space(R, c), Sq, space(Sq, c))
            K.quantize_group(x, codec, kc, kn, *((ks, kr) if Sq is not None else ()), offset=2)
        else:
            codec = K.CodecParams(bits=c.bits, rotation=R, centers=c.centers, boundaries=Bd)
            if Sq is None:
                K.quantize_mse(x, codec, kc, kn, offset=2)
            else:
                K.quantize_prod(x, codec, Sq, kc, kn, ks, kr, offset=2)
        h = [t.cpu().numpy() for t in (R, c.centers, Bd)]
        if Sq is None:
            compare(x, (kc, kn), O.encode_mse(rows, c.bits, h[0], h[2]), T)
        else:
            ref = O.encode_prod(rows, c.bits, h[0], h[1], h[2], Sq.cpu().numpy())
            if group:
                ref[3][ref[1] == 0x7C00] = 0x3C00  # as above
            compare(x, (kc, kn, ks, kr), ref, T)


@pytest.mark.parametrize("B,H,T", [(1, 1, 1), (2, 3, 17), (1, 8, 1000), (3, 2, 40001)])
def test_channel_energy_matches_fp64(cuda, B, H, T):
    """Strided keys and values, workgroups whose runs cross heads; fp32 sums of at most
    B * H * T / 4096 + 32 squares per thread, 512 of them: 1e-5 of each energy."""
    k = kv_bf16((B, T, H, D), seed=1, device=cuda).transpose(1, 2)
    v = kv_bf16((B, H, T, D), seed=2, device=cuda, outlier_channels=3)
    ref = sum(t.double().square().sum(dim=(0, 1, 2)) for t in (k, v))
    assert ((K.channel_energy(k, v).double() - ref).abs() <= 1e-5 * ref).all()
