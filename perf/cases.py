"""Timing cases of the TurboQuant hot path, through the package's public entry points.

The work a user of the package has it do, over the range of sizes it meets:

* ``step``    one decode step of one layer as a serving loop writes it: encode the new token's
              key and value into their slot, then attend over the packed cache;
* ``decode``  the attention backend's decode call (``turboquant.runtime.fused_attention``), over
              plain layers, outlier-split layers and layers with a dense tail of generated tokens;
* ``prefill`` compressing one layer's prompt keys and values
              (``PackedMSELayer.initialize_from_dense``), plain and outlier-split;
* ``chunked`` several query tokens against a packed layer (a second prompt on a packed cache, or
              drafted tokens to verify), with the causal mask the model hands the backend;
* ``rows``    decoding a packed layer back to bf16 rows (dense attention over a packed cache).

Every case has head dimension 128.  Keys and values have iid N(0, 1) directions and lognormal
norms around 20, queries are N(0, 1); all in bf16, as a bf16 model hands them over.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

ROOT = Path(__file__).resolve().parent.parent
for _p in (ROOT / "tq-local_amd", ROOT):
    if str(_p) not in sys.path:
        sys.path.insert(0, str(_p))

from turboquant.runtime import chunked_turboquant_attention, fused_attention  # noqa: E402
from turboquant.runtime import kernels as K  # noqa: E402
from turboquant.runtime.packed_qmse_cache import PackedMSELayer  # noqa: E402
from turboquant.runtime.params import layer_codecs  # noqa: E402
from turboquant.runtime.synthetic import kv_bf16  # noqa: E402

D = 128
DEV = "cuda"


def _case(name, op, B, Hq, Hkv, N, bits, qjl, outliers=0, dense=0, Sq=1):
    c = {"op": op, "B": B, "Hq": Hq, "Hkv": Hkv, "N": N, "bits": bits, "qjl": qjl, "outliers": outliers,
         "dense": dense, "Sq": Sq}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one token of a short chat on one GPU, the smallest call there is: 4-bit Q_prod, the
        # defaults of turboquant.activate()
        _case("step_short_chat", "step", 1, 32, 8, 1037, 4, True),
        # the benchmark's configurations: Llama-3.1-8B KV shape at 32K, batch 8
        _case("decode_8b_32k", "decode", 8, 32, 8, 32768, 4, True),
        # 3-bit Q_mse, batch 16 at 64K: the largest cache
        _case("decode_3bit_64k", "decode", 16, 32, 8, 65536, 3, False),
        # 7 query heads per KV head at 32K
        _case("decode_gqa7_32k", "decode", 4, 28, 4, 32768, 4, True),
        # 5 query heads per KV head, one long sequence
        _case("decode_gqa5_131k", "decode", 1, 40, 8, 131584, 4, True),
        # outlier-channel split, 4 channels one bit wider
        _case("decode_split_16k", "decode", 8, 32, 8, 16384, 4, True, outliers=4),
        # generated tokens kept dense, the defaults of TurboQuantSession: 3-bit Q_mse prompt
        _case("decode_dense_tail", "decode", 4, 32, 8, 8192, 3, False, dense=203),
        # compressing a full batch of 32K prompts, the largest call
        _case("prefill_8b_32k", "prefill", 8, 32, 8, 32768, 4, True),
        # compressing one short prompt of odd length
        _case("prefill_short", "prefill", 1, 32, 8, 301, 4, True),
        # compressing with the outlier-channel split
        _case("prefill_split_16k", "prefill", 2, 32, 8, 16384, 4, True, outliers=4),
        # a second prompt of 256 tokens on a packed conversation
        _case("chunked_second_prompt", "chunked", 1, 32, 8, 8192, 4, True, Sq=256),
        # a packed layer back to bf16 rows
        _case("rows_32k", "rows", 1, 32, 8, 32768, 4, True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(("step", "decode", "decode", "decode", "prefill", "prefill", "chunked", "rows"))
    qjl = rng.random() < 0.6
    bits = rng.choice((3, 4)) if not qjl else rng.choice((3, 4, 4))
    Hkv, g = rng.choice(((8, 4), (4, 7), (8, 5), (2, 8), (4, 1), (8, 2)))
    outliers = rng.choice((3, 4, 8)) if op in ("decode", "prefill") and rng.random() < 0.3 else 0
    dense, Sq = 0, 1
    if op == "step":
        B, N = rng.choice((1, 2, 5, 8)), _log(rng, 64, 8192)
    elif op == "decode":
        B, N = rng.choice((1, 2, 3, 4, 8)), _log(rng, 256, 65536)
        if rng.random() < 0.3:
            dense = _log(rng, 1, 1024)
    elif op == "prefill":
        B, N = rng.choice((1, 2, 3, 4)), _log(rng, 32, 32768)
    elif op == "chunked":
        B, N, Sq = rng.choice((1, 2)), _log(rng, 512, 8192), _log(rng, 2, 256)
    else:
        B, N = rng.choice((1, 2, 4)), _log(rng, 256, 32768)
    return _case(None, op, B, Hkv * g, Hkv, N, bits, qjl, outliers, dense, Sq)


# ---------------------------------------------------------------- preparing and running


def _kv(c, seed, n):
    shape = (c["B"], c["Hkv"], n, D)
    k = kv_bf16(shape, seed=seed, device=DEV)
    v = kv_bf16(shape, seed=seed + 1, device=DEV)
    if c["outliers"]:  # a few channels of large energy, the reason to split
        k[..., 5:128:128 // c["outliers"]] *= 8.0
    return k, v


def _layer(c, quantize_decode=True):
    return PackedMSELayer(bits=c["bits"], use_qjl_keys=c["qjl"], num_outlier_channels=c["outliers"],
                          quantize_decode=quantize_decode)


def prepare(case, seed):
    c = case
    seed = 16 * seed
    gen = torch.Generator(device=DEV).manual_seed(seed + 2)
    q = torch.randn(c["B"], c["Hq"], c["Sq"], D, generator=gen, device=DEV).to(torch.bfloat16)
    s = {"case": c, "q": q, "groups": c["Hq"] // c["Hkv"]}
    if c["op"] == "prefill":
        s["k"], s["v"] = _kv(c, seed, c["N"])
        return s
    k, v = _kv(c, seed, c["N"] + c["dense"])
    layer = _layer(c, quantize_decode=c["dense"] == 0)
    if c["dense"]:
        layer.initialize_from_dense(k[:, :, :c["N"]], v[:, :, :c["N"]])
        layer._lazy_update = True
        layer.update(k[:, :, c["N"]:], v[:, :, c["N"]:])
    else:
        layer.initialize_from_dense(k, v)
    s["layer"] = layer
    if c["op"] == "step":
        s["k"], s["v"] = _kv(c, seed + 4, 1)
    if c["op"] == "chunked":  # the last Sq tokens of the cache are the query's own
        i = torch.arange(c["Sq"], device=DEV)[:, None] + (c["N"] - c["Sq"])
        j = torch.arange(c["N"], device=DEV)[None, :]
        s["mask"] = (j <= i).expand(c["B"], 1, c["Sq"], c["N"]).contiguous()
    return s


def run(state):
    c = state["case"]
    if c["op"] == "decode":
        return fused_attention(state["q"], state["layer"], state["groups"])
    if c["op"] == "step":
        lc, st, n = state["layer"].codecs, state["layer"]._store, c["N"]
        if c["qjl"]:
            K.quantize_prod(state["k"], lc.key, lc.qjl, st.kc, st.kn, st.ks, st.kr, offset=n)
        else:
            K.quantize_mse(state["k"], lc.key, st.kc, st.kn, offset=n)
        K.quantize_mse(state["v"], lc.value, st.vc, st.vn, offset=n)
        return K.decode_attention(state["q"], k_codes=st.kc, k_norms=st.kn, v_codes=st.vc, v_norms=st.vn,
                                  n_tokens=n + 1, key=lc.key, value=lc.value, k_signs=st.ks, k_rnorms=st.kr,
                                  qjl=lc.qjl)
    if c["op"] == "prefill":
        layer = _layer(c)
        layer.initialize_from_dense(state["k"], state["v"])
        return _packed_outputs(layer)
    if c["op"] == "chunked":
        return chunked_turboquant_attention(state["q"], state["layer"], n_kv_groups=state["groups"],
                                            attention_mask=state["mask"])
    lc, st = state["layer"].codecs, state["layer"]._store
    if c["qjl"]:
        keys = K.dequantize_prod(st.kc, st.kn, st.ks, st.kr, c["N"], lc.key, lc.qjl)
    else:
        keys = K.dequantize_mse(st.kc, st.kn, c["N"], lc.key)
    return {"keys": keys, "values": K.dequantize_mse(st.vc, st.vn, c["N"], lc.value)}


def _packed_outputs(layer):
    out = {}
    for name, p in (("k", layer.keys_packed), ("v", layer.values_packed), ("ko", layer._keys_outlier),
                    ("vo", layer._values_outlier)):
        if p is not None:
            out[name + "_codes"], out[name + "_norms"] = p.packed_indices, p.norms
    for name, p in (("k", layer._keys_qjl), ("ko", layer._keys_outlier_qjl)):
        if p is not None:
            out[name + "_signs"], out[name + "_rnorms"] = p.packed_signs, p.residual_norms
    return out


# ---------------------------------------------------------------- what a pass cannot do without


def _packed_token_bytes(c):
    """Packed bytes of one token of one KV head, and its bits per value code."""
    groups = [(D - c["outliers"], c["bits"])]
    if c["outliers"]:
        groups.append((c["outliers"], c["bits"] + 1))
    n = 0
    for d, bits in groups:
        kb = bits - 1 if c["qjl"] else bits
        n += (d * kb + 7) // 8 + 2 + (d * bits + 7) // 8 + 2 + ((d + 7) // 8 + 2 if c["qjl"] else 0)
    return n


def work(case):
    c = case
    heads = c["B"] * c["Hkv"]
    per = _packed_token_bytes(c)
    mats = 3 if c["qjl"] else 1  # key products of a token: rotation, residual decode, QJL sketch
    mat = 2 * D * D
    io = 2 * c["B"] * c["Hq"] * c["Sq"] * D * 2
    params = (4 if c["qjl"] else 2) * D * D * 4
    if c["op"] == "prefill":
        return {"bytes": heads * c["N"] * (2 * D * 2 + per) + params, "flops": heads * c["N"] * (mats + 1) * mat}
    if c["op"] == "rows":
        return {"bytes": heads * c["N"] * (2 * D * 2 + per) + params,
                "flops": heads * c["N"] * ((2 if c["qjl"] else 1) + 1) * mat}
    tokens = c["N"] + c["dense"]
    flops = c["B"] * c["Hq"] * c["Sq"] * tokens * D * 4
    nbytes = heads * (c["N"] * per + c["dense"] * 2 * D * 2) + io + params
    if c["op"] == "step":
        nbytes += heads * (2 * D * 2 + per)
        flops += heads * (mats + 1) * mat
    if c["op"] == "chunked":
        nbytes += c["B"] * c["Sq"] * c["N"]
        flops += heads * c["N"] * ((2 if c["qjl"] else 1) + 1) * mat
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["op"] == "prefill":
        return "exact"  # codes, signs and fp16 norms are the oracle's, bit for bit
    if case["op"] == "rows":
        return {"rel": 2e-4, "max": 1e-2}  # a bf16 value rounded the other way now and then
    if case["op"] == "chunked":
        return {"rel": 2e-3, "max": 2e-2}  # bf16 output of fp32 sums
    return {"rel": 4e-3, "max": 3e-2}  # bf16 output


# ---------------------------------------------------------------- the same in 64 bits


def _unpack(codes, bits, dim):
    """[..., row] LSB-first bit streams -> int64 [..., dim]."""
    b = (codes.unsqueeze(-1) >> torch.arange(8, device=codes.device, dtype=torch.uint8)) & 1
    b = b.flatten(-2)[..., :dim * bits].unflatten(-1, (dim, bits)).to(torch.int16)
    return (b << torch.arange(bits, device=codes.device, dtype=torch.int16)).sum(-1)


def _groups(layer):
    """Per channel group: (channels, key codec, value codec, qjl matrix, buffer suffix)."""
    if layer._split is None:
        c = layer.codecs
        return [(slice(None), c.key, c.value, c.qjl, "")]
    sc = layer._split
    return [(sc.normal_indices, sc.key_normal, sc.value_normal, sc.key_normal.qjl, ""),
            (sc.outlier_indices, sc.key_outlier, sc.value_outlier, sc.key_outlier.qjl, "o")]


def _rows64(layer, b, h, n, bf16):
    """Keys and values [n, D] of one KV head in 64 bits; with ``bf16`` rounded to bf16 where the
    row decoder rounds (reconstruction, correction, sum)."""
    st = layer._store
    rnd = (lambda t: t.to(torch.bfloat16).double()) if bf16 else (lambda t: t)
    out = []
    for which in "kv":
        full = torch.zeros(n, D, dtype=torch.float64, device=DEV)
        for ch, kc, vc, S, sfx in _groups(layer):
            g = kc if which == "k" else vc
            d = g.rotation.shape[0]
            idx = _unpack(getattr(st, which + "c" + sfx)[b, h, :n], g.bits, d).long()
            nrm = getattr(st, which + "n" + sfx)[b, h, :n].double()[:, None]
            rows = rnd((g.centers.double()[idx] @ g.rotation.double()) * nrm)
            if which == "k" and S is not None:
                pm = 2.0 * _unpack(getattr(st, "ks" + sfx)[b, h, :n], 1, d).double() - 1.0
                rn = getattr(st, "kr" + sfx)[b, h, :n].double()[:, None]
                rows = rnd(rows + rnd((pm @ S.double()) * rn * (math.sqrt(math.pi / 2) / d)))
            full[:, ch] = rows
        out.append(full)
    return out


def exact(case, seed):
    c = case
    s = prepare(c, seed)
    if c["op"] == "prefill":
        out = {}
        for name, x in (("k", s["k"]), ("v", s["v"])):
            if c["outliers"]:
                continue  # the channel sets are the path's own result
            out[name + "_codes"] = None
            out[name + "_norms"] = x.double().square().sum(-1).sqrt()
        return out or None
    if c["op"] == "step":
        run(s)  # the appended token is part of the cache it attends to
    layer, n = s["layer"], c["N"] + (1 if c["op"] == "step" else 0)
    heads = [[_rows64(layer, b, h, n, c["op"] in ("rows", "chunked")) if c["op"] == "rows" else None
              for h in range(c["Hkv"])] for b in range(c["B"])]
    if c["op"] == "rows":
        return {name: torch.stack([torch.stack([kv[i] for kv in row]) for row in heads])
                for i, name in enumerate(("keys", "values"))}
    g = s["groups"]
    out = torch.empty(c["B"], c["Hq"], c["Sq"], D, dtype=torch.float64, device=DEV)
    for b in range(c["B"]):
        for h in range(c["Hkv"]):
            k, v = _rows64(layer, b, h, n, c["op"] == "chunked")
            if c["dense"]:
                k = torch.cat((k, layer._dense_keys[b, h].double()))
                v = torch.cat((v, layer._dense_values[b, h].double()))
            q = s["q"][b, h * g:(h + 1) * g].double().reshape(-1, D)
            logits = (q @ k.T / math.sqrt(D)).view(g, c["Sq"], -1)
            if c["op"] == "chunked":
                logits = logits.masked_fill(~s["mask"][b, 0], float("-inf"))
            out[b, h * g:(h + 1) * g] = torch.softmax(logits, -1) @ v
    return out.squeeze(2) if c["op"] == "step" else out
