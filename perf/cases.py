"""What the physical KV-cache engine is timed on: the calls a UniCache program
makes, through the package's public entry points.

One request of the BAGEL-style model (GQA 28/4, head_dim 128, 28 layers) goes
through these paths, and each is a kind of case here:

- ``decode_one``   one segment, one query token: packed_kivi_attention_summary.
- ``decode_batch`` a decode step over the packed caches of `layers` x `batch`
                   sequences: KiviDecodeBatch.run (one layer of a model loop,
                   or every layer at once).
- ``decode_mixed`` a decode step over packed prefix + dense tokens per layer:
                   MixedDecodeBatch.run.
- ``edit``         image editing: thousands of query tokens over packed,
                   H2O-retained and current keys; one sample through
                   run_fused_mixed_attention, the CFG samples of a step
                   through run_batched_physical_attention.
- ``pack``         a dense segment into a packed cache (PackedKIVICache.from_dense).
- ``unpack``       the way back (PackedKIVICache.dequantize), as a repack or an
                   offload does it.
- ``scores``       H2O scores of a prefill from Q and K (per_kv_head_scores_from_qk),
                   on its own softmax or against the attention pass's LSE.
- ``select``       the H2O segments of a layer chosen and gathered
                   (GQAH2OCache.from_dense_segments).
- ``observe``      the observed attention call: GQA logits, and from its
                   probabilities the output and the H2O score update.

Sizes come from the repository's own configurations (configs 0 to 4 of
bench.py) and, at the large end, from a 1024 x 1024 image (4096 latents, 4900
ViT tokens).
"""

from __future__ import annotations

import math

import torch

from unicache_amd.adapters.bagel import run_batched_physical_attention, run_fused_mixed_attention
from unicache_amd.operators.physical import per_kv_head_scores_from_probs, per_kv_head_scores_from_qk
from unicache_amd.storage.decode import KiviDecodeBatch, MixedDecodeBatch
from unicache_amd.storage.kivi_cuda import packed_kivi_attention_summary
from unicache_amd.storage.physical import (
    GQAH2OCache,
    PackedKIVICache,
    gqa_probability_value,
    gqa_query_key_logits,
)

D = 128
_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


# ------------------------------------------------------------------- cases --
def _case(name, kind, *, bits=2, group=32, residual=128, hq=28, hkv=4, dtype="bf16", **sizes):
    case = {"kind": kind, "hq": hq, "hkv": hkv, "dtype": dtype, **sizes}
    if kind not in ("scores", "select", "observe"):
        case.update(bits=bits, group=group, residual=residual)
    if name is not None:
        case["name"] = name
    return case


def listed():
    return [
        # one attention layer of a short chat turn: the smallest call, bound by latency
        _case("decode_one_2k", "decode_one", tokens=2048, lq=1),
        # one layer of a batched decode loop: a model runs its layers one after the other
        _case("decode_layer_8x8k", "decode_batch", layers=1, batch=8, tokens=8192, ragged=False),
        # a decode step over every layer and sequence in one call
        _case("decode_step_28x8x8k", "decode_batch", layers=28, batch=8, tokens=8192, ragged=False),
        # the same at 4 bits, the operators' default group and residual, fp16 and sequences of different lengths
        _case("decode_step_4bit_ragged", "decode_batch", layers=28, batch=3, tokens=12345, ragged=True, bits=4,
              group=64, residual=32, dtype="fp16"),
        # long-context decode over a packed segment and H2O-retained dense tokens
        _case("decode_mixed_32k", "decode_mixed", layers=28, tokens=20352, dense=2585),
        # one editing layer: the latents and text of a 512 x 512 image over 2304 keys
        _case("edit_1088", "edit", samples=1, lq=1088, tokens=1024, h2o=0, dense=1280),
        # the three CFG samples of a 1024 x 1024 edit: the largest call
        _case("edit_cfg_4098", "edit", samples=3, lq=4098, tokens=4900, h2o=819, dense=4354, bits=4, group=64,
              residual=32),
        # a long prompt's segment of one layer into the packed cache
        _case("pack_32k", "pack", tokens=32768),
        # a packed segment back into dense rows, 4 bits
        _case("unpack_20k", "unpack", tokens=20353, bits=4, group=64, residual=32),
        # H2O scores of a prefill layer
        _case("scores_512x4096", "scores", lq=512, tokens=4096, lse=False),
        # the instruction and ViT segments of a layer down to 20 %
        _case("select_4k_8k", "select", first=4096, second=8192),
        # the first call of a layer, with its probabilities observed
        _case("observe_512x4096", "observe", lq=512, tokens=4096),
    ]


def _log(rng, low, high):
    """A whole number spread over the logarithm of its range; every third one a multiple of 64."""

    n = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    return max(low, n // 64 * 64) if rng.random() < 0.34 and n >= 64 else n


def draw(rng):
    kind = rng.choice(["decode_one", "decode_batch", "decode_batch", "decode_mixed", "edit", "edit", "pack", "unpack",
                       "scores", "select", "observe"])
    heads = rng.choice([(28, 4), (28, 4), (28, 4), (32, 8), (16, 2)])
    common = dict(bits=rng.choice([2, 2, 4]), group=rng.choice([32, 32, 64, 128]), residual=rng.choice([0, 32, 100, 128]),
                  hq=heads[0], hkv=heads[1], dtype=rng.choice(["bf16", "bf16", "fp16"]))
    if kind == "decode_one":
        return _case(None, kind, tokens=_log(rng, 400, 65536), lq=rng.choice([1, 1, 2]), **common)
    if kind == "decode_batch":
        layers, batch = rng.choice([1, 1, 1, 7, 28]), rng.randint(1, 8)
        most = max(1024, 28 * 8 * 8192 // (layers * batch) // 2)
        return _case(None, kind, layers=layers, batch=batch, tokens=_log(rng, 600, min(32768, most)),
                     ragged=rng.random() < 0.5, **common)
    if kind == "decode_mixed":
        return _case(None, kind, layers=rng.choice([1, 4, 28]), tokens=_log(rng, 600, 20352), dense=_log(rng, 64, 4096),
                     **common)
    if kind == "edit":
        return _case(None, kind, samples=rng.choice([1, 1, 2, 3]), lq=_log(rng, 130, 4098), tokens=_log(rng, 500, 4900),
                     h2o=rng.choice([0, _log(rng, 51, 819)]), dense=_log(rng, 64, 4354), **common)
    if kind in ("pack", "unpack"):
        return _case(None, kind, tokens=_log(rng, 500, 65536), **common)
    if kind == "scores":
        return _case(None, kind, lq=_log(rng, 64, 2048), tokens=_log(rng, 300, 8192), lse=rng.random() < 0.5, **common)
    if kind == "select":
        return _case(None, kind, first=_log(rng, 256, 8192), second=_log(rng, 512, 16384), **common)
    return _case(None, kind, lq=_log(rng, 64, 1024), tokens=_log(rng, 300, 4900), **common)


# ------------------------------------------------------------------ inputs --
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _kv(gen, tokens, hkv, dtype):
    """K with 8 outlier channels (x10) per head as KIVI meets them, V normal."""

    key = torch.randn(tokens, hkv, D, generator=gen, device="cuda", dtype=dtype)
    value = torch.randn(tokens, hkv, D, generator=gen, device="cuda", dtype=dtype)
    gain = torch.ones(hkv, D, device="cuda", dtype=dtype)
    gain.scatter_(1, torch.rand(hkv, D, generator=gen, device="cuda").topk(8, dim=1).indices, 10.0)
    return key.mul_(gain), value


def _query(gen, lq, hq, dtype):
    return torch.randn(lq, hq, D, generator=gen, device="cuda", dtype=dtype)


def _pack(case, key, value):
    return PackedKIVICache.from_dense(
        key, value, logical_token_ids=torch.arange(int(key.shape[0]), device="cuda"), token_type_id=3,
        k_bits=case["bits"], v_bits=case["bits"], group_size=case["group"], residual_length=case["residual"],
        backend="cuda")


def _lengths(case):
    """Tokens of each sequence of a batch: equal, or evenly spread down to a fraction."""

    n, t = case["batch"], case["tokens"]
    return [max(case["residual"] + case["group"], t * (i + 1) // n - 3 * i) if case["ragged"] else t for i in range(n)]


def _edit_sample(case, gen, i):
    """Sample i of an edit: everything, then without the H2O segment, then with a quarter of the packed tokens."""

    dtype, hkv = _DTYPES[case["dtype"]], case["hkv"]
    tokens = max(case["residual"] + case["group"], case["tokens"] if i < 2 else case["tokens"] // 4)
    q = _query(gen, case["lq"], case["hq"], dtype)
    current = _kv(gen, case["dense"], hkv, dtype)
    packed = _kv(gen, tokens, hkv, dtype)
    kept = _kv(gen, case["h2o"], hkv, dtype) if case["h2o"] and i == 0 else None
    return q, current, packed, kept


def _scores_inputs(case, gen):
    dtype = _DTYPES[case["dtype"]]
    q = _query(gen, case["lq"], case["hq"], dtype)
    key, value = _kv(gen, case["tokens"], case["hkv"], dtype)
    return q, key, value


def _select_inputs(case, gen):
    """Two dense segments and their accumulated scores (a heavy tail, as column sums of softmax rows have)."""

    out = []
    for tokens in (case["first"], case["second"]):
        key, value = _kv(gen, tokens, case["hkv"], _DTYPES[case["dtype"]])
        scores = torch.randn(case["hkv"], tokens, generator=gen, device="cuda").mul_(1.5).exp_()
        target = max(1, round(tokens * 0.2))
        out.append(dict(key=key, value=value, logical_token_ids=torch.arange(tokens, device="cuda"), token_type_id=1,
                        per_kv_head_scores=scores, target_tokens=target, recent_tokens=round(target * 0.25),
                        selection_frozen=True))
    return out


def _probabilities(case, gen):
    """[Hq, Lq, T] softmax rows in the value dtype, as the adapter hands them on."""

    shape = (case["hq"], case["lq"], case["tokens"])
    x = torch.randn(shape, generator=gen, device="cuda", dtype=torch.bfloat16).float()
    return torch.softmax(x.mul_(2.7), dim=-1).to(_DTYPES[case["dtype"]])


def prepare(case, seed):
    gen, kind, dtype = _generator(seed), case["kind"], _DTYPES[case["dtype"]]
    hq, hkv = case["hq"], case["hkv"]
    if kind == "decode_one":
        key, value = _kv(gen, case["tokens"], hkv, dtype)
        return {"kind": kind, "cache": _pack(case, key, value), "query": _query(gen, case["lq"], hq, dtype)}
    if kind == "decode_batch":
        lengths = _lengths(case) * case["layers"]
        caches = [_pack(case, *_kv(gen, t, hkv, dtype)) for t in lengths]
        queries = _query(gen, len(caches), hq, dtype)
        batch = KiviDecodeBatch(caches, list(queries[:, None]))
        return _own_outputs(kind, batch)
    if kind == "decode_mixed":
        groups = []
        for _ in range(case["layers"]):
            cache = _pack(case, *_kv(gen, case["tokens"], hkv, dtype))
            groups.append([cache, _kv(gen, case["dense"], hkv, dtype)])
        queries = _query(gen, case["layers"], hq, dtype)
        return _own_outputs(kind, MixedDecodeBatch(groups, list(queries[:, None])))
    if kind == "edit":
        qs, ks, vs, segments = [], [], [], []
        for i in range(case["samples"]):
            q, current, packed, kept = _edit_sample(case, gen, i)
            own = [_pack(case, *packed)]
            if kept is not None:
                n = case["h2o"]
                own.append(GQAH2OCache(
                    key=kept[0].transpose(0, 1).contiguous(), value=kept[1].transpose(0, 1).contiguous(),
                    logical_token_ids=torch.arange(n, device="cuda").repeat(hkv, 1),
                    cumulative_scores=torch.ones(hkv, n, device="cuda"), token_type_id=1, original_tokens=5 * n,
                    heavy_tokens=n - n // 4, recent_tokens=n // 4, selection_frozen=True))
            qs.append(q)
            ks.append(current[0])
            vs.append(current[1])
            segments.append(own)
        cu_q = [case["lq"] * i for i in range(case["samples"] + 1)]
        cu_k = [case["dense"] * i for i in range(case["samples"] + 1)]
        return {"kind": kind, "q": torch.cat(qs), "k": torch.cat(ks), "v": torch.cat(vs), "segments": segments,
                "cu_q": cu_q, "cu_k": cu_k}
    if kind == "pack":
        key, value = _kv(gen, case["tokens"], hkv, dtype)
        return {"kind": kind, "case": case, "key": key, "value": value,
                "ids": torch.arange(case["tokens"], device="cuda")}
    if kind == "unpack":
        return {"kind": kind, "cache": _pack(case, *_kv(gen, case["tokens"], hkv, dtype)), "dtype": dtype}
    if kind == "scores":
        q, key, value = _scores_inputs(case, gen)
        return {"kind": kind, "q": q, "key": key, "lse": _lse(q, key).float() if case["lse"] else None}
    if kind == "select":
        return {"kind": kind, "segments": _select_inputs(case, gen)}
    q, key, value = _scores_inputs(case, gen)
    return {"kind": kind, "q": q, "key": key, "value": value, "probs": _probabilities(case, gen), "hkv": hkv}


def _own_outputs(kind, batch):
    """The batch with its outputs in one tensor each (a step's result as the next layer reads it)."""

    n, (lq, hq, d) = len(batch.outputs), batch.shape
    out = torch.zeros(n, lq, hq, d, dtype=batch.out_dtype, device="cuda")
    lse = torch.zeros(n, hq, lq, device="cuda")
    batch.outputs, batch.lses = list(out), list(lse)
    batch.refresh()
    return {"kind": kind, "batch": batch, "out": out, "lse": lse}


# -------------------------------------------------------------------- pass --
def run(state):
    kind = state["kind"]
    if kind == "decode_one":
        return packed_kivi_attention_summary(state["cache"], state["query"])
    if kind in ("decode_batch", "decode_mixed"):
        state["batch"].run()
        return state["out"], state["lse"]
    if kind == "edit":
        if len(state["segments"]) == 1:
            return run_fused_mixed_attention(state["q"], state["k"], state["v"], state["segments"][0])
        return run_batched_physical_attention(state["q"], state["k"], state["v"], state["cu_q"], state["cu_k"],
                                              state["segments"])
    if kind == "pack":
        case = state["case"]
        c = PackedKIVICache.from_dense(
            state["key"], state["value"], logical_token_ids=state["ids"], token_type_id=3, k_bits=case["bits"],
            v_bits=case["bits"], group_size=case["group"], residual_length=case["residual"], backend="cuda")
        return {"key_code": c.key_code, "key_scale": c.key_scale, "key_minimum": c.key_minimum,
                "value_code": c.value_code, "value_scale": c.value_scale, "value_minimum": c.value_minimum,
                "residual_key": c.residual_key, "residual_value": c.residual_value, "ids": c.logical_token_ids}
    if kind == "unpack":
        return state["cache"].dequantize(state["dtype"])
    if kind == "scores":
        return per_kv_head_scores_from_qk(state["q"], state["key"], lse=state["lse"])
    if kind == "select":
        return [(c.key, c.value, c.logical_token_ids, c.cumulative_scores)
                for c in GQAH2OCache.from_dense_segments(state["segments"])]
    logits = gqa_query_key_logits(state["q"], state["key"])
    return logits, gqa_probability_value(state["probs"], state["value"]), per_kv_head_scores_from_probs(
        state["probs"], state["hkv"])


# -------------------------------------------------------------------- work --
def _split(case, tokens):
    """(packed, residual) tokens of a segment."""

    packed = max(0, tokens - min(tokens, case["residual"])) // case["group"] * case["group"]
    return packed, tokens - packed


def _segment_bytes(case, tokens):
    """Packed codes and fp16 statistics plus the residual rows of one segment."""

    packed, rest = _split(case, tokens)
    per_token = 2 * D * case["bits"] / 8 + 2 * D * 4 / case["group"]
    return case["hkv"] * (packed * per_token + rest * 2 * D * 2)


def work(case):
    kind, hq, hkv = case["kind"], case["hq"], case["hkv"]
    row = hkv * D * 2  # bytes of one dense K or V row
    if kind == "decode_one":
        io = 2 * case["lq"] * hq * D * 2 + 4 * hq * case["lq"]
        return {"bytes": _segment_bytes(case, case["tokens"]) + io, "flops": 4 * case["lq"] * hq * D * case["tokens"]}
    if kind == "decode_batch":
        lengths = _lengths(case)
        nbytes = sum(_segment_bytes(case, t) for t in lengths) + len(lengths) * (2 * hq * D * 2 + 4 * hq)
        return {"bytes": case["layers"] * nbytes, "flops": case["layers"] * 4 * hq * D * sum(lengths)}
    if kind == "decode_mixed":
        nbytes = _segment_bytes(case, case["tokens"]) + case["dense"] * 2 * row + 2 * hq * D * 2 + 4 * hq
        return {"bytes": case["layers"] * nbytes,
                "flops": case["layers"] * 4 * hq * D * (case["tokens"] + case["dense"])}
    if kind == "edit":
        nbytes = flops = 0
        for i in range(case["samples"]):
            tokens = max(case["residual"] + case["group"], case["tokens"] if i < 2 else case["tokens"] // 4)
            dense = case["dense"] + (case["h2o"] if i == 0 else 0)
            nbytes += _segment_bytes(case, tokens) + dense * 2 * row + 2 * case["lq"] * hq * D * 2
            flops += 4 * case["lq"] * hq * D * (tokens + dense)
        return {"bytes": nbytes, "flops": flops}
    if kind == "pack":
        return {"bytes": case["tokens"] * (2 * row + 16) + _segment_bytes(case, case["tokens"]), "flops": 0}
    if kind == "unpack":
        return {"bytes": case["tokens"] * 2 * row + _segment_bytes(case, case["tokens"]), "flops": 0}
    if kind == "scores":
        nbytes = case["lq"] * hq * D * 2 + case["tokens"] * row + hkv * case["tokens"] * 4
        return {"bytes": nbytes + (hq * case["lq"] * 4 if case["lse"] else 0),
                "flops": 2 * case["lq"] * case["tokens"] * hq * D}
    if kind == "select":
        nbytes = 0
        for tokens in (case["first"], case["second"]):
            kept = max(1, round(tokens * 0.2))
            nbytes += hkv * tokens * 4 + hkv * kept * (2 * 2 * D * 2 + 8 + 8 + 4)
        return {"bytes": nbytes, "flops": 0}
    cells = hq * case["lq"] * case["tokens"]
    nbytes = cells * (4 + 2) + 2 * case["tokens"] * row + 2 * case["lq"] * hq * D * 2 + hkv * case["tokens"] * 4
    return {"bytes": nbytes, "flops": 4 * cells * D}


def tolerance(case):
    kind = case["kind"]
    if kind in ("pack", "unpack", "select"):
        return "exact"
    # four times the distance from exact() measured over listed and drawn cases:
    # scores 1.6e-4 to 2.9e-4 (probabilities in bf16), outputs 1.5e-3 to 2.4e-3 (16-bit results)
    return {"rel": 1.2e-3 if kind == "scores" else 1e-2}


# ------------------------------------------------------------------- exact --
def _quantized(x, bits, group, dim):
    """KIVI's grouped quantizer in fp32 (its definition: min/max per group, a
    correctly rounded division, half-even codes): (codes, fp16 scale, fp16
    minimum) with groups of x [T, H, D] along dim 0 or 2."""

    t, h, d = x.shape
    x = x.float()
    g = x.reshape(t // group, group, h, d) if dim == 0 else x.reshape(t, h, d // group, group)
    at = 1 if dim == 0 else 3
    low, high = g.amin(at, keepdim=True), g.amax(at, keepdim=True)
    # a tensor divisor: torch multiplies by the reciprocal of a plain number on the GPU
    steps = torch.full_like(low, float(2**bits - 1))
    scale = ((high - low) / steps).clamp_min(torch.finfo(torch.float32).eps)
    codes = ((g - low) / scale).round().clamp_(0, 2**bits - 1)
    return codes, scale.half(), low.half()


def _restored(x, case, dim):
    codes, scale, low = _quantized(x, case["bits"], case["group"], dim)
    return (codes.double() * scale.double() + low.double()).reshape(x.shape)


def _restored_kv(case, key, value):
    """What a packed cache of these tokens stands for, in 64 bits: [T, Hkv, D] K and V."""

    n = _split(case, int(key.shape[0]))[0]
    return (torch.cat([_restored(key[:n], case, 0), key[n:].double()]),
            torch.cat([_restored(value[:n], case, 2), value[n:].double()]))


def _rows(q, hkv, h):
    """Query rows of KV head h: [group * Lq, D], head-major."""

    group = int(q.shape[1]) // hkv
    return q[:, h * group:(h + 1) * group].transpose(0, 1).reshape(-1, D).double()


def _attend(q, key, value):
    """(out [Lq, Hq, D], lse [Hq, Lq]) in 64 bits."""

    lq, hq, _ = q.shape
    hkv = int(key.shape[1])
    group = hq // hkv
    out = torch.empty(hq, lq, D, dtype=torch.float64, device=q.device)
    lse = torch.empty(hq, lq, dtype=torch.float64, device=q.device)
    for h in range(hkv):
        k, v = key[:, h].double().t().contiguous(), value[:, h].double().contiguous()
        for j, rows in enumerate(_rows(q, hkv, h).split(lq)):
            x = (rows @ k).mul_(1.0 / math.sqrt(D))
            lse[h * group + j] = x.logsumexp(-1)
            out[h * group + j] = torch.softmax(x, -1) @ v
    return out.transpose(0, 1).contiguous(), lse


def _lse(q, key):
    hkv = int(key.shape[1])
    rows = [(_rows(q, hkv, h) @ key[:, h].double().t().contiguous()).mul_(1.0 / math.sqrt(D)).logsumexp(-1)
            for h in range(hkv)]
    return torch.cat(rows).reshape(int(q.shape[1]), int(q.shape[0]))


def exact(case, seed):
    gen, kind, dtype = _generator(seed), case["kind"], _DTYPES[case["dtype"]]
    hq, hkv = case["hq"], case["hkv"]
    if kind == "decode_one":
        kv = _restored_kv(case, *_kv(gen, case["tokens"], hkv, dtype))
        return _attend(_query(gen, case["lq"], hq, dtype), *kv)
    if kind == "decode_batch":
        lengths = _lengths(case) * case["layers"]
        kvs = [_kv(gen, t, hkv, dtype) for t in lengths]
        queries = _query(gen, len(lengths), hq, dtype)
        pairs = [_attend(queries[i][None], *_restored_kv(case, *kv)) for i, kv in enumerate(kvs)]
        return torch.stack([o for o, _ in pairs]), torch.stack([x for _, x in pairs])
    if kind == "decode_mixed":
        kvs = [(_kv(gen, case["tokens"], hkv, dtype), _kv(gen, case["dense"], hkv, dtype))
               for _ in range(case["layers"])]
        queries = _query(gen, case["layers"], hq, dtype)
        pairs = []
        for i, (packed, dense) in enumerate(kvs):
            key, value = _restored_kv(case, *packed)
            pairs.append(_attend(queries[i][None], torch.cat([key, dense[0].double()]),
                                 torch.cat([value, dense[1].double()])))
        return torch.stack([o for o, _ in pairs]), torch.stack([x for _, x in pairs])
    if kind == "edit":
        outs = []
        for i in range(case["samples"]):
            q, current, packed, kept = _edit_sample(case, gen, i)
            key, value = _restored_kv(case, *packed)
            keys, values = [key, current[0].double()], [value, current[1].double()]
            if kept is not None:
                keys.append(kept[0].double())
                values.append(kept[1].double())
            outs.append(_attend(q, torch.cat(keys), torch.cat(values))[0])
        return torch.cat(outs)
    if kind == "pack":
        key, value = _kv(gen, case["tokens"], hkv, dtype)
        n = _split(case, case["tokens"])[0]
        _, ks, km = _quantized(key[:n], case["bits"], case["group"], 0)
        _, vs, vm = _quantized(value[:n], case["bits"], case["group"], 2)
        return {"key_code": None, "key_scale": ks[:, 0].permute(1, 2, 0).double(),
                "key_minimum": km[:, 0].permute(1, 2, 0).double(), "value_code": None,
                "value_scale": vs[..., 0].transpose(0, 1).double(),
                "value_minimum": vm[..., 0].transpose(0, 1).double(), "residual_key": key[n:].double(),
                "residual_value": value[n:].double(), "ids": None}
    if kind == "unpack":
        return _restored_kv(case, *_kv(gen, case["tokens"], hkv, dtype))
    if kind == "scores":
        q, key, _ = _scores_inputs(case, gen)
        lse = _lse(q, key)
        out = []
        for h in range(hkv):
            x = (_rows(q, hkv, h) @ key[:, h].double().t().contiguous()).mul_(1.0 / math.sqrt(D))
            own = lse[h * (hq // hkv):(h + 1) * (hq // hkv)].reshape(-1, 1)
            out.append((x - own).exp().sum(0))
        return torch.stack(out)
    if kind == "select":
        out = []
        for seg in _select_inputs(case, gen):
            scores, tokens, recent = seg["per_kv_head_scores"], int(seg["key"].shape[0]), seg["recent_tokens"]
            best = scores[:, :tokens - recent].double().topk(seg["target_tokens"] - recent, dim=1).indices.sort(1).values
            kept = torch.cat([best, torch.arange(tokens - recent, tokens, device="cuda").repeat(hkv, 1)], dim=1)
            heads = torch.arange(hkv, device="cuda")[:, None]
            out.append((seg["key"][kept, heads].double(), seg["value"][kept, heads].double(), None,
                        scores.gather(1, kept).double()))
        return out
    q, key, value = _scores_inputs(case, gen)
    probs = _probabilities(case, gen)
    group = hq // hkv
    logits = torch.stack([_rows(q, hkv, j // group).split(case["lq"])[j % group]
                          @ key[:, j // group].double().t().contiguous() for j in range(hq)])
    out = torch.stack([probs[j].double() @ value[:, j // group].double().contiguous() for j in range(hq)])
    scores = torch.stack([sum(probs[j].double().sum(0) for j in range(h * group, (h + 1) * group)) for h in range(hkv)])
    return logits, out, scores
