"""GPU parity of the packed attention kernels against the oracle's fp32
dequant path: max abs <= 2e-2, mean abs <= 1e-3 (outputs), LSE within 1e-3."""

import math

import numpy as np
import pytest
import torch

from oracle import attention as A
from oracle import kivi as K
from tests.helpers import assert_close, f32, kv_pair, queries
from unicache_amd import _native as nat
from unicache_amd.adapters import merge_attention_summaries
from unicache_amd.storage import PackedKIVICache, gqa_probability_value, gqa_query_key_logits
from unicache_amd.storage.kivi_cuda import (
    packed_kivi_attention_summary,
    packed_kivi_quantized_attention_summary,
)

pytestmark = pytest.mark.gpu


def check_summary(out, lse, seg, q, *, include_residual=True, what="summary"):
    """Outputs within 2e-2 max / 1e-3 mean of the fp32 dequant path (the
    contract) and of the bf16-dequant runtime path of UniCache; the natural
    LSE within 1e-2 max / 1e-3 mean of the fp32 path."""

    eo, el = A.packed_summary(seg, f32(q), include_residual=include_residual, kv_dtype="fp32")
    assert_close(f32(out), eo, what=f"{what} out (fp32 path)")
    # the kernels round dequantized keys to fp16 before the MFMA (UniCache's
    # runtime rounds them to bf16, 8x coarser): with x10 outlier channels a key
    # of ~40 carries up to 0.016 of rounding, ~5e-3 on the largest of ~3e4 LSEs
    assert_close(f32(lse), el, max_abs=1e-2, mean_abs=1e-3, what=f"{what} lse (fp32 path)")
    # UniCache's runtime path rounds dequantized K/V to bf16 itself; over the
    # ~4e6 outputs of config 2 it strays from the fp32 path by up to ~3e-2, so
    # against it the bounds are looser
    bo, _ = A.packed_summary(seg, f32(q), include_residual=include_residual, kv_dtype="bf16")
    assert_close(f32(out), bo, max_abs=5e-2, mean_abs=2e-3, what=f"{what} out (bf16 path)")


def _pair(tokens, seed, bits, group, residual, device, heads=4, head_dim=128):
    key, value = kv_pair(tokens, heads=heads, head_dim=head_dim, seed=seed)
    cache = PackedKIVICache.from_dense(key.to(device), value.to(device), logical_token_ids=torch.arange(tokens),
                                       token_type_id=3, k_bits=bits, v_bits=bits, group_size=group,
                                       residual_length=residual, backend="cuda")
    seg = K.from_dense(f32(key), f32(value), k_bits=bits, v_bits=bits, group_size=group,
                       residual_length=residual, native=bits != 8)
    return cache, seg


@pytest.mark.parametrize("bits", [2, 4, 8])
@pytest.mark.parametrize("lq", [1, 37])
def test_attention_parts_qk_av(device, bits, lq):
    cache, seg = _pair(320, 5, bits, 64, 32, device)
    q = queries(lq, seed=7)
    logits, apply_value = cache.attention_parts(q.to(device))
    assert logits.dtype == torch.float32 and tuple(logits.shape) == (28, lq, 320)
    exp_logits = A.packed_logits(seg, f32(q), kv_dtype="fp32")
    assert_close(f32(logits), exp_logits, max_abs=2e-3, mean_abs=2e-4, what="logits")
    probs = torch.softmax(logits, dim=-1).to(torch.bfloat16)
    out = apply_value(probs)
    assert out.dtype == torch.bfloat16 and tuple(out.shape) == (28, lq, 128)
    exp = A.packed_pv(seg, f32(probs), kv_dtype="bf16")
    assert_close(f32(out), exp, what="av")


@pytest.mark.parametrize("bits,group,tokens,residual,lq", [(2, 16, 200, 32, 1), (4, 32, 250, 20, 3),
                                                         (2, 128, 1100, 60, 2), (4, 16, 2048, 128, 1)])
def test_attention_parts_tiles_groups_and_rows(device, bits, group, tokens, residual, lq):
    # token tiles that mix packed and residual tokens (groups 16 and 32 with
    # quantized counts of 160 and 224, not multiples of 64), groups 16 to 128,
    # several query rows per head and a second chunk of 16 rows (lq = 3: 21 rows
    # per KV head)
    cache, seg = _pair(tokens, 11, bits, group, residual, device)
    q = queries(lq, seed=13)
    logits, apply_value = cache.attention_parts(q.to(device))
    exp_logits = A.packed_logits(seg, f32(q), kv_dtype="fp32")
    assert_close(f32(logits), exp_logits, max_abs=2e-3, mean_abs=2e-4, what="logits")
    probs = torch.softmax(logits, dim=-1).to(torch.bfloat16)
    out = apply_value(probs)
    assert_close(f32(out), A.packed_pv(seg, f32(probs), kv_dtype="bf16"), what="av")
    # fp32 probabilities and an fp16 query
    logits16, apply16 = cache.attention_parts(q.half().to(device))
    assert_close(f32(logits16), A.packed_logits(seg, f32(q.half()), kv_dtype="fp32"), max_abs=2e-3,
                 mean_abs=2e-4, what="fp16-query logits")
    p32 = torch.softmax(logits16, dim=-1)
    assert_close(f32(apply16(p32)), A.packed_pv(seg, f32(p32), kv_dtype="bf16"), what="fp32-probability av")


@pytest.mark.parametrize("bits", [2, 4])
def test_decode_summary_config0(device, bits):
    # config 0: 2048 tokens (1920 packed + 128 residual), G=32, q [1, 28, 128]
    cache, seg = _pair(2048, 0, bits, 32, 128, device)
    q = queries(1, seed=1)
    out, lse = packed_kivi_attention_summary(cache, q.to(device))
    assert out.dtype == torch.bfloat16 and tuple(out.shape) == (1, 28, 128) and tuple(lse.shape) == (28, 1)
    check_summary(out, lse, seg, q, include_residual=True)
    # the packed prefix alone (kivi_cuda.py:96-120)
    po, pl = packed_kivi_quantized_attention_summary(cache, q.to(device))
    check_summary(po, pl, seg, q, include_residual=False)


def test_decode_summary_matches_parts_and_merge(device):
    cache, seg = _pair(1536, 9, 2, 32, 128, device)
    q = queries(1, seed=3).to(device)
    out, lse = packed_kivi_attention_summary(cache, q)
    logits, apply_value = cache.attention_parts(q)
    probs = torch.softmax(logits, dim=-1)
    ref = apply_value(probs.to(torch.bfloat16)).transpose(0, 1)
    assert_close(f32(out), f32(ref), what="summary vs parts")
    assert_close(f32(lse), f32(torch.logsumexp(logits, dim=-1)), max_abs=5e-3, mean_abs=1e-3, what="lse")


def test_multi_query_summary(device):
    cache, seg = _pair(1024, 4, 4, 32, 128, device)
    q = queries(37, seed=5)
    out, lse = packed_kivi_attention_summary(cache, q.to(device))
    check_summary(out, lse, seg, q, what="mq")


def test_batched_decode_items(device):
    from unicache_amd.storage.decode import KiviDecodeBatch

    caches, segs, qs = [], [], []
    for i, tokens in enumerate((1000, 2048, 700)):
        c, s = _pair(tokens, 30 + i, 2, 32, 128, device)
        caches.append(c)
        segs.append(s)
        qs.append(queries(1, seed=40 + i))
    batch = KiviDecodeBatch(caches, [q.to(device) for q in qs])
    batch.run()
    for i in range(3):
        check_summary(batch.outputs[i], batch.lses[i], segs[i], qs[i], what=f"item {i}")


@pytest.mark.parametrize("bits", [2, 4])
def test_batched_decode_many_units_ragged(device, bits):
    # 9 items x 4 KV heads = 36 units: the launch deals a unit's splits to one
    # XCD and interleaves their super-tiles (taken at >= 32 units); ragged
    # lengths leave splits with fewer super-tiles or none, one item packs a
    # single 32-token group and one has no residual
    from unicache_amd.storage.decode import KiviDecodeBatch

    lengths = (4500, 2048, 700, 3300, 1000, 6000, 513, 2600, 160)
    caches, segs, qs = [], [], []
    for i, tokens in enumerate(lengths):
        residual = 0 if i == 1 else 128
        c, s = _pair(tokens, 60 + i, bits, 32, residual, device)
        caches.append(c)
        segs.append(s)
        qs.append(queries(1, seed=70 + i))
    batch = KiviDecodeBatch(caches, [q.to(device) for q in qs])
    batch.run()
    for i in range(len(lengths)):
        check_summary(batch.outputs[i], batch.lses[i], segs[i], qs[i], what=f"item {i} ({lengths[i]} tokens)")


@pytest.mark.parametrize("residuals", [(1, 31, 32, 33, 64, 100, 127, 128), (1, 97, 128, 129, 200, 255, 256, 257)])
def test_batched_decode_residual_split_sizes(device, residuals):
    # residual splits take 32 tokens a wave when the longest residual of the
    # launch fits one split that way (<= 128 tokens) and 64 otherwise: lengths
    # around both rules, partial waves and tiles, and one item with a single
    # packed group (dense segments without packed tokens: the segment tables
    # of test_gpu_mixed.py)
    from unicache_amd.storage.decode import KiviDecodeBatch

    caches, segs, qs = [], [], []
    for i, tr in enumerate(residuals):
        packed = 32 if i == len(residuals) - 2 else 512
        c, s = _pair(packed + tr, 80 + i, 2, 32, tr, device)
        assert c.quantized_tokens == packed and c.residual_tokens == tr
        caches.append(c)
        segs.append(s)
        qs.append(queries(1, seed=90 + i))
    batch = KiviDecodeBatch(caches, [q.to(device) for q in qs])
    batch.run()
    for i, tr in enumerate(residuals):
        check_summary(batch.outputs[i], batch.lses[i], segs[i], qs[i], what=f"item {i} (residual {tr})")


@pytest.mark.parametrize("hq,hkv,lq", [(32, 4, 1), (8, 4, 2), (16, 2, 1), (28, 4, 2), (12, 4, 3)])
def test_decode_query_rows_around_the_fold(device, hq, hkv, lq):
    # 2-bit G=32 decode with at most 8 query rows per KV head (query heads per
    # KV head x query length) uses each MFMA column half for one of a wave's two
    # key groups; 9-16 rows use all 16 columns per group.  Lengths leave waves
    # whose second half has no packed token (544 and 2464 packed tokens).
    for tokens, seed in ((700, 140), (2600, 141)):
        cache, seg = _pair(tokens, seed, 2, 32, 128, device, heads=hkv)
        q = queries(lq, heads=hq, seed=seed + 10)
        out, lse = packed_kivi_attention_summary(cache, q.to(device))
        check_summary(out, lse, seg, q, what=f"Hq {hq} Hkv {hkv} Lq {lq} T {tokens}")


# packed tokens with group 32 and residual 100: none of two super-tiles (160), one (256 at 2 bits) and one group
# more (288), eight; 16 of 128 tokens at 4 bits; 129 super-tiles on one KV head
@pytest.mark.parametrize("bits,group,tokens,heads,packed", [(2, 32, 287, 4, 160), (2, 32, 356, 4, 256),
                                                            (2, 32, 388, 4, 288), (2, 32, 2148, 2, 2048),
                                                            (4, 64, 1999, 4, 1856), (2, 32, 33000, 1, 32896),
                                                            (4, 128, 9000, 8, 8832)])
def test_decode_results_do_not_depend_on_workspace(device, bits, group, tokens, heads, packed):
    # the calls that do not ask for finer splits give the same bits whatever the
    # workspace, and the call without one gives them too; the finer splits of a
    # small launch against the oracle, the same bits again with a larger workspace
    cache, seg = _pair(tokens, 150, bits, group, 100, device, heads=heads)
    assert cache.quantized_tokens == packed
    q = queries(1, heads=7 * heads, seed=151)
    qd = q.to(device)
    args = (bits, group, 7 * heads, heads, 128, 1)
    tr = cache.residual_tokens
    least, preferred = [f(1, *args, packed, tr)
                        for f in (nat.decode_workspace_bytes, nat.decode_preferred_workspace_bytes)]
    super_tiles = -(-packed // (16 * (32 // bits)))
    assert preferred > least if super_tiles > 1 else preferred == least

    def summary(entry, nbytes):
        out, lse = torch.empty_like(qd), torch.empty((7 * heads, 1), dtype=torch.float32, device=device)
        item = cache.native_item(qd.data_ptr(), out.data_ptr(), lse.data_ptr(),
                                 residual_key_ptr=cache.residual_key.data_ptr(),
                                 residual_value_ptr=cache.residual_value.data_ptr(), residual_tokens=tr)
        types = (nat.UC_BF16, nat.UC_BF16, nat.UC_BF16, 1.0 / math.sqrt(128))
        ws = nat.workspace(device, nbytes)
        room = (ws.data_ptr(), nbytes, nat.stream(device))
        if entry == "uc_kivi_attn_decode_static":
            nat.call(entry, item, *args, *types, nat.stream(device))
        elif entry == "uc_kivi_attn_decode_segments_host":
            nat.call(entry, item, 1, *args, *types, *room)
        elif entry == "uc_kivi_attn_decode":
            nat.call(entry, item, *args, *types, *room)
        else:
            nat.call(entry, item, None, 1, 1, *args, *types, 0, 0, *room)
        check_summary(out, lse, seg, q, what=f"{entry} with {nbytes} bytes of workspace")
        return out, lse

    want = summary("uc_kivi_attn_decode", least)
    for entry, nbytes in (("uc_kivi_attn_decode", preferred), ("uc_kivi_attn_decode", 8 << 20),
                          ("uc_kivi_attn_decode_static", 0), ("uc_kivi_attn_decode_segments_host", 8 << 20)):
        got = summary(entry, nbytes)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]), (entry, nbytes)
    fine = summary("uc_kivi_attn_decode_fine", preferred)
    more = summary("uc_kivi_attn_decode_fine", 8 << 20)
    assert torch.equal(fine[0], more[0]) and torch.equal(fine[1], more[1])
    with pytest.raises(ValueError, match="workspace too small"):
        summary("uc_kivi_attn_decode_fine", 4)


@pytest.mark.parametrize("bits,group,lengths", [(2, 32, (2500,) * 4), (4, 64, (4500,) * 4), (2, 32, (2048, 700, 4500, 287))])
def test_decode_tables_equal_single_calls(device, bits, group, lengths):
    # the C calls over device tables: a small batch gives segments as long as its
    # longest the bits of their own calls, and a group of segments has those of
    # uc_kivi_attn_decode_segments_host
    import ctypes

    caches, segs = zip(*(_pair(t, 200 + i, bits, group, 100, device) for i, t in enumerate(lengths)))
    qs = [queries(1, seed=210 + i).to(device) for i in range(4)]
    args = (bits, group, 28, 4, 128, 1, nat.UC_BF16, nat.UC_BF16, nat.UC_BF16, 1.0 / math.sqrt(128))
    ws = nat.workspace(device, 8 << 20)
    room = (ws.data_ptr(), 8 << 20, nat.stream(device))

    def results():
        return ([torch.full_like(q, float("nan")) for q in qs],
                [torch.full((28, 1), float("nan"), device=device) for _ in qs])

    def items(outs, lses, query=None):
        table = (nat.KiviItem * 4)()
        for i, c in enumerate(caches):
            q = qs[i] if query is None else query
            table[i] = c.native_item(q.data_ptr(), outs[i].data_ptr(), lses[i].data_ptr(),
                                     residual_key_ptr=c.residual_key.data_ptr(),
                                     residual_value_ptr=c.residual_value.data_ptr(),
                                     residual_tokens=c.residual_tokens)
        raw = bytearray(ctypes.string_at(ctypes.addressof(table), ctypes.sizeof(table)))
        return table, torch.frombuffer(raw, dtype=torch.uint8).to(device)

    tokens = (max(c.quantized_tokens for c in caches), max(c.residual_tokens for c in caches))
    want, got = results(), results()
    host, _ = items(*want)
    for i in range(4):
        nat.call("uc_kivi_attn_decode", host[i], *args, *room)
        check_summary(want[0][i], want[1][i], segs[i], qs[i].cpu(), what=f"item {i}")
    _, table = items(*got)
    nat.call("uc_kivi_attn_decode_batch", table.data_ptr(), 4, *args, *tokens, *room)
    for i in range(4):
        check_summary(got[0][i], got[1][i], segs[i], qs[i].cpu(), what=f"batch item {i}")
        if lengths[i] == lengths[0] == max(lengths):
            assert torch.equal(got[0][i], want[0][i]) and torch.equal(got[1][i], want[1][i]), f"item {i}"
    host, _ = items(*want, query=qs[0])
    nat.call("uc_kivi_attn_decode_segments_host", host, 4, *args, *room)
    _, table = items(*got, query=qs[0])
    nat.call("uc_kivi_attn_decode_segments", table.data_ptr(), 4, 4, *args, *tokens, *room)
    assert torch.equal(got[0][0], want[0][0]) and torch.equal(got[1][0], want[1][0])
    pairs = [K.dequantize(seg, "fp32") for seg in segs]
    eo, el = A.attention_summary(f32(qs[0]), np.concatenate([k for k, _ in pairs]), np.concatenate([v for _, v in pairs]))
    assert_close(f32(got[0][0]), eo, what="out")
    assert_close(f32(got[1][0]), el, max_abs=1e-2, mean_abs=1e-3, what="lse")


@pytest.mark.parametrize("bits,group,hq,lq,lengths", [(2, 32, 28, 1, (2048,)), (2, 64, 28, 2, (2048, 1024, 256)),
                                                      (4, 64, 16, 1, (1024,)), (4, 128, 32, 2, (8192,) * 4),
                                                      (2, 32, 12, 1, (32768, 512)), (2, 32, 32, 1, (8192,) * 8)])
def test_finer_splits_hand_over_fp32_partials(device, bits, group, hq, lq, lengths):
    # zero keys weigh all tokens alike and V alternates between two fp16 values
    # whose mean is none: every product and sum is exact in fp32, an fp16 partial
    # is off by 2^-11.  3 to 16 query rows per KV head, 1 to 128 super-tiles
    from unicache_amd.storage.decode import KiviDecodeBatch

    caches = []
    for tokens in lengths:
        value = torch.ones(tokens, 4, 128, dtype=torch.float16, device=device)
        value[1::2] += 2.0 ** -10
        caches.append(PackedKIVICache.from_dense(
            torch.zeros_like(value), value, logical_token_ids=torch.arange(tokens), token_type_id=3, k_bits=bits,
            v_bits=bits, group_size=group, residual_length=0, backend="cuda"))
    q = [queries(lq, heads=hq, seed=160 + i, dtype=torch.float16).to(device) for i in range(len(caches))]
    args = (len(caches), bits, group, hq, 4, 128, lq, max(lengths), 0)
    assert nat.decode_preferred_workspace_bytes(*args) > nat.decode_workspace_bytes(*args)
    batch = KiviDecodeBatch(caches, q, out_dtype=torch.float32)
    batch.run()
    for i, tokens in enumerate(lengths):
        # the normalisations and the weighted sum: a few fp32 roundings each
        assert float((batch.outputs[i] - (1 + 2.0 ** -11)).abs().max()) <= 2.0 ** -20
        assert float((batch.lses[i] - math.log(tokens)).abs().max()) <= 1e-5
    one = KiviDecodeBatch(caches[:1], q[:1])
    one.run()
    out, lse = packed_kivi_attention_summary(caches[0], q[0])  # the item in the kernel arguments
    assert torch.equal(out, one.outputs[0]) and torch.equal(lse, one.lses[0])


def test_finer_splits_in_a_graph(device):
    # a captured run of finer splits, replayed over changing queries with eager
    # work in between, gives what the eager run gives
    from unicache_amd.storage.decode import KiviDecodeBatch

    caches = [_pair(t, 220 + i, 2, 32, 128, device)[0] for i, t in enumerate((2500, 700))]
    qs = [queries(1, seed=230 + i).to(device) for i in range(2)]
    batch = KiviDecodeBatch(caches, qs)
    batch.run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        batch.run()
    for step in range(4):
        for i, q in enumerate(qs):
            q.copy_(queries(1, seed=240 + 2 * step + i))
        batch.run()
        want = [x.clone() for x in batch.outputs + batch.lses]
        for x in batch.outputs + batch.lses:
            x.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for x, exp in zip(batch.outputs + batch.lses, want):
            assert torch.equal(x, exp), f"replay {step}"


def test_decode_combine_of_many_splits(device):
    # one packed segment and 7 dense ones of up to 13 splits at 4 query rows per
    # KV head: 112 splits, the 16 parts a combine block takes at most
    from unicache_amd.storage.kivi_cuda import decode_segments_summary

    cache, seg = _pair(64, 170, 2, 32, 0, device, heads=8)
    parts = [kv_pair(3300 - 50 * i, heads=8, seed=171 + i) for i in range(7)]
    q = queries(1, heads=32, seed=180)
    out, lse = decode_segments_summary([cache], q.to(device), [(k.to(device), v.to(device)) for k, v in parts])
    key, value = K.dequantize(seg, "fp32")
    eo, el = A.attention_summary(f32(q), np.concatenate([key] + [f32(k) for k, _ in parts]),
                                 np.concatenate([value] + [f32(v) for _, v in parts]))
    assert_close(f32(out), eo, what="out")
    assert_close(f32(lse), el, max_abs=1e-2, mean_abs=1e-3, what="lse")


def test_decode_is_deterministic(device):
    cache, _ = _pair(4096, 11, 2, 32, 128, device)
    q = queries(1, seed=2).to(device)
    a = packed_kivi_attention_summary(cache, q)
    b = packed_kivi_attention_summary(cache, q)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


def test_gqa_helpers(device):
    key, value = kv_pair(77, seed=8)
    q = queries(5, seed=9)
    logits = gqa_query_key_logits(q.to(device), key.to(device))
    assert_close(f32(logits), A.gqa_logits(f32(q), f32(key)), max_abs=1e-3, mean_abs=1e-4, what="qk")
    p = torch.softmax(logits / math.sqrt(128), dim=-1)
    pv = gqa_probability_value(p, value.to(device))
    assert pv.dtype == torch.bfloat16
    assert_close(f32(pv), A.gqa_pv(f32(p), f32(value)), what="pv")


@pytest.mark.parametrize("lq,tokens,dtype", [(100, 300, torch.bfloat16), (70, 1000, torch.float16),
                                             (90, 301, torch.bfloat16)])
def test_gqa_logits_mfma_tiles(device, lq, tokens, dtype):
    # >= 64 query rows per KV head take the MFMA logits kernel: ragged row
    # blocks and key chunks; fp32 accumulation of up to ~100-sized products.
    # 301 keys: rows that do not start on 16 bytes take the 4-byte stores
    key, _ = kv_pair(tokens, seed=31, dtype=dtype)
    q = queries(lq, seed=32, dtype=dtype)
    got = gqa_query_key_logits(q.to(device), key.to(device))
    assert_close(f32(got), A.gqa_logits(f32(q), f32(key)), max_abs=2e-3, mean_abs=1e-4, what="qk mfma")
    # head-major storage read through strides (the H2O segment layout): same tiles, same bits
    kh = key.transpose(0, 1).contiguous().to(device).transpose(0, 1)
    assert torch.equal(gqa_query_key_logits(q.to(device), kh), got)


# Waves with all of their 64 rows (whole-line stores), with some of them and
# with none; one tile a workgroup and several; a last tile that is not full;
# rows that do and do not start on 16 bytes.
@pytest.mark.parametrize("lq,tokens,dtype", [(64, 64, torch.bfloat16), (10, 132, torch.bfloat16), (37, 192, torch.float16),
                                             (128, 191, torch.bfloat16), (97, 4096, torch.bfloat16),
                                             (130, 8196, torch.float16)])
def test_gqa_logits_store_paths(device, lq, tokens, dtype):
    key, _ = kv_pair(tokens, seed=33, dtype=dtype)
    q = queries(lq, seed=34, dtype=dtype)
    got = f32(gqa_query_key_logits(q.to(device), key.to(device)))
    # exact products, 128 additions in fp32 each way, and the same again for the oracle
    bound = 2 * 130 * 2.0 ** -24 * A.gqa_logits(np.abs(f32(q)), np.abs(f32(key)))
    assert (np.abs(got - A.gqa_logits(f32(q), f32(key))) <= bound).all()


@pytest.mark.parametrize("pdtype,vdtype", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.bfloat16),
                                           (torch.float32, torch.float16)])
def test_gqa_pv_mfma_tiles(device, pdtype, vdtype):
    # >= 64 query rows per KV head take the MFMA P.V kernel, P cast to the value
    # dtype first (physical.py:59); 301 keys end inside a 64-key tile and inside an
    # 8-key run, and the row padding past them holds NaN that must not leak in
    lq, t = 100, 301
    _, value = kv_pair(t, seed=33, dtype=vdtype)
    g = torch.Generator().manual_seed(34)
    probs = torch.softmax(torch.randn(28, lq, t, generator=g) * 3, -1)
    wide = torch.full((28, lq, 304), float("nan"))
    wide[..., :t] = probs
    got = gqa_probability_value(wide.to(pdtype).to(device)[..., :t], value.to(device))
    assert got.dtype == vdtype
    exp = A.gqa_pv(f32(probs.to(pdtype).to(vdtype)), f32(value))
    assert_close(f32(got), exp, max_abs=1e-2, mean_abs=1e-3, what="pv mfma")


def test_gqa_generic_and_mfma_routes_agree(device):
    # the same products through the MFMA tiles (contiguous inputs, >= 64 rows per
    # KV head) and through the generic kernels (fp32 query; key-strided P): both
    # within tolerance of the oracle and of each other
    key, value = kv_pair(200, seed=35)
    q = queries(80, seed=36)
    mfma = gqa_query_key_logits(q.to(device), key.to(device))
    generic = gqa_query_key_logits(q.float().to(device), key.float().to(device))
    exp = A.gqa_logits(f32(q), f32(key))
    assert_close(f32(mfma), exp, max_abs=2e-3, mean_abs=1e-4, what="qk mfma")
    assert_close(f32(generic), exp, max_abs=2e-3, mean_abs=1e-4, what="qk generic")
    p = torch.softmax(mfma / math.sqrt(128), -1).to(torch.bfloat16)
    pv_mfma = gqa_probability_value(p, value.to(device))
    pt = p.transpose(1, 2).contiguous().transpose(1, 2)  # same values, key stride != 1
    pv_generic = gqa_probability_value(pt, value.to(device))
    assert_close(f32(pv_mfma), f32(pv_generic), max_abs=1e-2, mean_abs=1e-3, what="pv routes")
    assert_close(f32(pv_mfma), A.gqa_pv(f32(p), f32(value)), what="pv oracle")


def test_lse_merge(device):
    # test_physical.py:181-202 on the GPU kernel
    torch.manual_seed(11)
    sa, sb = torch.randn(4, 3, 7), torch.randn(4, 3, 5)
    va, vb = torch.randn(4, 7, 8), torch.randn(4, 5, 8)
    summaries = [
        (torch.matmul(torch.softmax(sa, -1), va).transpose(0, 1).to(device), torch.logsumexp(sa, -1).to(device)),
        (torch.matmul(torch.softmax(sb, -1), vb).transpose(0, 1).to(device), torch.logsumexp(sb, -1).to(device)),
    ]
    out, lse = merge_attention_summaries(summaries)
    allsc = torch.cat([sa, sb], -1)
    expected = torch.matmul(torch.softmax(allsc, -1), torch.cat([va, vb], 1)).transpose(0, 1)
    assert torch.allclose(out.cpu(), expected, atol=1e-5, rtol=1e-5)
    assert torch.allclose(lse.cpu(), torch.logsumexp(allsc, -1), atol=1e-6)
    eo, el = A.merge_summaries([(f32(o), f32(l)) for o, l in summaries])
    assert np.allclose(f32(out), eo, atol=1e-6) and np.allclose(f32(lse), el, atol=1e-6)


def test_lse_merge_vector_and_row_kernels_agree(device):
    # 16-byte aligned summaries take the vector kernel, 2-byte offset ones the
    # per-row kernel: the same arithmetic, so equal bits; both match the oracle
    torch.manual_seed(12)
    lq, hq, d = 37, 28, 128
    outs = [torch.randn(lq, hq, d).to(torch.bfloat16) for _ in range(3)]
    lses = [torch.randn(hq, lq) * 4 for _ in range(3)]
    lses[1][0, :5] = -math.inf  # rows where one segment is empty
    a, la = merge_attention_summaries([(o.to(device), l.to(device)) for o, l in zip(outs, lses)])
    shifted = []
    for o in outs:
        buf = torch.empty(o.numel() + 1, dtype=torch.bfloat16, device=device)
        view = buf[1:].view(lq, hq, d)
        view.copy_(o.to(device))
        shifted.append(view)
    b, lb = merge_attention_summaries([(o, l.to(device)) for o, l in zip(shifted, lses)])
    assert torch.equal(a, b) and torch.equal(la, lb)
    eo, el = A.merge_summaries([(f32(o), f32(l)) for o, l in zip(outs, lses)])
    assert_close(f32(a), eo, what="merge")
    assert np.allclose(f32(la), el, atol=1e-5)


def test_summaries_merge_to_full_attention(device):
    # packed+residual summary merged with a dense bf16 segment equals attention over all keys
    cache, seg = _pair(1024, 12, 2, 32, 128, device)
    dk, dv = kv_pair(256, seed=13)
    q = queries(1, seed=14)
    s1 = packed_kivi_attention_summary(cache, q.to(device))
    logits = gqa_query_key_logits(q.to(device), dk.to(device)) / math.sqrt(128)
    p = torch.softmax(logits, -1)
    s2 = (gqa_probability_value(p, dv.to(device)).transpose(0, 1), torch.logsumexp(logits, -1))
    out, _ = merge_attention_summaries([s1, s2])
    key, value = K.dequantize(seg, "bf16")
    eo, _ = A.attention_summary(f32(q), np.concatenate([key, f32(dk)]), np.concatenate([value, f32(dv)]))
    assert_close(f32(out), eo, what="merged")


@pytest.mark.parametrize("bits,group,tokens,residual", [(2, 64, 3000, 300), (4, 128, 2500, 40), (2, 128, 640, 0),
                                                        (4, 32, 5000, 600)])
def test_decode_summary_groups_and_long_residual(device, bits, group, tokens, residual):
    cache, seg = _pair(tokens, 50 + bits, bits, group, residual, device)
    for lq in (1, 2):
        q = queries(lq, seed=60 + lq)
        out, lse = packed_kivi_attention_summary(cache, q.to(device))
        check_summary(out, lse, seg, q, what=f"G{group} Lq{lq}")


@pytest.mark.parametrize("bits", [2, 4])
def test_mq_config2_editing(device, bits):
    # config 2's packed segment: 1024 source-VAE tokens (896 packed + 128 residual),
    # 1088 queries x 28 heads (7616 query rows per KV head) through uc_kivi_attn_mq
    cache, seg = _pair(1024, 70 + bits, bits, 32, 128, device)
    assert (cache.quantized_tokens, cache.residual_tokens) == (896, 128)
    q = queries(1088, seed=71)
    out, lse = packed_kivi_attention_summary(cache, q.to(device))
    assert tuple(out.shape) == (1088, 28, 128) and tuple(lse.shape) == (28, 1088)
    check_summary(out, lse, seg, q, what=f"mq c2 {bits}-bit")
    po, pl = packed_kivi_quantized_attention_summary(cache, q.to(device))
    check_summary(po, pl, seg, q, include_residual=False, what=f"mq c2 packed-only {bits}-bit")


@pytest.mark.parametrize("bits,group,tokens,residual,lq", [(2, 32, 500, 20, 20), (4, 128, 700, 50, 3),
                                                           (2, 64, 1300, 130, 130), (4, 32, 96, 64, 300)])
def test_mq_ragged_tiles_and_rows(device, bits, group, tokens, residual, lq):
    # packed and residual lengths that end inside a 64-key tile, query rows that
    # end inside a 128-row workgroup
    cache, seg = _pair(tokens, 80 + lq, bits, group, residual, device)
    q = queries(lq, seed=81)
    out, lse = packed_kivi_attention_summary(cache, q.to(device))
    check_summary(out, lse, seg, q, what=f"mq G{group} T{tokens} Lq{lq}")


@pytest.mark.parametrize("lq,tokens,dense,qdtype", [(1171, 128 + 100, 1, torch.bfloat16), (1180, 700, 65, torch.float16),
                                                    (2345, 64, 300, torch.bfloat16), (3520, 200, 0, torch.bfloat16)])
def test_mq_workgroups_of_one_and_two_halves(device, lq, tokens, dense, qdtype):
    # 28/4 heads: 260 work items (4-wave workgroups: every tile in one half),
    # 516 (8 waves, two halves) and 772 (4 waves again), over 1 to 12 key tiles
    # that end inside a tile, all or none of them packed but one
    from unicache_amd.storage.kivi_cuda import packed_segments_summary

    cache, seg = _pair(tokens, 97, 2, 32, 37 if tokens > 100 else 0, device)
    dk, dv = kv_pair(dense, seed=98, dtype=qdtype)
    q = queries(lq, seed=99, dtype=qdtype)
    out, lse = packed_segments_summary([cache], q.to(device), [(dk.to(device), dv.to(device))])
    key, value = K.dequantize(seg, "fp32")
    rows = np.r_[0:40, lq // 2:lq // 2 + 40, lq - 40:lq]  # the oracle on a few rows of the first and last blocks
    eo, el = A.attention_summary(f32(q)[rows], np.concatenate([key, f32(dk)]), np.concatenate([value, f32(dv)]))
    assert_close(f32(out)[rows], eo, what="out")
    assert_close(f32(lse)[:, rows], el, max_abs=1e-2, mean_abs=1e-3, what="lse")
    # the other rows: every query row written, rows of one query head independent of their block
    assert torch.isfinite(out.float()).all() and torch.isfinite(lse).all()
    part, _ = packed_segments_summary([cache], q[5:700].to(device), [(dk.to(device), dv.to(device))])
    # (the fp32 results differ by rounding, so a bf16 output moves by one step at
    # most: 2^-5 = 0.03125 for outputs below 8, which an average of N(0,1) values is)
    assert float(out.abs().max()) < 8
    assert_close(f32(part), f32(out)[5:700], max_abs=0.0313, mean_abs=5e-4, what="part of the rows")


@pytest.mark.parametrize("dtype,tokens", [(torch.bfloat16, 4096), (torch.float16, 4096), (torch.bfloat16, 700)])
def test_mq_one_half_is_as_close_as_two(device, dtype, tokens):
    # 1200 queries (264 work items: one half) against two calls of 600 (132 items
    # each: two halves) on the same rows: fp32 outputs no further from 64 bits
    key, value = (x.to(device) for x in kv_pair(tokens, seed=190, dtype=dtype))
    q = queries(1200, seed=191, dtype=dtype).to(device)

    def attend(rows):
        out = torch.empty(rows.shape, dtype=torch.float32, device=device)
        seg = (nat.DenseSegment * 1)(nat.DenseSegment(key.data_ptr(), value.data_ptr(), tokens, 4 * 128, 128))
        nat.call("uc_kivi_attn_mq_segments", (nat.KiviItem * 1)(), 0, seg, 1, rows.data_ptr(), out.data_ptr(), None, 2, 32,
                 28, 4, 128, int(rows.shape[0]), nat.dtype_code(dtype), nat.dtype_code(dtype), nat.UC_FP32,
                 1.0 / math.sqrt(128), nat.stream(device))
        return out

    one, two = attend(q), torch.cat([attend(q[:600]), attend(q[600:])])
    assert not torch.equal(one, two)  # two kinds of workgroup
    exact = torch.empty(1200, 28, 128, dtype=torch.float64, device=device)
    for h in range(28):
        k, v = key[:, h // 7].double().t().contiguous(), value[:, h // 7].double().contiguous()
        exact[:, h] = torch.softmax((q[:, h].double().contiguous() @ k) / math.sqrt(128), -1) @ v
    assert float((one - exact).norm()) <= float((two - exact).norm())


def _kernels_of(run):
    """Kernel launches of run(), counted as the nodes of its captured graph."""

    import ctypes

    with open("/proc/self/maps") as maps:  # the HIP runtime that torch loaded
        hip = ctypes.CDLL(next(line.split()[-1] for line in maps if "libamdhip64" in line))
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        run()
    count = ctypes.c_size_t()
    assert hip.hipGraphGetNodes(ctypes.c_void_p(graph.raw_cuda_graph()), None, ctypes.byref(count)) == 0
    return count.value


# work items (128 rows x KV head) at 28/4 heads: 1200 queries 264, 1171 260 (an odd number of row blocks: the last
# pair has one), 4098 900 (one half each); 90, 300, 500 and 1088 at most 240, 2345 516 (two halves each)
@pytest.mark.parametrize("lens,odt,launches", [((300, 1200, 90), torch.bfloat16, 1), ((1171, 500), torch.float32, 1),
                                               ((2345, 1171), torch.float16, 1), ((300, 4098), torch.bfloat16, 1),
                                               ((1088, 1200), torch.float32, 2), ((1171, 1200), torch.float32, 1)])
def test_mq_table_of_both_kinds(device, lens, odt, launches):
    # one table call whose queries take workgroups of one half and of two: each
    # query equals its own call bit for bit
    cache, _ = _pair(600, 100, 2, 32, 40, device)
    qs = [queries(lq, seed=101 + i).to(device) for i, lq in enumerate(lens)]
    dense = [tuple(x.to(device) for x in kv_pair(70 + 64 * i, seed=110 + i)) for i in range(len(lens))]
    codes = (nat.UC_BF16, nat.UC_BF16, nat.dtype_code(odt), 1.0 / math.sqrt(128))

    def table(which, outs, lses):
        queries_ = (nat.MqQuery * len(which))()
        items, segs = (nat.KiviItem * len(which))(), (nat.DenseSegment * len(which))()
        for j, i in enumerate(which):
            queries_[j] = nat.MqQuery(qs[i].data_ptr(), outs[i].data_ptr(), lses[i].data_ptr(), lens[i], j, 1, j, 1)
            items[j] = cache.native_item(None, None, None, residual_key_ptr=cache.residual_key.data_ptr(),
                                         residual_value_ptr=cache.residual_value.data_ptr(),
                                         residual_tokens=cache.residual_tokens)
            key, value = dense[i]
            segs[j] = nat.DenseSegment(key.data_ptr(), value.data_ptr(), int(key.shape[0]), 4 * 128, 128)
        nat.call("uc_kivi_attn_mq_table", queries_, len(which), items, len(which), segs, len(which), 2, 32, 28, 4, 128,
                 *codes, nat.stream(device))

    def results():
        return ([torch.full(q.shape, float("nan"), dtype=odt, device=device) for q in qs],
                [torch.full((28, lq), float("nan"), device=device) for lq in lens])

    want, got = results(), results()
    for i in range(len(lens)):
        table([i], *want)
    assert _kernels_of(lambda: table(range(len(lens)), *got)) == launches
    for i in range(len(lens)):
        assert torch.isfinite(want[0][i].float()).all()
        assert torch.equal(got[0][i], want[0][i]) and torch.equal(got[1][i], want[1][i]), f"query {i}"


def test_mq_fp16_inputs(device):
    key, value = kv_pair(800, seed=90, dtype=torch.float16)
    cache = PackedKIVICache.from_dense(key.to(device), value.to(device), logical_token_ids=torch.arange(800),
                                       token_type_id=3, k_bits=2, v_bits=2, group_size=32,
                                       residual_length=128, backend="cuda")
    seg = K.from_dense(f32(key), f32(value), k_bits=2, v_bits=2, group_size=32, residual_length=128,
                       in_dtype="fp16")
    q = queries(64, seed=91, dtype=torch.float16)
    out, lse = packed_kivi_attention_summary(cache, q.to(device))
    assert out.dtype == torch.float16
    eo, el = A.packed_summary(seg, f32(q), include_residual=True, kv_dtype="fp32")
    assert_close(f32(out), eo, what="mq fp16")
    assert_close(f32(lse), el, max_abs=5e-3, mean_abs=1e-3, what="mq fp16 lse")


def test_mq_is_deterministic(device):
    cache, _ = _pair(1024, 95, 2, 32, 128, device)
    q = queries(200, seed=96).to(device)
    a, la = packed_kivi_attention_summary(cache, q)
    b, lb = packed_kivi_attention_summary(cache, q)
    assert torch.equal(a, b) and torch.equal(la, lb)


def test_batched_decode_doubled_split(device):
    # 100 items x 4 KV heads of 4096 packed + 128 residual tokens: 3 splits per
    # unit (1200 workgroups) exceed one round of slots, 2 splits (800) fit, so the
    # batch runs 16 super-tiles per split; each item alone runs 8
    from unicache_amd.storage.decode import KiviDecodeBatch

    g = torch.Generator(device=device).manual_seed(61)
    caches, qs = [], []
    for i in range(100):
        k = torch.randn(4224, 4, 128, generator=g, device=device).to(torch.bfloat16)
        v = torch.randn(4224, 4, 128, generator=g, device=device).to(torch.bfloat16)
        caches.append(PackedKIVICache.from_dense(k, v, logical_token_ids=torch.arange(4224, device=device),
                                                 token_type_id=3, k_bits=2, v_bits=2, group_size=32,
                                                 residual_length=128, backend="cuda"))
        qs.append(torch.randn(1, 28, 128, generator=g, device=device).to(torch.bfloat16))
    assert caches[0].quantized_tokens == 4096
    batch = KiviDecodeBatch(caches, qs)
    batch.run()
    for i in (0, 37, 99):
        out, lse = packed_kivi_attention_summary(caches[i], qs[i])
        assert_close(f32(batch.outputs[i]), f32(out), max_abs=5e-3, mean_abs=2e-4, what=f"item {i}")
        assert_close(f32(batch.lses[i]), f32(lse), max_abs=1e-4, mean_abs=1e-5, what=f"lse {i}")
