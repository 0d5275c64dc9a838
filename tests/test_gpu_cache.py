"""The compressed cache that grows (packkv_amd/cache.py) against the restated reference cache
(oracle/cache.py): dense view bit-exact, decode step within the attention tolerance, streams equal to a
one-shot encode."""
import numpy as np
import pytest
import torch

from oracle import cache as oc
from oracle import quant as oq
from packkv_amd import ops, synth
from packkv_amd.cache import PackKVCacheConfig, PackKVCompressedCache
from attn_bounds import check_fast, check_reference_mode, say as _say

pytestmark = pytest.mark.gpu


def _attend_parity(cache, layer, q, wk, wv, ek, ev, dtype, cuda, label):
    """cache.attend in the checking mode against the reference path at the contract, and the fast decode step
    against exact arithmetic, its distance to the reference path printed beside the contract (tests/attn_bounds.py).
    wk, wv: what the reference's update returns; ek, ev: the same tokens before their rounding to 16 bits (fp64).
    Only the tokens already in the streams are attended unrounded: a pending 64-token cut sits in the 16-bit window
    in dequantised form, like the buffer."""
    n = cache.layers[layer].k.tokens
    ek, ev = torch.cat([ek[:, :, :n], wk[:, :, n:].double()], dim=2), torch.cat([ev[:, :, :n], wv[:, :, n:].double()], dim=2)
    ref = oq.attention_f32(q.unsqueeze(2), wk, wv).squeeze(2)
    exact = oq.attention_f64_np(q.unsqueeze(2), ek, ev).squeeze(2)
    chk = cache.attend(q.to(cuda), layer, variant=1, ref_rounding=True, out_f32=True)
    check_reference_mode(chk, ref, label)
    check_fast(cache.attend(q.to(cuda), layer), ref, exact, dtype, label=label)


def _rope_tables(B, pos0, n, dtype):
    pos = torch.arange(pos0, pos0 + n, dtype=torch.float32)
    inv = 1.0 / (10000.0 ** (torch.arange(0, 128, 2, dtype=torch.float32) / 128))
    f = torch.outer(pos, inv)
    emb = torch.cat((f, f), dim=-1)
    return emb.cos().to(dtype).expand(B, n, 128).contiguous(), emb.sin().to(dtype).expand(B, n, 128).contiguous()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rope", [False, True])
def test_cache_matches_restated_reference(cuda, dtype, rope):
    B, Hq, H, T0, steps = 2, 8, 4, 300, 200
    k, v = synth.make_kv(B, H, T0 + steps, seed=90, dtype=dtype)
    want = oc.SimulatedCache(1, 64, 192, 0.1, 0.1, track_exact=True)
    got = PackKVCompressedCache(B, H, 128, 1, PackKVCacheConfig(64, 192, 0.1, 0.1), max_tokens=1024, dtype=dtype,
                                device=cuda)
    check_at = {0, 1, 18, 19, 20, 82, 83, 84, 146, 147, 148, 199}   # around the cuts at steps 19, 83, 147
    pos, tok = 0, 0
    for step in range(-1, steps):
        n = T0 if step < 0 else 1
        ks, vs = k[:, :, tok:tok + n], v[:, :, tok:tok + n]
        cos = sin = None
        if rope:
            cos, sin = _rope_tables(B, pos, n, dtype)
        wk, wv = want.update(ks, vs, 0, cos, sin)
        kw = {"cos": cos.to(cuda), "sin": sin.to(cuda)} if rope else None
        got.update(ks.to(cuda), vs.to(cuda), 0, kw, return_dense=False)
        tok += n
        pos += n
        assert got.get_seq_length(0) == want.get_seq_length(0) == tok
        if step in check_at or step < 0:
            _say("cache case", dtype, "rope" if rope else "plain", "step", step, "tokens", tok,
                 "compressed", got.layers[0].k.tokens, "window", got.layers[0].win_len)
            gk, gv = got.materialize(0)
            assert torch.equal(gk.cpu().view(torch.int16), wk.view(torch.int16))
            assert torch.equal(gv.cpu().view(torch.int16), wv.view(torch.int16))
            q = synth.make_q(B, Hq, seed=300 + step, dtype=dtype)
            ek, ev = want.exact(0)
            _attend_parity(got, 0, q, wk, wv, ek, ev, dtype, cuda, "step %d" % step)
    L = got.layers[0]
    # 500 tokens: 320 have been cut (128 at the prefill, then at steps 19, 83, 147) = 2 tiles + one pending cut
    assert L.k.tokens == L.v.tokens == 256 and L.pend == 64 and L.win_len == T0 + steps - 256


def test_append_equals_one_shot_encode(cuda):
    """Chunk-by-chunk append (K in cuts of 64 and 128 tokens, V of 128 and 256) gives the stream, block_info and
    parameters of one encode over all tokens."""
    B, H, T = 2, 4, 512
    k, v = synth.make_kv(B, H, T, seed=95, device=cuda)
    for is_k, x, chunks in ((True, k, (64, 128, 64, 256)), (False, v, (128, 256, 128))):
        one = ops.k_quant_encode(x, 0.1) if is_k else ops.v_quant_encode(x, 0.1)
        per_tok = (B * H) if is_k else (B * H * 2)
        nblk = T // (64 if is_k else 128) * per_tok
        stream = torch.zeros(one["size"] + 64, dtype=torch.uint8, device=cuda)
        info = torch.zeros(nblk, 2, dtype=torch.uint32, device=cuda)
        scale = torch.zeros(B, T + 128, dtype=x.dtype, device=cuda)     # rows longer than the token count
        zero = torch.zeros_like(scale)
        used, tok = 0, 0
        for n in chunks:
            _say("append case", "K" if is_k else "V", "tokens", tok, "+", n)
            used = ops.quant_encode_append(is_k, x[:, :, tok:tok + n].contiguous(), 0.1, one["bits"], stream, used,
                                           info, tok, scale, zero)
            tok += n
        assert tok == T and used == one["size"]
        assert torch.equal(stream[:used], one["stream"][:used])
        assert torch.equal(info.view(torch.int32), one["info"].view(torch.int32))
        assert torch.equal(scale[:, :T].view(torch.int16), one["scale"].view(torch.int16))
        assert torch.equal(zero[:, :T].view(torch.int16), one["zero"].view(torch.int16))


def test_append_reports_a_full_buffer(cuda):
    B, H = 1, 2
    k, _ = synth.make_kv(B, H, 128, seed=96, device=cuda)
    stream = torch.zeros(256, dtype=torch.uint8, device=cuda)
    info = torch.zeros(4, 2, dtype=torch.uint32, device=cuda)
    scale = torch.zeros(B, 128, dtype=k.dtype, device=cuda)
    with pytest.raises(RuntimeError):
        ops.quant_encode_append(True, k, 0.1, 4, stream, 0, info, 0, scale, torch.zeros_like(scale))


def test_cache_bytes_and_prefill_only(cuda):
    """A prompt below buffer_size stays uncompressed (utils/compute.py:54-67); a long prefill compresses all but
    128..191 tokens, in whole tiles."""
    B, H = 1, 8
    k, v = synth.make_kv(B, H, 1000, seed=97, device=cuda)
    c = PackKVCompressedCache(B, H, 128, 2, max_tokens=2048, device=cuda)
    c.update(k[:, :, :191], v[:, :, :191], 0, return_dense=False)
    assert c.layers[0].k.tokens == 0 and c.layers[0].win_len == 191
    assert c.cache_bytes(0) == 2 * B * H * 191 * 128 * 2
    c.update(k, v, 1, return_dense=False)     # 1000 tokens: 832 cut = 6 tiles + one pending cut of 64, 168 buffered
    L = c.layers[1]
    assert L.k.tokens == 768 and L.pend == 64 and L.win_len == 64 + 168 and c.get_seq_length(1) == 1000
    fp16_bytes = 2 * B * H * 1000 * 128 * 2
    assert c.cache_bytes(1) < 0.45 * fp16_bytes
    q = synth.make_q(B, 32, seed=98, device=cuda)
    gk, gv = c.materialize(1)
    ref = oq.attention_f32(q.cpu().unsqueeze(2), gk.cpu(), gv.cpu()).squeeze(2)
    out = c.attend(q.unsqueeze(2), 1)
    assert out.shape == (B, 32, 1, 128)
    # the reference path on the dense view: the checking mode at the contract; the fast step within the bound the
    # oracle gives (exact arithmetic = the restated quantiser's unrounded values for the 832 cut tokens)
    sim = oc.SimulatedCache(1, 64, 192, 0.1, 0.1, track_exact=True)
    wk, wv = sim.update(k.cpu(), v.cpu(), 0)
    assert torch.equal(gk.cpu().view(torch.int16), wk.view(torch.int16))
    ek, ev = sim.exact(0)
    ek, ev = torch.cat([ek[:, :, :768], wk[:, :, 768:].double()], dim=2), torch.cat([ev[:, :, :768], wv[:, :, 768:].double()], dim=2)
    exact = oq.attention_f64_np(q.cpu().unsqueeze(2), ek, ev).squeeze(2)
    check_reference_mode(c.attend(q, 1, variant=1, ref_rounding=True, out_f32=True), ref, "prefill 1000")
    check_fast(out[:, :, 0], ref, exact, torch.float16, label="prefill 1000")


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_window_append_is_the_reference_chain_bit_for_bit(cuda, dtype):
    """Rotary embedding of the new keys + append, one launch, against the reference's chain of 16-bit elementwise ops
    (utils/compute.py:35-43, restated in oracle/cache.py) evaluated by torch on the device: equal bits; contiguous
    and strided inputs (a transposed projection output, an expanded cos / sin table), one and several new tokens,
    with and without the embedding."""
    from oracle import cache as oc
    g = torch.Generator().manual_seed(400)
    B, H, cap = 3, 4, 40
    for n, pos, strided in ((1, 0, False), (1, 17, True), (5, 30, True), (8, 32, False)):
        _say("append case", dtype, n, pos, strided)
        if strided:     # [B, n, H, 128] storage seen as [B, H, n, 128], like a projection output after transpose(1, 2)
            k = (torch.randn(B, n, H, 128, generator=g) * 3).to(dtype).to(cuda).transpose(1, 2)
            v = torch.randn(B, n, H, 128, generator=g).to(dtype).to(cuda).transpose(1, 2)
            cos1, sin1 = _rope_tables(1, 100 + pos, n, dtype)
            cos, sin = cos1.to(cuda).expand(B, n, 128), sin1.to(cuda).expand(B, n, 128)
        else:
            k = (torch.randn(B, H, n, 128, generator=g) * 3).to(dtype).to(cuda)
            v = torch.randn(B, H, n, 128, generator=g).to(dtype).to(cuda)
            cos, sin = (t.to(cuda) for t in _rope_tables(B, 100 + pos, n, dtype))
        for rotary in (True, False):
            k_win = torch.full((B, H, cap, 128), 7.0, dtype=dtype, device=cuda)
            v_win = torch.full((B, H, cap, 128), 7.0, dtype=dtype, device=cuda)
            ops.window_append(k, v, cos if rotary else None, sin if rotary else None, k_win, v_win, pos)
            want_k = oc.apply_rotary_pos_emb_single(k, cos, sin) if rotary else k
            assert torch.equal(k_win[:, :, pos:pos + n].view(torch.int16), want_k.contiguous().view(torch.int16))
            assert torch.equal(v_win[:, :, pos:pos + n], v)
            rest = torch.ones(cap, dtype=torch.bool)
            rest[pos:pos + n] = False
            assert (k_win[:, :, rest] == 7.0).all() and (v_win[:, :, rest] == 7.0).all()     # nothing else written
    with pytest.raises(Exception):
        ops.window_append(k, v, None, None, k_win, v_win, cap - 2)                           # 8 rows do not fit


def test_cache_with_five_bit_codes(cuda):
    """rel 0.05 (5-bit codes, the format extension) through the growing cache: the fused encoders append, the
    asynchronous-copy attention kernel reads; dense view bit-exact with the restated reference cache, the decode
    step within the attention tolerance, across one cut."""
    B, Hq, H, T0, steps = 2, 8, 4, 300, 40
    dtype = torch.float16
    k, v = synth.make_kv(B, H, T0 + steps, seed=96, dtype=dtype)
    want = oc.SimulatedCache(1, 64, 192, 0.05, 0.05, track_exact=True)
    got = PackKVCompressedCache(B, H, 128, 1, PackKVCacheConfig(64, 192, 0.05, 0.05), max_tokens=1024, dtype=dtype,
                                device=cuda)
    assert got.config.k_bits == 5 and got.config.v_bits == 5
    tok = 0
    for step in range(-1, steps):
        n = T0 if step < 0 else 1
        ks, vs = k[:, :, tok:tok + n], v[:, :, tok:tok + n]
        wk, wv = want.update(ks, vs, 0, None, None)
        got.update(ks.to(cuda), vs.to(cuda), 0, None, return_dense=False)
        tok += n
        if step in (-1, 0, 19, 20, 39):
            _say("5-bit cache case step", step, "tokens", tok, "compressed", got.layers[0].k.tokens)
            gk, gv = got.materialize(0)
            assert torch.equal(gk.cpu().view(torch.int16), wk.view(torch.int16))
            assert torch.equal(gv.cpu().view(torch.int16), wv.view(torch.int16))
            q = synth.make_q(B, Hq, seed=500 + step, dtype=dtype)
            ek, ev = want.exact(0)
            _attend_parity(got, 0, q, wk, wv, ek, ev, dtype, cuda, "5-bit step %d" % step)
    assert got.layers[0].k.tokens == 128 and got.layers[0].pend == 64      # 128 at the prefill, one more cut waiting for its partner


def test_reference_cache_class_and_its_two_line_hook(cuda):
    """The reference builds ``PackKVCache(batch, heads, head_dim, layers)`` (models/llama.py:830-833), configured
    through ``PackKVCacheConfigStatic.config``, and its attention modules run (models/llama.py:260-261)

        cache_kwargs = {"sin": sin, "cos": cos, "cache_position": cache_position}
        key_states, value_states = past_key_value.update(key_states, value_states, self.layer_idx, cache_kwargs)

    The drop-in class takes both lines as they stand: it is a transformers.Cache, and update returns the dense K and V
    of the restated reference cache bit for bit -- prompt pass and decode steps across a cut, two layers."""
    import transformers
    from packkv_amd.cache import PackKVCache, PackKVCacheConfigStatic
    dtype = torch.float16
    B, H, T0, steps, layers = 2, 4, 300, 70, 2
    k, v = synth.make_kv(B, H, T0 + steps, seed=610, dtype=dtype)
    PackKVCacheConfigStatic.config = PackKVCacheConfig(64, 192, 0.1, 0.1)
    PackKVCacheConfigStatic.max_tokens = 1024
    try:
        past_key_value = PackKVCache(B, H, 128, layers)
        assert isinstance(past_key_value, transformers.Cache)
        want = oc.SimulatedCache(layers, 64, 192, 0.1, 0.1)
        pos = 0
        for step in range(-1, steps):
            n = T0 if step < 0 else 1
            cos, sin = _rope_tables(B, pos, n, dtype)
            cache_position = torch.arange(pos, pos + n)
            for layer_idx in range(layers):
                key_states = (k[:, :, pos:pos + n] * (1 + layer_idx)).to(cuda)
                value_states = v[:, :, pos:pos + n].to(cuda)
                wk, wv = want.update(key_states.cpu(), value_states.cpu(), layer_idx, cos, sin)
                sin_d, cos_d = sin.to(cuda), cos.to(cuda)
                # the reference's two lines, with sin / cos on the device
                cache_kwargs = {"sin": sin_d, "cos": cos_d, "cache_position": cache_position}
                key_states, value_states = past_key_value.update(key_states, value_states, layer_idx, cache_kwargs)
                if step < 0 or step in (0, 18, 19, 20, 69):
                    _say("reference hook: step", step, "layer", layer_idx, "K", tuple(key_states.shape))
                    assert key_states.shape == wk.shape and value_states.shape == wv.shape
                    assert torch.equal(key_states.cpu().view(torch.int16), wk.view(torch.int16))
                    assert torch.equal(value_states.cpu().view(torch.int16), wv.view(torch.int16))
            pos += n
            assert past_key_value.get_seq_length(0) == past_key_value.get_seq_length(1) == pos
    finally:
        PackKVCacheConfigStatic.config = None
        PackKVCacheConfigStatic.max_tokens = 32768


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rel,T_c,T_w", [(0.5, 128, 1), (0.2, 384, 64), (0.1, 256, 65), (0.1, 0, 191), (0.05, 128, 0), (0.025, 256, 63),
                                         (0.0125, 128, 130), (0.00625, 128, 5)])
def test_dense_view_equals_the_restated_dequantisation(cuda, dtype, rel, T_c, T_w):
    """Widths 2..8, with and without compressed tokens, window rows around the 64-row pieces: bit for bit (the window
    is a copy, and every dequantised element is two single roundings of exact values)."""
    B, H, cap = 2, 3, 200
    k, v = synth.make_kv(B, H, max(T_c, 128), seed=77, dtype=dtype)
    kw, vw = synth.make_kv(B, H, cap, seed=78, dtype=dtype)
    sides, want = [], []
    for x, w, enc in ((k, kw, ops.k_quant_encode), (v, vw, ops.v_quant_encode)):
        parts = [w[:, :, :T_w]]
        if T_c:
            c, z, s = oq.quant_ints(x, 64, rel)
            parts.insert(0, oq.dequant(c, z, s))
        want.append(torch.cat(parts, dim=2))
        sides.append(dict(enc(x.to(cuda), rel), heads=H) if T_c else None)
    got = ops.dense_view(sides[0], sides[1], kw.to(cuda), vw.to(cuda), T_w)
    for g, w in zip(got, want):
        assert g.shape == w.shape and torch.equal(g.cpu().view(torch.int16), w.view(torch.int16))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,T,rel", [(1, 1, 128, 0.1), (3, 3, 256, 0.1), (2, 4, 384, 0.05), (2, 8, 256, 0.1), (1, 8, 128, 0.05), (2, 12, 256, 0.1)])
def test_append_reads_the_rows_where_they_are(cuda, dtype, B, H, T, rel):
    """K and V as transposed projection outputs ([B, T, heads, 128] slices, heads beside them) appended in two pieces,
    one wait for both sides: the streams, tables and parameters of one encode of the contiguous tensors."""
    k, v = synth.make_kv(B, H, T, seed=31, dtype=dtype, device=cuda)
    both = torch.stack((k, v), dim=2).permute(0, 3, 1, 2, 4).reshape(B, T, 2 * H, 128).contiguous()
    kt, vt = both[:, :, 0::2].transpose(1, 2), both[:, :, 1::2].transpose(1, 2)
    assert not kt.is_contiguous() and torch.equal(kt, k) and torch.equal(vt, v)
    want = (ops.k_quant_encode(k, rel), ops.v_quant_encode(v, rel))
    bits, row = want[0]["bits"], T + 128
    sides = []
    for w in want:
        sides.append([rel, bits, torch.empty(w["stream"].numel() + 64, dtype=torch.uint8, device=cuda), 0,
                      torch.empty(2 * w["info"].size(0), 2, dtype=torch.uint32, device=cuda),
                      torch.empty(B, row, dtype=dtype, device=cuda), torch.empty(B, row, dtype=dtype, device=cuda)])
    first = T // 2 // 128 * 128
    for lo, n in ((0, first), (first, T - first)):
        if n:
            sides[0][3], sides[1][3] = ops.kv_quant_encode_append(kt[:, :, lo:], vt[:, :, lo:], n, sides[0], sides[1], lo)
    for w, s in zip(want, sides):
        assert s[3] == w["size"] and torch.equal(s[2][:s[3]], w["stream"][:w["size"]])
        assert torch.equal(s[4][:w["info"].size(0)].view(torch.int32), w["info"].view(torch.int32))
        assert torch.equal(s[5][:, :T], w["scale"]) and torch.equal(s[6][:, :T], w["zero"])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("pend,buf,n,rope", [(0, 0, 300, True), (0, 0, 1, False), (64, 150, 70, True), (64, 64, 257, False), (0, 191, 1, True)])
def test_window_cut_moves_every_row(cuda, dtype, pend, buf, n, rope):
    """The rows of a cut against the same chain of torch operations (rotary embedding, concatenation, slices): staged
    tokens, the new pending originals and the window are copies or single 16-bit roundings, hence bit for bit; the
    pending rows of the window are quant_params / quantize / dequantize of those originals."""
    from packkv_amd.cache import apply_rotary_pos_emb_single
    B, H, cap = 2, 3, 320
    k, v = synth.make_kv(B, H, 64 + cap + n, seed=41, dtype=dtype, device=cuda)
    kp, vp, kw, vw = k[:, :, :64].contiguous(), v[:, :, :64].contiguous(), k[:, :, 64:64 + cap].contiguous(), v[:, :, 64:64 + cap].contiguous()
    kn, vn = k[:, :, 64 + cap:], v[:, :, 64 + cap:]
    cos, sin = (t.to(cuda) for t in _rope_tables(B, 7, n, dtype)) if rope else (None, None)
    kr = apply_rotary_pos_emb_single(kn, cos, sin) if rope else kn
    ks = torch.cat(([kp] if pend else []) + [kw[:, :, pend:pend + buf], kr], dim=2)
    vs = torch.cat(([vp] if pend else []) + [vw[:, :, pend:pend + buf], vn], dim=2)
    stage, pend_out = max(0, ks.size(2) - 200) // 128 * 128, 64 if ks.size(2) >= 64 else 0
    got = ops.window_cut(kn, vn, cos, sin, kp if pend else None, vp if pend else None, kw, vw, pend + buf, stage, pend_out, 0.1, 0.05)
    for x, st, po, w, rel in ((ks, got[0], got[2], got[4], 0.1), (vs, got[1], got[3], got[5], 0.05)):
        assert torch.equal(st[:, :, :stage], x[:, :, :stage])
        if pend_out:
            cut = x[:, :, stage:stage + 64].contiguous()
            assert torch.equal(po, cut)
            scale, zero = ops.quant_params(cut, rel)
            want = ops.dequantize(ops.quantize(cut, scale, zero)[0], scale, zero, B, H)
            assert torch.equal(w[:, :, :64], want)
        assert torch.equal(w[:, :, pend_out:x.size(2) - stage], x[:, :, stage + pend_out:])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,T,rel", [(1, 5, 128, 0.1), (2, 8, 256, 0.1), (3, 7, 128, 0.05), (1, 8, 384, 0.2), (2, 12, 256, 0.1), (1, 32, 128, 0.05)])
def test_keys_rotated_by_the_encoder(cuda, dtype, B, H, T, rel):
    """K appended with cos / sin tables -- one table for all sequences, one each, a prompt laid out [B, T, H, 128], and the
    second half of a prompt's rows -- gives the stream, table and parameters of encoding the keys rotated by torch, a
    negative zero and a subnormal among them (bit for bit: the roundings are the same)."""
    from packkv_amd.cache import apply_rotary_pos_emb_single
    k, v = synth.make_kv(B, H, T, seed=61, dtype=dtype, device=cuda)
    k[:, :, 3, 5] = -0.0
    k[:, :, 4, 70] = 6e-8
    kt = k.transpose(1, 2).contiguous().transpose(1, 2)
    for shared, x, lo in ((True, k, 0), (False, kt, 0), (True, kt, 128)):
        n = T - lo
        if n <= 0:
            continue
        _say("rotated keys", dtype, B, H, T, rel, "shared table", shared, "from", lo)
        cos, sin = (t.to(cuda) for t in _rope_tables(1 if shared else B, 9, n, dtype))
        cos, sin = cos.expand(B, n, 128), sin.expand(B, n, 128)
        kr = apply_rotary_pos_emb_single(x[:, :, lo:], cos, sin).contiguous()
        want = (ops.k_quant_encode(kr, rel), ops.v_quant_encode(v[:, :, lo:].contiguous(), rel))
        sides = [[rel, w["bits"], torch.empty(w["stream"].numel() + 64, dtype=torch.uint8, device=cuda), 0, torch.empty_like(w["info"]),
                  torch.empty_like(w["scale"]), torch.empty_like(w["zero"])] for w in want]
        vx = v if x is k else v.transpose(1, 2).contiguous().transpose(1, 2)
        sizes = ops.kv_quant_encode_append(x[:, :, lo:], vx[:, :, lo:], n, sides[0], sides[1], 0, cos, sin)
        for w, s, size in zip(want, sides, sizes):
            assert size == w["size"] and torch.equal(s[2][:size], w["stream"][:size])
            assert torch.equal(s[4].view(torch.int32), w["info"].view(torch.int32))
            assert torch.equal(s[5], w["scale"]) and torch.equal(s[6], w["zero"])


def test_a_cut_on_another_stream_keeps_the_window_it_reads(cuda):
    """The prompt on one stream, a cut that waits for nothing queued on a second one: the first stream's next allocations
    must not get the window that the cut has still to read (and may write to what they get)."""
    B, H = 2, 4
    k, v = synth.make_kv(B, H, 230, seed=17, device=cuda)
    want = PackKVCompressedCache(B, H, 128, 1, max_tokens=512, device=cuda)
    for lo, hi in ((0, 130), (130, 230)):
        want.update(k[:, :, lo:hi], v[:, :, lo:hi], 0, return_dense=False)
    want = want.materialize(0)
    torch.cuda.synchronize()
    prompt, decode = torch.cuda.Stream(), torch.cuda.Stream()
    got = PackKVCompressedCache(B, H, 128, 1, max_tokens=512, device=cuda)
    with torch.cuda.stream(prompt):
        got.update(k[:, :, :130], v[:, :, :130], 0, return_dense=False)
    L = got.layers[0]
    old, shape = {L.k_win.data_ptr(), L.v_win.data_ptr()}, L.k_win.shape
    decode.wait_stream(prompt)
    with torch.cuda.stream(decode):
        torch.cuda._sleep(50_000_000)
        got.update(k[:, :, 130:], v[:, :, 130:], 0, return_dense=False)
        done = decode.record_event()
    assert L.k.tokens == 0 and L.pend == 64                   # a pending block only: nothing was waited for
    with torch.cuda.stream(prompt):
        others = [torch.full(shape, 7.0, dtype=torch.float16, device=cuda) for _ in range(4)]
        early = not done.query()
    assert early, "the cut had run before the other stream allocated"
    assert not old & {t.data_ptr() for t in others}
    prompt.wait_event(done)
    with torch.cuda.stream(prompt):
        dense = got.materialize(0)
    torch.cuda.synchronize()
    assert torch.equal(dense[0], want[0]) and torch.equal(dense[1], want[1])


def _placed(x, how):
    """x where an encoder cannot read it in 16-byte rows: contiguous but 8 bytes past a 16-byte boundary, or with an odd
    stride in a dimension of one element."""
    if how == "offset":
        out = torch.empty(x.numel() + 4, dtype=x.dtype, device=x.device)[4:].view(x.shape)
    else:
        out = torch.empty(x.numel(), dtype=x.dtype, device=x.device).as_strided(x.shape, (x.numel() // x.size(0) + 3,) + x.stride()[1:])
    assert out.is_contiguous() and (out.data_ptr() % 16 == 8 or out.stride(0) % 8 == 3)
    return out.copy_(x)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("B,how", [(2, "offset"), (1, "stride")])
def test_cuts_take_tokens_and_tables_at_any_address(cuda, dtype, rope, B, how):
    """A prompt that is encoded, a cut that makes a pending block, one that joins it and a prompt that ends in one, each
    from tensors that are contiguous in torch's eyes only: the streams, pending originals and windows of a cache that was
    given ordinary tensors."""
    H, sizes = 5, (300, 1, 82, 64, 257)
    k, v = synth.make_kv(B, H, sum(sizes), seed=51, dtype=dtype, device=cuda)
    caches = [PackKVCompressedCache(B, H, 128, 1, max_tokens=1024, dtype=dtype, device=cuda) for _ in range(2)]
    pos, states = 0, []
    for n in sizes:
        _say("tokens", pos, n, dtype, rope, B, how)
        ks, vs = k[:, :, pos:pos + n].contiguous(), v[:, :, pos:pos + n].contiguous()
        kw = dict(zip(("cos", "sin"), (t.to(cuda) for t in _rope_tables(B, pos, n, dtype)))) if rope else None
        caches[0].update(ks, vs, 0, kw, return_dense=False)
        caches[1].update(_placed(ks, how), _placed(vs, how), 0, kw and {a: _placed(t, how) for a, t in kw.items()}, return_dense=False)
        pos += n
        a, b = caches[0].layers[0], caches[1].layers[0]
        states.append((b.k.tokens, b.pend))
        assert (a.k.used, a.v.used, a.k.tokens, a.win_len, a.pend) == (b.k.used, b.v.used, b.k.tokens, b.win_len, b.pend)
        for x, y in zip(caches[0].materialize(0), caches[1].materialize(0)):
            assert torch.equal(x, y)
        if a.pend:
            assert torch.equal(a.k_pend, b.k_pend) and torch.equal(a.v_pend, b.v_pend)
    assert states == [(128, 0), (128, 0), (128, 64), (256, 0), (512, 64)]


def test_tensors_on_another_device_are_refused_before_a_launch(cuda):
    """Host tables, windows, parameters and streams beside device tokens: an error, on the append between cuts, on a cut, in
    the encode and in the dense view."""
    B, H = 1, 5
    k, v = synth.make_kv(B, H, 256, seed=5, device=cuda)
    host = torch.empty(B, H, 320, 128, dtype=torch.float16)
    for n in (1, 256):                                        # an append, a cut
        cos, sin = _rope_tables(B, 0, n, torch.float16)
        for c, s in ((cos, sin), (cos.to(cuda), sin), (cos, sin.to(cuda))):
            cache = PackKVCompressedCache(B, H, 128, 1, max_tokens=512, device=cuda)
            with pytest.raises(RuntimeError, match="one device"):
                cache.update(k[:, :, :n], v[:, :, :n], 0, {"cos": c, "sin": s}, return_dense=False)
    win = host.to(cuda)
    for kw, vw in ((host, win), (win, host)):
        with pytest.raises(RuntimeError, match="one device"):
            ops.window_append(k[:, :, :1], v[:, :, :1], None, None, kw, vw, 0)
        with pytest.raises(RuntimeError, match="one device"):
            ops.window_cut(k, v, None, None, None, None, kw, vw, 0, 128, 0, 0.1, 0.1)
    ke, ve = ops.k_quant_encode(k, 0.1), ops.v_quant_encode(v, 0.1)
    side = lambda e: [0.1, e["bits"], e["stream"], 0, e["info"], e["scale"], e["zero"]]
    for f in (5, 6):
        ks, vs = side(ke), side(ve)
        vs[f] = vs[f].cpu()
        with pytest.raises(RuntimeError, match="one device"):
            ops.kv_quant_encode_append(k, v, 256, ks, vs, 0)
        with pytest.raises(RuntimeError, match="one device"):
            ops.dense_view(ke, dict(ve, **{("scale", "zero")[f - 5]: vs[f]}))
    for kw, vw in ((win, host), (host, win)):
        with pytest.raises(RuntimeError, match="one device"):
            ops.dense_view(ke, ve, kw, vw, 1)


@pytest.mark.parametrize("side", ["k", "v"])
@pytest.mark.parametrize("why", ["capacity", "bits"])
def test_encode_status_after_a_joint_append_that_failed(cuda, side, why):
    """A stream of K or of V that does not fit its buffer, or codes that do not fit their width: the append raises, and so
    does encode_status behind it.  After one that went well it gives V's size."""
    k, v = synth.make_kv(1, 5, 256, seed=23, device=cuda)
    enc = {"k": ops.k_quant_encode(k, 0.1), "v": ops.v_quant_encode(v, 0.1)}
    sides = {s: [0.1, e["bits"], torch.empty_like(e["stream"]), 0, e["info"], e["scale"], e["zero"]] for s, e in enc.items()}
    assert ops.kv_quant_encode_append(k, v, 256, sides["k"], sides["v"], 0) == (enc["k"]["size"], enc["v"]["size"])
    assert ops.encode_status(cuda, bits=4) == enc["v"]["size"]
    if why == "capacity":
        sides[side][2] = sides[side][2][:1024]
    else:
        sides[side][1] = 2
    for call in (lambda: ops.kv_quant_encode_append(k, v, 256, sides["k"], sides["v"], 0), lambda: ops.encode_status(cuda, bits=sides["v"][1])):
        with pytest.raises(ops.PackKVError) as e:
            call()
        assert e.value.code == (4 if why == "capacity" else 1)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,n,layout,shared", [(1, 5, 320, "bhnd", True), (2, 5, 363, "bnhd", True), (2, 8, 300, "bnhd", False),
                                                 (2, 8, 512, "bhnd", False), (1, 12, 380, "bnhd", True), (2, 12, 447, "bhnd", False)])
def test_prompt_rotated_in_the_encoder_or_before_it(cuda, monkeypatch, dtype, B, H, n, layout, shared):
    """A first prompt by both routes, with a whole number of tiles and with a pending cut behind them, as [B, H, n, 128] and
    as a transposed [B, n, H, 128], one rotary table for all sequences and one each: the same streams, tables, parameters,
    pending originals and window, and the dense view of the restated reference cache."""
    from packkv_amd import cache as cache_mod
    k, v = synth.make_kv(B, H, n, seed=71, dtype=dtype)
    cos, sin = _rope_tables(1 if shared else B, 5, n, dtype)
    if not shared:
        for b in range(1, B):
            cos[b], sin[b] = (t[0] for t in _rope_tables(1, 5 + 40 * b, n, dtype))
    cos, sin = cos.expand(B, n, 128), sin.expand(B, n, 128)
    want = oc.SimulatedCache(1, 64, 192, 0.1, 0.1).update(k, v, 0, cos, sin)
    place = (lambda x: x.to(cuda)) if layout == "bhnd" else (lambda x: x.to(cuda).transpose(1, 2).contiguous().transpose(1, 2))
    dev = [place(k), place(v), (cos[:1] if shared else cos).to(cuda).expand(B, n, 128), (sin[:1] if shared else sin).to(cuda).expand(B, n, 128)]
    cut, routes = ops.window_cut, []

    def spy(*args, rotary_later=False, **kw):
        routes.append(rotary_later)
        return cut(*args, rotary_later=rotary_later, **kw)

    monkeypatch.setattr(ops, "window_cut", spy)
    layers = []
    for limit in (0, 1 << 62):
        monkeypatch.setattr(cache_mod, "ROTATE_IN_ENCODER", limit)
        cache = PackKVCompressedCache(B, H, 128, 1, max_tokens=512, dtype=dtype, device=cuda)
        _say("prompt", dtype, B, H, n, layout, "one table" if shared else "a table each", "limit", limit)
        dense = cache.update(dev[0], dev[1], 0, {"cos": dev[2], "sin": dev[3]})
        for g, w in zip(dense, want):
            assert torch.equal(g.cpu().view(torch.int16), w.view(torch.int16))
        layers.append(cache.layers[0])
    assert routes == [True, False]
    a, b = layers
    assert a.k.tokens and (a.k.tokens, a.pend, a.win_len) == (b.k.tokens, b.pend, b.win_len)
    for x, y in ((a.k, b.k), (a.v, b.v)):
        blocks = x.tokens // 128 * x.blocks_per_tile
        assert x.used == y.used and torch.equal(x.stream[:x.used], y.stream[:x.used])
        assert torch.equal(x.info[:blocks].view(torch.int32), y.info[:blocks].view(torch.int32))
        assert torch.equal(x.scale[:, :x.tokens], y.scale[:, :x.tokens]) and torch.equal(x.zero[:, :x.tokens], y.zero[:, :x.tokens])
    assert (a.k_pend is None) == (a.pend == 0) and (a.pend == 0 or torch.equal(a.k_pend, b.k_pend) and torch.equal(a.v_pend, b.v_pend))
    assert torch.equal(a.k_win[:, :, :a.win_len], b.k_win[:, :, :a.win_len]) and torch.equal(a.v_win[:, :, :a.win_len], b.v_win[:, :, :a.win_len])
