"""GPU parity of the quantizer and the fused quantize+encode kernels: integer codes, scale, zero,
dequantised values and the packed stream are bit-exact against the CPU oracle."""
import ctypes

import numpy as np
import pytest
import torch

from oracle import quant as oq
from packkv_amd import _lib, ops, synth

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, flush=True)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rel", [0.1, 0.2, 0.14])
def test_quantizer_bit_exact(cuda, dtype, rel):
    B, H, T = 2, 8, 256
    k, v = synth.make_kv(B, H, T, seed=21, dtype=dtype)
    for name, x in (("k", k), ("v", v)):
        _say("quant case", name, dtype, rel)
        c, z, s = oq.quant_ints(x, 64, rel)
        want_codes = oq.code_matrix(c)
        xd = x.to(cuda)
        scale, zero = ops.quant_params(xd, rel)
        assert torch.equal(scale.cpu().view(torch.int16), s.reshape(B, T).view(torch.int16))
        assert torch.equal(zero.cpu().view(torch.int16), z.reshape(B, T).view(torch.int16))
        codes, mx = ops.quantize(xd, scale, zero)
        assert torch.equal(codes.cpu(), want_codes)
        assert mx == int(want_codes.max())
        y = ops.dequantize(codes, scale, zero, B, H)
        want_y = oq.dequant(c, z, s)
        assert torch.equal(y.cpu().view(torch.int16), want_y.view(torch.int16))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,T", [(1, 1, 1), (2, 8, 37), (3, 9, 64), (1, 20, 100)])
def test_parameters_and_codes_in_one_pass(cuda, dtype, B, H, T):
    """As quant_params and quantize give them, bit for bit: rows in registers, more heads than those hold, a last workgroup
    of fewer than 16 tokens, and tokens with NaN and infinities."""
    k, v = synth.make_kv(B, H, T, seed=22, dtype=dtype, device=cuda)
    if T > 3:
        k[0, 0, 1, 5], v[0, H - 1, 2], v[0, :, 3], k[B - 1, 0, T - 1, 127] = float("nan"), float("nan"), float("inf"), -float("inf")
    rels = (0.1, 0.03)
    for (codes, scale, zero), x, rel in zip(ops.quant_codes_pair(k, v, *rels), (k, v), rels):
        _say("one pass", dtype, B, H, T, rel)
        ws, wz = ops.quant_params(x, rel)
        want, _ = ops.quantize(x, ws, wz)
        one = ops.quant_codes(x, rel)
        for c, s, z in ((codes, scale, zero), one):
            assert torch.equal(s.view(torch.int16), ws.view(torch.int16)) and torch.equal(z.view(torch.int16), wz.view(torch.int16))
            assert torch.equal(c, want)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_fused_quant_encode_stream_bit_exact(cuda, oracle_codec, dtype):
    for (B, H, T, rel) in ((1, 2, 128, 0.1), (2, 8, 256, 0.1), (1, 32, 128, 0.1), (2, 4, 256, 0.2), (1, 8, 128, 0.34),
                           (1, 3, 128, 0.1), (2, 5, 256, 0.14), (3, 1, 128, 0.1),
                           # five to eight heads: the kernels that read x once as cells (unused head slots repeat a head)
                           (1, 6, 256, 0.1), (3, 7, 128, 0.2), (2, 7, 256, 0.05), (1, 6, 128, 0.03),
                           # few heads: several groups to a workgroup, the last workgroup partly filled
                           (3, 2, 384, 0.1), (5, 1, 256, 0.1), (3, 3, 384, 0.2), (3, 4, 128, 0.1),
                           # widths 5 and 6 (format extension): cells / round-major kernels up to eight heads, runs of eight beyond
                           (2, 8, 256, 0.05), (1, 4, 384, 0.03), (1, 3, 128, 0.05), (1, 16, 128, 0.05), (2, 12, 256, 0.03)):
        k, v = synth.make_kv(B, H, T, seed=31 + H, dtype=dtype)
        for is_k, x in ((1, k), (0, v)):
            _say("fused quant+encode", "K" if is_k else "V", dtype, B, H, T, rel)
            c, z, s = oq.quant_ints(x, 64, rel)
            cm = oq.code_matrix(c).numpy()
            W = ops.bits_for_rel(rel)
            assert oq.bits_for_codes(torch.from_numpy(cm)) <= W
            cb, hb = (64, 128) if is_k else (128, 64)
            so, io, zo = oracle_codec.encode(is_k, cm, cb, hb, W)
            r = (ops.k_quant_encode if is_k else ops.v_quant_encode)(x.to(cuda), rel, W)
            assert r["size"] == zo
            assert np.array_equal(r["info"].cpu().numpy(), io)
            assert np.array_equal(r["stream"][:zo].cpu().numpy(), so[:zo])
            assert torch.equal(r["scale"].cpu().view(torch.int16), s.reshape(B, T).view(torch.int16))
            assert torch.equal(r["zero"].cpu().view(torch.int16), z.reshape(B, T).view(torch.int16))


def test_fused_quant_encode_more_than_eight_heads(cuda, oracle_codec):
    """More than eight KV heads: the heads of a (context block, sequence) are cut into runs of eight, one workgroup
    each, that exchange their minima and maxima through memory; hundreds of runs in flight, groups of 3, 4 and 5 runs,
    a last run of fewer than eight heads."""
    for (B, H, T, rel, dtype) in ((4, 32, 2048, 0.1, torch.float16), (2, 24, 1024, 0.2, torch.bfloat16),
                                  (1, 40, 512, 0.1, torch.float16), (3, 20, 512, 0.05, torch.float16)):
        k, v = synth.make_kv(B, H, T, seed=3 + H, dtype=dtype)
        for is_k, x in ((1, k), (0, v)):
            _say("fused quant+encode, many heads", "K" if is_k else "V", dtype, B, H, T, rel)
            c, z, s = oq.quant_ints(x, 64, rel)
            cm = oq.code_matrix(c).numpy()
            W = ops.bits_for_rel(rel)
            cb, hb = (64, 128) if is_k else (128, 64)
            so, io, zo = oracle_codec.encode(is_k, cm, cb, hb, W)
            for rep in range(2):                      # (twice: the exchange words of the first call must not leak into the second)
                r = (ops.k_quant_encode if is_k else ops.v_quant_encode)(x.to(cuda), rel, W)
                assert r["size"] == zo
                assert np.array_equal(r["info"].cpu().numpy(), io)
                assert np.array_equal(r["stream"][:zo].cpu().numpy(), so[:zo])
                assert torch.equal(r["scale"].cpu().view(torch.int16), s.reshape(B, T).view(torch.int16))
                assert torch.equal(r["zero"].cpu().view(torch.int16), z.reshape(B, T).view(torch.int16))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_fused_quant_encode_offset_rows_bit_exact(cuda, oracle_codec, dtype):
    """Rows far from zero: the zero point is large (here about -750 and +750, and a few hundred for the smaller
    shift), which takes the encoders' general rounding sequence for some tokens and the short one for others;
    ties (quotients at exactly k + 0.5) are common because the shifted fp16 values are multiples of 0.5."""
    B, H, T, rel = 2, 4, 256, 0.1
    k, v = synth.make_kv(B, H, T, seed=77)
    shift = torch.zeros(B, 1, T, 1)
    big, small = (600.0, 150.0) if dtype == torch.float16 else (48.0, 12.0)    # bf16 keeps 8 bits: stay where it resolves the rows
    shift[:, :, 0:128:3] = -big          # first half: every 16-token round holds tokens of both kinds
    shift[:, :, 1:128:3] = big
    shift[:, :, 2:128:6] = small
    shift[:, :, 128::2] = big            # second half: large positive zero points only (the short sequence)
    shift[:, :, 129::4] = small
    for is_k, x0 in ((1, v), (0, v)):          # unit-variance rows, so that the codes stay within 4 bits
        x = (x0.float() + shift).to(dtype)
        c, z, s = oq.quant_ints(x, 64, rel)
        zi = z.float().flatten()
        if dtype == torch.float16:
            assert (zi.abs() > 600).any() and (zi.abs() < 400).any()
        else:
            assert (zi.abs() > 40).any()
        cm = oq.code_matrix(c).numpy()
        assert int(cm.max()) <= 15
        cb, hb = (64, 128) if is_k else (128, 64)
        so, io, zo = oracle_codec.encode(is_k, cm, cb, hb, 4)
        r = (ops.k_quant_encode if is_k else ops.v_quant_encode)(x.to(cuda), rel, 4)
        assert r["size"] == zo
        assert np.array_equal(r["stream"][:zo].cpu().numpy(), so[:zo])
        assert torch.equal(r["zero"].cpu().view(torch.int16), z.reshape(B, T).view(torch.int16))
        codes, _ = ops.quantize(x.to(cuda), r["scale"], r["zero"])
        assert np.array_equal(codes.cpu().numpy(), cm)


def test_code_wider_than_bits_is_reported(cuda):
    k, _ = synth.make_kv(1, 2, 128, seed=5)
    with pytest.raises(ops.PackKVError) as e:
        ops.k_quant_encode(k.to(cuda), 0.1, 3)     # codes reach 10..11: needs 4 bits
    assert e.value.code == 1 and "does not fit" in str(e.value)


@pytest.mark.gpu
def test_fused_quant_encode_round_trip_medium(cuda):
    """Size-independent property at a size the CPU oracle would take minutes for: unpacking the fused
    encoder's stream gives back exactly the codes of the stand-alone quantizer."""
    B, H, T, rel = 4, 8, 4096, 0.1
    k, v = synth.make_kv(B, H, T, seed=77)
    for is_k, x in ((True, k), (False, v)):
        x = x.to(cuda)
        r = (ops.k_quant_encode if is_k else ops.v_quant_encode)(x, rel, 4)
        scale, zero = ops.quant_params(x, rel)
        assert torch.equal(scale, r["scale"]) and torch.equal(zero, r["zero"])
        codes, _ = ops.quantize(x, scale, zero)
        back = torch.empty_like(codes)
        if is_k:
            ops.k_decode(r["stream"], r["info"], back, 64, 128, 4)
        else:
            ops.v_decode(r["stream"], r["info"], back, 128, 64, 4)
        assert torch.equal(back, codes)


@pytest.mark.gpu
def test_fused_quant_encode_round_trip_full_size(cuda):
    """The benchmark workload itself (16 x 8 heads x 32768 tokens, 1 GiB of fp16 per tensor): block_info tiles the
    stream without gaps, and unpacking the stream reproduces the stand-alone quantizer's codes."""
    B, H, T, rel = 16, 8, 32768, 0.1
    k, v = synth.make_kv(B, H, T, seed=0, device=cuda)
    for is_k, x in ((True, k), (False, v)):
        r = (ops.k_quant_encode if is_k else ops.v_quant_encode)(x, rel, 4)
        info = r["info"].view(-1, 2).to(torch.int64)
        assert int(info[0, 0]) == 0
        assert torch.equal(info[1:, 0], torch.cumsum(info[:-1, 1], 0))          # back to back, in block order
        assert int(info[-1, 0] + info[-1, 1]) == r["size"]
        scale, zero = ops.quant_params(x, rel)
        assert torch.equal(scale, r["scale"]) and torch.equal(zero, r["zero"])
        codes, _ = ops.quantize(x, scale, zero)
        back = torch.empty_like(codes)
        if is_k:
            ops.k_decode(r["stream"], r["info"], back, 64, 128, 4)
        else:
            ops.v_decode(r["stream"], r["info"], back, 128, 64, 4)
        assert torch.equal(back, codes)
        del r, codes, back


@pytest.mark.parametrize("B,H,T,dtype,rel", [(16, 8, 32768, torch.bfloat16, 0.1), (8, 7, 16384, torch.bfloat16, 0.2),
                                             (2, 40, 8192, torch.float16, 0.05)])
def test_fused_quant_encode_large_shapes_repeat_and_round_trip(cuda, B, H, T, dtype, rel):
    """Thousands of workgroups in flight (the in-order stream offsets, the exchange between runs of eight heads, the
    wavefronts' shared minima and maxima): three launches give the same bytes, the parameters are the stand-alone
    quantizer's, and the stream unpacks to its codes."""
    k, v = synth.make_kv(B, H, T, seed=5, device=cuda, dtype=dtype)
    bits = ops.bits_for_rel(rel)
    for is_k, x in ((True, k), (False, v)):
        scale, zero = ops.quant_params(x, rel)
        codes, _ = ops.quantize(x, scale, zero)
        first = None
        for _ in range(3):
            r = (ops.k_quant_encode if is_k else ops.v_quant_encode)(x, rel, bits)
            assert torch.equal(scale, r["scale"]) and torch.equal(zero, r["zero"])
            got = (r["size"], r["stream"][:r["size"]].clone(), r["info"].clone())
            if first is None:
                first = got
            else:
                assert got[0] == first[0] and torch.equal(got[1], first[1]) and torch.equal(got[2], first[2])
        back = torch.empty_like(codes)
        if is_k:
            ops.k_decode(r["stream"], r["info"], back, 64, 128, bits)
        else:
            ops.v_decode(r["stream"], r["info"], back, 128, 64, bits)
        assert torch.equal(back, codes)
        del r, codes, back, first, got


def test_asynchronous_encode_reports_through_encode_status(cuda):
    """want_size=False keeps the launch asynchronous and reports nothing by itself; ops.encode_status then gives the
    size, or raises what the synchronous form raises: a stream that does not fit, a code wider than bits_len.  A
    compressed buffer at an odd address is refused up front (blocks are written in 2-byte units)."""
    B, H, T = 2, 4, 512
    k, _ = synth.make_kv(B, H, T, seed=620, device=cuda)
    sync = ops.k_quant_encode(k, 0.1)
    a = ops.k_quant_encode(k, 0.1, want_size=False)
    assert a["size"] == 0
    q = synth.make_q(B, 4 * H, seed=621, device=cuda)
    ops.attn_decode(q, sync, ops.v_quant_encode(k, 0.1))          # other work on the stream does not disturb the status
    assert ops.encode_status(cuda, bits=4) == sync["size"]
    assert torch.equal(a["stream"][:sync["size"]], sync["stream"][:sync["size"]])
    small = torch.empty(1024, dtype=torch.uint8, device=cuda)
    ops.k_quant_encode(k, 0.1, stream=small, want_size=False)     # does not fit: silent until asked
    with pytest.raises(ops.PackKVError) as e:
        ops.encode_status(cuda)
    assert e.value.code == 4
    ops.k_quant_encode(k, 0.1, bits=2, want_size=False)           # codes up to 11 do not fit 2 bits
    with pytest.raises(ops.PackKVError) as e:
        ops.encode_status(cuda, bits=2)
    assert e.value.code == 1
    odd = torch.empty(B * H * T * 128 + 1, dtype=torch.uint8, device=cuda)[1:]
    with pytest.raises(ops.PackKVError) as e:
        ops.k_quant_encode(k, 0.1, stream=odd)
    assert e.value.code == 2 and "even address" in str(e.value)
    codes = torch.zeros(64, 128, dtype=torch.uint8, device=cuda)
    with pytest.raises(RuntimeError, match="even address"):
        ops.k_encode(codes, odd, torch.zeros(1, 2, dtype=torch.uint32, device=cuda))


def test_encodes_that_wait_are_refused_while_their_stream_is_capturing(cuda):
    """A call that hands a size or a time back is refused before it records anything, so the capture goes on: an encode
    without them joins the graph, whose replays give what the eager call gives."""
    B, H, T = 1, 5, 256
    k, v = synth.make_kv(B, H, T, seed=630, device=cuda)
    room = lambda: (torch.zeros(B * H * T * 128, dtype=torch.uint8, device=cuda), torch.zeros(T // 64 * B * H, 2, dtype=torch.uint32, device=cuda))
    want, (stream, info), (other, oinfo) = ops.k_quant_encode(k, 0.1), room(), room()
    codes, long_codes = ops.quantize(k, want["scale"], want["zero"])[0], torch.zeros(512, 128, dtype=torch.uint8, device=cuda)
    side = lambda: [0.1, 4, other, 0, oinfo, torch.empty_like(want["scale"]), torch.empty_like(want["scale"])]
    ksd, vsd = side(), side()
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        ops.k_quant_encode(k, 0.1, stream=stream, info=info)
    g = torch.cuda.CUDAGraph()
    calls = [lambda: ops.k_quant_encode(k, 0.1, stream=other, info=oinfo), lambda: ops.k_quant_encode(k, 0.1, stream=other, info=oinfo, want_size=False, timed=True),
             lambda: ops.k_encode(codes, other, oinfo), lambda: ops.kv_quant_encode_append(k, v, T, ksd, vsd, 0),
             lambda: ops.encode_p(True, long_codes, other, oinfo[:2], 64, 4), lambda: ops.code_stats(codes, 16)]
    with torch.cuda.graph(g, stream=s):
        for i, call in enumerate(calls):
            _say("while capturing: call", i)
            with pytest.raises(ops.PackKVError, match="capturing"):
                call()
        got = ops.k_quant_encode(k, 0.1, stream=stream, info=info, want_size=False)
    for i in range(3):
        for t in (stream, info.view(torch.int32), got["scale"], got["zero"]):
            t.zero_()
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(stream[:want["size"]], want["stream"][:want["size"]]) and torch.equal(info.view(torch.int32), want["info"].view(torch.int32))
        assert torch.equal(got["scale"], want["scale"]) and torch.equal(got["zero"], want["zero"])
        with torch.cuda.stream(s):
            assert ops.encode_status(cuda, bits=4) == want["size"]
            assert ops.k_quant_encode(k, 0.1)["size"] == want["size"]


def test_an_encode_that_fails_after_its_launch_leaves_the_look_back_state_clear(cuda):
    """The encoder is launched but the call fails behind it (an error that an earlier HIP call of the thread left is found
    there): a graph that holds an encode, a capture made next and eager encodes give what they gave before.  Where the
    clearing of a new state is what fails, nothing is captured before an eager call, and the stream has no status."""
    B, H, T = 1, 5, 512
    k, _ = synth.make_kv(B, H, T, seed=640, device=cuda)
    want = ops.k_quant_encode(k, 0.1)
    e = {n: torch.empty_like(want[n]) for n in ("stream", "info", "scale", "zero")}
    lib, s = _lib.load(), torch.cuda.Stream()
    with open("/proc/self/maps") as f:
        hip = ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))
    torch.cuda.synchronize()

    def fail():
        assert hip.hipSetDevice(4096) != 0                    # no such device: the error stays for the thread
        p = {n: ctypes.c_void_p(t.data_ptr()) for n, t in e.items()}
        rc = lib.pkv_k_quant_encode(ctypes.c_void_p(k.data_ptr()), _lib.F16, B, H, T, 0.1, want["bits"], p["stream"], e["stream"].numel(), p["info"],
                                    p["scale"], p["zero"], None, None, ctypes.c_void_p(s.cuda_stream))
        assert rc == 3, (rc, lib.pkv_last_error())

    def check():
        torch.cuda.synchronize()
        assert torch.equal(e["stream"][:want["size"]], want["stream"][:want["size"]])
        for n in ("info", "scale", "zero"):
            assert torch.equal(e[n].view(torch.int16), want[n].view(torch.int16))
            e[n].zero_()
        e["stream"].zero_()
        torch.cuda.synchronize()

    def capture():
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            got = ops.k_quant_encode(k, 0.1, stream=e["stream"], info=e["info"], want_size=False)
            e["scale"].copy_(got["scale"])
            e["zero"].copy_(got["zero"])
        return g, got

    fail()                                                    # the first call of the stream: its state is not even clear
    with torch.cuda.stream(s), pytest.raises(ops.PackKVError, match="no encode has run"):
        ops.encode_status(cuda)
    with torch.cuda.graph(torch.cuda.CUDAGraph(), stream=s):
        e["stream"].zero_()
        with pytest.raises(ops.PackKVError, match="eager call"):
            ops.k_quant_encode(k, 0.1, stream=e["stream"], info=e["info"], want_size=False)
    with torch.cuda.stream(s):
        assert ops.k_quant_encode(k, 0.1)["size"] == want["size"]
    graphs = [capture()]
    for i in range(3):
        _say("after a failed call", i)
        fail()
        for g, _ in graphs:
            with torch.cuda.stream(s):                        # (the state is the stream's: a replay elsewhere would race with it)
                g.replay()
            check()
        fail()
        graphs.append(capture())
        with torch.cuda.stream(s):
            got = ops.k_quant_encode(k, 0.1, stream=e["stream"], info=e["info"])
            e["scale"].copy_(got["scale"])
            e["zero"].copy_(got["zero"])
        assert got["size"] == want["size"]
        check()


# Either side of the lines between the kernels: 256 workgroups of 256 threads, 256 of 1024 threads, the kernels that walk.
@pytest.mark.parametrize("B,H,T,rel", [(1, 8, 4096, 0.1), (1, 8, 4224, 0.05), (1, 8, 16384, 0.1), (1, 8, 16512, 0.1), (3, 3, 2816, 0.1),
                                       (2, 1, 16384, 0.2), (1, 20, 1536, 0.1), (1, 9, 3712, 0.05), (5, 7, 128, 0.03)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_fused_quant_encode_by_group_count(cuda, oracle_codec, B, H, T, rel, dtype):
    k, v = synth.make_kv(B, H, T, seed=H + T, dtype=dtype)
    W = ops.bits_for_rel(rel)
    for is_k, x in ((1, k), (0, v)):
        _say("fused quant+encode by groups", "K" if is_k else "V", dtype, B, H, T, rel)
        c, z, s = oq.quant_ints(x, 64, rel)
        so, io, zo = oracle_codec.encode(is_k, oq.code_matrix(c).numpy(), *((64, 128) if is_k else (128, 64)), W)
        for rep in range(2):                      # (twice: nothing of the first call's exchange may be left)
            r = (ops.k_quant_encode if is_k else ops.v_quant_encode)(x.to(cuda), rel, W)
            assert r["size"] == zo
            assert np.array_equal(r["info"].cpu().numpy(), io)
            assert np.array_equal(r["stream"][:zo].cpu().numpy(), so[:zo])
            assert torch.equal(r["scale"].cpu().view(torch.int16), s.reshape(B, T).view(torch.int16))
            assert torch.equal(r["zero"].cpu().view(torch.int16), z.reshape(B, T).view(torch.int16))


@pytest.mark.parametrize("T", [128, 4096, 4224, 16512])
def test_encodes_at_once_report_codes_and_capacity(cuda, T):
    """A code wider than the stream's width and a stream that does not fit are reported, and the next encode is right."""
    k, v = synth.make_kv(1, 8, T, seed=T, device=cuda)
    for fn, x in ((ops.k_quant_encode, k), (ops.v_quant_encode, v)):
        good = fn(x, 0.1)
        with pytest.raises(RuntimeError, match="does not fit bits_len"):
            fn(x, 0.03, bits=4)
        small = torch.full((good["size"] + 62,), 77, dtype=torch.uint8, device=cuda)
        with pytest.raises(RuntimeError, match="does not fit the output buffer"):
            fn(x, 0.1, stream=small[:good["size"] - 2])
        torch.cuda.synchronize()
        assert bool((small[good["size"] - 2:] == 77).all())
        again = fn(x, 0.1, stream=small[:good["size"]])
        assert again["size"] == good["size"] and torch.equal(again["stream"], good["stream"][:good["size"]])
        assert torch.equal(again["info"].view(torch.int32), good["info"].view(torch.int32)) and bool((small[good["size"]:] == 77).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("H", [3, 8, 12])
def test_nan_parameters_do_not_depend_on_the_launch(cuda, dtype, H):
    """Tokens with NaN and infinities get the same scale, zero and codes from a launch of one group and from one that fills
    the chip (257 groups of V: other kernels)."""
    g = torch.Generator(device=cuda).manual_seed(5)
    big = torch.randn(1, H, 128 * 257, 128, generator=g, device=cuda).to(dtype)
    nan, inf = float("nan"), float("inf")
    big[0, 1, 5, 7] = nan                                # one value
    big[0, :, 9] = nan                                   # a whole token
    big[0, 0, 20] = nan                                  # a whole head of a token
    big[0, H - 1, 40, 3], big[0, 0, 41, 100] = inf, -inf
    big[0, 2, 50, 1], big[0, 1, 50, 2] = nan, inf
    big[0, H - 1, 77, 64:] = -torch.tensor(nan)
    for enc in (ops.k_quant_encode, ops.v_quant_encode):
        small, whole = enc(big[:, :, :128].contiguous(), 0.1, want_size=False), enc(big, 0.1, want_size=False)
        torch.cuda.synchronize()
        for name in ("scale", "zero"):
            a, b = small[name].cpu(), whole[name][:, :128].cpu()
            same = (a.view(torch.int16) == b.view(torch.int16)) | (a.isnan() & b.isnan())
            assert bool(same.all()), (enc.__name__, name, (~same).nonzero().tolist())
        info = small["info"].view(torch.int32)                # the same blocks at the same place: the group comes first in both streams
        assert torch.equal(info, whole["info"].view(torch.int32)[:info.size(0)]), enc.__name__
        end = int(info[-1].sum())
        differ = (small["stream"][:end] != whole["stream"][:end]).nonzero().flatten().tolist()
        assert not differ, (enc.__name__, len(differ), differ[:8])


# Runs of two heads of K and one of V (256 threads), of eight and four (1024), one launch for both sides and two.
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,T,rels,block", [(1, 8, 512, (0.1, 0.1), 0), (2, 3, 256, (0.05, 0.1), 0), (1, 32, 128, (0.1, 0.1), 0), (1, 8, 4224, (0.05, 0.05), 0),
                                              (1, 20, 4096, (0.1, 0.2), 0), (1, 8, 512, (0.1, 0.1), 64), (3, 5, 256, (0.05, 0.05), 128)])
def test_a_run_that_waits_for_no_other_gives_the_same_stream(cuda, dtype, B, H, T, rels, block):
    """The encode of few groups with no look at what the other runs of a group found, as when they do not start."""
    x = list(synth.make_kv(B, H, T, seed=H + T, dtype=dtype, device=cuda))
    for i in range(2):           # (at 4 bits only: codes that do not fit write packs of 4 bits or of 6, which must not outgrow a block's slot)
        if rels[i] == 0.1:
            x[i][0, 1, 5, 7], x[i][0, :, 9], x[i][0, H - 1, 40, 3], x[i][0, 0, 41, 100] = float("nan"), float("nan"), float("inf"), -float("inf")
    perm = None
    if block:
        perm = torch.stack([torch.randperm(block, generator=torch.Generator().manual_seed(i)) for i in range(T // block)]).to(torch.int32).reshape(-1).to(cuda)
    want = [ops._quant_encode(i == 0, x[i], rels[i], ops.bits_for_rel(rels[i]), None, None, False, False, perm, block) for i in range(2)]
    got, sides = [], []
    for i in range(2):
        stream, info = ops._stream_and_info(i == 0, x[i], want[i]["bits"])
        scale, zero = torch.zeros(B, T, dtype=dtype, device=cuda), torch.zeros(B, T, dtype=dtype, device=cuda)
        got.append({"stream": stream, "info": info, "scale": scale, "zero": zero})
        sides.append(_lib.AppendSide(x[i].data_ptr(), *x[i].stride()[:3], stream.data_ptr(), stream.numel(), 0, info.data_ptr(), scale.data_ptr(),
                                     zero.data_ptr(), rels[i], want[i]["bits"]))
    sizes = [ctypes.c_uint64(0), ctypes.c_uint64(0)]
    rc = _lib.load().pkv_kv_quant_encode_alone(ctypes.byref(sides[0]), ctypes.byref(sides[1]), _lib.F16 if dtype == torch.float16 else _lib.BF16, B, H, T, T,
                                               None if perm is None else ctypes.c_void_p(perm.data_ptr()), block, ctypes.byref(sizes[0]),
                                               ctypes.byref(sizes[1]), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    torch.cuda.synchronize()
    assert rc in (0, 1), _lib.load().pkv_last_error()         # (1: codes of the tokens with infinities that are too wide)
    for i in range(2):
        end = want[i]["info"].view(torch.int32)[-1].cpu().sum().item()
        assert end > 0 and (rc or sizes[i].value == end)
        assert torch.equal(got[i]["stream"][:end], want[i]["stream"][:end])
        for name in ("info", "scale", "zero"):
            assert torch.equal(got[i][name].view(torch.int16), want[i][name].view(torch.int16)), name


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("H,T", [(1, 128), (3, 128), (2, 128), (1, 16640), (3, 16640)])
def test_padding_of_one_sequence_leaves_the_others_alone(cuda, dtype, H, T):
    """Tokens of zeros (scale 0) and tokens far below zero in one sequence: the codes of the other one are those of its own
    parameters, whichever groups share a wavefront."""
    for is_k in (True, False):
        x = torch.randn(2, H, T, 128, generator=torch.Generator(device=cuda).manual_seed(H + T), device=cuda).to(dtype)
        x[0, :, T // 2 + 3:] = 0
        x[0, :, 2:T // 2:3] -= 100
        enc, dec = (ops.k_quant_encode, ops.k_decode) if is_k else (ops.v_quant_encode, ops.v_decode)
        e = enc(x, 0.1, want_size=False)
        codes = torch.zeros(T, 2 * H * 128, dtype=torch.uint8, device=cuda)
        dec(e["stream"], e["info"], codes, bits=4)
        c, z, s = oq.quant_ints(x[1:].cpu(), 64, 0.1)
        assert torch.equal(codes[:, H * 128:].cpu(), oq.code_matrix(c)), "K" if is_k else "V"


@pytest.mark.parametrize("H,T", [(2, 128), (2, 1920), (2, 2048), (2, 2176), (8, 2048), (16, 1024), (8, 16384), (40, 640)])
def test_encoders_that_close_by_themselves(cuda, H, T):
    """Launches of up to 256 workgroups that hand no size back leave their outcome and clear the look-back state without a kernel
    behind them, counted in sixteens: one workgroup, counts around a multiple of sixteen, the most there are.  Each encode finds the
    state clear, whatever the one before was -- fused K and V, K and V in one launch, codes, with and without a size, a stream that does
    not fit -- and gives what encodes of 64 and 128 tokens appended one by one give."""
    k, v = synth.make_kv(1, H, T, seed=H + T, device=cuda)

    def side(x, is_k):
        nblk = T // (64 if is_k else 128) * H * (1 if is_k else 2)
        return [0.1, 4, torch.zeros(T * H * 128 + 16, dtype=torch.uint8, device=cuda), 0, torch.zeros(nblk, 2, dtype=torch.uint32, device=cuda),
                torch.zeros(1, T, dtype=x.dtype, device=cuda), torch.zeros(1, T, dtype=x.dtype, device=cuda)]
    want = {}
    for is_k, x in ((True, k), (False, v)):
        s, step = side(x, is_k), 64 if is_k else 128
        for t in range(0, T, step):
            s[3] = ops.quant_encode_append(is_k, x[:, :, t:t + step].contiguous(), 0.1, 4, s[2], s[3], s[4], t, s[5], s[6])
        want[is_k] = s

    def check(is_k, size, stream, info, what):
        w = want[is_k]
        assert size == w[3], (what, is_k)
        assert torch.equal(stream[:size], w[2][:size]) and torch.equal(info.view(torch.int32), w[4].view(torch.int32)), (what, is_k)
    for turn in range(3):
        ks, vs = side(k, True), side(v, False)
        kn, vn = ops.kv_quant_encode_append(k, v, T, ks, vs, 0)
        check(True, kn, ks[2], ks[4], "both")
        check(False, vn, vs[2], vs[4], "both")
        for is_k, x, enc, code_enc in ((True, k, ops.k_quant_encode, ops.k_encode), (False, v, ops.v_quant_encode, ops.v_encode)):
            e = enc(x, 0.1)
            check(is_k, e["size"], e["stream"], e["info"], "alone")
            u = enc(x, 0.1, want_size=False)
            check(is_k, ops.encode_status(cuda, bits=4), u["stream"], u["info"], "no size")
            codes = ops.quantize(x, e["scale"], e["zero"])[0]
            s = side(x, is_k)
            check(is_k, code_enc(codes, s[2], s[4]), s[2], s[4], "codes")
            s[2].zero_()
            code_enc(codes, s[2], s[4], want_size=False)
            check(is_k, ops.encode_status(cuda, bits=4), s[2], s[4], "codes, no size")
            with pytest.raises(ops.PackKVError, match="fit"):
                code_enc(codes, s[2][:e["size"] - 2], s[4])
            with pytest.raises(ops.PackKVError, match="fit"):
                enc(x, 0.1, stream=s[2][:e["size"] - 2], info=s[4])
            enc(x, 0.1, stream=s[2][:e["size"] - 2], info=s[4], want_size=False)
            with pytest.raises(ops.PackKVError, match="fit"):
                ops.encode_status(cuda, bits=4)


# V of 5 and 6 bits beyond the encodes at once: two segments of a block side by side; idle head slots, runs of eight heads.
@pytest.mark.parametrize("B,H,T,rel", [(1, 8, 16512, 0.05), (3, 5, 5632, 0.03), (1, 12, 11136, 0.05), (129, 8, 128, 0.05)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_wide_v_with_both_segments_at_once(cuda, oracle_codec, B, H, T, rel, dtype):
    k, v = synth.make_kv(B, H, T, seed=H + T, dtype=dtype)
    W = ops.bits_for_rel(rel)
    c, z, s = oq.quant_ints(v, 64, rel)
    codes = oq.code_matrix(c)
    so, io, zo = oracle_codec.encode(0, codes.numpy(), 128, 64, W)
    _say("wide V", B, H, T, rel, dtype)
    vd = v.to(cuda)
    r = ops.v_quant_encode(vd, rel, W)
    assert r["size"] == zo
    assert np.array_equal(r["info"].cpu().numpy(), io)
    assert np.array_equal(r["stream"][:zo].cpu().numpy(), so[:zo])
    assert torch.equal(r["scale"].cpu().view(torch.int16), s.reshape(B, T).view(torch.int16))
    assert torch.equal(r["zero"].cpu().view(torch.int16), z.reshape(B, T).view(torch.int16))
    if H % 8 == 0:                                     # the same from the code matrix
        stream, info = torch.zeros_like(r["stream"]), torch.zeros_like(r["info"])
        assert ops.encode_p(False, codes.to(cuda), stream, info, 16, W) == zo
        assert torch.equal(stream[:zo], r["stream"][:zo]) and torch.equal(info.view(torch.int32), r["info"].view(torch.int32))
    if H <= 8:                                         # in the order of a repacking: as the rows in that order
        _, ve, perm = ops.repack_quant_encode(k.to(cuda), vd, rel, rel, "median")
        block = 64
        src = torch.arange(T, device=cuda) // block * block + perm.view(torch.int32).long()
        want = ops.v_quant_encode(vd[:, :, src].contiguous(), rel, W)
        n = want["size"]
        assert ve["size"] == n and torch.equal(ve["stream"][:n], want["stream"][:n])
        for name in ("info", "scale", "zero"):
            assert torch.equal(ve[name].view(torch.int16), want[name].view(torch.int16)), name


# K and V of five to eight heads in one launch: idle head slots, V first and in turns of 256 groups with a rest, one type and both
# kinds of rows, each as the encodes of one side.
@pytest.mark.parametrize("B,H,T", [(1, 8, 17408), (2, 5, 17280), (9, 7, 4864), (21, 6, 6272)])
@pytest.mark.parametrize("form", ["order", "rows", "rotary"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_both_sides_in_one_launch(cuda, B, H, T, form, dtype):
    k, v = synth.make_kv(B, H, T, seed=H + T, dtype=dtype, device=cuda)
    rels = (0.1, 0.2)
    _say("both sides", B, H, T, form, dtype)
    if form == "order":
        ke, ve, perm = ops.repack_quant_encode(k, v, *rels, "median")
        for e, x, is_k in ((ke, k, True), (ve, v, False)):
            want = ops._quant_encode(is_k, x, rels[not is_k], e["bits"], None, None, True, False, perm, 64)
            n = want["size"]
            assert e["size"] == n and torch.equal(e["stream"][:n], want["stream"][:n])
            assert all(torch.equal(e[f].view(torch.int16), want[f].view(torch.int16)) for f in ("info", "scale", "zero"))
        return
    used, before = 1002, 128
    cos = sin = None
    kr = k
    if form == "rotary":
        cos, sin = (torch.randn(1, T, 128, device=cuda).to(dtype).expand(B, -1, -1) for _ in range(2))
        kr = (k * cos.unsqueeze(1)) + (torch.cat((-k[..., 64:], k[..., :64]), dim=-1) * sin.unsqueeze(1))
    want = [ops.k_quant_encode(kr, rels[0]), ops.v_quant_encode(v, rels[1])]
    sides, blocks = [], []
    for i in range(2):
        per_tile, ctx = (B * H, 64) if i == 0 else (2 * B * H, 128)
        blocks.append(before // ctx * per_tile)
        sides.append((rels[i], want[i]["bits"], torch.zeros(used + want[i]["stream"].numel(), dtype=torch.uint8, device=cuda), used,
                      torch.zeros((before + T) // ctx * per_tile, 2, dtype=torch.uint32, device=cuda),
                      torch.zeros(B, before + T + 64, dtype=dtype, device=cuda), torch.zeros(B, before + T + 64, dtype=dtype, device=cuda)))
    rows = [x.transpose(1, 2).contiguous().transpose(1, 2) for x in (k, v)] if form == "rows" else [k, v]
    for rep in range(2):                               # (twice: nothing of the first call's look-back may be left)
        sizes = ops.kv_quant_encode_append(*rows, T, *sides, before, cos, sin)
        for i in range(2):
            n = want[i]["size"]
            _, _, stream, _, info, scale, zero = sides[i]
            assert sizes[i] == used + n and torch.equal(stream[used:used + n], want[i]["stream"][:n])
            got, ref = info.view(torch.int32)[blocks[i]:], want[i]["info"].view(torch.int32)
            assert torch.equal(got[:, 0], ref[:, 0] + used) and torch.equal(got[:, 1], ref[:, 1])
            assert torch.equal(scale[:, before:before + T], want[i]["scale"]) and torch.equal(zero[:, before:before + T], want[i]["zero"])
            assert not scale[:, :before].any() and not scale[:, before + T:].any() and not stream[:used].any()


# Either side of the sizes up to which the encoders that walk close by themselves: 2048 workgroups of K, 2048 of V.
@pytest.mark.parametrize("H,T", [(5, 131072), (5, 131200), (6, 262144), (6, 262272)])
def test_encoders_that_walk_and_close_by_themselves(cuda, H, T):
    k, v = synth.make_kv(1, H, T, seed=T, device=cuda)
    for is_k, x, enc in ((True, k, ops.k_quant_encode), (False, v, ops.v_quant_encode)):
        _say("closing", H, T, is_k)
        first = enc(x, 0.1)
        with pytest.raises(RuntimeError, match="does not fit bits_len 3"):
            enc(x, 0.1, 3)
        enc(x, 0.1, 3, want_size=False)
        with pytest.raises(RuntimeError, match="does not fit bits_len 3"):
            ops.encode_status(cuda, bits=3)
        for rep in range(4):                           # (after an error, and after a launch of its own kind: the state is clear)
            r = enc(x, 0.1, want_size=rep < 2)
            r["size"] = r["size"] or ops.encode_status(cuda, bits=4)
            assert r["size"] == first["size"] and torch.equal(r["stream"][:r["size"]], first["stream"][:r["size"]])
            assert all(torch.equal(r[f].view(torch.int16), first[f].view(torch.int16)) for f in ("info", "scale", "zero"))
        codes = torch.empty(T, H * 128, dtype=torch.uint8, device=cuda)
        (ops.k_decode if is_k else ops.v_decode)(r["stream"], r["info"], codes, *((64, 128) if is_k else (128, 64)), r["bits"])
        assert torch.equal(codes, ops.quant_codes(x, 0.1)[0])


@pytest.mark.parametrize("T", [32768, 131072, 131200])
@pytest.mark.parametrize("bits", [4, 5])
def test_code_encoders_that_walk_and_close_by_themselves(cuda, T, bits):
    g = torch.Generator(device=cuda).manual_seed(T + bits)
    codes = torch.randint(0, 1 << bits, (T, 1024), generator=g, dtype=torch.uint8, device=cuda)
    codes[T // 2:] &= 3
    stream, info = torch.zeros(T * 1024, dtype=torch.uint8, device=cuda), torch.zeros(T // 8, 2, dtype=torch.uint32, device=cuda)
    back = torch.empty_like(codes)
    for is_k in (True, False):
        _say("codes, closing", T, bits, is_k)
        size = ops.encode_p(is_k, codes, stream, info, 16, bits)
        ops.decode_p(is_k, stream, info, back, 16, bits)
        assert torch.equal(back, codes)
        want, table = stream[:size].clone(), info.clone()
        with pytest.raises(RuntimeError):              # (a stream that does not fit; the state is clear behind it)
            ops.encode_p(is_k, codes, stream[:size - 2], info, 16, bits)
        ops.encode_p(is_k, codes, stream[:size - 2], info, 16, bits, want_size=False)
        with pytest.raises(RuntimeError, match="fit"):
            ops.encode_status(cuda)
        for want_size in (True, False, False):
            stream.zero_()
            got = ops.encode_p(is_k, codes, stream, info, 16, bits, want_size=want_size)
            assert (got if want_size else ops.encode_status(cuda)) == size
            assert torch.equal(stream[:size], want) and torch.equal(info.view(torch.int32), table.view(torch.int32))


@pytest.fixture(scope="module")
def other():
    return torch.cuda.Stream()           # (one for all cases: torch hands out 32 in turn, and some tests want one without a past)


@pytest.mark.parametrize("B,T", [(1, 512), (2, 4096), (16, 8192)])
@pytest.mark.parametrize("kind", ["k", "v", "append", "repack", "k codes", "v codes"])
def test_a_size_says_that_the_output_is_there_for_any_stream(cuda, other, kind, B, T):
    """A call that hands its size back is synchronous: the stream's bytes, block_info and the parameters can be read through
    another stream at once, without an event.  (In launches of a few, of some hundred and of 2048 workgroups; every pass has
    other inputs, in zeroed buffers.)"""
    H = 8
    for seed in range(3):
        k, v = synth.make_kv(B, H, T, seed=650 + seed, device=cuda)
        sides = []
        for blocks, bound in ((T // 64 * B * H, ops.block_bound(True, 64, 128, 4)), (T // 128 * 2 * B * H, ops.block_bound(False, 128, 64, 4))):
            sides.append([torch.zeros(blocks * bound + 16, dtype=torch.uint8, device=cuda), torch.zeros(blocks, 2, dtype=torch.uint32, device=cuda),
                          torch.zeros(B, T, dtype=k.dtype, device=cuda), torch.zeros(B, T, dtype=k.dtype, device=cuda)])
        codes = [ops.quantize(x, *ops.quant_params(x, 0.1))[0] for x in (k, v)]
        torch.cuda.synchronize()
        if kind in ("k", "v"):
            r = (ops.k_quant_encode if kind == "k" else ops.v_quant_encode)(k if kind == "k" else v, 0.1, stream=sides[kind == "v"][0], info=sides[kind == "v"][1])
            out = [r["stream"][:r["size"]], r["info"], r["scale"], r["zero"]]
        elif kind == "append":
            sizes = ops.kv_quant_encode_append(k, v, T, *((0.1, 4, st, 0, *rest) for st, *rest in sides), 0)
            out = [t for side, size in zip(sides, sizes) for t in (side[0][:size], *side[1:])]
        elif kind == "repack":
            out = [t for r in ops.repack_quant_encode(k, v, 0.1, 0.1)[:2] for t in (r["stream"][:r["size"]], r["info"], r["scale"], r["zero"])]
        else:
            i = int(kind == "v codes")
            size = ops.encode_p(i == 0, codes[i], *sides[i][:2], 16, 4)
            out = [sides[i][0][:size], sides[i][1]]
        with torch.cuda.stream(other):
            seen = [t.view(torch.uint8).clone() for t in out]
        torch.cuda.synchronize()
        assert all(t.numel() for t in out) and all(torch.equal(a, b.view(torch.uint8)) for a, b in zip(seen, out)), seed


@pytest.mark.parametrize("B,H,T", [(1, 8, 128), (1, 2, 256), (33, 8, 1024)])
@pytest.mark.parametrize("rel", [0.1, 0.03])
def test_a_pack_of_nans_of_both_signs_has_the_full_width(cuda, B, H, T, rel):
    """The codes of such a pack lie 0x8000 apart: it is stored at the width of one whose codes span the whole range (the call
    reports the overflow when it is asked), 4 and 6 bits, in the encoders at once and in those that walk."""
    base = torch.linspace(-1, 1, 128, device=cuda).half().expand(B, H, T, 128)
    for enc in (ops.k_quant_encode, ops.v_quant_encode):
        sizes = []
        for even, odd in ((0x7E00, -0x200), (-0x4400, 0x3C00)):           # NaN and -NaN; -1 and 1, the limits of every token
            x = base.clone()
            x.view(torch.int16)[:, H - 1, 0::2, 5], x.view(torch.int16)[:, H - 1, 1::2, 5] = even, odd
            sizes.append(enc(x, rel, want_size=False)["info"].view(torch.int32)[:, 1].clone())
        assert torch.equal(*sizes)
        with pytest.raises(ops.PackKVError):
            x = base.clone()
            x.view(torch.int16)[:, H - 1, 0::2, 5], x.view(torch.int16)[:, H - 1, 1::2, 5] = 0x7E00, -0x200
            enc(x, rel)
