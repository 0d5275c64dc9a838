"""Python op surface over the C ABI: the reference's eight ``packkv_cuda`` functions with the
same positional signatures (packkv_cuda_ext/packkv_cuda.pyi:4-86, bound in
packkv_cuda_ext/export_packkv.cpp:9-18), plus the device-native ops the reference does not
have (GPU encode / unpack, fused quantize+encode, fused decompress-attention).

All tensors are caller-allocated and written in place, as in the reference.  PyTorch is used
for device memory and the current stream only; every computation happens in
libpackkv_hip.so.
"""
import contextlib
import ctypes
import math

import torch

from . import _lib
from ._lib import AttnArgs, PackKVError  # noqa: F401  (re-exported)

__all__ = [
    "k_encode_cpu", "k_decode_cpu", "v_encode_cpu", "v_decode_cpu",
    "kq_mat_vec_mul", "wv_mat_vec_mul", "fused_kq", "fused_wv",
    "k_encode", "v_encode", "k_decode", "v_decode",
    "quant_params", "quantize", "dequantize", "k_quant_encode", "v_quant_encode",
    "attn_decode", "AttnPlan", "block_bound", "bits_for_rel", "repack_quant_encode", "encode_status",
]


def _dtype_code(t):
    if t.dtype == torch.float16:
        return _lib.F16
    if t.dtype == torch.bfloat16:
        return _lib.BF16
    raise RuntimeError("Unsupported data type")


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr()) if t is not None else ctypes.c_void_p(0)


def _host():
    """The native side of the calls a decode loop repeats (csrc/pkv_host.cpp): its functions return None for a call that they do
    not serve, which then takes the general code below them."""
    return _lib.host or _first_host()


def _first_host():
    try:
        _lib.load()
    except ImportError:          # (the general code says so where it needs the library, and refuses what it refuses without it)
        return _lib.NO_HOST
    return _lib.host


# Every op makes `dev` current and passes on its current stream.  A stream object and a device context that is entered
# although the device is current take 3.5 us of host time a call -- a decode step is two calls and 13 us of GPU time --
# these two take 0.5.  (They are not part of torch's public surface: without them the public functions serve.)
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None) or (lambda index: torch.cuda.current_stream(index).cuda_stream)
_current_device = getattr(torch._C, "_cuda_getDevice", None) or torch.cuda.current_device
_here = contextlib.nullcontext()


def _stream(dev):
    return _raw_stream(_current_device() if dev.index is None else dev.index)


def _on(dev):
    return _here if dev.type == "cuda" and dev.index in (None, _current_device()) else torch.cuda.device(dev)


def _require(cond, msg):
    if not cond:
        raise RuntimeError("PackKV Assertion failed: " + msg)


# The kernels get bare addresses: a tensor on another device than the one they run on must not get that far.  (Compared as
# get_device() of tensors that are on a GPU: -1 on the host; two torch.device objects take three times as long.)
_ONE_DEVICE = "all tensors must be on one device"


def _device_of(*tensors):
    dev = None
    for t in tensors:
        if t.is_cuda:
            dev = t.device
    if dev is None:
        if not torch.cuda.is_available():
            raise RuntimeError("packkv needs a GPU: the ops run in libpackkv_hip.so, there is no CPU path")
        dev = torch.device("cuda", torch.cuda.current_device())
    return dev


def block_bound(is_k, ctx_blk, hid_blk, bits):
    return int(_lib.load().pkv_block_bound(int(is_k), ctx_blk, hid_blk, bits))


def bits_for_rel(rel):
    """Raw code width W for a relative quant step: codes span 0..ceil(1/rel), plus at most one
    more level from rounding the quotient to the storage type."""
    import math
    top = math.ceil(1.0 / rel - 1e-9) + 1
    return max(2, top.bit_length())


# ------------------------------------------------------------------ codec ------------

def _check_codec_args(codes, stream, info, ctx_len, hidden_dim, ctx_blk, hid_blk, bits, is_k, max_bits=4):
    # mirrors k_encode_cpu_assert / v_encode_cpu_assert (src/k_encode_cpu.cpp:247-284,
    # src/v_encode_cpu.cpp:262-299); raises instead of aborting the process
    _require(codes.dim() == 2 and codes.size(0) == ctx_len, "ctx_len mismatch")
    _require(codes.size(1) == hidden_dim, "hidden_dim mismatch")
    _require(ctx_blk > 0, "ctx_len_block_size must be greater than 0")
    _require(hid_blk > 0, "hidden_dim_block_size must be greater than 0")
    _require(ctx_len % ctx_blk == 0, "ctx_len must be divisible by ctx_len_block_size")
    _require(hidden_dim % hid_blk == 0, "hidden_dim must be divisible by hidden_dim_block_size")
    nblk = (ctx_len // ctx_blk) * (hidden_dim // hid_blk)
    _require(info.dim() == 2 and info.size(0) == nblk, "block_info_buffer block num mismatch")
    _require(info.size(1) == 2, "block_info_buffer.size(1) must be 2")
    _require(bits <= max_bits, "bits_len must be less than or equal to %d" % max_bits)
    _require(ctx_blk % 16 == 0, "ctx_len_block_size must be divisible by PACK_ELE_NUM")
    if is_k:
        _require(hid_blk == 128, "hidden_dim_block_size must be 128, because this is most common head dim")
    _require(codes.dtype == torch.uint8, "quant_ints_tensor must be a UInt8 tensor")
    _require(stream.dtype == torch.uint8, "compressed_buffer must be a UInt8 tensor")
    _require(stream.numel() > 0, "compressed_buffer must be a non-empty tensor")
    _require(info.dtype == torch.uint32, "block_info_buffer must be a UInt32 tensor")
    _require(codes.is_contiguous() and stream.is_contiguous() and info.is_contiguous(),
             "tensors must be contiguous")
    _require(not stream.is_cuda or stream.data_ptr() % 2 == 0, "compressed_buffer must start at an even address")


# Host tensors go through page-locked memory from torch's host allocator, at most two pieces of this size at a time: the
# link moves 8 MiB between it and the device in 155 us, where a copy from or to pageable memory takes 246 and 460 us (574
# into a fresh tensor); the copy on the host is 16 us.  Smaller tensors are copied as they are, the buffer and the event cost
# more than they save there.  Up / down in us, as they are and staged: 128 KiB 17 / 18 and 30 / 42, 512 KiB 28 / 34 and
# 37 / 51, 1 MiB 57 / 66 and 47 / 63, 8 MiB 250 / 523 and 201 / 235.  Tensors that the caller holds in page-locked memory go
# over the link as they are (8 MiB 160 / 160, staged 191 / 244).  The allocator keeps the pieces, at most 2 x 32 MiB of them for
# each host thread that copies at a time.  No pageable tensor is made here any more, so that a program finds no pages that such
# ones left behind: the host tensors it allocates between calls are as slow as elsewhere until it has freed some of its own
# (4 x 8 MiB and their buffers: 5.2 ms while they are fresh, 1.4 ms in memory used before).
_STAGE_BYTES = 32 << 20
_STAGE_FROM = 1 << 20


def _bytes(t):
    return t.reshape(-1).view(torch.uint8)


def _staged(n, pieces, step):
    """step(piece buffer, from, to) over 0..n in pieces of _STAGE_BYTES, `pieces` buffers in turn; step returns what is
    left to do with a buffer before it is used again and after the last piece, or None."""
    bufs, todo = [None] * pieces, [None] * pieces
    for i, at in enumerate(range(0, n, _STAGE_BYTES)):
        m, j = min(_STAGE_BYTES, n - at), i % pieces
        if todo[j] is not None:
            todo[j]()
        if bufs[j] is None:
            bufs[j] = torch.empty(m, dtype=torch.uint8, pin_memory=True)
        todo[j] = step(bufs[j][:m], at, at + m)
    order = range((n + _STAGE_BYTES - 1) // _STAGE_BYTES)
    for i in order[-pieces:]:
        if todo[i % pieces] is not None:
            todo[i % pieces]()


def _upload(dst, src):
    """Device bytes dst = host bytes src, on the current stream of dst's device; src may be reused at once."""
    if src.numel() < _STAGE_FROM or src.is_pinned():
        dst.copy_(src)
        return
    last = src.numel() <= _STAGE_BYTES

    def step(buf, a, b):
        buf.copy_(src[a:b])
        dst[a:b].copy_(buf, non_blocking=True)
        if last:                     # (the allocator keeps a buffer until the copies from it are done)
            return None
        return torch.cuda.current_stream(dst.device).record_event().synchronize
    _staged(src.numel(), 2, step)


def _download(dst, src):
    """Host bytes dst = device bytes src, there when this returns."""
    if src.numel() < _STAGE_FROM or dst.is_pinned():
        dst.copy_(src)
        return

    def step(buf, a, b):
        buf.copy_(src[a:b], non_blocking=True)
        there = torch.cuda.current_stream(src.device).record_event()

        def take():
            there.synchronize()
            dst[a:b].copy_(buf)
        return take
    _staged(src.numel(), 2, step)


def _encode(is_k, codes, stream, info, ctx_len, hidden_dim, ctx_blk, hid_blk, bits, want_size=True,
            timed=False, max_bits=4):
    _check_codec_args(codes, stream, info, ctx_len, hidden_dim, ctx_blk, hid_blk, bits, is_k, max_bits)
    lib = _lib.load()
    dev = _device_of(codes, stream, info)
    on_host = not codes.is_cuda
    _require(stream.is_cuda != on_host and info.is_cuda != on_host, "all tensors must be on one device")
    d_codes = torch.empty_like(codes, device=dev) if on_host else codes
    d_stream = torch.empty(stream.numel(), dtype=torch.uint8, device=dev) if on_host else stream
    d_info = torch.empty_like(info, device=dev) if on_host else info
    size = ctypes.c_uint64(0)
    ms = ctypes.c_float(0.0)
    fn = lib.pkv_k_encode if is_k else lib.pkv_v_encode
    with _on(dev):
        if on_host:
            _upload(_bytes(d_codes), _bytes(codes))
        rc = fn(_ptr(d_codes), _ptr(d_stream), d_stream.numel() * d_stream.element_size(), _ptr(d_info), ctx_len, hidden_dim,
                ctx_blk, hid_blk, bits, ctypes.byref(size) if (want_size or on_host) else None,
                ctypes.byref(ms) if timed else None, _stream(dev))
        _lib.check(rc)
        if on_host:
            n = int(size.value)
            _download(_bytes(stream)[:n], d_stream[:n])
            _download(_bytes(info), _bytes(d_info))
    return (int(size.value), float(ms.value)) if timed else int(size.value)


def _decode(is_k, stream, info, codes, ctx_len, hidden_dim, ctx_blk, hid_blk, bits, timed=False, max_bits=4):
    _check_codec_args(codes, stream, info, ctx_len, hidden_dim, ctx_blk, hid_blk, bits, is_k, max_bits)
    lib = _lib.load()
    dev = _device_of(codes, stream, info)
    on_host = not codes.is_cuda
    _require(stream.is_cuda != on_host and info.is_cuda != on_host, "all tensors must be on one device")
    d_stream, d_info, d_codes = stream, info, codes
    ms = ctypes.c_float(0.0)
    fn = lib.pkv_k_decode if is_k else lib.pkv_v_decode
    with _on(dev):
        if on_host:          # the part of the buffer that block_info points into, where that is worth its sum (9 us)
            used = stream.numel()
            if info.numel() and used >= _STAGE_FROM:
                used = min(used, max(1, int(info.view(torch.int32).to(torch.int64).bitwise_and_(0xFFFFFFFF).sum(1).max())))
            d_stream = torch.empty(used, dtype=torch.uint8, device=dev)
            d_info, d_codes = torch.empty_like(info, device=dev), torch.empty_like(codes, device=dev)
            _upload(d_stream, _bytes(stream)[:used])
            _upload(_bytes(d_info), _bytes(info))
        rc = fn(_ptr(d_stream), d_stream.numel() * d_stream.element_size(), _ptr(d_info), _ptr(d_codes), ctx_len, hidden_dim, ctx_blk, hid_blk, bits,
                ctypes.byref(ms) if timed else None, _stream(dev))
        _lib.check(rc)
        if on_host:
            _download(_bytes(codes), _bytes(d_codes))
    return float(ms.value) if timed else None


def stream_release(stream=None):
    """Gives back the device memory the library keeps for `stream` (a torch.cuda.Stream; default: the current one) --
    scratch buffers, tile counters and the buffers it has outgrown.  For callers that create and destroy streams:
    call it before the stream goes away, and only when no HIP graph captured on it will be replayed again."""
    st = torch.cuda.current_stream() if stream is None else stream
    with _on(st.device):
        rc = _lib.load().pkv_stream_release(ctypes.c_void_p(st.cuda_stream))
    _lib.check(rc)


def encode_status(device=None, bits=0):
    """Stream size of the last encode launched on the current stream of `device` with want_size=False; waits for the
    stream and raises what the encode would have raised (a stream that did not fit, a code wider than `bits`)."""
    dev = torch.device("cuda", torch.cuda.current_device()) if device is None else torch.device(device)
    size = ctypes.c_uint64(0)
    with _on(dev):
        rc = _lib.load().pkv_encode_status(_stream(dev), int(bits), ctypes.byref(size))
    _lib.check(rc)
    return int(size.value)


def k_encode_cpu(quant_ints_tensor, compressed_buffer, block_info_buffer, ctx_len, hidden_dim,
                 ctx_len_block_size, hidden_dim_block_size, bits_len):
    """Drop-in for packkv_cuda.k_encode_cpu (packkv_cuda.pyi:4-13): host tensors in, host tensors
    written in place, stream size returned -- but encoded on the GPU (staged through device
    memory).  Device tensors are accepted too and then nothing is copied."""
    return _encode(True, quant_ints_tensor, compressed_buffer, block_info_buffer, ctx_len, hidden_dim,
                   ctx_len_block_size, hidden_dim_block_size, bits_len)


def v_encode_cpu(quant_ints_tensor, compressed_buffer, block_info_buffer, ctx_len, hidden_dim,
                 ctx_len_block_size, hidden_dim_block_size, bits_len):
    """Drop-in for packkv_cuda.v_encode_cpu (packkv_cuda.pyi:38-47)."""
    return _encode(False, quant_ints_tensor, compressed_buffer, block_info_buffer, ctx_len, hidden_dim,
                   ctx_len_block_size, hidden_dim_block_size, bits_len)


def k_decode_cpu(compressed_buffer, block_info_buffer, quant_ints_tensor, ctx_len, hidden_dim,
                 ctx_len_block_size, hidden_dim_block_size, bits_len):
    """Drop-in for packkv_cuda.k_decode_cpu (packkv_cuda.pyi:15-24)."""
    _decode(True, compressed_buffer, block_info_buffer, quant_ints_tensor, ctx_len, hidden_dim,
            ctx_len_block_size, hidden_dim_block_size, bits_len)


def v_decode_cpu(compressed_buffer, block_info_buffer, quant_ints_tensor, ctx_len, hidden_dim,
                 ctx_len_block_size, hidden_dim_block_size, bits_len):
    """Drop-in for packkv_cuda.v_decode_cpu (packkv_cuda.pyi:49-58)."""
    _decode(False, compressed_buffer, block_info_buffer, quant_ints_tensor, ctx_len, hidden_dim,
            ctx_len_block_size, hidden_dim_block_size, bits_len)


MAX_BITS = 8     # widths 5..8 are this library's extension of the format (the reference stops at 4)


def k_encode(codes, stream, info, ctx_blk=64, hid_blk=128, bits=4, want_size=True, timed=False):
    """Device encode of a uint8 code matrix [ctx_len, hidden]; returns the stream size (and ms).  bits 2..8."""
    return _encode(True, codes, stream, info, codes.size(0), codes.size(1), ctx_blk, hid_blk, bits,
                   want_size, timed, MAX_BITS)


def v_encode(codes, stream, info, ctx_blk=128, hid_blk=64, bits=4, want_size=True, timed=False):
    return _encode(False, codes, stream, info, codes.size(0), codes.size(1), ctx_blk, hid_blk, bits,
                   want_size, timed, MAX_BITS)


def k_decode(stream, info, codes, ctx_blk=64, hid_blk=128, bits=4, timed=False):
    return _decode(True, stream, info, codes, codes.size(0), codes.size(1), ctx_blk, hid_blk, bits, timed, MAX_BITS)


def v_decode(stream, info, codes, ctx_blk=128, hid_blk=64, bits=4, timed=False):
    return _decode(False, stream, info, codes, codes.size(0), codes.size(1), ctx_blk, hid_blk, bits, timed, MAX_BITS)


# ---- packs longer than 16 tokens (an extension of the format: the reference only prices them, utils/compute.py:272-297) ----

PACK_LENS = (16, 32, 64, 128, 256)


def long_block_shape(is_k, pack_len):
    """(tokens, channels) of a block with packs of `pack_len` tokens: the reference's 64 x 128 / 128 x 64 scaled."""
    return ((4 * pack_len, 128) if is_k else (8 * pack_len, 64))


def block_bound_p(pack_len, bits):
    return int(_lib.load().pkv_block_bound_p(pack_len, bits))


def _check_long(is_k, codes, stream, info, pack_len, bits):
    _require(pack_len in PACK_LENS, "not supported: pack_len %d (16, 32, 64, 128 or 256)" % pack_len)
    ctx_blk, hid_blk = long_block_shape(is_k, pack_len)
    _require(codes.dim() == 2 and codes.dtype == torch.uint8, "quant_ints_tensor must be a 2-D UInt8 tensor")
    _require(codes.size(0) % ctx_blk == 0, "ctx_len must be divisible by %d (the block's tokens at this pack_len)" % ctx_blk)
    _require(codes.size(1) % hid_blk == 0, "hidden_dim must be divisible by hidden_dim_block_size")
    nblk = (codes.size(0) // ctx_blk) * (codes.size(1) // hid_blk)
    _require(info.dim() == 2 and info.size(0) == nblk and info.size(1) == 2, "block_info_buffer block num mismatch")
    _require(stream.dtype == torch.uint8 and stream.numel() > 0, "compressed_buffer must be a non-empty UInt8 tensor")
    _require(info.dtype == torch.uint32, "block_info_buffer must be a UInt32 tensor")
    _require(2 <= bits <= MAX_BITS, "bits_len must be 2..%d" % MAX_BITS)
    _require(codes.is_cuda and stream.is_cuda and info.is_cuda, "tensors must be on the GPU")
    _require(codes.is_contiguous() and stream.is_contiguous() and info.is_contiguous(), "tensors must be contiguous")
    _require(stream.data_ptr() % 2 == 0, "compressed_buffer must start at an even address")


def encode_p(is_k, codes, stream, info, pack_len, bits, want_size=True, timed=False):
    """Encode a uint8 code matrix [ctx_len, hidden] with packs of `pack_len` tokens (16 = the reference's format with
    its block shapes).  Returns the stream size (and ms)."""
    _check_long(is_k, codes, stream, info, pack_len, bits)
    dev = _device_of(codes, stream, info)
    size, ms = ctypes.c_uint64(0), ctypes.c_float(0.0)
    fn = _lib.load().pkv_k_encode_p if is_k else _lib.load().pkv_v_encode_p
    with _on(dev):
        rc = fn(_ptr(codes), _ptr(stream), stream.numel(), _ptr(info), codes.size(0), codes.size(1), pack_len, bits,
                ctypes.byref(size) if want_size else None, ctypes.byref(ms) if timed else None, _stream(dev))
    _lib.check(rc)
    return (int(size.value), float(ms.value)) if timed else int(size.value)


def decode_p(is_k, stream, info, codes, pack_len, bits, timed=False):
    _check_long(is_k, codes, stream, info, pack_len, bits)
    dev = _device_of(codes, stream, info)
    ms = ctypes.c_float(0.0)
    fn = _lib.load().pkv_k_decode_p if is_k else _lib.load().pkv_v_decode_p
    with _on(dev):
        rc = fn(_ptr(stream), stream.numel(), _ptr(info), _ptr(codes), codes.size(0), codes.size(1), pack_len, bits,
                ctypes.byref(ms) if timed else None, _stream(dev))
    _lib.check(rc)
    return float(ms.value) if timed else None


# --------------------------------------------------------------- quantizer -----------

def _check_x(x):
    _require(x.is_cuda and x.dim() == 4 and x.size(3) == 128 and x.is_contiguous(),
             "x must be a contiguous device tensor [B, H, T, 128]")
    return x.size(0), x.size(1), x.size(2)


def _check_params(scale, zero, B, T, dtype, device):
    for name, t in (("scale", scale), ("zero", zero)):
        _require(t.is_cuda and t.device == device and t.dtype == dtype and t.dtype in (torch.float16, torch.bfloat16) and
                 t.numel() == B * T and t.is_contiguous(),
                 name + " must be a contiguous device tensor of B*T values in the tensor's 16-bit dtype")


def quant_params(x, rel, timed=False):
    """Per-(batch, token) scale and zero of quant_ints(TokenQuant) (utils/compute.py:84-112);
    returns (scale, zero) as [B, T] tensors of x.dtype."""
    B, H, T = _check_x(x)
    scale = torch.empty(B, T, dtype=x.dtype, device=x.device)
    zero = torch.empty(B, T, dtype=x.dtype, device=x.device)
    ms = ctypes.c_float(0.0)
    with _on(x.device):
        rc = _lib.load().pkv_quant_params(_ptr(x), _dtype_code(x), B, H, T, float(rel), _ptr(scale),
                                          _ptr(zero), ctypes.byref(ms) if timed else None, _stream(x.device))
    _lib.check(rc)
    return (scale, zero, float(ms.value)) if timed else (scale, zero)


def quantize(x, scale, zero):
    """uint8 code matrix [T, B*H*128] (layout of evaluation/evaluation.py:406) and the largest code."""
    B, H, T = _check_x(x)
    _check_params(scale, zero, B, T, x.dtype, x.device)
    mx = torch.zeros(1, dtype=torch.int32, device=x.device)
    codes = _quantize(x, scale, zero, B, H, T, mx)
    return codes, int(mx.item())


def _quantize(x, scale, zero, B, H, T, mx):
    codes = torch.empty(T, B * H * 128, dtype=torch.uint8, device=x.device)
    with _on(x.device):
        rc = _lib.load().pkv_quantize(_ptr(x), _dtype_code(x), B, H, T, _ptr(scale), _ptr(zero), _ptr(codes),
                                      _ptr(mx), None, _stream(x.device))
    _lib.check(rc)
    return codes


def quant_codes(x, rel):
    """(codes, scale, zero) of quant_params and quantize, without the largest code: nothing is waited for."""
    return _quant_codes((x,), (rel,))[0]


def quant_codes_pair(k, v, k_rel, v_rel):
    """quant_codes of K and of V, in one launch where they are alike."""
    if v.shape == k.shape and v.dtype == k.dtype and v.device == k.device:
        return _quant_codes((k, v), (k_rel, v_rel))
    return [quant_codes(k, k_rel), quant_codes(v, v_rel)]


def _quant_codes(xs, rels):
    out, args = [], []
    for x in xs:
        B, H, T = _check_x(x)
        codes = torch.empty(T, B * H * 128, dtype=torch.uint8, device=x.device)
        scale, zero = (torch.empty(B, T, dtype=x.dtype, device=x.device) for _ in range(2))
        out.append((codes, scale, zero))
        args += [_ptr(scale), _ptr(zero), _ptr(codes)]
    both, dev = len(xs) == 2, xs[0].device
    with _on(dev):
        rc = _lib.load().pkv_quant_codes(_ptr(xs[0]), _ptr(xs[1]) if both else None, _dtype_code(xs[0]), B, H, T, float(rels[0]),
                                         float(rels[-1]), *args, *(() if both else (None,) * 3), _stream(dev))
    _lib.check(rc)
    return out


def dequantize(codes, scale, zero, B, H):
    """(code + zero) * scale in the storage dtype -> [B, H, T, 128] (utils/compute.py:173-179)."""
    _require(codes.is_cuda and codes.dtype == torch.uint8 and codes.dim() == 2 and codes.is_contiguous() and
             codes.size(1) == B * H * 128, "codes must be a contiguous uint8 device tensor [T, B*H*128]")
    T = codes.size(0)
    _check_params(scale, zero, B, T, scale.dtype, codes.device)
    x = torch.empty(B, H, T, 128, dtype=scale.dtype, device=codes.device)
    with _on(codes.device):
        rc = _lib.load().pkv_dequantize(_ptr(codes), _dtype_code(scale), B, H, T, _ptr(scale), _ptr(zero),
                                        _ptr(x), None, _stream(codes.device))
    _lib.check(rc)
    return x


def _quant_encode(is_k, x, rel, bits, stream, info, want_size, timed, perm=None, perm_block=0, params=None):
    B, H, T = _check_x(x)
    _require(perm is None or (bits <= 6 and H <= 8), "a token order is taken by the fused encoders only (bits <= 6, H <= 8)")
    hidden = B * H * 128
    ctx_blk, hid_blk = (64, 128) if is_k else (128, 64)
    nblk = (T // ctx_blk) * (hidden // hid_blk)
    if stream is None:     # sized like the code matrix as the reference does; the extension widths can need more
        stream = torch.empty(max(T * hidden, nblk * block_bound(is_k, ctx_blk, hid_blk, bits) + 16) if bits > 4
                             else T * hidden, dtype=torch.uint8, device=x.device)
    if info is None:
        info = torch.empty(nblk, 2, dtype=torch.uint32, device=x.device)
    _require(info.numel() == 2 * nblk and info.dtype == torch.uint32, "block_info_buffer block num mismatch")
    if bits > 6:
        # widths 7..8 (format extension): quantize to the code matrix, then the block codec -- three kernels instead
        # of the fused one
        scale, zero = quant_params(x, rel)
        codes, mx = quantize(x, scale, zero)
        if mx >= (1 << bits):
            raise PackKVError(1, "not supported: code %d does not fit bits_len %d" % (mx, bits))
        res = _encode(is_k, codes, stream, info, T, hidden, ctx_blk, hid_blk, bits, want_size, timed, MAX_BITS)
        size, ms = res if timed else (res, 0.0)
        return {"stream": stream, "info": info, "scale": scale, "zero": zero, "size": int(size), "ms": float(ms),
                "bits": bits}
    scale = torch.empty(B, T, dtype=x.dtype, device=x.device)
    zero = torch.empty(B, T, dtype=x.dtype, device=x.device)
    size = ctypes.c_uint64(0)
    ms = ctypes.c_float(0.0)
    with _on(x.device):
        tail = (_ptr(stream), stream.numel(), _ptr(info), _ptr(scale), _ptr(zero), ctypes.byref(size) if want_size else None,
                ctypes.byref(ms) if timed else None, _stream(x.device))
        if perm is None:
            fn = _lib.load().pkv_k_quant_encode if is_k else _lib.load().pkv_v_quant_encode
            rc = fn(_ptr(x), _dtype_code(x), B, H, T, float(rel), bits, *tail)
        else:
            _require(perm.is_cuda and perm.dtype in (torch.uint32, torch.int32) and perm.numel() == T and perm.is_contiguous(),
                     "perm must hold one 32-bit index per token")
            if is_k:
                rc = _lib.load().pkv_k_quant_encode_perm(_ptr(x), _dtype_code(x), B, H, T, float(rel), bits, _ptr(perm),
                                                         int(perm_block), *tail)
            else:       # params: V's (scale, zero) [B, T] in the order of x, as median_order writes them
                sp, zp = (None, None) if params is None else (_ptr(params[0]), _ptr(params[1]))
                rc = _lib.load().pkv_v_quant_encode_perm(_ptr(x), _dtype_code(x), B, H, T, float(rel), bits, _ptr(perm),
                                                         int(perm_block), sp, zp, *tail)
    _lib.check(rc)
    return {"stream": stream, "info": info, "scale": scale, "zero": zero, "size": int(size.value),
            "ms": float(ms.value), "bits": bits}


def _stream_and_info(is_k, x, bits):
    """A stream buffer and block_info for x [B, H, T, 128]: sized like the code matrix as the reference does; the extension
    widths can need more."""
    B, H, T = x.size(0), x.size(1), x.size(2)
    hidden = B * H * 128
    ctx_blk, hid_blk = (64, 128) if is_k else (128, 64)
    nblk = (T // ctx_blk) * (hidden // hid_blk)
    room = max(T * hidden, nblk * block_bound(is_k, ctx_blk, hid_blk, bits) + 16) if bits > 4 else T * hidden
    return torch.empty(room, dtype=torch.uint8, device=x.device), torch.empty(nblk, 2, dtype=torch.uint32, device=x.device)


def _kv_quant_encode_perm(k, v, k_rel, v_rel, k_bits, v_bits, perm, perm_block, v_scale, v_zero):
    """Both sides of a repacked encode with one wait: dicts like k_quant_encode / v_quant_encode.  v_scale / v_zero: V's
    parameters [B, T] in the order of v."""
    B, H, T = _check_x(k)
    _require(k.get_device() == v.get_device() == perm.get_device() == v_scale.get_device() == v_zero.get_device(), _ONE_DEVICE)
    sides, out = [], []
    for is_k, x, rel, bits in ((True, k, k_rel, k_bits), (False, v, v_rel, v_bits)):
        stream, info = _stream_and_info(is_k, x, bits)
        scale = torch.empty(B, T, dtype=x.dtype, device=x.device)
        zero = torch.empty(B, T, dtype=x.dtype, device=x.device)
        a = _lib.AppendSide()
        a.x, a.stream, a.capacity, a.info_tail = x.data_ptr(), stream.data_ptr(), stream.numel(), info.data_ptr()
        a.scale_tail, a.zero_tail, a.rel, a.bits = scale.data_ptr(), zero.data_ptr(), float(rel), int(bits)
        sides.append(a)
        out.append({"stream": stream, "info": info, "scale": scale, "zero": zero, "size": 0, "ms": 0.0, "bits": bits})
    ks, vs = ctypes.c_uint64(0), ctypes.c_uint64(0)
    with _on(k.device):
        rc = _lib.load().pkv_kv_quant_encode_perm(ctypes.byref(sides[0]), ctypes.byref(sides[1]), _dtype_code(k), B, H, T, _ptr(perm),
                                                  int(perm_block), _ptr(v_scale), _ptr(v_zero), ctypes.byref(ks), ctypes.byref(vs),
                                                  _stream(k.device))
    _lib.check(rc)
    out[0]["size"], out[1]["size"] = int(ks.value), int(vs.value)
    return out[0], out[1]


def k_quant_encode(x, rel, bits=None, stream=None, info=None, want_size=True, timed=False):
    """Fused quantize + K encode of x [B, H, T, 128]; returns a dict with stream, info (block_info),
    scale, zero [B, T], size (bytes), ms and bits."""
    return _quant_encode(True, x, rel, bits or bits_for_rel(rel), stream, info, want_size, timed)


def v_quant_encode(x, rel, bits=None, stream=None, info=None, want_size=True, timed=False):
    return _quant_encode(False, x, rel, bits or bits_for_rel(rel), stream, info, want_size, timed)


def quant_encode_append(is_k, x, rel, bits, stream, used, info, tokens, scale, zero):
    """Append the tokens x [B, H, n, 128] (n a multiple of 64 for K, 128 for V) to a stream that holds
    ``tokens`` tokens in its first ``used`` bytes.  ``info`` [blocks, 2] and ``scale`` / ``zero``
    [B, row] are allocated for the cache's full length and filled behind what is there; the new blocks'
    offsets count from the start of ``stream``.  Returns the bytes in use afterwards."""
    B, H, n = _check_x(x)
    ctx_blk, hid_blk = (64, 128) if is_k else (128, 64)
    per_row = B * H * 128 // hid_blk
    _require(n % ctx_blk == 0 and tokens % ctx_blk == 0, "token counts must be multiples of the block length")
    nblk_done, nblk_new = tokens // ctx_blk * per_row, n // ctx_blk * per_row
    _require(info.is_cuda and info.dtype == torch.uint32 and info.is_contiguous()
             and info.numel() >= 2 * (nblk_done + nblk_new), "block_info_buffer too small")
    _require(scale.shape == zero.shape and scale.dim() == 2 and scale.size(0) == B and scale.dtype == x.dtype
             and zero.dtype == x.dtype and scale.is_contiguous() and zero.is_contiguous()
             and scale.size(1) >= tokens + n, "scale / zero must be contiguous [B, row] with room for the new tokens")
    _require(stream.is_cuda and stream.dtype == torch.uint8 and stream.is_contiguous() and 0 <= used <= stream.numel(),
             "compressed_buffer must be a contiguous device UInt8 tensor holding the bytes in use")
    es = scale.element_size()
    size = ctypes.c_uint64(0)
    fn = _lib.load().pkv_k_quant_encode_append if is_k else _lib.load().pkv_v_quant_encode_append
    with _on(x.device):
        rc = fn(_ptr(x), _dtype_code(x), B, H, n, float(rel), int(bits), _ptr(stream), stream.numel(), int(used),
                ctypes.c_void_p(info.data_ptr() + 8 * nblk_done), ctypes.c_void_p(scale.data_ptr() + es * tokens),
                ctypes.c_void_p(zero.data_ptr() + es * tokens), scale.size(1), ctypes.byref(size), None,
                _stream(x.device))
    _lib.check(rc)
    return int(size.value)


def window_append(k_new, v_new, cos, sin, k_win, v_win, win_pos):
    """Write the new tokens k_new / v_new [B, H, n, 128] into rows win_pos.. of the 16-bit windows k_win / v_win
    [B, H, cap, 128]; with cos / sin [B, n, 128] the keys get the rotary embedding first, rounded like the reference's
    chain of 16-bit elementwise ops (utils/compute.py:35-43).  One launch; strided views (a transposed projection
    output, an expanded cos / sin table) are read in place."""
    rc = _host().window_append(k_new, v_new, cos, sin, k_win, v_win, win_pos)
    if rc is not None:
        return _lib.check(rc)
    B, H, n, D = k_new.shape
    dev, at, dtype, win = k_new.device, k_new.get_device(), k_new.dtype, k_win.shape
    _require(D == 128 and v_new.shape == k_new.shape and k_new.is_cuda and v_new.dtype == dtype,
             "K and V must be device tensors [B, H, n, 128] of one dtype")
    _require(k_win.is_contiguous() and v_win.is_contiguous() and v_win.shape == win and len(win) == 4
             and win[0] == B and win[1] == H and win[3] == 128 and k_win.dtype == dtype,
             "windows must be contiguous [B, H, cap, 128] of the tokens' dtype")
    _require(v_new.get_device() == at and k_win.get_device() == at and v_win.get_device() == at, _ONE_DEVICE)
    ks = k_new.stride()
    if ks[3] != 1 or ks != v_new.stride():
        k_new, v_new = k_new.contiguous(), v_new.contiguous()
        ks = k_new.stride()
    rot_sb = 0
    if cos is not None:
        _require(cos.shape == (B, n, 128) and sin.shape == (B, n, 128) and cos.dtype == dtype
                 and sin.dtype == dtype, "cos / sin must be [B, n, 128] of the tokens' dtype")
        _require(cos.get_device() == at and sin.get_device() == at, _ONE_DEVICE)
        cs = cos.stride()
        if cs[2] != 1 or (n > 1 and cs[1] != 128) or cs != sin.stride():
            cos, sin = cos.contiguous(), sin.contiguous()
            cs = cos.stride()
        rot_sb = cs[0] if B > 1 else 0
    with _on(dev):
        rc = _lib.load().pkv_window_append(k_new.data_ptr(), v_new.data_ptr(), cos.data_ptr() if cos is not None else None,
                                           sin.data_ptr() if cos is not None else None, _dtype_code(k_new), B, H, n, ks[0], ks[1],
                                           ks[2], rot_sb, k_win.data_ptr(), v_win.data_ptr(), int(win_pos), win[2], _stream(dev))
    _lib.check(rc)


def _strides(t):
    """Element strides, those of one-element dimensions as 0: they mean nothing and can be any number."""
    st, shape = t.stride(), t.shape
    return tuple(s if size > 1 else 0 for s, size in zip(st, shape)) if 1 in shape else st


def _rows16(t, st):
    """Whether the rows of t [B, n, 128] or [B, H, n, 128] (strides `st`) can be read 16 bytes at a time where they are."""
    return st[-1] == 1 and t.data_ptr() % 16 == 0 and (st[0] | st[-3] | st[-2]) % 8 == 0


def _encodable(x, st):
    """Whether the encoders can read the rows of x [B, H, n, 128] (strides `st`) where they are: the limits of
    pkv_kv_quant_encode_append (token stride; K's head stride for five heads or more, where rows 128 apart have none)."""
    return _rows16(x, st) and st[2] < 1 << 25 and (x.size(1) <= 4 or st[2] == 128 or st[1] < (1 << 31) - 128)


def _copy(t):
    """A contiguous copy in memory of its own (contiguous() hands back a tensor that is contiguous at any address)."""
    return t.clone(memory_format=torch.contiguous_format)


def _rotary_rows(cos, sin, like):
    """cos / sin as [B, n, 128] tables the kernels read in place: (cos, sin, elements from one sequence's table to the next)."""
    B, n, dev, dtype = like.size(0), like.size(2), like.device, like.dtype
    _require(cos.device == dev and sin.device == dev, _ONE_DEVICE)
    cos, sin = cos.expand(B, n, 128), sin.expand(B, n, 128)
    _require(cos.dtype == dtype and sin.dtype == dtype, "cos / sin must be [B, n, 128] of the tokens' dtype")
    cs = _strides(cos)
    if (n > 1 and cs[1] != 128) or cs != _strides(sin) or not _rows16(cos, cs) or not _rows16(sin, cs):
        cos, sin = _copy(cos), _copy(sin)
        cs = _strides(cos)
    return cos, sin, cs[0]


def kv_quant_encode_append(k, v, n, k_side, v_side, tokens, cos=None, sin=None):
    """quant_encode_append for the first n tokens (a multiple of 128) of k and of v [B, H, >= n, 128], with one wait for
    both.  The rows are read where they are (any strides whose rows start on 16-byte boundaries).  k_side / v_side:
    (rel, bits, stream, used, info, scale, zero) as quant_encode_append takes them.  With cos / sin (tables of k's rows;
    five heads or more) the encoder applies the rotary embedding to K.  Returns the bytes in use of K and V."""
    B, H, dev, at = k.size(0), k.size(1), k.device, k.get_device()
    _require(n % 128 == 0 and tokens % 128 == 0, "token counts must be multiples of the block length")
    sides, sizes = [], (ctypes.c_uint64(0), ctypes.c_uint64(0))
    for x, (rel, bits, stream, used, info, scale, zero), per_tile, ctx_blk in ((k, k_side, B * H, 64), (v, v_side, 2 * B * H, 128)):
        st = _strides(x)
        _require(x.is_cuda and x.dim() == 4 and x.size(0) == B and x.size(1) == H and x.size(2) >= n and x.size(3) == 128 and _rows16(x, st),
                 "x must be a device tensor [B, H, n, 128] with rows on 16-byte boundaries")
        _require(x.get_device() == at and stream.get_device() == at and info.get_device() == at and scale.get_device() == at and zero.get_device() == at, _ONE_DEVICE)
        _require(info.dtype == torch.uint32 and info.is_contiguous()
                 and info.numel() >= 2 * ((tokens + n) // ctx_blk * per_tile), "block_info_buffer too small")
        _require(scale.shape == zero.shape == k_side[5].shape and scale.dim() == 2 and scale.size(0) == B and scale.dtype == x.dtype
                 and zero.dtype == x.dtype and scale.is_contiguous() and zero.is_contiguous() and scale.size(1) >= tokens + n,
                 "scale / zero must be contiguous [B, row] with room for the new tokens")
        _require(stream.dtype == torch.uint8 and stream.is_contiguous() and 0 <= used <= stream.numel(),
                 "compressed_buffer must be a contiguous device UInt8 tensor holding the bytes in use")
        es = scale.element_size()
        sides.append(_lib.AppendSide(x.data_ptr(), *st[:3], stream.data_ptr(), stream.numel(), int(used),
                                     info.data_ptr() + 8 * (tokens // ctx_blk * per_tile), scale.data_ptr() + es * tokens,
                                     zero.data_ptr() + es * tokens, float(rel), int(bits)))
    if cos is not None:
        cos, sin, sides[0].rot_stride_b = _rotary_rows(cos, sin, k)
        sides[0].cos, sides[0].sin = cos.data_ptr(), sin.data_ptr()
    with _on(dev):
        rc = _lib.load().pkv_kv_quant_encode_append(ctypes.byref(sides[0]), ctypes.byref(sides[1]), _dtype_code(k), B, H, n,
                                                    k_side[5].size(1), ctypes.byref(sizes[0]), ctypes.byref(sizes[1]), _stream(dev))
    _lib.check(rc)
    return int(sizes[0].value), int(sizes[1].value)


def window_cut(k_new, v_new, cos, sin, k_pend, v_pend, k_win, v_win, win_len, stage, pend_out, k_rel, v_rel,
               rotary_later=False):
    """The write into the cache's window when its first tokens leave for the streams (utils/compute.py:54-67,
    models/cache/packkv_quant.py:59-83).  Tokens in order: the pending cut's originals k_pend / v_pend [B, H, 64, 128] or
    None, the window rows behind them up to win_len, the new tokens [B, H, n, 128] (keys with their rotary embedding when
    cos / sin [B, n, 128] are given).  The first `stage` go to the encoder, `pend_out` (0 or 64) wait as the next pending
    cut, the rest are the new window.  Returns (k_stage, v_stage, k_pend, v_pend, k_win, v_win): what the encoder reads
    (the new tokens themselves where nothing has to be done to them, or where, with nothing in the window, rotary_later
    leaves the embedding of the staged keys to the encoder), the new pending originals or None, the new windows."""
    B, H, n, D = k_new.shape
    _require(D == 128 and v_new.shape == k_new.shape and k_new.is_cuda and v_new.is_cuda and v_new.dtype == k_new.dtype,
             "K and V must be device tensors [B, H, n, 128] of one dtype")
    _require(k_win.is_contiguous() and v_win.is_contiguous() and k_win.shape == v_win.shape and k_win.dim() == 4
             and k_win.size(0) == B and k_win.size(1) == H and k_win.size(3) == 128 and k_win.dtype == k_new.dtype,
             "windows must be contiguous [B, H, cap, 128] of the tokens' dtype")
    dev, at = k_new.device, k_new.get_device()
    _require(v_new.get_device() == at and k_win.get_device() == at and v_win.get_device() == at
             and (k_pend is None or k_pend.get_device() == at and v_pend.get_device() == at), _ONE_DEVICE)
    ks = _strides(k_new)
    if ks != _strides(v_new) or not _encodable(k_new, ks) or not _encodable(v_new, ks):
        k_new, v_new = _copy(k_new), _copy(v_new)
        ks = _strides(k_new)
    pend = 64 if k_pend is not None else 0
    buf = win_len - pend
    a = _lib.CutArgs()
    if cos is not None:
        cos, sin, a.rot_stride_b = _rotary_rows(cos, sin, k_new)
        a.cos, a.sin = cos.data_ptr(), sin.data_ptr()
    empty = lambda rows: torch.empty(B, H, rows, 128, dtype=k_new.dtype, device=dev)
    k_stage, v_stage = k_new, v_new
    if stage and (pend + buf or (cos is not None and not rotary_later)):
        k_stage = empty(stage)
        a.k_stage = k_stage.data_ptr()
    if stage and pend + buf:
        v_stage = empty(stage)
        a.v_stage = v_stage.data_ptr()
    kp, vp = (empty(64), empty(64)) if pend_out else (None, None)
    kw, vw = (torch.empty_like(k_win), torch.empty_like(v_win)) if win_len else (k_win, v_win)
    a.k_new, a.v_new = k_new.data_ptr(), v_new.data_ptr()
    a.stride_b, a.stride_h, a.stride_t = ks[:3]
    if pend:
        a.k_pend, a.v_pend = k_pend.data_ptr(), v_pend.data_ptr()
    if win_len:
        a.k_win, a.v_win = k_win.data_ptr(), v_win.data_ptr()
    if pend_out:
        a.k_pend_out, a.v_pend_out = kp.data_ptr(), vp.data_ptr()
    a.k_win_out, a.v_win_out, a.win_stride = kw.data_ptr(), vw.data_ptr(), k_win.size(2)
    a.dtype, a.B, a.H, a.n, a.pend, a.buf, a.stage, a.pend_out = _dtype_code(k_new), B, H, n, pend, buf, stage, pend_out
    a.k_rel, a.v_rel = float(k_rel), float(v_rel)
    with _on(dev):
        rc = _lib.load().pkv_window_cut(ctypes.byref(a), _stream(dev))
    _lib.check(rc)
    return k_stage, v_stage, kp, vp, kw, vw


# ------------------------------------------------- repacking and analytic size ------

def _check_code_matrix(c, name):
    _require(c.is_cuda and c.dim() == 2 and c.dtype == torch.uint8 and c.is_contiguous(),
             "%s must be a contiguous device UInt8 code matrix [ctx_len, hidden]" % name)


def code_stats(codes, pack_len, timed=False):
    """(sum over packs of bit_length(max - min), number of distinct code values) of a code matrix [ctx_len, hidden]
    for packs of `pack_len` consecutive tokens of one channel: the two data-dependent terms of `bit_pack`
    (utils/compute.py:272-297)."""
    _check_code_matrix(codes, "codes")
    ctx, hidden = codes.shape
    len_sum, n_unique, ms = ctypes.c_uint64(0), ctypes.c_uint32(0), ctypes.c_float(0.0)
    with _on(codes.device):
        rc = _lib.load().pkv_bit_pack_size(_ptr(codes), ctx, hidden, int(pack_len), ctypes.byref(len_sum),
                                           ctypes.byref(n_unique), ctypes.byref(ms) if timed else None,
                                           _stream(codes.device))
    _lib.check(rc)
    out = (int(len_sum.value), int(n_unique.value))
    return out + (float(ms.value),) if timed else out


def code_stats_pair(k_codes, v_codes, pack_len, perm=None, block_size=0):
    """code_stats of K and of V (one shape) with one wait; with `perm` [ctx_len] (32 bits, as the repackings return it) of the
    matrices in that order, which are not written: blocks of `block_size` tokens, a multiple of pack_len."""
    _check_code_matrix(k_codes, "k_codes")
    _check_code_matrix(v_codes, "v_codes")
    _require(k_codes.shape == v_codes.shape, "K and V code matrices must have one shape")
    _require(k_codes.get_device() == v_codes.get_device(), _ONE_DEVICE)
    ctx, hidden = k_codes.shape
    _require(perm is None or (perm.get_device() == k_codes.get_device() and perm.dtype in (torch.int32, torch.uint32) and perm.numel() == ctx
                              and perm.is_contiguous()), "perm must hold one 32-bit index per token")
    len_sum, n_unique = (ctypes.c_uint64 * 2)(), (ctypes.c_uint32 * 2)()
    with _on(k_codes.device):
        rc = _lib.load().pkv_bit_pack_size_pair(_ptr(k_codes), _ptr(v_codes), None if perm is None else _ptr(perm), int(block_size), ctx, hidden,
                                                int(pack_len), len_sum, n_unique, _stream(k_codes.device))
    _lib.check(rc)
    return (len_sum[0], n_unique[0]), (len_sum[1], n_unique[1])


def bit_pack_bytes(codes, pack_len, timed=False):
    """Analytic size of ONE code matrix [ctx_len, hidden] in bytes, as `bit_pack` prices each half
    (utils/compute.py:272-297): packs of `pack_len` consecutive tokens of one channel cost
    pack_len * bit_length(max - min) payload bits + W + ceil(log2(W + 1)) metadata bits, W = ceil(log2(#codes))."""
    stats = code_stats(codes, pack_len, timed=timed)
    size = _packed_bytes(codes, pack_len, *stats[:2])
    return (size, stats[2]) if timed else size


def _packed_bytes(codes, pack_len, len_sum, n_unique):
    ctx, hidden = codes.shape
    w = math.ceil(math.log2(n_unique))
    n_packs = (ctx // pack_len) * hidden
    return (len_sum * pack_len + n_packs * (w + math.ceil(math.log2(w + 1)))) // 8


def bit_pack(k_codes, v_codes, pack_len):
    """(k_bytes, v_bytes) of `bit_pack(blocks, pack_len)` (utils/compute.py:272-297) for blocks = K and V codes
    side by side."""
    if k_codes.shape != v_codes.shape or k_codes.get_device() != v_codes.get_device():
        return bit_pack_bytes(k_codes, pack_len), bit_pack_bytes(v_codes, pack_len)
    k, v = code_stats_pair(k_codes, v_codes, pack_len)
    return _packed_bytes(k_codes, pack_len, *k), _packed_bytes(v_codes, pack_len, *v)


def median_repacking(k_codes, v_codes, block_size=64, timed=False):
    """`median_repacking` (utils/compute.py:262-270) on the device: inside every block of `block_size` tokens, K and
    V rows are reordered together by descending median of the token's V codes; equal medians keep their order.
    Returns (k_repacked, v_repacked, perm) with perm [ctx_len] int32: perm[blk * block_size + r] = position inside the
    block the token at r came from."""
    _check_code_matrix(k_codes, "k_codes")
    _check_code_matrix(v_codes, "v_codes")
    _require(k_codes.shape == v_codes.shape, "K and V code matrices must have one shape")
    ctx, hidden = k_codes.shape
    k_out, v_out = torch.empty_like(k_codes), torch.empty_like(v_codes)
    perm = torch.empty(ctx, dtype=torch.int32, device=k_codes.device)
    ms = ctypes.c_float(0.0)
    with _on(k_codes.device):
        rc = _lib.load().pkv_median_repack(_ptr(k_codes), _ptr(v_codes), _ptr(k_out), _ptr(v_out), _ptr(perm), ctx,
                                           hidden, int(block_size), ctypes.byref(ms) if timed else None,
                                           _stream(k_codes.device))
    _lib.check(rc)
    return (k_out, v_out, perm, float(ms.value)) if timed else (k_out, v_out, perm)


def greedy_repacking(k_codes, v_codes, pack_len=16, block_size=64, timed=False):
    """`greedy_repacking` (utils/compute.py:210-260) on the device: every block of `block_size` tokens is rebuilt pack
    by pack -- seed = the remaining token closest (cosine) to the rounded mean of the remaining tokens, then
    pack_len - 1 times the remaining token that adds the fewest payload bits -- jointly for K and V.  Exact integer
    arithmetic; ties go to the earlier token.  Returns (k_repacked, v_repacked, perm) like median_repacking."""
    _check_code_matrix(k_codes, "k_codes")
    _check_code_matrix(v_codes, "v_codes")
    _require(k_codes.shape == v_codes.shape, "K and V code matrices must have one shape")
    ctx, hidden = k_codes.shape
    k_out, v_out = torch.empty_like(k_codes), torch.empty_like(v_codes)
    perm = torch.empty(ctx, dtype=torch.int32, device=k_codes.device)
    ms = ctypes.c_float(0.0)
    with _on(k_codes.device):
        rc = _lib.load().pkv_greedy_repack(_ptr(k_codes), _ptr(v_codes), _ptr(k_out), _ptr(v_out), _ptr(perm), ctx,
                                           hidden, int(block_size), int(pack_len), ctypes.byref(ms) if timed else None,
                                           _stream(k_codes.device))
    _lib.check(rc)
    return (k_out, v_out, perm, float(ms.value)) if timed else (k_out, v_out, perm)


def _median_code_order(k_codes, v_codes, block_size):
    """perm [ctx] int32 of median_repacking without the repacked matrices."""
    _check_code_matrix(k_codes, "k_codes")
    _check_code_matrix(v_codes, "v_codes")
    _require(k_codes.shape == v_codes.shape, "K and V code matrices must have one shape")
    ctx, hidden = k_codes.shape
    perm = torch.empty(ctx, dtype=torch.int32, device=k_codes.device)
    with _on(k_codes.device):
        rc = _lib.load().pkv_median_repack(_ptr(k_codes), _ptr(v_codes), None, None, _ptr(perm), ctx, hidden, int(block_size), None,
                                           _stream(k_codes.device))
    _lib.check(rc)
    return perm


def greedy_order(k_codes, v_codes, pack_len=16, block_size=64):
    """perm [ctx] int32 of greedy_repacking without the repacked matrices (for the fused encoders, which gather the
    rows of K and V themselves)."""
    _check_code_matrix(k_codes, "k_codes")
    _check_code_matrix(v_codes, "v_codes")
    _require(k_codes.shape == v_codes.shape, "K and V code matrices must have one shape")
    ctx, hidden = k_codes.shape
    perm = torch.empty(ctx, dtype=torch.int32, device=k_codes.device)
    with _on(k_codes.device):
        rc = _lib.load().pkv_greedy_repack(_ptr(k_codes), _ptr(v_codes), None, None, _ptr(perm), ctx, hidden,
                                           int(block_size), int(pack_len), None, _stream(k_codes.device))
    _lib.check(rc)
    return perm


def repack_and_encode(k_codes, v_codes, pack_size, repack_method="none", block_size=64):
    """`repack_and_encode` (utils/compute.py:329-357) on code matrices: (k_size_pre, v_size_pre, k_size_aft,
    v_size_aft) in bytes.  repack_method: "none", "median" or "greedy"."""
    return _repack_and_encode(k_codes, v_codes, pack_size, repack_method, block_size, bit_pack(k_codes, v_codes, pack_size))


def _repack_and_encode(k_codes, v_codes, pack_size, repack_method, block_size, pre):
    """repack_and_encode with the sizes before repacking at hand."""
    k_pre, v_pre = pre
    if repack_method in ("median", "greedy") and block_size % pack_size == 0:       # priced where they lie
        order = greedy_order(k_codes, v_codes, pack_size, block_size) if repack_method == "greedy" else _median_code_order(k_codes, v_codes, block_size)
        k_aft, v_aft = code_stats_pair(k_codes, v_codes, pack_size, order, block_size)
        return k_pre, v_pre, _packed_bytes(k_codes, pack_size, *k_aft), _packed_bytes(v_codes, pack_size, *v_aft)
    if repack_method == "median":
        k_codes, v_codes, _ = median_repacking(k_codes, v_codes, block_size)
    elif repack_method == "greedy":
        k_codes, v_codes, _ = greedy_repacking(k_codes, v_codes, pack_size, block_size)
    elif repack_method == "none":
        return k_pre, v_pre, k_pre, v_pre
    else:
        raise ValueError("repack_method must be one of none, median, greedy")
    k_aft, v_aft = bit_pack(k_codes, v_codes, pack_size)
    return k_pre, v_pre, k_aft, v_aft


def median_order(v, rel, bits=None, block_size=64, timed=False, want_params=False):
    """perm [T] int32 of `median_repacking` (utils/compute.py:262-270) for V [B, H, T, 128] quantised at `rel`,
    counted straight from V: perm[blk * block_size + r] = index inside the block of the token that moves to r."""
    B, H, T = _check_x(v)
    bits = bits or bits_for_rel(rel)
    perm = torch.empty(T, dtype=torch.int32, device=v.device)
    scale = torch.empty(B, T, dtype=v.dtype, device=v.device) if want_params else None
    zero = torch.empty(B, T, dtype=v.dtype, device=v.device) if want_params else None
    ms = ctypes.c_float(0.0)
    with _on(v.device):
        rc = _lib.load().pkv_median_order(_ptr(v), _dtype_code(v), B, H, T, float(rel), bits, int(block_size), _ptr(perm),
                                          _ptr(scale) if want_params else None, _ptr(zero) if want_params else None,
                                          ctypes.byref(ms) if timed else None, _stream(v.device))
    _lib.check(rc)
    out = (perm, scale, zero) if want_params else perm          # want_params: V's (scale, zero) in the order of v
    return (out, float(ms.value)) if timed else out


def repack_quant_encode(k, v, k_rel, v_rel, repack_method="median", block_size=64, k_bits=None, v_bits=None, fused=None):
    """Quantize K and V [B, H, T, 128], reorder the tokens of every quantisation block (jointly for K and V, as the
    reference's repacking does before it prices the packs, utils/compute.py:329-357) and encode.  Returns (k, v,
    perm): dicts like k_quant_encode / v_quant_encode -- stream, info, scale, zero in the REPACKED token order, so
    attn_decode takes them as they are (attention does not depend on the order of the cached tokens) -- and the
    permutation [T] int32 (perm[blk * block_size + r] = position inside the block the token at r came from).
    `fused` (default: whenever it applies -- median or greedy method, H <= 8, codes of at most 6 bits) runs the fused
    encoders on the permuted tokens: the median order is counted from V itself (median_order, no code matrix at all),
    the greedy order from the code matrices (greedy_order), which are then dropped instead of being repacked and
    encoded; fused=False goes through the code matrices (quantize, repack, block codec), which gives the same streams."""
    B, H, T = _check_x(k)
    _require(v.shape == k.shape and v.dtype == k.dtype and v.is_cuda and v.is_contiguous(), "K and V must have one shape")
    _require(T % 128 == 0 and T % block_size == 0, "the token count must be a multiple of 128 and of block_size")
    k_bits, v_bits = k_bits or bits_for_rel(k_rel), v_bits or bits_for_rel(v_rel)
    can_fuse = (repack_method in ("median", "greedy") and H <= 8 and max(k_bits, v_bits) <= 6 and block_size % 64 == 0 and
                block_size <= (1024 if repack_method == "median" else 256))
    if fused is None:
        fused = can_fuse
    if fused:
        # the order from V itself, then the fused encoders on the tokens in that order: no code matrix in HBM
        _require(can_fuse, "the fused path takes the median or greedy method, at most 8 KV heads, codes of at most 6 bits and "
                           "blocks of a multiple of 64 tokens")
        if repack_method == "median":
            perm, vs, vz = median_order(v, v_rel, v_bits, block_size, want_params=True)
        else:
            (kc, _, _), (vc, vs, vz) = quant_codes_pair(k, v, k_rel, v_rel)
            perm = greedy_order(kc, vc, 16, block_size)      # the codecs' packs are 16 tokens
            del kc, vc                                       # (codes too wide for the stream are the encoders' to report)
        return _kv_quant_encode_perm(k, v, k_rel, v_rel, k_bits, v_bits, perm, block_size, vs, vz) + (perm,)
    ks, kz = quant_params(k, k_rel)
    vs, vz = quant_params(v, v_rel)
    kc, kmx = quantize(k, ks, kz)
    vc, vmx = quantize(v, vs, vz)
    for mx, bits in ((kmx, k_bits), (vmx, v_bits)):
        if mx >= (1 << bits):
            raise PackKVError(1, "not supported: code %d does not fit bits_len %d" % (mx, bits))
    if repack_method in ("median", "greedy"):
        if repack_method == "median":
            kc, vc, perm = median_repacking(kc, vc, block_size)
        else:
            kc, vc, perm = greedy_repacking(kc, vc, 16, block_size)      # the codecs' packs are 16 tokens
        src = (torch.arange(T, device=k.device, dtype=torch.int64) // block_size) * block_size + perm.to(torch.int64)
        ks, kz, vs, vz = (p[:, src].contiguous() for p in (ks, kz, vs, vz))
    elif repack_method == "none":
        perm = (torch.arange(T, device=k.device, dtype=torch.int32) % block_size)
    else:
        raise ValueError("repack_method must be one of none, median, greedy")
    hidden = B * H * 128
    out = []
    for is_k, codes, scale, zero, bits in ((True, kc, ks, kz, k_bits), (False, vc, vs, vz, v_bits)):
        ctx_blk, hid_blk = (64, 128) if is_k else (128, 64)
        nblk = (T // ctx_blk) * (hidden // hid_blk)
        stream = torch.empty(max(T * hidden, nblk * block_bound(is_k, ctx_blk, hid_blk, bits) + 16) if bits > 4
                             else T * hidden, dtype=torch.uint8, device=k.device)
        info = torch.empty(nblk, 2, dtype=torch.uint32, device=k.device)
        size = _encode(is_k, codes, stream, info, T, hidden, ctx_blk, hid_blk, bits, True, False, MAX_BITS)
        out.append({"stream": stream, "info": info, "scale": scale, "zero": zero, "size": int(size), "ms": 0.0,
                    "bits": bits})
    return out[0], out[1], perm


# ------------------------------------------------------- reference GEMV surface ------

def _timed(served, raises=False):
    """What the native side of a timed op returned: milliseconds, or a status -- an unsupported shape prints and takes no time."""
    if type(served) is float:
        return served
    if served == _lib.ERR_UNSUPPORTED and not raises:
        print("no such case")
        return 0.0
    return _lib.check(served)


def _require_cuda(*ts):
    for t in ts:
        if not t.is_cuda:
            raise RuntimeError("tensor must be a CUDA tensor")


def kq_mat_vec_mul(compressed_buffer, block_info_buffer, q, kq_out, ctx_len, hidden_dim,
                   ctx_len_block_size, hidden_dim_block_size, bits_len, q_interleaved=True):
    """Drop-in for packkv_cuda.kq_mat_vec_mul (packkv_cuda.pyi:26-36): kq_out[h, tok] =
    sum_d q[h, d] * code[tok, h*128 + d]; returns kernel milliseconds.  `q` is expected in the
    reference's lane-interleaved layout (evaluation/evaluation.py:465-468) unless
    q_interleaved=False.  Like the reference, an unsupported shape or dtype prints a message
    and returns 0.0 (src/kernels.cu:586-589, :626-629)."""
    served = _host().mat_vec(True, compressed_buffer, block_info_buffer, q, kq_out, ctx_len, hidden_dim, ctx_len_block_size, hidden_dim_block_size,
                             bits_len, q_interleaved)
    if served is not None:
        return _timed(served)
    _require_cuda(compressed_buffer, block_info_buffer, q, kq_out)
    if q.dtype not in (torch.float16, torch.bfloat16):
        print("Unsupported data type")
        return 0.0
    ms = ctypes.c_float(0.0)
    with _on(q.device):
        rc = _lib.load().pkv_kq_mat_vec_mul(_ptr(compressed_buffer), compressed_buffer.numel() * compressed_buffer.element_size(), _ptr(block_info_buffer), _ptr(q),
                                            _ptr(kq_out), ctx_len, hidden_dim, ctx_len_block_size,
                                            hidden_dim_block_size, bits_len, _dtype_code(q),
                                            int(bool(q_interleaved)), ctypes.byref(ms), _stream(q.device))
    if rc == _lib.ERR_UNSUPPORTED:
        print("no such case")
        return 0.0
    _lib.check(rc)
    return float(ms.value)


def wv_mat_vec_mul(compressed_buffer, block_info_buffer, w, wv_out, ctx_len, hidden_dim,
                   ctx_len_block_size, hidden_dim_block_size, bits_len):
    """Drop-in for packkv_cuda.wv_mat_vec_mul (packkv_cuda.pyi:60-70): wv_out (fp32, caller-zeroed,
    [hidden_dim] or [H, 128]) += sum_tok w[c // 128, tok] * code[tok, c]; returns milliseconds."""
    served = _host().mat_vec(False, compressed_buffer, block_info_buffer, w, wv_out, ctx_len, hidden_dim, ctx_len_block_size, hidden_dim_block_size,
                             bits_len, False)
    if served is not None:
        return _timed(served)
    _require_cuda(compressed_buffer, block_info_buffer, w, wv_out)
    if w.dtype not in (torch.float16, torch.bfloat16):
        print("Unsupported data type")
        return 0.0
    if wv_out.dtype != torch.float32:
        raise RuntimeError("wv_out must be a float32 tensor")
    ms = ctypes.c_float(0.0)
    with _on(w.device):
        rc = _lib.load().pkv_wv_mat_vec_mul(_ptr(compressed_buffer), compressed_buffer.numel() * compressed_buffer.element_size(), _ptr(block_info_buffer), _ptr(w),
                                            _ptr(wv_out), ctx_len, hidden_dim, ctx_len_block_size,
                                            hidden_dim_block_size, bits_len, _dtype_code(w),
                                            ctypes.byref(ms), _stream(w.device))
    if rc == _lib.ERR_UNSUPPORTED:
        print("no such case")
        return 0.0
    _lib.check(rc)
    return float(ms.value)


def fused_kq(our_kq, q, k_quant_zero, k_quant_scale, t):
    """Drop-in for packkv_cuda.fused_kq (packkv_cuda.pyi:72-78; checks of
    src/fused_kernels.cu:90-108): our_kq[m, n] = (sum(q[m]) * zero[n] + t[m, n]) * scale[n]."""
    served = _host().fused(True, our_kq, q, k_quant_zero, k_quant_scale, t)
    if served is not None:
        return _timed(served, raises=True)
    if q.dtype not in (torch.float16, torch.bfloat16):
        raise RuntimeError("Unsupported data type for fused_kq_launcher")
    if q.dim() != 2: raise RuntimeError("q must be a 2D tensor")
    if t.dim() != 2: raise RuntimeError("t must be a 2D tensor")
    if k_quant_zero.dim() != 1: raise RuntimeError("k_quant_zero must be a 1D tensor")
    if k_quant_scale.dim() != 1: raise RuntimeError("k_quant_scale must be a 1D tensor")
    if our_kq.dim() != 2: raise RuntimeError("our_kq must be a 2D tensor")
    M, K = q.shape
    N = t.size(1)
    if t.size(0) != M: raise RuntimeError("t.size(0) must be equal to q.size(0)")
    if k_quant_zero.size(0) != N: raise RuntimeError("k_quant_zero.size(0) must be equal to t.size(1)")
    if k_quant_scale.size(0) != N: raise RuntimeError("k_quant_scale.size(0) must be equal to t.size(1)")
    if our_kq.size(0) != M: raise RuntimeError("our_kq.size(0) must be equal to q.size(0)")
    if our_kq.size(1) != N: raise RuntimeError("our_kq.size(1) must be equal to t.size(1)")
    for name, x in (("q", q), ("t", t), ("k_quant_zero", k_quant_zero), ("k_quant_scale", k_quant_scale),
                    ("our_kq", our_kq)):
        if not x.is_cuda:
            raise RuntimeError("%s must be a CUDA tensor" % name)
    if not our_kq.is_contiguous(): raise RuntimeError("our_kq must be contiguous")
    ms = ctypes.c_float(0.0)
    # contiguous copies of strided inputs must outlive the call: a temporary released between two .contiguous() calls
    # can be handed the same memory again
    q_c, z_c, s_c, t_c = q.contiguous(), k_quant_zero.contiguous(), k_quant_scale.contiguous(), t.contiguous()
    with _on(q.device):
        rc = _lib.load().pkv_fused_kq(_ptr(our_kq), _ptr(q_c), _ptr(z_c), _ptr(s_c), _ptr(t_c), M, K, N,
                                      _dtype_code(q), ctypes.byref(ms), _stream(q.device))
    del q_c, z_c, s_c, t_c
    _lib.check(rc)
    return float(ms.value)


def fused_wv(our_wv, w, v_quant_zero, v_quant_scale, term1):
    """Drop-in for packkv_cuda.fused_wv (packkv_cuda.pyi:80-86; checks of
    src/fused_kernels.cu:275-293): our_wv[m, d] = sum_n w[m, n] * zero[n] * scale[n] + term1[m, d]."""
    served = _host().fused(False, our_wv, w, v_quant_zero, v_quant_scale, term1)
    if served is not None:
        return _timed(served, raises=True)
    if w.dtype not in (torch.float16, torch.bfloat16):
        raise RuntimeError("Unsupported data type for fused_wv_launcher")
    if w.dim() != 2: raise RuntimeError("w must be a 2D tensor")
    if term1.dim() != 2: raise RuntimeError("term1 must be a 2D tensor")
    if v_quant_zero.dim() != 1: raise RuntimeError("v_quant_zero must be a 1D tensor")
    if v_quant_scale.dim() != 1: raise RuntimeError("v_quant_scale must be a 1D tensor")
    if our_wv.dim() != 2: raise RuntimeError("our_wv must be a 2D tensor")
    M, N = w.shape
    D = term1.size(1)
    if term1.size(0) != M: raise RuntimeError("term1.size(0) must be equal to w.size(0)")
    if v_quant_zero.size(0) != N: raise RuntimeError("v_quant_zero.size(0) must be equal to w.size(1)")
    if v_quant_scale.size(0) != N: raise RuntimeError("v_quant_scale.size(0) must be equal to w.size(1)")
    if tuple(our_wv.shape) != (M, D): raise RuntimeError("our_wv shape must match term1")
    if term1.dtype != w.dtype: raise RuntimeError("term1 must have the dtype of w")
    for name, x in (("w", w), ("term1", term1), ("v_quant_zero", v_quant_zero),
                    ("v_quant_scale", v_quant_scale), ("our_wv", our_wv)):
        if not x.is_cuda:
            raise RuntimeError("%s must be a CUDA tensor" % name)
    if not our_wv.is_contiguous(): raise RuntimeError("our_wv must be contiguous")
    ms = ctypes.c_float(0.0)
    w_c, z_c, s_c, t_c = w.contiguous(), v_quant_zero.contiguous(), v_quant_scale.contiguous(), term1.contiguous()
    with _on(w.device):
        rc = _lib.load().pkv_fused_wv(_ptr(our_wv), _ptr(w_c), _ptr(z_c), _ptr(s_c), _ptr(t_c), M, N, D,
                                      _dtype_code(w), ctypes.byref(ms), _stream(w.device))
    del w_c, z_c, s_c, t_c
    _lib.check(rc)
    return float(ms.value)


# ------------------------------------------------- fused decompress-attention --------

def dense_view(k, v, k_win=None, v_win=None, win_len=None):
    """(K, V) [B, H, T, 128] behind a compressed cache: k and v as attn_decode takes them (stream, info, scale, zero,
    bits, ``tokens``, ``heads``) or None, dequantised as the reference stores them (utils/compute.py:173-179), followed
    by the `win_len` rows in use of the 16-bit windows k_win / v_win [B, H, cap, 128].  One launch."""
    served = _host().dense_view(k, v, k_win, v_win, win_len)
    if served is not None:
        return served if type(served) is tuple else _lib.check(served)
    a = AttnArgs()
    like = k["scale"] if k is not None else k_win
    dev, at = like.device, like.get_device()
    _require(like.is_cuda, "a compressed cache is on a GPU")
    if k is not None:
        T_c, B = int(k.get("tokens", k["scale"].size(1))), k["scale"].size(0)
        H = int(k["heads"]) if "heads" in k else k["info"].numel() // 2 // (T_c // 64) // B
        a.k_stream, a.k_info, a.k_scale, a.k_zero = _ptr(k["stream"]), _ptr(k["info"]), _ptr(k["scale"]), _ptr(k["zero"])
        a.v_stream, a.v_info, a.v_scale, a.v_zero = _ptr(v["stream"]), _ptr(v["info"]), _ptr(v["scale"]), _ptr(v["zero"])
        a.k_bytes, a.v_bytes = k["stream"].numel(), v["stream"].numel()
        a.k_bits, a.v_bits, a.par_stride = int(k["bits"]), int(v["bits"]), k["scale"].size(1)
        for d in (k, v):
            _require(d["scale"].shape == k["scale"].shape and d["zero"].shape == k["scale"].shape and d["scale"].size(1) >= T_c
                     and d["info"].numel() // 2 >= T_c // 64 * B * H and all(d[f].get_device() == at and d[f].is_contiguous()
                                                                             for f in ("stream", "info", "scale", "zero")),
                     "stream, info, scale and zero must be contiguous tensors on one device that hold the tokens in use")
    else:
        T_c, H, B = 0, k_win.size(1), k_win.size(0)
    T_w = 0
    if k_win is not None:
        T_w = k_win.size(2) if win_len is None else int(win_len)
        _require(k_win.get_device() == at and v_win.get_device() == at and k_win.is_contiguous() and v_win.is_contiguous() and k_win.shape == v_win.shape
                 and k_win.shape[:2] == (B, H) and k_win.size(3) == 128 and 0 <= T_w <= k_win.size(2) and k_win.dtype == like.dtype
                 and v_win.dtype == like.dtype, "window tensors must be contiguous [B, H, cap, 128] of the cache's dtype, all on one device")
        a.k_win, a.v_win, a.win_stride = _ptr(k_win), _ptr(v_win), k_win.size(2)
    a.B, a.Hkv, a.T_c, a.T_w, a.dtype = B, H, T_c, T_w, _dtype_code(like)
    k_out = torch.empty(B, H, T_c + T_w, 128, dtype=like.dtype, device=dev)
    v_out = torch.empty_like(k_out)
    with _on(dev):
        rc = _lib.load().pkv_dense_view(ctypes.byref(a), _ptr(k_out), _ptr(v_out), _stream(dev))
    _lib.check(rc)
    return k_out, v_out


class AttnPlan:
    """The checked, filled-in arguments of one decode step, kept for callers that repeat it (a decode loop over the
    same layer): ``plan()`` launches again without re-validating; ``plan(q=..., out=...)`` swaps the query / output
    tensors (same shape and dtype).  The tensors given at construction must stay alive and in place; build a new
    plan when a buffer is reallocated or the token counts change."""

    def __init__(self, q, k, v, k_win=None, v_win=None, sm_scale=None, out=None, variant=0, win_len=None,
                 ref_rounding=False, out_f32=False, noalloc=False):
        _require(q.is_cuda and q.dim() == 3 and q.size(2) == 128 and q.is_contiguous(),
                 "q must be a contiguous device tensor [B, Hq, 128]")
        B, Hq, _ = q.shape
        a = AttnArgs()
        T_c = 0
        Hkv = None
        if k is not None:
            T_c = int(k.get("tokens", k["scale"].size(1)))
            _require(int(v.get("tokens", v["scale"].size(1))) == T_c, "K and V hold different token counts")
            _require(0 < T_c <= k["scale"].size(1) and k["scale"].shape == v["scale"].shape,
                     "scale / zero rows shorter than the token count")
            a.par_stride = k["scale"].size(1)
            for name, d in (("k", k), ("v", v)):
                for f in ("stream", "info", "scale", "zero"):
                    if not (d[f].is_cuda and d[f].is_contiguous()):
                        _require(False, "%s.%s must be a contiguous device tensor" % (name, f))
            nblk_k = k["info"].numel() // 2
            Hkv = int(k["heads"]) if "heads" in k else nblk_k // (T_c // 64) // B
            _require(nblk_k >= (T_c // 64) * B * Hkv and v["info"].numel() // 2 >= (T_c // 128) * B * Hkv * 2,
                     "block_info_buffer block num mismatch")
            a.k_stream, a.k_info = k["stream"].data_ptr(), k["info"].data_ptr()
            a.v_stream, a.v_info = v["stream"].data_ptr(), v["info"].data_ptr()
            # readable bytes of each buffer.  The default kernel copies whole dwords and needs no slack; the gather
            # kernel (variant 2, and variant 0 on streams that are not 16-byte aligned) fetches pack words as whole
            # 8-byte words and needs 7 readable bytes behind the encoded size: without them the plain kernel runs
            gathers = int(variant) == 2 or (int(variant) == 0 and (k["stream"].data_ptr() | v["stream"].data_ptr()) % 16 != 0)
            if gathers and any(d.get("size") and d["stream"].numel() < int(d["size"]) + 7 for d in (k, v)):
                variant = 1
            a.k_bytes, a.v_bytes = k["stream"].numel(), v["stream"].numel()
            a.k_scale, a.k_zero = k["scale"].data_ptr(), k["zero"].data_ptr()
            a.v_scale, a.v_zero = v["scale"].data_ptr(), v["zero"].data_ptr()
            a.k_bits, a.v_bits = int(k["bits"]), int(v["bits"])
        T_w = 0
        if k_win is not None:
            _require(k_win.is_cuda and v_win.is_cuda and k_win.is_contiguous() and v_win.is_contiguous()
                     and k_win.shape == v_win.shape and k_win.dim() == 4 and k_win.size(3) == 128
                     and k_win.dtype == q.dtype and v_win.dtype == q.dtype,
                     "window tensors must be contiguous [B, Hkv, T_w, 128] of q's dtype")
            T_w = k_win.size(2) if win_len is None else int(win_len)
            _require(0 < T_w <= k_win.size(2), "win_len outside the window tensors")
            a.win_stride = k_win.size(2)
            _require(Hkv is None or Hkv == k_win.size(1), "window head count mismatch")
            Hkv = k_win.size(1)
            a.k_win, a.v_win = k_win.data_ptr(), v_win.data_ptr()
        _require(Hkv is not None, "empty cache")
        out_dtype = torch.float32 if out_f32 else q.dtype
        if out is None:
            out = torch.empty(q.shape, dtype=out_dtype, device=q.device)
        _require(out.is_cuda and out.shape == q.shape and out.dtype == out_dtype and out.is_contiguous(),
                 "out must be a contiguous device tensor of q's shape (fp32 with out_f32, else q's dtype)")
        a.flags = (_lib.ATTN_REF_ROUNDING if ref_rounding else 0) | (_lib.ATTN_OUT_F32 if out_f32 else 0)
        a.q, a.out = q.data_ptr(), out.data_ptr()
        a.B, a.Hq, a.Hkv, a.T_c, a.T_w = B, Hq, Hkv, T_c, T_w
        a.dtype = _dtype_code(q)
        a.sm_scale = float(sm_scale if sm_scale is not None else 128 ** -0.5)
        a.variant = int(variant)
        self.args, self.out, self.device = a, out, q.device
        self._shape, self._dtype, self._out_dtype = q.shape, q.dtype, out_dtype
        self._keep = (q, k, v, k_win, v_win, out)          # the buffers the pointers refer to
        self._fn = _lib.load().pkv_attn_decode
        self._fn_noalloc = _lib.load().pkv_attn_decode_noalloc if noalloc else None
        self._ref = ctypes.byref(a)
        self._where = (ctypes.addressof(a), q.get_device())

    def step(self, q, win_len):
        """The result of the step for `q` -- [B, Hq, 128], or [B, Hq, 1, 128] -- with `win_len` window rows in use, in q's shape;
        None where q is not what the plan was made for as it lies, and for plans of the checking kernels (flags, noalloc).  The
        plan's own query, output and window rows stay as they are."""
        if self._fn_noalloc is not None:
            return None
        served = _host().plan_step(*self._where, win_len, q)
        return _lib.check(served) if type(served) is int else served

    def set_window_rows(self, win_len):
        """Window rows in use (the window tensors are allocated longer and fill up between cuts)."""
        self.args.T_w = int(win_len)

    def __call__(self, q=None, out=None, timed=False):
        a = self.args
        if q is not None:
            _require(q.is_cuda and q.shape == self._shape and q.dtype == self._dtype and q.is_contiguous(),
                     "q must match the plan's query tensor")
            a.q = q.data_ptr()
        if out is not None:
            _require(out.is_cuda and out.shape == self._shape and out.dtype == self._out_dtype and out.is_contiguous(),
                     "out must match the plan's output tensor")
            a.out = out.data_ptr()
            self.out = out
        ms = ctypes.c_float(0.0) if timed else None
        with _on(self.device):
            if self._fn_noalloc is not None:
                _require(not timed, "the entry point that allocates nothing does not time its launch")
                rc = self._fn_noalloc(self._ref, _stream(self.device))
            else:
                rc = self._fn(self._ref, ctypes.byref(ms) if timed else None, _stream(self.device))
        if rc:
            _lib.check(rc)
        return (self.out, float(ms.value)) if timed else self.out


def attn_decode(q, k, v, k_win=None, v_win=None, sm_scale=None, out=None, variant=0, timed=False, win_len=None,
                ref_rounding=False, out_f32=False, noalloc=False):
    """One decode step over a compressed cache.

    q [B, Hq, 128]; k and v are the dicts returned by k_quant_encode / v_quant_encode (stream,
    info, scale, zero, bits) or None when only the 16-bit window exists; k_win / v_win are
    optional [B, Hkv, T_w, 128] tails.  Returns out [B, Hq, 128] (and ms when timed).

    Buffers allocated for a cache that grows: the dicts may carry ``tokens`` (compressed tokens in use;
    scale / zero rows and block_info are then longer than that) and ``heads`` (KV heads); ``win_len``
    gives the window rows in use when k_win / v_win are allocated longer.  AttnPlan keeps the checked
    arguments for callers that repeat the step.

    out_f32: the result as fp32, before its rounding to q's dtype.  ref_rounding (variant 1 only): the checking
    mode -- every K and V element is formed as the reference stores it, dtype(dtype(code + zero) * scale)
    (utils/compute.py:173-179), before the fp32 dot products.  noalloc: go through pkv_attn_decode_noalloc (the
    partial results in the library's fixed 8 MiB device array; the caller passes `out`, or torch allocates it)."""
    if out is None and not (variant or timed or ref_rounding or out_f32 or noalloc):
        served = _host().attn_decode(q, k, v, k_win, v_win, sm_scale, win_len)
        if served is not None:
            return _lib.check(served) if type(served) is int else served
    return AttnPlan(q, k, v, k_win, v_win, sm_scale, out, variant, win_len, ref_rounding, out_f32, noalloc)(timed=timed)
