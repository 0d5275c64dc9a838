"""The native host side (csrc/pkv_host.cpp) against the general code of ops.py: every call once through both, over the forms
that the native side takes and those that it must leave to the general code -- same results, same refusals."""
import contextlib

import pytest
import torch

from packkv_amd import _lib, cache as pc, ops, synth

pytestmark = pytest.mark.gpu


class _Counting:
    """The native side, counting what it serves; or nothing served at all."""

    def __init__(self, host, serve):
        self.host, self.serve, self.served = host, serve, 0

    def __getattr__(self, name):
        def call(*a):
            res = getattr(self.host, name)(*a) if self.serve else None
            self.served += res is not None
            return res
        return call


@contextlib.contextmanager
def _through(serve):
    _lib.load()
    old = _lib.host
    _lib.host = c = _Counting(old, serve)
    try:
        yield c
    finally:
        _lib.host = old


def _both(call, served):
    """call() natively and through the general code; the two results.  `served`: calls the native side is to take (None: any)."""
    out = []
    for serve in (True, False):
        with _through(serve) as c:
            out.append(call())
        assert c.served == (served if serve else 0) or (serve and served is None), c.served
    return out


def _same(a, b):
    if isinstance(a, (tuple, list)):
        return all(_same(x, y) for x, y in zip(a, b))
    return a.shape == b.shape and a.stride() == b.stride() and a.dtype == b.dtype and a.device == b.device and torch.equal(a, b)


def _cache(cuda, dtype, B=2, H=4, T=256, win=70, cap=96, rel=0.1):
    k, v = synth.make_kv(B, H, T + cap, seed=B + H, dtype=dtype, device=cuda)
    ke, ve = ops.k_quant_encode(k[:, :, :T].contiguous(), rel), ops.v_quant_encode(v[:, :, :T].contiguous(), rel)
    return ke, ve, k[:, :, T:].contiguous(), v[:, :, T:].contiguous(), synth.make_q(B, 2 * H, seed=3, dtype=dtype, device=cuda)


def _odd(t):
    """t's values at an address that is only its element's."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    return buf[1:].view(t.shape).copy_(t)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_attn_decode(cuda, dtype):
    ke, ve, kw, vw, q = _cache(cuda, dtype)
    grown = [dict(d, tokens=256, heads=4, scale=torch.cat([d["scale"], d["scale"]], 1), zero=torch.cat([d["zero"], d["zero"]], 1),
                  info=torch.cat([d["info"].view(torch.int32)] * 2).view(torch.uint32)) for d in (ke, ve)]
    shifted = dict(ke, stream=_odd(ke["stream"]))
    for args, kw_args, served in (((q, ke, ve), {}, 1), ((q, ke, ve, kw, vw), {}, 1), ((q, ke, ve, kw, vw), {"win_len": 3}, 1),
                                  ((q, None, None, kw, vw), {"win_len": 96}, 1), ((q, *grown, kw, vw), {"win_len": 70, "sm_scale": 0.25}, 1),
                                  ((_odd(q), ke, ve, kw, _odd(vw)), {}, 1), ((q, ke, ve), {"sm_scale": 1}, 0), ((q, shifted, ve), {}, 0),
                                  ((q, ke, ve), {"variant": 1}, 0), ((q, ke, ve), {"out_f32": True}, 0), ((q, ke, ve), {"noalloc": True}, 0),
                                  ((torch.nn.Parameter(q), ke, ve), {}, None)):
        a, b = _both(lambda: ops.attn_decode(*args, **kw_args), served)
        # (with a window of its own workgroups a head's partials can be added in any order: 1 ulp)
        assert a.shape == b.shape and a.dtype == b.dtype and (a.float() - b.float()).abs().max() <= 2e-3 * b.float().abs().max() + 2e-3
    bad = [(q.transpose(1, 2).contiguous().transpose(1, 2), ke, ve), (q.float(), ke, ve), (q, ke, ve, kw[:, :, ::2], vw[:, :, ::2]), (q, ke, ve, kw.float(), vw.float()),
           (q, None, None), (q.cpu(), ke, ve), (q[:, :, :64].contiguous(), ke, ve), (q, dict(ke, tokens=128), ve), (q, dict(ke, info=ke["info"][:3]), ve),
           (q, ke, ve, kw[:, :3].contiguous(), vw[:, :3].contiguous()), (q, dict(ke, tokens=64), dict(ve, tokens=64))]
    for args in bad:
        errors = []
        for serve in (True, False):
            with _through(serve) as c, pytest.raises(Exception) as e:
                ops.attn_decode(*args)
            errors.append((type(e.value), str(e.value)))
            assert c.served <= 1
        assert errors[0] == errors[1], args
    for win_len in (0, 97):
        for serve in (True, False):
            with _through(serve), pytest.raises(RuntimeError):
                ops.attn_decode(q, ke, ve, kw, vw, win_len=win_len)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_dense_view(cuda, dtype):
    ke, ve, kw, vw, _ = _cache(cuda, dtype, rel=0.05)
    for args, served in (((ke, ve), 1), ((ke, ve, kw, vw), 1), ((ke, ve, kw, vw, 5), 1), ((ke, ve, kw, vw, 0), 0), ((None, None, kw, vw, 7), 0)):
        assert _same(*_both(lambda: ops.dense_view(*args), served))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,H,n", [(1, 8, 1), (3, 2, 1), (2, 4, 5)])
def test_window_append(cuda, dtype, B, H, n):
    g = torch.Generator(device=cuda)
    g.manual_seed(n)
    new = lambda *s: torch.randn(*s, generator=g, device=cuda).to(dtype)
    k, v, table = new(B, H, n, 128), new(B, H, n, 128), new(n + 4, 128)
    projected = [new(B, n, H, 128).transpose(1, 2) for _ in range(2)]
    expanded = [table[i:i + n].unsqueeze(0).expand(B, -1, -1) for i in (0, 4)]
    for a, b, cos, sin, served in ((k, v, None, None, 1), (k, v, *expanded, 1), (*projected, *expanded, 1), (*projected, new(B, n, 128), new(B, n, 128), 1),
                                   (_odd(k), _odd(v), *expanded, 1), (k, projected[1], None, None, 0),
                                   (new(B, H, 128, n).transpose(2, 3), new(B, H, 128, n).transpose(2, 3), None, None, None),
                                   (k, v, new(B, n, 256)[..., ::2], new(B, n, 256)[..., ::2], 0)):
        def call():
            win = [torch.zeros(B, H, 9, 128, dtype=dtype, device=cuda) for _ in range(2)]
            ops.window_append(a, b, cos, sin, *win, 3)
            return win
        assert _same(*_both(call, served))
    for bad in ((k, v.float(), None, None), (k.cpu(), v.cpu(), None, None), (k[..., :64], v[..., :64], None, None), (k, v, table[:n], table[:n])):
        for serve in (True, False):
            win = [torch.zeros(B, H, 9, 128, dtype=dtype, device=cuda) for _ in range(2)]
            with _through(serve) as c, pytest.raises(RuntimeError):
                ops.window_append(*bad, *win, 3)
            assert c.served == 0 and not win[0].any()
    for serve in (True, False):           # (past the window's end: refused by the library)
        win = [torch.zeros(B, H, 9, 128, dtype=dtype, device=cuda) for _ in range(2)]
        with _through(serve), pytest.raises(ops.PackKVError):
            ops.window_append(k, v, None, None, *win, 9)


def test_a_growing_cache_through_both(cuda):
    B, Hq, H, steps = 2, 8, 2, 70
    k, v = synth.make_kv(B, H, 300 + steps, seed=9, device=cuda)
    q = torch.randn(steps, B, Hq, 1, 128, device=cuda).half()

    def run():
        cache, out = pc.PackKVCompressedCache(B, H, 128, 1, pc.PackKVCacheConfig(64, 192, 0.1, 0.1), max_tokens=512, device=cuda), []
        cache.update(k[:, :, :300], v[:, :, :300], 0, return_dense=False)
        for t in range(steps):
            cache.update(k[:, :, 300 + t:301 + t], v[:, :, 300 + t:301 + t], 0, return_dense=False)
            qt = q[t] if t % 3 else q[t, :, :, 0]
            out.append(cache.attend(qt, 0))
            assert out[-1].shape == qt.shape and out[-1].is_contiguous()
            if t % 16 == 5:
                given = torch.empty(B, Hq, 128, dtype=torch.float16, device=cuda)
                out += [cache.attend(qt, 0, out=given).reshape(qt.shape), cache.attend(qt, 0, sm_scale=0.5),
                        cache.attend(q[t].transpose(1, 2).contiguous().transpose(1, 2), 0), cache.attend(q[t].repeat(1, 1, 3, 1)[:, :, :1], 0)]
        return out, cache.materialize(0)
    (a, da), (b, db) = _both(run, None)
    assert _same(da, db) and len(a) == len(b)
    for x, y in zip(a, b):
        assert x.shape == y.shape and (x.float() - y.float()).abs().max() <= 2e-3


def test_on_a_side_stream_and_while_capturing(cuda):
    ke, ve, kw, vw, q = _cache(cuda, torch.float16)
    want = ops.attn_decode(q, ke, ve, kw, vw)
    s, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        ops.attn_decode(q, ke, ve, kw, vw)
    with _through(True) as c, torch.cuda.graph(graph, stream=s):
        got = ops.attn_decode(q, ke, ve, kw, vw)
    assert c.served == 1
    for _ in range(3):
        got.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert (got.float() - want.float()).abs().max() <= 2e-3
        assert (ops.attn_decode(q, ke, ve, kw, vw).float() - want.float()).abs().max() <= 2e-3


def test_a_step_leaves_the_plan_as_it_is(cuda):
    ke, ve, kw, vw, q = _cache(cuda, torch.float16)
    other = q.flip(0).contiguous()
    for form in ({"out_f32": True}, {"ref_rounding": True, "variant": 1}, {"noalloc": True}):
        assert ops.AttnPlan(q, ke, ve, kw, vw, win_len=33, **form).step(q, 33) is None
    plan = ops.AttnPlan(q, ke, ve, kw, vw, win_len=33)
    want = plan().clone()
    before, out = bytes(plan.args), plan.out
    got = plan.step(other, 70)
    assert bytes(plan.args) == before and (got.float() - ops.attn_decode(other, ke, ve, kw, vw, win_len=70).float()).abs().max() <= 2e-3
    out.zero_()
    again = plan()
    assert again is out and (again.float() - want.float()).abs().max() <= 2e-3


def test_a_function_mode_sees_the_general_code(cuda):
    ke, ve, _, _, q = _cache(cuda, torch.float16)

    class Seen(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))
    with _through(True) as c, Seen():
        ops.attn_decode(q, ke, ve)
    assert c.served == 0


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_matrix_vector_ops(cuda, dtype, capsys):
    H, T = 2, 256
    ke, ve, *_ = _cache(cuda, dtype, 1, H, T)
    new = lambda *s: torch.randn(*s, device=cuda).to(dtype)
    q, w = new(H, 128), new(H, T)

    def all_four(zero=lambda d: d["zero"].reshape(-1), q=q, w=w):
        t, kq, term, wv = (torch.zeros(H, T, dtype=dtype, device=cuda), torch.zeros(H, T, dtype=dtype, device=cuda),
                           torch.zeros(H, 128, device=cuda), torch.zeros(H, 128, dtype=dtype, device=cuda))
        ms = [ops.kq_mat_vec_mul(ke["stream"], ke["info"], q, t, T, H * 128, 64, 128, 4), ops.fused_kq(kq, q, zero(ke), ke["scale"].reshape(-1), t),
              ops.wv_mat_vec_mul(ve["stream"], ve["info"], w, term, T, H * 128, 128, 64, 4), ops.fused_wv(wv, w, zero(ve), ve["scale"].reshape(-1), term.to(dtype))]
        assert all(m > 0 for m in ms)
        return t, kq, term, wv
    a, b = _both(all_four, 4)
    assert _same(a[:2], b[:2]) and all(torch.allclose(x.float(), y.float(), rtol=2e-2, atol=1e-2) for x, y in zip(a[2:], b[2:]))
    strided = lambda d: torch.stack([d["zero"].reshape(-1)] * 2, 1)[:, 0]
    a, b = _both(lambda: all_four(strided), 2)
    assert _same(a[:2], b[:2])
    for serve in (True, False):
        with _through(serve):
            assert ops.kq_mat_vec_mul(ke["stream"], ke["info"], q, new(H, T), T, H * 128, 64, 128, 7) == 0.0
            assert "no such case" in capsys.readouterr().out
            assert ops.kq_mat_vec_mul(ke["stream"], ke["info"], q.float(), new(H, T), T, H * 128, 64, 128, 4) == 0.0
            assert "Unsupported" in capsys.readouterr().out
            with pytest.raises(RuntimeError):
                ops.fused_kq(new(H, T + 1), q, ke["zero"].reshape(-1), ke["scale"].reshape(-1), new(H, T))
            with pytest.raises(RuntimeError):
                ops.wv_mat_vec_mul(ve["stream"], ve["info"], w, new(H, 128), T, H * 128, 128, 64, 4)


def test_a_tensor_that_does_not_give_its_address(cuda):
    """data_ptr() may throw: the error is the general code's, whichever tensor it is, and the interpreter goes on."""
    ke, ve, kw, vw, q = _cache(cuda, torch.float16, 1, 2, 256)
    new = lambda *s: torch.zeros(*s, dtype=torch.float16, device=cuda)
    win = [new(1, 2, 9, 128) for _ in range(2)]
    rows, par = [new(1, 2, 1, 128) for _ in range(2)], [d[f].reshape(-1) for d in (ke, ve) for f in ("zero", "scale")]
    table = [new(1, 1, 128) for _ in range(2)]
    calls = {"append": (lambda a: ops.window_append(*a, 3), [*rows, *table, *win]),
             "kq": (lambda a: ops.kq_mat_vec_mul(*a, 256, 256, 64, 128, 4), [ke["stream"], ke["info"], new(2, 128), new(2, 256)]),
             "wv": (lambda a: ops.wv_mat_vec_mul(*a, 256, 256, 128, 64, 4), [ve["stream"], ve["info"], new(2, 256), torch.zeros(2, 128, device=cuda)]),
             "fused_kq": (lambda a: ops.fused_kq(*a), [new(2, 256), new(2, 128), *par[:2], new(2, 256)]),
             "fused_wv": (lambda a: ops.fused_wv(*a), [new(2, 128), new(2, 256), *par[2:], new(2, 128)]),
             "attn": (lambda a: ops.attn_decode(a[0], ke, ve, *a[1:]), [q, kw, vw]),
             "dense": (lambda a: ops.dense_view(ke, ve, *a), [kw, vw])}
    for name, (call, tensors) in calls.items():
        for i in range(len(tensors)):
            closed = tensors[i].clone()
            torch._C._set_throw_on_mutable_data_ptr(closed)
            args = tensors[:i] + [closed] + tensors[i + 1:]
            for serve in (True, False):
                with _through(serve), pytest.raises(RuntimeError, match="data pointer"):
                    call(args)
        call(tensors)
    torch.cuda.synchronize()
