"""GPU parity of the reference's GEMV surface (kq_mat_vec_mul, fused_kq, wv_mat_vec_mul, fused_wv),
following the reference call sequences (evaluation/evaluation.py:398-524, :587-715) and checked
against fp64 NumPy on the same codes."""
import numpy as np
import pytest
import torch

import packkv_cuda
from oracle import quant as oq
from packkv_amd import ops, synth

pytestmark = pytest.mark.gpu


def _setup(cuda, H, T, rel, is_k, dtype, seed):
    k, v = synth.make_kv(1, H, T, seed=seed, dtype=dtype)
    x = k if is_k else v
    c, z, s = oq.quant_ints(x, 64, rel)
    cm = oq.code_matrix(c)
    W = ops.bits_for_rel(rel)
    cb, hb = (64, 128) if is_k else (128, 64)
    info = torch.zeros((T // cb) * (H * 128 // hb), 2, dtype=torch.uint32)
    comp = torch.zeros_like(cm)
    size = (packkv_cuda.k_encode_cpu if is_k else packkv_cuda.v_encode_cpu)(cm, comp, info, T, H * 128, cb, hb, W)
    assert size > 0
    return cm, z.flatten(), s.flatten(), comp.to(cuda), info.to(cuda), W, cb, hb


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("H", [8, 32, 40])
def test_kq_path(cuda, dtype, H):
    T, rel = 512, 0.1
    cm, zero, scale, comp, info, W, cb, hb = _setup(cuda, H, T, rel, True, dtype, 41)
    torch.manual_seed(0)
    q = torch.randn(H, 128).to(dtype)
    t = torch.zeros(H, T, dtype=dtype, device=cuda)
    ms = packkv_cuda.kq_mat_vec_mul(comp, info, oq.q_interleave(q).to(cuda), t, T, H * 128, cb, hb, W)
    assert ms > 0
    codes = cm.numpy().astype(np.float64).reshape(T, H, 128)
    want_t = np.einsum("thd,hd->ht", codes, q.double().numpy())
    tol = 2 ** -9 if dtype == torch.float16 else 2 ** -6      # one rounding of the output to dtype
    assert np.abs(t.cpu().double().numpy() - want_t).max() <= tol * np.abs(want_t).max()
    # plain (non-interleaved) q gives the same result
    t2 = torch.zeros_like(t)
    ops.kq_mat_vec_mul(comp, info, q.to(cuda), t2, T, H * 128, cb, hb, W, q_interleaved=False)
    assert torch.equal(t, t2)
    our_kq = torch.empty_like(t)
    ms2 = packkv_cuda.fused_kq(our_kq, q.to(cuda), zero.to(cuda), scale.to(cuda), t)
    assert ms2 > 0
    want = (q.double().sum(1, keepdim=True) * zero.double()[None] + t.cpu().double()) * scale.double()[None]
    assert np.abs(our_kq.cpu().double().numpy() - want.numpy()).max() <= tol * want.abs().max().item()
    # against the dequantised-K matmul the reference uses as its target (10 % acceptance there)
    kd = ((cm.double().reshape(T, H, 128) + zero.double().view(T, 1, 1)) * scale.double().view(T, 1, 1))
    target = np.einsum("thd,hd->ht", kd.numpy(), q.double().numpy())
    assert np.abs(our_kq.cpu().double().numpy() - target).max() <= 4 * tol * np.abs(target).max()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("H,rel", [(8, 0.2), (40, 0.2), (32, 0.1)])
def test_wv_path(cuda, dtype, H, rel):
    T = 512
    cm, zero, scale, comp, info, W, cb, hb = _setup(cuda, H, T, rel, False, dtype, 43)
    torch.manual_seed(1)
    w = torch.randn(H, T).to(dtype).pow(2).softmax(dim=1)
    w_prime = (w * scale.unsqueeze(0)).to(cuda)
    term1 = torch.zeros(H, 128, dtype=torch.float32, device=cuda)
    ms = packkv_cuda.wv_mat_vec_mul(comp, info, w_prime, term1, T, H * 128, cb, hb, W)
    assert ms > 0
    codes = cm.numpy().astype(np.float64).reshape(T, H, 128)
    want1 = np.einsum("ht,thd->hd", w_prime.cpu().double().numpy(), codes)
    assert np.abs(term1.cpu().double().numpy() - want1).max() <= 1e-5 * np.abs(want1).max()
    term1_t = term1.to(dtype)
    our_wv = torch.empty_like(term1_t)
    ms2 = packkv_cuda.fused_wv(our_wv, w.to(cuda), zero.to(cuda), scale.to(cuda), term1_t)
    assert ms2 > 0
    c_m = (w.double() * zero.double()[None] * scale.double()[None]).sum(1, keepdim=True)
    want = c_m + term1_t.cpu().double()
    tol = 2 ** -9 if dtype == torch.float16 else 2 ** -6
    assert np.abs(our_wv.cpu().double().numpy() - want.numpy()).max() <= tol * max(want.abs().max().item(), 1.0)


def test_unsupported_case_returns_zero(cuda, capsys):
    comp = torch.zeros(64 * 128, dtype=torch.uint8, device=cuda)
    info = torch.zeros(1, 2, dtype=torch.uint32, device=cuda)
    q = torch.zeros(1, 128, dtype=torch.float16, device=cuda)
    t = torch.zeros(1, 64, dtype=torch.float16, device=cuda)
    assert packkv_cuda.kq_mat_vec_mul(comp, info, q, t, 64, 128, 64, 128, 7) == 0.0
    assert "no such case" in capsys.readouterr().out
    assert packkv_cuda.kq_mat_vec_mul(comp, info, q.float(), t, 64, 128, 64, 128, 4) == 0.0
    assert "Unsupported data type" in capsys.readouterr().out
    with pytest.raises(RuntimeError, match="2D"):
        packkv_cuda.fused_kq(t, q[0], t[0], t[0], t)


def test_fused_fixups_take_strided_tensors(cuda):
    """fused_kq / fused_wv on transposed and sliced views (every operand non-contiguous at once): the contiguous
    copies the binding makes must all be alive during the call, so the results equal those of contiguous inputs."""
    g = torch.Generator().manual_seed(77)
    M, N = 8, 1024
    q = torch.randn(128, M, generator=g).to(torch.float16).to(cuda).t()                 # [M, 128] view of [128, M]
    t = torch.randn(N, M, generator=g).to(torch.float16).to(cuda).t()                   # [M, N] view
    zero = torch.randn(2 * N, generator=g).round().to(torch.float16).to(cuda)[::2]      # stride 2
    scale = (torch.rand(2 * N, generator=g) + 0.5).to(torch.float16).to(cuda)[::2]
    assert not (q.is_contiguous() or t.is_contiguous() or zero.is_contiguous() or scale.is_contiguous())
    got, want = torch.empty(M, N, dtype=torch.float16, device=cuda), torch.empty(M, N, dtype=torch.float16, device=cuda)
    packkv_cuda.fused_kq(got, q, zero, scale, t)
    packkv_cuda.fused_kq(want, q.contiguous(), zero.contiguous(), scale.contiguous(), t.contiguous())
    assert torch.equal(got, want)
    w = torch.rand(N, M, generator=g).to(torch.float16).to(cuda).t()
    term1 = torch.randn(128, M, generator=g).to(torch.float16).to(cuda).t()
    got, want = torch.empty(M, 128, dtype=torch.float16, device=cuda), torch.empty(M, 128, dtype=torch.float16, device=cuda)
    packkv_cuda.fused_wv(got, w, zero, scale, term1)
    packkv_cuda.fused_wv(want, w.contiguous(), zero.contiguous(), scale.contiguous(), term1.contiguous())
    assert torch.equal(got, want)


def test_damaged_block_info_is_survived(cuda):
    """Entries of block_info that point outside the compressed buffer give arbitrary products for their blocks;
    nothing outside the buffer is read and the other blocks' results stand."""
    H, T = 8, 512
    cm, zero, scale, comp, info, W, cb, hb = _setup(cuda, H, T, 0.1, True, torch.float16, 43)
    torch.manual_seed(1)
    q = torch.randn(H, 128).to(torch.float16).to(cuda)
    good = torch.zeros(H, T, dtype=torch.float16, device=cuda)
    ops.kq_mat_vec_mul(comp, info, q, good, T, H * 128, cb, hb, W, q_interleaved=False)
    bad_info = info.cpu().numpy().astype(np.int64)
    bad_info[3] = (comp.numel() + 999, 3000)
    bad_info[9] = (0xFFFFFFF0, 0xFFFFFFFF)
    t = torch.zeros(H, T, dtype=torch.float16, device=cuda)
    ops.kq_mat_vec_mul(comp, torch.from_numpy(bad_info.astype(np.uint32)).to(cuda), q, t, T, H * 128, cb, hb, W,
                       q_interleaved=False)
    torch.cuda.synchronize()
    keep = torch.ones(H, T, dtype=torch.bool)
    for b in (3, 9):                                      # block b = (context block b // H, head b % H)
        keep[b % H, (b // H) * cb:(b // H + 1) * cb] = False
    assert torch.equal(t.cpu()[keep], good.cpu()[keep])
    cm, zero, scale, comp, info, W, cb, hb = _setup(cuda, H, T, 0.1, False, torch.float16, 44)
    w = torch.rand(H, T).to(torch.float16).to(cuda)
    bad_info = info.cpu().numpy().astype(np.int64)
    bad_info[0] = (comp.numel(), 1 << 20)
    bad_info[7] = (comp.numel() - 1, 77)
    out = torch.zeros(H, 128, dtype=torch.float32, device=cuda)
    ops.wv_mat_vec_mul(comp, torch.from_numpy(bad_info.astype(np.uint32)).to(cuda), w, out, T, H * 128, cb, hb, W)
    torch.cuda.synchronize()
    assert out.shape == (H, 128)


# Blocks of other lengths and widths, odd round counts, blocks and context blocks that do not fill the last workgroup.
KQ_SHAPES = [(1, 16, 16, 2), (3, 48, 48, 3), (8, 768, 48, 4), (2, 1024, 256, 4), (5, 192, 64, 2), (1, 64, 64, 4)]
WV_SHAPES = [(1, 128, 32, 2), (3, 384, 64, 3), (2, 640, 128, 4), (5, 1152, 64, 2), (1, 512, 128, 3)]


def _block_codec(cuda, is_k, H, T, cb, hb, bits, seed):
    g = torch.Generator().manual_seed(seed)
    codes = torch.randint(0, 1 << bits, (T, H * 128), generator=g, dtype=torch.uint8)
    codes[:, ::5] = codes[0, ::5]                                   # packs of width 0 among them
    codes = codes.to(cuda)
    n = (T // cb) * (H * 128 // hb)
    stream = torch.zeros(n * ops.block_bound(is_k, cb, hb, bits) + 16, dtype=torch.uint8, device=cuda)
    info = torch.zeros(n, 2, dtype=torch.uint32, device=cuda)
    (ops.k_encode if is_k else ops.v_encode)(codes, stream, info, cb, hb, bits)
    return codes.cpu().double().view(T, H, 128), stream, info


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("H,T,cb,bits", KQ_SHAPES)
def test_kq_block_shapes(cuda, H, T, cb, bits, dtype):
    codes, stream, info = _block_codec(cuda, True, H, T, cb, 128, bits, 5)
    q = torch.randn(H, 128, generator=torch.Generator().manual_seed(6)).to(dtype)
    t = torch.full((H, T), float("nan"), dtype=dtype, device=cuda)
    ops.kq_mat_vec_mul(stream, info, q.to(cuda), t, T, H * 128, cb, 128, bits, q_interleaved=False)
    want = torch.einsum("thd,hd->ht", codes, q.double())
    # fp32 sums of 128 exact products (at most 128 roundings of 2^-24 of the sum of magnitudes), one rounding to dtype
    mag = torch.einsum("thd,hd->ht", codes, q.double().abs())
    half_ulp = 2 ** -11 if dtype == torch.float16 else 2 ** -8
    assert bool(((t.cpu().double() - want).abs() <= half_ulp * want.abs() * 1.01 + 2 ** -17 * mag).all())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("H,T,hb,bits", WV_SHAPES)
def test_wv_block_shapes(cuda, H, T, hb, bits, dtype):
    codes, stream, info = _block_codec(cuda, False, H, T, 128, hb, bits, 7)
    w = torch.rand(H, T, generator=torch.Generator().manual_seed(8)).to(dtype)
    out = torch.ones(H, 128, dtype=torch.float32, device=cuda)      # the sums are added to what is there
    ops.wv_mat_vec_mul(stream, info, w.to(cuda), out, T, H * 128, 128, hb, bits)
    want = 1.0 + torch.einsum("ht,thd->hd", w.double(), codes)
    # every term is non-negative: at most T + 8 roundings of 2^-24 of the result
    assert bool(((out.cpu().double() - want).abs() <= (T + 8) * 2 ** -24 * want).all())


@pytest.mark.parametrize("N,off", [(1, 0), (1023, 0), (1024, 1), (1028, 0), (4100, 3), (2050, 0)])
def test_fused_fixups_any_length_and_alignment(cuda, N, off):
    """Rows that start off an 8-byte boundary or are no multiple of four long are read one value at a time."""
    g = torch.Generator().manual_seed(N)
    M, K, D = 3, 128, 100

    def rows(shape, fn):
        n = int(np.prod(shape))
        return fn(n + off).to(torch.float16).to(cuda)[off:].view(shape)
    q, t = rows((M, K), lambda n: torch.randn(n, generator=g)), rows((M, N), lambda n: torch.randn(n, generator=g))
    zero, scale = rows((N,), lambda n: torch.randn(n, generator=g).round()), rows((N,), lambda n: torch.rand(n, generator=g) + 0.5)
    w, term1 = rows((M, N), lambda n: torch.rand(n, generator=g)), rows((M, D), lambda n: torch.randn(n, generator=g))
    guard = torch.full((M * N + off + 8,), 7.0, dtype=torch.float16, device=cuda)
    kq = guard[off:off + M * N].view(M, N)
    packkv_cuda.fused_kq(kq, q, zero, scale, t)
    want = (q.double().sum(1, keepdim=True) * zero.double() + t.double()) * scale.double()
    mag = (q.double().abs().sum(1, keepdim=True) * zero.double().abs() + t.double().abs()) * scale.double()
    assert bool(((kq.double() - want).abs() <= 2 ** -11 * want.abs() * 1.01 + 2 ** -17 * mag + 2 ** -24).all())
    assert bool((guard[:off] == 7.0).all()) and bool((guard[off + M * N:] == 7.0).all())
    wv = torch.empty(M, D, dtype=torch.float16, device=cuda)
    packkv_cuda.fused_wv(wv, w, zero, scale, term1)
    c = w.double() * zero.double() * scale.double()
    want = c.sum(1, keepdim=True) + term1.double()
    mag = c.abs().sum(1, keepdim=True) + term1.double().abs()
    assert bool(((wv.double() - want).abs() <= 2 ** -11 * want.abs() * 1.01 + 2 ** -14 * mag + 2 ** -24).all())


@pytest.mark.parametrize("bits", [2, 3, 4])
@pytest.mark.parametrize("low,high", [(-126, -116), (-126, 110), (100, 115)])
def test_bf16_factors_of_any_size(cuda, low, high, bits):
    """bf16 q and weights near the ends of the exponent range, and both ends in one row (the large ones over channels and
    tokens whose codes are zero, so that the small ones make the result)."""
    H, T = 3, 256
    g = torch.Generator().manual_seed(bits)
    codes = torch.randint(1, 1 << bits, (T, H * 128), generator=g, dtype=torch.uint8)
    mixed = high - low > 100
    if mixed:
        codes[:, ::8], codes[::8] = 0, 0

    def factors(n, zero):
        e = torch.randint(low, low + 10, (H, n), generator=g).double()
        f = (1 + torch.rand(H, n, generator=g).double()) * 2 ** e
        if mixed:
            f[:, zero] = 2.0 ** high
        return f.to(torch.bfloat16)
    q, w = factors(128, slice(0, None, 8)), factors(T, slice(0, None, 8))
    c = codes.double().view(T, H, 128)
    for is_k, cb, hb in ((True, 64, 128), (False, 128, 64)):
        n = codes.numel() // (cb * hb)
        stream = torch.zeros(n * ops.block_bound(is_k, cb, hb, bits) + 16, dtype=torch.uint8, device=cuda)
        info = torch.zeros(n, 2, dtype=torch.uint32, device=cuda)
        (ops.k_encode if is_k else ops.v_encode)(codes.to(cuda), stream, info, cb, hb, bits)
        # all terms are non-negative: the fp32 sums of exact products are off by at most a rounding of 2^-24 a term; bf16 rounds
            # to 8 bits
        if is_k:
            got = torch.empty(H, T, dtype=torch.bfloat16, device=cuda)
            ops.kq_mat_vec_mul(stream, info, q.to(cuda), got, T, H * 128, cb, hb, bits, q_interleaved=False)
            want = torch.einsum("thd,hd->ht", c, q.double())
            bound = (2 ** -8 + 136 * 2 ** -24) * 1.01
        else:
            got = torch.zeros(H, 128, dtype=torch.float32, device=cuda)
            ops.wv_mat_vec_mul(stream, info, w.to(cuda), got, T, H * 128, cb, hb, bits)
            want = torch.einsum("ht,thd->hd", w.double(), c)
            bound = (T + 8) * 2 ** -24
        assert bool(((got.cpu().double() - want).abs() <= bound * want).all()), is_k


def test_times_and_results_of_ops_on_several_streams_at_once(cuda):
    """Each op waits for its own kernel and returns its own time, whoever else is waiting; while a stream is capturing there is
    no time to wait for, and the op is refused before it records anything."""
    import threading
    H, T = 8, 4096
    g = torch.Generator(device=cuda)
    g.manual_seed(3)
    z, sc = (torch.randn(T, generator=g, device=cuda).half() for _ in range(2))
    jobs = [(torch.randn(H, 128, generator=g, device=cuda).half(), torch.randn(H, T, generator=g, device=cuda).half()) for _ in range(4)]
    want = [torch.empty(H, T, dtype=torch.float16, device=cuda) for _ in jobs]
    for (q, t), out in zip(jobs, want):
        assert ops.fused_kq(out, q, z, sc, t) > 0
    torch.cuda.synchronize()
    bad = []

    def work(i):
        st, (q, t) = torch.cuda.Stream(), jobs[i]
        with torch.cuda.stream(st):
            for _ in range(50):
                out = torch.zeros_like(want[i])
                ms = ops.fused_kq(out, q, z, sc, t)
                if not (0 < ms < 20 and torch.equal(out, want[i])):
                    bad.append((i, ms))
    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not bad
    st, graph, out = torch.cuda.Stream(), torch.cuda.CUDAGraph(), torch.empty_like(want[0])
    with torch.cuda.stream(st):
        graph.capture_begin()
        try:
            with pytest.raises(ops.PackKVError, match="capturing"):
                ops.fused_kq(out, jobs[0][0], z, sc, jobs[0][1])
            out.zero_()
        finally:
            graph.capture_end()
    graph.replay()
    torch.cuda.synchronize()
    assert not out.any()
    assert ops.fused_kq(out, jobs[0][0], z, sc, jobs[0][1]) > 0 and torch.equal(out, want[0])
