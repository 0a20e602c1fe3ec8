"""Kernels chosen by a size rule, at the sizes where the rule changes: edges of
tiles and teams, remainders, unaligned rows, the smallest and largest of each
range.  References are the oracle, or torch on the CPU in float64."""

import types

import numpy as np
import pytest
import torch

from oracle import bf16, ops

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K(cuda):
    from mi355x_pjrt import kernels

    kernels.lib()
    return kernels


def shifted(t, off):
    """t on the GPU, off elements past a 16-byte boundary."""
    buf = torch.empty(t.numel() + off, dtype=t.dtype, device="cuda")
    view = buf[off:].view(t.shape)
    view.copy_(t)
    return view


# rows x columns around a wave's, a 4-wave and a 16-wave team's shares (64, 512, 2048 and 8192
# vectors), tails of every kind, and past the registers (65536 bf16, 32768 fp32)
ROW_SHAPES = [(1, 1, 0), (4, 7, 1), (2050, 511, 1), (700, 4097, 0), (511, 4105, 3), (2, 16384, 1), (33, 16391, 0),
              (5, 50257, 0), (4, 65529, 1), (2, 65551, 0), (2, 140003, 1)]
# one wave with 3 - 4 and 5 - 8 vectors per lane, four waves with 5 - 8 (softmax, LayerNorm), of either type
ROW_SHAPES += [(2049, 601, 1), (2051, 1100, 0), (2051, 2043, 1), (2049, 4091, 1), (600, 6001, 1), (600, 12301, 0)]


@pytest.mark.parametrize("rows,cols,off", ROW_SHAPES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_row_kernels_any_width(K, rows, cols, off, dtype):
    """Sum, max, argmax, softmax and LayerNorm of odd rows: argmax exact, the
    rest within fp32 summation error (2^-24 sqrt(cols) of the magnitudes, with
    a factor of 16) and one rounding to the stored type."""
    print(f"case: rows [{rows},{cols}] off={off} {dtype}", flush=True)
    g = torch.Generator().manual_seed(rows * 7 + cols)
    x = torch.randn(rows, cols, generator=g).to(dtype)
    x[0, cols // 2] = x[0].max() + 1 if cols > 1 else 1.0
    x[0, cols - 1] = x[0, cols // 2]  # a tie: the lower index wins
    if rows > 2:
        x[1, cols // 3] = float("nan")
        x[2] = -float("inf")
    xd, xf = shifted(x, off), x.double().numpy()
    index, value = K.row_argmax(xd)
    want, _ = ops.argmax_rows(x.float().numpy())
    np.testing.assert_array_equal(index.cpu().numpy(), want)
    bits = torch.int16 if dtype == torch.bfloat16 else torch.int32
    picked = x[torch.arange(rows), torch.from_numpy(want.astype(np.int64))]
    assert torch.equal(value.cpu().view(bits), picked.view(bits))
    low, _ = K.row_argmax(xd, is_min=True, index_dtype=torch.int64)
    np.testing.assert_array_equal(low.cpu().numpy(), ops.argmax_rows(x.float().numpy(), True)[0])
    np.testing.assert_array_equal(K.row_reduce(xd, "max").cpu().numpy().astype(np.float64), xf.max(-1))

    ok = slice(3, None) if rows > 2 else slice(None)  # the finite rows
    assert x[ok].numel() > 0
    xs, xf = shifted(x[ok], off), xf[ok]
    # unit roundoff of the stored type: bf16 has 8 significant bits, so half an ulp is up to 2^-8 of the value
    eps, out = 16 * 2.0 ** -24 * np.sqrt(cols), 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -24
    got = K.row_reduce(xs, "sum").cpu().double().numpy()
    assert np.all(np.abs(got - xf.sum(-1)) <= eps * np.abs(xf).sum(-1) / np.sqrt(cols))
    want = ops.softmax_rows(xf)
    got = K.softmax_rows(xs).cpu().double().numpy()
    # __expf: 2 ulp plus the rounding of its argument, |x - max| * 2^-24
    assert np.all(np.abs(got - want) <= (out + eps + 32 * 2.0 ** -24) * want + 1e-38)
    gamma, beta = (1 + 0.1 * torch.randn(cols, generator=g)).to(dtype), torch.randn(cols, generator=g).to(dtype)
    want = ops.layernorm(xf, gamma.double().numpy(), beta.double().numpy())
    got = K.layernorm(xs, shifted(gamma, off), shifted(beta, 0)).cpu().double().numpy()
    scale = np.abs(gamma.double().numpy()) * 8 + np.abs(beta.double().numpy())
    assert np.all(np.abs(got - want) <= out * np.abs(want) + 1e-5 * scale)


# short rows, read by element (up to 64, or 128 that are no whole vectors), and the row counts from
# which rows take fewer waves
@pytest.mark.parametrize("rows,cols,off", [(9, 1, 0), (4097, 63, 1), (70, 64, 0), (70, 64, 1), (4100, 65, 0), (9, 127, 1),
                                           (9, 128, 0), (4096, 4100, 0), (4095, 4100, 1)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_row_kernels_short_and_many(K, rows, cols, off, dtype):
    test_row_kernels_any_width(K, rows, cols, off, dtype)
    x = torch.randn(rows, cols, generator=torch.Generator().manual_seed(cols)).to(torch.float16)
    xd = shifted(x, off)
    np.testing.assert_array_equal(K.row_reduce(xd, "max").cpu().numpy(), x.float().numpy().max(-1))
    np.testing.assert_array_equal(K.row_argmax(xd)[0].cpu().numpy(), ops.argmax_rows(x.float().numpy())[0])


@pytest.mark.parametrize("rows,cols", [(5, 2052), (3, 4099), (2, 33000)])
def test_add_layernorm_f32_wide(K, rows, cols):
    """The fp32 residual add inside the LayerNorm of rows the one-wave kernel
    does not hold: the stored sum is the one fp32 add, bit for bit."""
    g = torch.Generator().manual_seed(cols)
    a, b = torch.randn(rows, cols, generator=g), torch.randn(rows, cols, generator=g)
    gamma, beta = torch.randn(cols, generator=g), torch.randn(cols, generator=g)
    s, y = K.add_layernorm(a.cuda(), b.cuda(), None, gamma.cuda(), beta.cuda())
    assert torch.equal(s.cpu(), a + b)
    want = ops.layernorm((a + b).double().numpy(), gamma.double().numpy(), beta.double().numpy())
    scale = gamma.abs().double().numpy() * 8 + beta.abs().double().numpy()
    assert np.all(np.abs(y.cpu().double().numpy() - want) <= 1e-5 * scale)
    _, y16 = K.add_layernorm(a.cuda(), b.cuda(), None, gamma.cuda(), beta.cuda(), out_dtype=torch.bfloat16)
    assert torch.equal(y16.cpu(), y.cpu().bfloat16())


# few-row products: rows around the 16-row blocks, columns around the 16/32/64-column tiles, k
# around the 32-deep steps and the waves' shares, both orientations of B, rows off alignment
SKINNY = [(1, 16, 1), (1, 17, 31), (5, 63, 33), (16, 100, 96), (17, 64, 1000), (33, 129, 515), (64, 4096, 256),
          (64, 33, 40), (3, 12352, 130), (49, 12301, 64)]


@pytest.mark.parametrize("M,N,K_", SKINNY)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("b_kc", [False, True])
def test_gemm_few_rows(K, M, N, K_, dtype, b_kc):
    """C = relu(A B + bias) with NaN past every row end in memory: fp32 sums
    within 2^-23 sqrt(K) of the magnitudes (factor 8), one rounding to C."""
    print(f"case: gemm {M}x{N}x{K_} {dtype} b_kc={b_kc}", flush=True)
    g = torch.Generator().manual_seed(M * 1000 + N + K_)
    a, b, bias = torch.randn(M, K_, generator=g), torch.randn(K_, N, generator=g), torch.randn(N, generator=g)
    a, b, bias = a.to(dtype), b.to(dtype), bias.to(dtype)
    nan = float("nan")
    ad = torch.full((M, K_ + 3), nan, dtype=dtype, device="cuda")[:, 1:K_ + 1]
    ad.copy_(a)
    rows, cols = (N, K_) if b_kc else (K_, N)
    bd = torch.full((rows, cols + 5), nan, dtype=dtype, device="cuda")[:, 2:cols + 2]
    bd.copy_(b.t() if b_kc else b)
    out = torch.full((M + 1, N + 1), 7.0, dtype=dtype, device="cuda")
    K.gemm(ad, bd.t() if b_kc else bd, bias=bias.cuda(), relu=True, out=out[:M, :N])
    ad_, bd_ = a.double(), b.double()
    want = torch.relu(ad_ @ bd_ + bias.double())
    mag = ad_.abs() @ bd_.abs() + bias.double().abs()
    bound = 8 * 2.0 ** -23 * mag + (2.0 ** -8 if dtype == torch.bfloat16 else 0) * want.abs()
    assert bool(((out[:M, :N].cpu().double() - want).abs() <= bound).all())
    assert bool((out[M] == 7).all()) and bool((out[:, N] == 7).all())


# deep products of few rows: k cut over workgroups (the workspace function says so) and, where C's
# rows are off the grid, in one launch whose waves run their pipelined loop; k's remainder owned by
# the first and by later slices (281 steps of 32 in 16 slices of 8 or 16 waves: slice 1 or 3)
@pytest.mark.parametrize("M,N,K_", [(1, 256, 4300), (16, 768, 9003), (17, 64, 4127), (33, 500, 6200), (64, 132, 12301),
                                    (5, 2048, 16411)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("b_kc", [False, True])
@pytest.mark.parametrize("sliced", [True, False])
def test_gemm_few_rows_deep(K, M, N, K_, dtype, b_kc, sliced):
    """relu(A B + bias) through gemm, and A B through gemm_splitk, against
    float64, with NaN past every row end: fp32 sums within 8 * 2^-23 of the
    magnitudes (at most 0.01 here; a lost element of k is worth 0.6 on
    average) and one rounding to C."""
    print(f"case: gemm {M}x{N}x{K_} {dtype} b_kc={b_kc} sliced={sliced}", flush=True)
    g = torch.Generator().manual_seed(M + N + K_)
    a, b = torch.randn(M, K_, generator=g).to(dtype), torch.randn(K_, N, generator=g).to(dtype)
    bias = torch.randn(N, generator=g).to(dtype)
    ad = torch.full((M, K_ + 3), float("nan"), dtype=dtype, device="cuda")[:, 1:K_ + 1]
    ad.copy_(a)
    rows, cols = (N, K_) if b_kc else (K_, N)
    bd = torch.full((rows, cols + 5), float("nan"), dtype=dtype, device="cuda")[:, 2:cols + 2]
    bd.copy_(b.t() if b_kc else b)
    bd = bd.t() if b_kc else bd
    need = K.lib().mk_gemm_few_rows_workspace_bytes(K.mk_dtype(dtype), M, N, K_, 1, *bd.stride())
    assert need >= 2 * M * N * 4
    want, mag = a.double() @ b.double(), a.double().abs() @ b.double().abs()
    for out_dtype in (torch.float32, dtype):
        u = 2.0 ** -8 if out_dtype == torch.bfloat16 else 2.0 ** -24
        out = torch.full((M + 1, N + (4 if sliced else 1)), 7.0, dtype=out_dtype, device="cuda")
        K.gemm(ad, bd, out_dtype=out_dtype, bias=bias.cuda().to(out_dtype), relu=True, out=out[:M, :N])
        top = torch.relu(want + bias.double())
        bound = 8 * 2.0 ** -23 * (mag + bias.double().abs()) + u * top
        assert bool(((out[:M, :N].cpu().double() - top).abs() <= bound).all())
        assert bool((out[M] == 7).all()) and bool((out[:, N:] == 7).all())
        if sliced:
            for splits in (3, 16):
                got = K.gemm_splitk(ad, bd, splits, out_dtype=out_dtype)
                assert bool(((got.cpu().double() - want).abs() <= 8 * 2.0 ** -23 * mag + u * want.abs()).all())
                assert torch.equal(got, K.gemm_splitk(ad, bd, splits, out_dtype=out_dtype))


@pytest.mark.parametrize("dtype,depth", [(torch.bfloat16, 4096), (torch.float32, 2048)])
def test_gemm_few_rows_cut_from_its_depth_on(K, dtype, depth, monkeypatch):
    """A product too shallow to pay for a workspace and a second kernel takes
    neither; from 4096 bf16 (2048 fp32) deep on it is cut."""
    taken, scratch = [], K._scratch
    monkeypatch.setattr(K, "_scratch", lambda n, *rest: (taken.append(n), scratch(n, *rest))[1])
    for k in (depth - 8, depth):
        x, w = torch.ones(4, k, dtype=dtype, device="cuda"), torch.ones(k, 768, dtype=dtype, device="cuda")
        assert bool((K.gemm(x, w, out_dtype=torch.float32) == k).all())
        assert len(taken) == (k >= depth), k


def test_gemm_few_rows_batched_and_split(K):
    """Batches with a broadcast B, and the split-K entry at few rows (too
    shallow a k to be cut)."""
    g = torch.Generator().manual_seed(3)
    a, b = torch.randn(5, 7, 100, generator=g), torch.randn(100, 48, generator=g)
    got = K.gemm(a.cuda(), b.cuda())
    want = a.double() @ b.double()
    assert bool(((got.cpu().double() - want).abs() <= 8 * 2.0 ** -23 * (a.double().abs() @ b.double().abs())).all())
    x, w = torch.randn(9, 1024, generator=g).bfloat16(), torch.randn(1024, 64, generator=g).bfloat16()
    got = K.gemm_splitk(x.cuda(), w.cuda(), 4)
    want = x.double() @ w.double()
    assert bool(((got.cpu().double() - want).abs() <= 8 * 2.0 ** -23 * (x.double().abs() @ w.double().abs())).all())


# few queries: key counts around the 32-key steps, the 4 waves' shares and the 256-key slices
@pytest.mark.parametrize("B,H,Sq,Sk,D", [(1, 1, 1, 1, 128), (2, 3, 1, 31, 64), (1, 2, 7, 33, 128), (1, 2, 16, 129, 64),
                                         (2, 2, 1, 511, 128), (1, 2, 2, 513, 128), (1, 3, 16, 2049, 128),
                                         (3, 5, 4, 1000, 64), (1, 1, 1, 16391, 128), (32, 16, 1, 300, 64),
                                         (3, 5, 4, 1025, 64), (1, 2, 2, 769, 128), (8, 16, 1, 2048, 128),
                                         (1, 2, 10, 64, 128), (2, 3, 11, 33, 128), (1, 2, 16, 64, 128),
                                         (1, 2, 16, 65, 128), (32, 16, 16, 64, 128), (16, 16, 12, 1, 128)])
@pytest.mark.parametrize("slices", [True, False])
def test_sdpa_few_queries(K, B, H, Sq, Sk, D, slices):
    """O and lse against float64 softmax; the cache holds NaN past its keys.
    Each probability is rounded to bf16 (2^-8) in numerator and sum, O once."""
    print(f"case: sdpa {B}x{H} Sq={Sq} Sk={Sk} D={D} slices={slices}", flush=True)
    g = torch.Generator().manual_seed(Sk * 31 + Sq)
    q = torch.randn(B, Sq, H, D, generator=g).bfloat16().transpose(1, 2)
    k, v = (torch.randn(B, H, Sk, D, generator=g).bfloat16() for _ in range(2))
    q[:, :, 0] *= 6  # a peaked row beside flat ones
    room = torch.full((2, B, H, Sk + 40, D), float("nan"), dtype=torch.bfloat16, device="cuda")
    kd, vd = room[0, :, :, :Sk], room[1, :, :, :Sk]
    kd.copy_(k)
    vd.copy_(v)
    out = torch.full((B, H, Sq, D), float("nan"), dtype=torch.bfloat16, device="cuda")
    lse = torch.full((B, H, Sq), float("nan"), device="cuda")
    if slices:
        K.sdpa_fwd(q.cuda(), kd, vd, D ** -0.5, causal=False, out=out, lse=lse)
    else:  # the entry without a workspace: one workgroup per head
        qd = q.cuda()
        strides = [[t.data_ptr(), *t.stride()[:3]] for t in (qd, kd, vd, out)]
        assert K.lib().mk_sdpa_fwd(K._stream(), B, H, Sq, Sk, D, *sum(strides, []), D ** -0.5, 0, lse.data_ptr()) == 0
    s = (q.double() @ k.double().transpose(-1, -2)) * D ** -0.5
    p = torch.softmax(s, -1)
    want, u = p @ v.double(), 2.0 ** -8
    bound = 2 * u * (p @ v.double().abs()) + u * want.abs() + 1e-6
    assert bool(((out.cpu().double() - want).abs() <= bound).all())
    assert bool(((lse.cpu().double() - torch.logsumexp(s, -1)).abs() <= u + 1e-5).all())


def test_few_rows_and_queries_on_an_explicit_stream(K):
    """The cuts along the contraction and the keys don't depend on how the
    stream is named or on a batch dimension of one: the same bits.  The
    workspace is the stream's own memory."""
    g = torch.Generator().manual_seed(8)
    x, w = torch.randn(16, 8192, generator=g).bfloat16().cuda(), torch.randn(8192, 512, generator=g).bfloat16().cuda()
    assert K.lib().mk_gemm_few_rows_workspace_bytes(K.mk_dtype(x.dtype), 16, 512, 8192, 1, 512, 1) > 0
    q, k, v = (torch.randn(1, 4, s, 128, generator=g).bfloat16().cuda() for s in (2, 8192, 8192))
    assert K.lib().mk_sdpa_fwd_workspace_bytes(1, 4, 2, 8192, 128, 0) > 0
    y, o = K.gemm(x, w), K.sdpa_fwd(q, k, v, 0.1, causal=False)
    torch.cuda.synchronize()
    s = torch.cuda.Stream()
    for stream in (torch.cuda.current_stream(), s):
        ys = K.gemm(x, w, stream=stream)
        os = K.sdpa_fwd(q, k, v, 0.1, causal=False, stream=stream)
        stream.synchronize()
        assert torch.equal(ys, y) and torch.equal(os, o)
    assert torch.equal(K.gemm(x[None], w), y[None]) and torch.equal(K.gemm(x[None], w[None]), y[None])
    held = K._scratch(1 << 22, x.device, s).data_ptr()  # freed at once: the current stream must not get it
    blocks = [torch.empty(1 << 22, dtype=torch.uint8, device="cuda") for _ in range(4)]
    assert all(b.data_ptr() != held for b in blocks)
    assert K._scratch(1 << 22, x.device, s).data_ptr() == held
    bare = types.SimpleNamespace(cuda_stream=s.cuda_stream)  # any object with a stream's handle
    for ys, want in ((K.gemm(x, w, stream=bare), y), (K.gemm_splitk(x, w, 16, stream=bare, out_dtype=x.dtype), y),
                     (K.sdpa_fwd(q, k, v, 0.1, causal=False, stream=bare), o)):
        s.synchronize()
        assert torch.equal(ys, want)


def test_sdpa_few_queries_infinities(K):
    """Scores of -inf at the first keys do not poison later ones, and a NaN
    key makes exactly its head NaN."""
    q = torch.ones(1, 3, 2, 64, dtype=torch.bfloat16, device="cuda")
    k = torch.ones(1, 3, 700, 64, dtype=torch.bfloat16, device="cuda")
    v = torch.ones(1, 3, 700, 64, dtype=torch.bfloat16, device="cuda") * 2
    k[0, 0, :650] = -float("inf")
    k[0, 1, 699, 3] = float("nan")
    o = K.sdpa_fwd(q, k, v, 0.125, causal=False)
    assert bool((o[0, 0] == 2).all()) and bool(o[0, 1].isnan().all()) and bool((o[0, 2] == 2).all())
    # a head without a score above -inf has no weights, a query of scores at the type's lowest value has
    k[0, 0] = -float("inf")
    k[0, 1] = 0
    k[0, 1, :, 0] = torch.finfo(torch.bfloat16).min
    q[0, 1] = 0
    q[0, 1, 0, 0] = 1
    lse = torch.empty(1, 3, 2, device="cuda")
    for scale in (0.69, 0.125):  # 0.69 log2(e) leaves the scores finite
        for n in (700, 40):
            o = K.sdpa_fwd(q, k[:, :, :n], v[:, :, :n], scale, causal=False, lse=lse)
            assert bool(o[0, 0].isnan().all()) and bool((lse[0, 0] == -float("inf")).all())
            assert bool((o[0, 1] == 2).all()) and bool(lse[0, 1].isfinite().all()) and bool((o[0, 2] == 2).all())


def test_gpt2_steps_on_several_streams(cuda):
    """Captured steps replayed at once on streams of their own give the bits
    each gives alone, and none of their calls shares a library workspace."""
    from mi355x_pjrt import gpt2

    cfg = gpt2.GPT2Config(n_layer=1, d_model=256, n_head=4, seq=256, batch=4, vocab=5003)
    steps, alone = [], []
    for i in range(3):
        step = gpt2.GPT2TrainStep(cfg, seed=i, stream=torch.cuda.Stream())
        assert not any("blas" in c.name for c in step.calls)
        g = torch.Generator().manual_seed(i)
        step.set_batch(torch.randint(cfg.vocab, (cfg.tokens,), generator=g),
                       torch.randint(cfg.vocab, (cfg.tokens,), generator=g))
        torch.cuda.synchronize()
        step.step()
        step.stream.synchronize()
        step.capture()
        steps.append(step)
        start = [t.clone() for t in (step.master, step.param, step.m, step.v)]
        torch.cuda.synchronize()
        for _ in range(3):
            step.replay()
        torch.cuda.synchronize()
        alone.append(step.master.clone())
        for t, s0 in zip((step.master, step.param, step.m, step.v), start):
            t.copy_(s0)
        step.t = 1
    torch.cuda.synchronize()
    for _ in range(3):
        for step in steps:
            step.replay()
    torch.cuda.synchronize()
    for step, want in zip(steps, alone):
        assert torch.equal(step.master, want)


@pytest.mark.parametrize("M,N,Kd,splits", [(200, 136, 1000, 8), (128, 256, 4120, 8), (130, 132, 520, 4), (256, 768, 50256, 8),
                                           (128, 128, 400, 8), (129, 128, 36, 4), (300, 256, 1004, 4)])
def test_gemm_splitk_slices_off_the_16_byte_grid(K, M, N, Kd, splits):
    """Slice counts that divide K into slices that are no multiple of 8, on
    the uneven slices (400 in 8: slices of 56 are too short for the tiled
    kernel; 36 and 1004: rows off the grid, the even form), each operand
    k-contiguous in turn with NaN past K.  fp32 sums within 8 * 2^-23 of the
    magnitudes, bit for bit the slices' own products added in order."""
    assert Kd % splits == 0 and Kd // splits % 8 != 0
    g = torch.Generator().manual_seed(Kd)
    a, b = torch.randn(M, Kd, generator=g).bfloat16(), torch.randn(Kd, N, generator=g).bfloat16()
    want, norm = a.double() @ b.double(), a.double().abs() @ b.double().abs()

    def k_rows(t):  # t's rows of K on the GPU, 8 NaN behind each
        rows = torch.full((t.shape[0], Kd + 8), float("nan"), dtype=torch.bfloat16, device="cuda")[:, :Kd]
        rows.copy_(t)
        return rows

    for ad, bd in ((k_rows(a), b.cuda()), (k_rows(a), k_rows(b.t()).t()), (a.t().contiguous().cuda().t(), k_rows(b.t()).t())):
        got = K.gemm_splitk(ad, bd, splits)
        assert bool(((got.cpu().double() - want).abs() <= 8 * 2.0 ** -23 * norm).all())
        ks = ((Kd + splits - 1) // splits + 7) // 8 * 8
        if ks < 64 or any(max(t.stride()) % 8 for t in (ad, bd)):
            ks = Kd // splits
        total = None
        for k0 in range(0, Kd, ks):
            part = K.gemm(ad[:, k0:k0 + ks], bd[k0:k0 + ks], out_dtype=torch.float32)
            total = part if total is None else total + part
        assert torch.equal(got, total)
        assert torch.equal(got, K.gemm_splitk(ad, bd, splits))
        low = K.gemm_splitk(ad, bd, splits, out_dtype=torch.bfloat16)
        assert torch.equal(low, got.bfloat16())
