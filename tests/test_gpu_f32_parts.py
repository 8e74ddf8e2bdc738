"""fp32 products from three bf16 parts (gemm, convolutions, attention) against float64: sizes at the
edges of the tiles, wide ranges down to fp32's smallest normal number, and operands that are infinite, NaN or
round to infinity in bf16.

Tolerance (2-norm of the error over the result's): the parts are exact and the products left out are
below 3 * 2^-26; what is left are the roundings of the sum, at most six for every 16 values of K, each
below 2^-24 of the sum and independent: 2^-24 sqrt(6 K / 16).
"""
import numpy as np
import pytest

from conftest import report

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import splathip


def _tol(K):
    return 2.0 ** -24 * (6 * max(K, 16) / 16) ** 0.5 + 3 * 2.0 ** -26


def _rand(g, *shape):
    return torch.randn(*shape, generator=g).cuda()


def _gemm(ctx, A, W, bias):
    M, K = A.shape
    N = W.shape[0]
    ldw = (K + 63) // 64 * 64
    Wp = torch.zeros(N, ldw, device="cuda")
    Wp[:, :K] = W
    out = torch.full((M, N), -7.0, device="cuda")
    torch.cuda.synchronize()
    ctx.kernel_gemm(splathip.F32, A.data_ptr(), M, K, Wp.data_ptr(), N, ldw, bias.data_ptr(), 0, out.data_ptr(), True)
    ctx.synchronize()
    return out


def f32_plan(M, N, K, conv=False, ln=False):
    """csrc/gemm.hip f32_plan for N > 32, 8-column runs and the row epilogues: (rows, columns of the tile, K slices)."""
    tiles = [(64, 64, 16, 2.9, 0.45, 0.49, 0.07, 0.47, 4.7, 0.61, 0.53),
             (128, 64, 1, 1.9, 1.9, 0.785, 0.20, 0.75, 5.6, 0.90, 0.83),
             (128, 128, 8, 1.4, 3.9, 0.985, 0.31, 1.05, 4.2, 1.17, 1.10)]
    nk, best, plan = -(-K // 32), 1e30, None
    for bm, bn, cap, start, tile, step, fill, steps, cstart, cstep, csteps in tiles:
        if N <= 64 and bn > 64:
            continue
        if conv:
            start, step, steps = cstart, cstep, csteps
        mn = -(-M // bm) * -(-N // bn)
        cap = 1 if ln else max(1, min(cap, nk // 2, 1024 // mn))
        for s in (1, 2, 3, 4, 6, 8, 12, 16):
            kper = -(-nk // s)
            if s > cap or -(-nk // kper) != s:
                continue
            n = -(-mn * s // 256)
            t = start + n * tile + kper * (step + fill * min(1.0, mn * s / 256) if n == 1 else n * steps)
            if s > 1:
                t = 1.02 * (t + 3.2 + 0.3 * s + 0.16e-6 * 4.0 * s * M * N)
            if t < best * 0.999:
                best, plan = t, (bm, bn, s)
    return plan


@pytest.mark.parametrize("M,N,K,tile", [
    (1, 8, 4, None), (31, 32, 32, None), (33, 24, 68, None),                   # 128x32, K tails
    (64, 64, 96, (64, 64, 1)), (65, 72, 36, (64, 64, 1)), (1297, 384, 384, (64, 64, 1)),
    (200, 64, 1536, (64, 64, 8)), (65, 64, 3456, (64, 64, 12)), (1297, 384, 1536, (64, 64, 4)),   # K split
    (1200, 1096, 384, (128, 64, 1)), (1150, 1152, 420, (128, 64, 1)), (3893, 384, 388, (128, 64, 1)),   # 128x64, ragged
    (2100, 1152, 68, (64, 64, 1)), (5188, 1152, 384, (128, 128, 1)), (4097, 1544, 132, (128, 128, 1)),
    (2000, 3072, 1024, (128, 128, 1)), (3893, 384, 1540, (128, 128, 2)), (1296, 256, 6912, (64, 64, 6)),
])
def test_gemm_matches_float64(ctx, M, N, K, tile):
    assert tile is None or f32_plan(M, N, K) == tile
    g = torch.Generator().manual_seed(M + 3 * N + 7 * K)
    A, W, b = _rand(g, M, K), _rand(g, N, K) * K ** -0.5, _rand(g, N)
    out = _gemm(ctx, A, W, b).double()
    ref = A.double() @ W.double().t() + b.double()
    err = float((out - ref).norm() / ref.norm())
    report("f32.gemm", M=M, N=N, K=K, err=f"{err:.2e}", tol=f"{_tol(K):.2e}")
    assert err <= _tol(K)


@pytest.mark.parametrize("M,N,act,tile", [(640, 384, 0, (64, 64, 1)), (1200, 1152, 0, (128, 64, 1)),
                                          (1000, 1536, 2, (128, 64, 1)), (3892, 1536, 2, (128, 128, 1))])
def test_folded_layer_norm_matches_float64(ctx, M, N, act, tile):
    """Statistics and the folded-LayerNorm GEMM on each tile. Beside the sum's roundings: the row's mean, variance
    and their use, the bias and the activation, within eight more of 2^-24."""
    K = 384
    assert f32_plan(M, N, K, ln=True) == tile
    g = torch.Generator().manual_seed(M)
    x, W, b = _rand(g, M, K) + 0.1, _rand(g, N, K) * K ** -0.5, _rand(g, N)
    gamma, beta = 1 + 0.1 * _rand(g, K), 0.1 * _rand(g, K)
    Wf = (W * gamma).contiguous()
    c1, bf = Wf.double().sum(1).float(), (b.double() + W.double() @ beta.double()).float()
    stats, out = torch.empty(M, K // 64, 2, device="cuda"), torch.empty(M, N, device="cuda")
    torch.cuda.synchronize()
    ctx.kernel_ln_stats(x.data_ptr(), M, K, 64, stats.data_ptr(), splathip.F32)
    ctx.kernel_gemm_ln(splathip.F32, x.data_ptr(), M, K, Wf.data_ptr(), N, K, bf.data_ptr(), act, out.data_ptr(), True,
                       ln_in=stats.data_ptr(), c1=c1.data_ptr(), eps=1e-6)
    ctx.synchronize()
    ref = torch.nn.functional.layer_norm(x.double(), (K,), None, None, 1e-6) @ Wf.double().t() + bf.double()
    if act == 2:
        ref = torch.nn.functional.gelu(ref)
    err = float((out.double() - ref).norm() / ref.norm())
    report("f32.gemm_ln", M=M, N=N, act=act, err=f"{err:.2e}")
    assert err <= 2.0 ** -24 * ((6 * K / 16) ** 0.5 + 8)


@pytest.mark.parametrize("M,K,tile", [(1297, 384, (64, 64, 1)), (3892, 384, (128, 64, 1)), (5838, 384, (128, 128, 1)),
                                      (1297, 1536, (64, 64, 4)), (3892, 1536, (128, 128, 2))])
def test_residual_statistics_match_float64(ctx, M, K, tile):
    """out = res + gamma (A W^T + b) and its row statistics on each tile, whole and split: the sum's roundings and
    three of the epilogue; a group's sums take 64 more."""
    N = 384
    assert f32_plan(M, N, K) == tile
    g = torch.Generator().manual_seed(M + K)
    A, W, b, gam, res = _rand(g, M, K), _rand(g, N, K) * K ** -0.5, _rand(g, N), _rand(g, N), _rand(g, M, N)
    out, stats = torch.empty(M, N, device="cuda"), torch.empty(M, N // 64, 2, device="cuda")
    torch.cuda.synchronize()
    ctx.kernel_gemm_ln(splathip.F32, A.data_ptr(), M, K, W.data_ptr(), N, K, b.data_ptr(), 0, out.data_ptr(), True,
                       gamma=gam.data_ptr(), res=res.data_ptr(), ln_out=stats.data_ptr(), group=64)
    ctx.synchronize()
    ref = res.double() + gam.double() * (A.double() @ W.double().t() + b.double())
    err = float((out.double() - ref).norm() / ref.norm())
    o = out.double().view(M, N // 64, 64)
    want = torch.stack([o.sum(-1), (o * o).sum(-1)], -1)
    serr = ((stats.double() - want).abs() / torch.stack([o.abs().sum(-1), (o * o).sum(-1)], -1)).max()
    report("f32.gemm_res", M=M, K=K, err=f"{err:.2e}", stats=f"{float(serr):.2e}")
    assert err <= 2.0 ** -24 * ((6 * K / 16) ** 0.5 + 3)
    assert float(serr) <= 64 * 2.0 ** -24


def test_qkv_epilogue_on_128x64_tiles(ctx, tmp_path):
    """DA3-Small on 2 views of 21x28 patches: the cross-view blocks' qkv (1178 rows) runs the folded LayerNorm
    with qk-norm and RoPE on 128x64 tiles. Against the CPU oracle, both in fp32."""
    from oracle import da3 as OD
    from splathip import specs, synth
    assert f32_plan(2 * (21 * 28 + 1), 1152, 384, ln=True) == (128, 64, 1)
    spec = specs.DA3_VARIANTS["small"]
    w = synth.generate(synth.da3_shapes(spec), seed=1, layer_scale=1.0)
    path = str(tmp_path / "da3.safetensors")
    synth.save(path, w)
    images = synth.procedural_images(2, 294, 392, seed=2)
    ctx.load_da3(path, "small", "f32")
    out, ref = ctx.da3_forward_raw(images), OD.forward_raw(w, spec, images)
    want = ref["depth"].numpy()
    err = float(np.max(np.abs(out["depth"] - want) / want))
    report("f32.da3", err=f"{err:.2e}")
    assert err < 1e-4


@pytest.mark.parametrize("exp", [-55, 40])
def test_gemm_wide_range(ctx, exp):
    """Rows and columns spread over 2^+-20 around 2^exp: every row is right by itself."""
    g = torch.Generator().manual_seed(5)
    A = _rand(g, 130, 256) * torch.exp2(torch.randint(-20, 21, (130, 1), generator=g).float() + exp).cuda()
    W = _rand(g, 96, 256) * torch.exp2(torch.randint(-20, 21, (96, 1), generator=g).float()).cuda()
    out = _gemm(ctx, A, W, torch.zeros(96, device="cuda")).double()
    ref = A.double() @ W.double().t()
    scale = A.double().norm(dim=1)[:, None] * W.double().norm(dim=1)[None]
    err = float(((out - ref) / scale).norm() / (ref / scale).norm())
    assert err <= _tol(256)


@pytest.mark.parametrize("M,N,K", [(130, 96, 256), (140, 64, 1536), (1200, 1152, 68), (4097, 1544, 132)])
@pytest.mark.parametrize("side", ["a", "w"])
def test_gemm_tiny_values(ctx, M, N, K, side):
    """One operand's rows (of A, or of W) lie at 2^-126 to 2^-90, where the third part of a split falls under
    bf16's smallest subnormal; the other operand brings the results back to ordinary sizes. Every
    row is right by itself: the fp32 instructions keep all 24 bits there."""
    g = torch.Generator().manual_seed(M + K)
    A, W = _rand(g, M, K), _rand(g, N, K)
    small, big = (A, W) if side == "a" else (W, A)
    e = torch.linspace(-124, -90, small.shape[0]).floor()
    small.mul_(torch.exp2(e)[:, None].cuda())
    small[small.abs() < 2.0 ** -126] = 0.0
    big.mul_(2.0 ** 100)
    out = _gemm(ctx, A, W, torch.zeros(N, device="cuda")).double()
    ref = A.double() @ W.double().t()
    dim = 1 if side == "a" else 0
    err = ((out - ref).norm(dim=dim) / ref.norm(dim=dim)).max()
    report("f32.tiny", M=M, N=N, K=K, side=side, err=f"{float(err):.2e}")
    assert float(err) <= 2 * _tol(K)   # the worst row, not the whole matrix


def test_gemm_few_tiny_values(ctx):
    """Ordinary operands with a tiny value here and there: the waves that redo their sums agree."""
    g = torch.Generator().manual_seed(4)
    A, W = _rand(g, 300, 384), _rand(g, 200, 384)
    A[::7, 3], W[::5, 9] = 1.2345e-37, -3.21e-36
    out = _gemm(ctx, A, W, torch.zeros(200, device="cuda")).double()
    ref = A.double() @ W.double().t()
    assert float((out - ref).norm() / ref.norm()) <= _tol(384)


def _same(out, ref, tol):
    """NaN, infinities and their signs in the same places; the rest within tol."""
    out, ref = out.double(), ref.double()
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    assert torch.equal(out[torch.isinf(ref)], ref[torch.isinf(ref)])
    fine = torch.isfinite(ref)
    assert torch.isfinite(out[fine]).all()
    err = float((out[fine] - ref[fine]).norm() / ref[fine].norm())
    assert err <= tol, err


@pytest.mark.parametrize("M,N,K", [(70, 96, 64), (140, 64, 1536), (1200, 1152, 384), (4097, 1544, 132)])
def test_gemm_special_values(ctx, M, N, K):
    """64x64 tiles, whole and split, 128x64 and 128x128."""
    assert f32_plan(M, N, K)[:2] == ((64, 64) if M < 200 else (128, 64) if M == 1200 else (128, 128))
    g = torch.Generator().manual_seed(9)
    A, W = _rand(g, M, K), _rand(g, N, K)
    A[3, 5], A[40, 7], A[41, K - 1] = float("inf"), float("nan"), float("-inf")
    W[9, 2] = float("inf")
    A[50] = 0.0
    A[50, 1], W[:, 1] = 3.4e38, W[:, 1].clamp(-0.5, 0.5)   # rounds to infinity in bf16, the product is finite
    W[9, 1] = 0.25
    out = _gemm(ctx, A, W, torch.zeros(N, device="cuda"))
    ref = A.double().cpu() @ W.double().cpu().t()
    rows = [r for r in range(M) if r != 50]
    _same(out.cpu()[rows], ref[rows], _tol(K))
    keep = [c for c in range(N) if c != 9]
    _same(out.cpu()[50, keep], ref[50, keep].float(), 1e-6)


@pytest.mark.parametrize("V,H,W,C,N,relu", [(1, 5, 7, 64, 64, 1), (2, 18, 18, 96, 64, 0), (1, 70, 66, 32, 32, 0),
                                            (1, 40, 33, 48, 40, 0), (3, 108, 144, 64, 64, 1)])
def test_conv_matches_float64(ctx, V, H, W, C, N, relu):
    g = torch.Generator().manual_seed(H * W + C)
    x, w, b = _rand(g, V, H, W, C), _rand(g, N, C, 3, 3) * (9 * C) ** -0.5, _rand(g, N)
    ldw = (9 * C + 63) // 64 * 64
    wp = torch.zeros(N, ldw, device="cuda")
    wp[:, :9 * C] = w.permute(0, 2, 3, 1).reshape(N, -1)
    out = torch.empty(V, H, W, N, device="cuda")
    torch.cuda.synchronize()
    ctx.kernel_conv2d(splathip.F32, x.data_ptr(), V, H, W, C, wp.data_ptr(), N, ldw, 3, 1, b.data_ptr(), relu, 0, 0,
                      out.data_ptr())
    ctx.synchronize()
    xin = (x.clamp(min=0) if relu else x).cpu().double().permute(0, 3, 1, 2)
    ref = torch.nn.functional.conv2d(xin, w.cpu().double(), b.cpu().double(), padding=1).permute(0, 2, 3, 1)
    err = float((out.cpu().double() - ref).norm() / ref.norm())
    report("f32.conv", V=V, H=H, W=W, C=C, N=N, err=f"{err:.2e}")
    assert err <= _tol(9 * C)


def _attention(ctx, qkv, S, L, heads):
    out = torch.full((S * L, heads * 64), -7.0, device="cuda")
    torch.cuda.synchronize()
    ctx.kernel_attention(splathip.F32, qkv.data_ptr(), out.data_ptr(), S, L, heads)
    ctx.synchronize()
    return out.cpu().double().reshape(S, L, heads, 64).permute(0, 2, 1, 3)


def _attention_ref(qkv, S, L, heads):
    q, k, v = qkv.cpu().double().reshape(S, L, 3, heads, 64).permute(2, 0, 3, 1, 4)
    return torch.softmax(q @ k.transpose(-1, -2) / 8, -1) @ v


@pytest.mark.parametrize("S,L,heads", [(1, 1, 1), (2, 31, 2), (1, 33, 3), (3, 64, 1), (2, 129, 2), (1, 257, 6),
                                       (1, 1297, 6), (2, 700, 3)])
def test_attention_matches_float64(ctx, S, L, heads):
    """The scores' roundings reach the weights as they are, the weighted sum takes six for every 16
    keys: within 2^-24 (sqrt(6 L / 16) + 64), the 64 for scores up to about 8 and the exponential."""
    g = torch.Generator().manual_seed(L)
    qkv = _rand(g, S * L, 3 * heads * 64)
    out, ref = _attention(ctx, qkv, S, L, heads), _attention_ref(qkv, S, L, heads)
    err = float((out - ref).norm() / ref.norm())
    report("f32.attention", S=S, L=L, heads=heads, err=f"{err:.2e}")
    assert err <= 2.0 ** -24 * ((6 * max(L, 16) / 16) ** 0.5 + 64)


@pytest.mark.parametrize("S,L,heads", [(1, 40, 2), (1, 1297, 2)])   # unsplit; key slices
@pytest.mark.parametrize("which", ["k", "v"])
def test_attention_tiny_values(ctx, S, L, heads, which):
    """K at 2^-115 against Q at 2^115 (scores of ordinary size), and V at 2^-112: the tolerance of
    ordinary values, the scores' dominated by their own rounding."""
    g = torch.Generator().manual_seed(L)
    qkv = _rand(g, S * L, 3 * heads * 64)
    q, k, v = qkv.view(S * L, 3, heads, 64).unbind(1)
    if which == "k":
        q.mul_(2.0 ** 115)
        k.mul_(2.0 ** -115)
    else:
        v.mul_(2.0 ** -112)
    out, ref = _attention(ctx, qkv, S, L, heads), _attention_ref(qkv, S, L, heads)
    err = float((out - ref).norm() / ref.norm())
    report("f32.attention.tiny", L=L, which=which, err=f"{err:.2e}")
    assert err <= 2.0 ** -24 * ((6 * max(L, 16) / 16) ** 0.5 + 64)


def test_attention_special_values(ctx):
    """An infinite value reaches its channel of every query and no other."""
    S, L, heads = 1, 300, 2
    g = torch.Generator().manual_seed(2)
    qkv = _rand(g, S * L, 3 * heads * 64)
    v = qkv.view(L, 3, heads, 64)[:, 2]
    v[17, 0, 5] = float("inf")
    v[290, 0, 40] = float("-inf")
    out = _attention(ctx, qkv, S, L, heads)
    ref = _attention_ref(qkv, S, L, heads)
    report("f32.attention.special", inf=int(torch.isinf(out).sum()), ref=int(torch.isinf(ref).sum()),
           nan=int(torch.isnan(out).sum()))
    assert torch.equal(torch.isinf(out), torch.isinf(ref)) and not torch.isnan(out).any()
    assert torch.equal(out[torch.isinf(ref)], ref[torch.isinf(ref)])
    fine = torch.isfinite(ref)
    assert float(((out[fine] - ref[fine]).abs() / (ref[fine].abs() + 1.0)).max()) < 1e-5


@pytest.mark.parametrize("S,L,heads", [(1, 40, 2), (1, 1297, 2)])   # unsplit; key slices
@pytest.mark.parametrize("which", ["nan_q", "inf_k", "nan_k", "big_k", "big_v", "nan_v"])
def test_attention_operands_outside_bf16(ctx, S, L, heads, which):
    """One operand value that bf16 parts cannot hold, in head 0: what float64 gives, NaN and infinities in the
    same places. big: finite, rounds to infinity in bf16; Q is a power of two there, so that no other
    check sees it."""
    g = torch.Generator().manual_seed(L + 1)
    qkv = _rand(g, S * L, 3 * heads * 64)
    q, k, v = qkv.view(S * L, 3, heads, 64).unbind(1)
    if which == "nan_q":
        q[L // 2, 0, 7] = float("nan")
    elif which in ("inf_k", "nan_k"):
        k[L // 3, 0, 9] = float(which[:3])
    elif which == "big_k":
        q[:, 0, 9] = torch.where(q[:, 0, 9] > 0, 2.0 ** -124, -2.0 ** -124)
        k[L // 3, 0, 9] = 3.4e38
    else:
        v[L // 3, 0, 9] = 3.4e38 if which == "big_v" else float("nan")
        k[L // 3, 0] = 0.0   # a weight of at most 1 before the division: the sum stays finite
    out, ref = _attention(ctx, qkv, S, L, heads), _attention_ref(qkv, S, L, heads)
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    fine = ~torch.isnan(ref)
    scale = ref.abs() + 1.0
    assert float(((out[fine] - ref[fine]).abs() / scale[fine]).max()) <= 2.0 ** -24 * ((6 * max(L, 16) / 16) ** 0.5 + 64)


@pytest.mark.parametrize("V,H,W,C,N,stride,relu", [
    (1, 18, 18, 96, 64, 1, 0), (1, 18, 18, 96, 64, 1, 1), (1, 18, 18, 96, 64, 2, 1),   # K in slices
    (3, 108, 144, 32, 64, 1, 1), (1, 60, 60, 64, 32, 1, 0),                         # whole; 128x32
    (4, 100, 130, 64, 64, 1, 1), (2, 66, 70, 64, 256, 1, 0), (2, 66, 70, 64, 256, 2, 1),   # 128x64; wider
    (1, 40, 33, 48, 40, 1, 0), (1, 40, 33, 36, 72, 2, 0), (3, 108, 144, 20, 130, 1, 0),    # per-lane addressing
])
def test_conv_special_values(ctx, V, H, W, C, N, stride, relu):
    """An infinite, a NaN and a 3.4e38 pixel, at a corner and inside: such waves redo their sums with a convolution
    of their own. Every output within K 2^-24 of the sum of its products' magnitudes (any order of an
    fp32 sum), the others' NaN and infinities in the same places."""
    g = torch.Generator().manual_seed(H * W + C)
    x, w, b = _rand(g, V, H, W, C), _rand(g, N, C, 3, 3) * (9 * C) ** -0.5, _rand(g, N)
    x[0, 0, 0, 3], x[V - 1, H // 2, W // 3, 1] = float("inf"), float("nan")
    x[0, H - 1, W - 1, 2] = 3.4e38
    x[V - 1, 3, 5, 0], x[0, 9, 2, 4] = float("-inf"), -3.4e38
    w[:, 2] *= 0.01
    w[:, 4] *= 0.01
    ldw = (9 * C + 63) // 64 * 64
    wp = torch.zeros(N, ldw, device="cuda")
    wp[:, :9 * C] = w.permute(0, 2, 3, 1).reshape(N, -1)
    Ho, Wo = (H - 1) // stride + 1, (W - 1) // stride + 1
    out = torch.empty(V, Ho, Wo, N, device="cuda")
    torch.cuda.synchronize()
    ctx.kernel_conv2d(splathip.F32, x.data_ptr(), V, H, W, C, wp.data_ptr(), N, ldw, 3, stride, b.data_ptr(), relu, 0, 0,
                      out.data_ptr())
    ctx.synchronize()
    xd = x.cpu().double()
    xd = torch.where(xd < 0, 0.0, xd) if relu else xd   # keeps NaN
    cols = torch.nn.functional.unfold(xd.permute(0, 3, 1, 2), 3, padding=1, stride=stride).transpose(1, 2)   # [V, P, 9 C]
    wd = w.cpu().double().reshape(N, -1).t()
    ref = (cols @ wd + b.cpu().double()).float().reshape(V, Ho, Wo, N)
    mag = (cols.abs() @ wd.abs()).reshape(V, Ho, Wo, N) + b.cpu().double().abs()
    out = out.cpu()
    assert torch.equal(torch.isnan(out), torch.isnan(ref))
    assert torch.equal(out[torch.isinf(ref)], ref[torch.isinf(ref)])
    fine = torch.isfinite(ref)
    assert 0 < int((~fine).sum()) < fine.numel() // 2
    err = float(((out - ref).double().abs()[fine] / mag[fine]).max())
    report("f32.conv.special", H=H, W=W, C=C, N=N, stride=stride, relu=relu, err=f"{err:.2e}")
    assert err <= (9 * C + 2) * 2.0 ** -24
