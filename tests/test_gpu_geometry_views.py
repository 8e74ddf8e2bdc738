"""The one-pass geometry kernel at view counts on either side of the cameras it keeps in LDS (64), at
sizes that leave ragged blocks and turns, on maps below and above the L2s' size, and with the cleaned
confidences written over the given ones, against oracle/geometry.py. Points are f64 results stored as f32,
cameras f64 (1e-6 and 1e-9 of their scale, as tests/test_gpu_geometry.py); the confidences are equal:
a projection within f64's rounding of a pixel boundary has a chance of about 1e-6 in these scenes."""
import numpy as np
import pytest

from conftest import report

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import geometry as OG


@pytest.mark.parametrize("V,H,W,in_place", [(1, 3, 5, False), (2, 17, 31, True), (64, 14, 18, False), (65, 14, 18, True),
                                            (130, 9, 11, False), (6, 810, 810, True), (66, 243, 243, False)])
def test_views(ctx, V, H, W, in_place):
    rng = np.random.default_rng(V)
    pose = np.zeros((V, 9), np.float32)
    pose[:, :3] = rng.normal(scale=0.05, size=(V, 3))
    pose[:, 3:6] = rng.normal(scale=0.02, size=(V, 3))
    pose[:, 6] = 1.0
    pose[:, 7:] = rng.uniform(0.9, 1.0, (V, 2))
    depth = (2 + 0.3 * rng.standard_normal((V, H, W))).astype(np.float32)
    conf = (1 + np.exp(rng.standard_normal((V, H, W)))).astype(np.float32)
    fg = (rng.random((V, H, W)) < 0.9).astype(np.uint8)
    d = {k: torch.from_numpy(a).cuda() for k, a in (("depth", depth), ("pose_encoding", pose), ("conf", conf), ("foreground", fg))}
    cams = torch.empty(V, 16, dtype=torch.float64, device="cuda")
    pts = torch.empty(V, H, W, 3, device="cuda")
    outs = []
    for out in [torch.empty_like(d["conf"])] + ([d["conf"]] if in_place else []):
        torch.cuda.synchronize()
        ctx.kernel_reconstruct(V, H, W, **{k: t.data_ptr() for k, t in d.items()}, cameras=cams.data_ptr(),
                               points=pts.data_ptr(), conf_out=out.data_ptr())
        ctx.synchronize()
        outs.append(out)
    assert torch.equal(outs[0], outs[-1])
    out = outs[0]
    ref = OG.da3_reconstruct(depth, conf, pose, fg)
    c = cams.cpu().numpy()
    for key, got in (("rotation", c[:, :9].reshape(V, 3, 3)), ("translation", c[:, 9:12]), ("focal", c[:, 12:14])):
        assert np.abs(got - ref[key]).max() <= 1e-9 * max(np.abs(ref[key]).max(), 1e-30)
    assert np.abs(pts.cpu().numpy() - ref["points"]).max() <= 1e-6 * np.abs(ref["points"]).max()
    differ = float(np.mean(out.cpu().numpy() != ref["conf"]))
    report("geometry.views", V=V, in_place=in_place, differ=differ, zeroed=float(np.mean(ref["conf"] == 0)))
    assert differ == 0


def test_points_over_their_source(ctx):
    """MapAnything's points written over the camera-frame points: what separate buffers give."""
    V, H, W = 4, 70, 98
    g = torch.Generator().manual_seed(1)
    y, x = torch.meshgrid(torch.linspace(-0.4, 0.4, H), torch.linspace(-0.5, 0.5, W), indexing="ij")
    z = 2 + 0.1 * torch.randn(V, H, W, generator=g)
    pts = torch.stack([x * z, y * z, z], -1).cuda()
    quat = torch.tensor([[0.0, 0.0, 0.0, 1.0]]).repeat(V, 1).cuda()
    trans = torch.randn(V, 3, generator=g).mul(0.05).cuda()
    trans[:, 2] -= 0.5 * torch.arange(V).cuda()   # the views' depths differ from view 0's
    conf = (1 + torch.exp(torch.randn(V, H, W, generator=g))).cuda()
    mask = (torch.rand(V, H, W, generator=g) < 0.9).to(torch.uint8).cuda()

    def call(source, points):
        cams, out = torch.empty(V, 16, dtype=torch.float64, device="cuda"), torch.empty_like(conf)
        torch.cuda.synchronize()
        ctx.kernel_reconstruct(V, H, W, points_in_camera=source.data_ptr(), quaternion=quat.data_ptr(),
                               translation=trans.data_ptr(), conf=conf.data_ptr(), mask=mask.data_ptr(),
                               cameras=cams.data_ptr(), points=points.data_ptr(), conf_out=out.data_ptr())
        ctx.synchronize()
        return cams, points, out

    ref = call(pts, torch.empty_like(pts))
    both = pts.clone()
    got = call(both, both)
    assert all(torch.equal(a, b) for a, b in zip(got, ref))
    assert 0 < int((ref[2] == 0).sum()) < conf.numel()


@pytest.mark.parametrize("mode,inputs,over", [
    ("da3", ("pose_encoding",), "points"), ("da3", ("foreground", "pose_encoding"), "conf_out"), ("da3", ("depth",), "points"),
    ("da3", ("conf",), "points"), ("ma", ("mask", "foreground"), "conf_out"), ("ma", ("quaternion", "translation"), "points"),
    ("ma", ("mask", "quaternion"), "points"), ("ma", ("translation",), "cameras"),
])
def test_inputs_in_an_output_s_memory(ctx, mode, inputs, over):
    """Inputs that lie, one after the other and off its start, in an output's memory: what separate buffers give."""
    V, H, W = 3, 70, 98
    g = torch.Generator().manual_seed(3)
    z = 2 + 0.2 * torch.randn(V, H, W, generator=g)
    conf = 1 + torch.exp(torch.randn(V, H, W, generator=g))
    fg = (torch.rand(V, H, W, generator=g) < 0.9).to(torch.uint8)
    shift = torch.randn(V, 3, generator=g).mul(0.05)
    turn = torch.cat([torch.randn(V, 3, generator=g).mul(0.02), torch.ones(V, 1)], 1)
    if mode == "da3":
        d = {"depth": z, "pose_encoding": torch.cat([shift, turn, torch.full((V, 2), 0.9)], 1), "conf": conf, "foreground": fg}
    else:
        y, x = torch.meshgrid(torch.linspace(-0.4, 0.4, H), torch.linspace(-0.5, 0.5, W), indexing="ij")
        d = {"points_in_camera": torch.stack([x * z, y * z, z], -1), "quaternion": turn, "translation": shift, "conf": conf,
             "mask": (torch.rand(V, H, W, generator=g) < 0.9).to(torch.uint8), "foreground": fg}
    d = {k: t.contiguous().cuda() for k, t in d.items()}

    def call(shared):
        out = {"cameras": torch.zeros(V, 16, dtype=torch.float64, device="cuda"), "points": torch.zeros(V, H, W, 3, device="cuda"),
               "conf_out": torch.zeros(V, H, W, device="cuda")}
        ptr = {k: t.data_ptr() for k, t in {**d, **out}.items()}
        at = 16
        for k in inputs if shared else ():
            raw = out[over].view(-1).view(torch.uint8)
            n = d[k].numel() * d[k].element_size()
            raw[at:at + n] = d[k].reshape(-1).view(torch.uint8)
            ptr[k] = raw.data_ptr() + at
            at += (n + 15) // 16 * 16
        torch.cuda.synchronize()
        ctx.kernel_reconstruct(V, H, W, **ptr)
        ctx.synchronize()
        return out

    want, got = call(False), call(True)
    assert 0 < int((want["conf_out"] == 0).sum()) < conf.numel()
    assert all(torch.equal(want[k], got[k]) for k in want)


def test_half_pixels_round_away_from_zero(ctx):
    """Every projection of view 0 into view 1 lies exactly half way between two columns (focal length 64, depths
    that divide 43065, a translation of 43065 / 128: all exact in fp32, and the fitted intrinsics in f64),
    and view 1's columns are in turn more and less confident: the confidences are f64::round's."""
    Z = 43065
    z = np.array([d for d in range(1, Z + 1, 2) if Z % d == 0 and Z // d < 90], np.float64)
    H, W, cx = len(z), 48, 24.0
    cy = H / 2
    rows, cols = np.meshgrid(np.arange(H), np.arange(W), indexing="ij")
    pts = np.empty((2, H, W, 3), np.float32)
    for v, k in ((0, 1), (1, 4)):   # view 1 sees everything four times as far
        depth = k * z[:, None] * np.ones((1, W))
        pts[v] = np.stack([(cols - cx) * depth / 64, (rows - cy) * depth / 64, depth], -1)
    conf = np.full((2, H, W), 2.0, np.float32)
    conf[1] = np.where(cols % 2, 3.0, 1.0)
    trans = np.zeros((2, 3), np.float32)
    trans[1, 0] = Z / 128
    quat = np.tile(np.array([0, 0, 0, 1], np.float32), (2, 1))
    d = {k: torch.from_numpy(a).cuda() for k, a in (("points_in_camera", pts), ("quaternion", quat), ("translation", trans),
                                                    ("conf", conf), ("mask", np.ones((2, H, W), np.uint8)))}
    cams = torch.empty(2, 16, dtype=torch.float64, device="cuda")
    points, out = torch.empty(2, H, W, 3, device="cuda"), torch.empty(2, H, W, device="cuda")
    torch.cuda.synchronize()
    ctx.kernel_reconstruct(2, H, W, **{k: t.data_ptr() for k, t in d.items()}, cameras=cams.data_ptr(),
                           points=points.data_ptr(), conf_out=out.data_ptr())
    ctx.synchronize()
    assert cams[:, 12:].tolist() == [[64.0, 64.0, cx, cy]] * 2
    twice = 2 * cols - (Z / z).astype(int)[:, None]            # 2 u, odd
    column = np.where(twice >= 0, (twice + 1) // 2, (twice - 1) // 2)
    seen = (column >= 0) & (column < W)
    want = conf.copy()
    want[0][seen & (column % 2 == 1)] = 0.0
    assert np.array_equal(out.cpu().numpy(), want)


@pytest.mark.parametrize("H,W", [(46340, 46340), (46342, 46341)])   # within a turn of 2^31 pixels, and past it
def test_largest_view(ctx, H, W):
    """One view whose pixel numbers pass 32 bits on the last turn, or are longer: every confidence is kept, and
    the points of the last rows and of a sample of pixels are the unprojected depths."""
    n = H * W
    if torch.cuda.mem_get_info()[0] < 28 * n:
        pytest.skip("needs 60 GB of GPU memory")
    depth = torch.rand(n, device="cuda").add_(1.0)
    conf = torch.rand(n, device="cuda").add_(1.0)
    pose = torch.tensor([[0, 0, 0, 0, 0, 0, 1, 0.9, 1.0]], device="cuda")
    cams = torch.empty(1, 16, dtype=torch.float64, device="cuda")
    pts, out = torch.full((n, 3), -7.0, device="cuda"), torch.full((n,), -7.0, device="cuda")
    torch.cuda.synchronize()
    ctx.kernel_reconstruct(1, H, W, depth=depth.data_ptr(), pose_encoding=pose.data_ptr(), conf=conf.data_ptr(),
                           cameras=cams.data_ptr(), points=pts.data_ptr(), conf_out=out.data_ptr())
    ctx.synchronize()
    assert torch.equal(out, conf)
    fx, fy, cx, cy = (float(v) for v in cams[0, 12:])
    for idx in (torch.arange(n - 600000, n, device="cuda"),
                torch.randint(0, n, (600000,), device="cuda", generator=torch.Generator("cuda").manual_seed(1))):
        d = depth[idx].double()
        x, y = (idx % W).double(), torch.div(idx, W, rounding_mode="floor").double()
        want = torch.stack([(x - cx) / fx * d, (y - cy) / fy * d, d], -1)
        assert float((pts[idx].double() - want).abs().max()) <= 2.0 ** -23 * float(want.abs().max())
    del depth, conf, pts, out
    torch.cuda.empty_cache()
