"""The one-pass geometry kernel at view counts on either side of the cameras it keeps in LDS (64), at
sizes that leave ragged blocks and turns, and with the cleaned confidences written over the given
ones, against oracle/geometry.py. Points are f64 results stored as f32, cameras f64 (1e-6 and 1e-9 of
their scale, as tests/test_gpu_geometry.py); a confidence may differ only where a projection falls
within rounding of a pixel boundary."""
import numpy as np
import pytest

from conftest import report

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import geometry as OG


@pytest.mark.parametrize("V,H,W,in_place", [(1, 3, 5, False), (2, 17, 31, True), (64, 14, 18, False), (65, 14, 18, True),
                                            (130, 9, 11, False)])
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
    out = d["conf"] if in_place else torch.empty_like(d["conf"])
    torch.cuda.synchronize()
    ctx.kernel_reconstruct(V, H, W, **{k: t.data_ptr() for k, t in d.items()}, cameras=cams.data_ptr(),
                           points=pts.data_ptr(), conf_out=out.data_ptr())
    ctx.synchronize()
    ref = OG.da3_reconstruct(depth, conf, pose, fg)
    c = cams.cpu().numpy()
    for key, got in (("rotation", c[:, :9].reshape(V, 3, 3)), ("translation", c[:, 9:12]), ("focal", c[:, 12:14])):
        assert np.abs(got - ref[key]).max() <= 1e-9 * max(np.abs(ref[key]).max(), 1e-30)
    assert np.abs(pts.cpu().numpy() - ref["points"]).max() <= 1e-6 * np.abs(ref["points"]).max()
    differ = float(np.mean(out.cpu().numpy() != ref["conf"]))
    report("geometry.views", V=V, in_place=in_place, differ=differ, zeroed=float(np.mean(ref["conf"] == 0)))
    assert differ <= 1e-3
