"""Photo batches through the pinned upload ring (16 MB in 2 MB chunks, two device buffers in turn):
batches that wrap it, end in part of a chunk, hold one photo or photos of several sizes, and one
below the ring's threshold. Each photo must come out as the single-image resize (itself checked
against the oracle in tests/test_gpu_preprocess.py) gives it, byte for byte."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

import splathip
from oracle import preprocess as P
from oracle.common import to_model_input


@pytest.mark.parametrize("sizes", [
    [(1100, 1200)] * 5,                                    # 26 MB: wraps the ring, chunks of 2 MB and a part
    [(2000, 1801)],                                        # one photo
    [(900, 1000), (518, 392), (1300, 900), (700, 1201)],   # several sizes, one copied as it is
    [(300, 260), (280, 300)],                              # 0.6 MB: without the ring
])
def test_batches(ctx, sizes):
    rng = np.random.default_rng(len(sizes))
    photos = []
    for w, h in sizes:
        p = rng.integers(0, 256, size=(h, w, 4), dtype=np.uint8)
        p[..., 3] |= 128
        photos.append(p)
    W, H = splathip.ma_input_size(sizes)
    img = torch.empty(len(sizes), 3, H, W, device="cuda")
    fg = torch.empty(len(sizes), H, W, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    for _ in range(2):   # the second call reuses the ring and the buffers
        img.zero_()
        torch.cuda.synchronize()
        assert ctx.ma_model_inputs_device(photos, img.data_ptr(), fg.data_ptr()) == (H, W)
        ctx.synchronize()
        for k, p in enumerate(photos):
            (rw, rh), (left, top), f = P.cover(p.shape[1], p.shape[0], (W, H))
            r = ctx.resize_rgba8(p, rw, rh, f)
            want, want_fg = to_model_input(np.ascontiguousarray(r[None, top:top + H, left:left + W]))
            assert np.array_equal(img[k].cpu().numpy(), want[0]), k
            assert np.array_equal(fg[k].cpu().numpy().astype(bool), want_fg[0]), k
