"""Photo batches through the pinned upload ring (16 MB in 2 MB chunks, two device buffers in turn):
batches that wrap it, end in part of a chunk, hold one photo or photos of several sizes, page-locked ones
among them, and one below the ring's threshold; MapAnything's inputs (one resize a photo) and DA3's
(two, which alternate between two buffers). Each photo must come out as the single-image resizes (themselves
checked against the oracle in tests/test_gpu_preprocess.py) give it, byte for byte."""
import os

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


DA3_SIZES = [(2100, 1403), (1201, 1900), (2000, 1300), (1600, 1100)]   # 38 MB, every size of its own


def _photos(sizes, pinned=()):
    rng = np.random.default_rng(len(sizes))
    photos = []
    for k, (w, h) in enumerate(sizes):
        p = torch.empty(h, w, 4, dtype=torch.uint8, pin_memory=k in pinned).numpy()
        p[:] = rng.integers(0, 256, size=(h, w, 4), dtype=np.uint8)
        p[..., 3] |= 128
        photos.append(p)
    return photos


def _da3(ctx, photos):
    W, H = splathip.da3_model_inputs_size([(p.shape[1], p.shape[0]) for p in photos])
    img = torch.zeros(len(photos), 3, H, W, device="cuda")
    fg = torch.zeros(len(photos), H, W, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    assert ctx.da3_model_inputs_device(photos, img.data_ptr(), fg.data_ptr()) == (H, W)
    ctx.synchronize()
    return img.cpu().numpy(), fg.cpu().numpy()


def _da3_one_by_one(ctx, photos):
    """The two resizes of each photo through splat_resize_rgba8, then the common crop."""
    W, H = splathip.da3_model_inputs_size([(p.shape[1], p.shape[0]) for p in photos])
    out = []
    for p in photos:
        (bw, bh), (w, h) = P.model_input_size(p.shape[1], p.shape[0])
        resized = 0
        for nw, nh in ((bw, bh), (w, h)):
            if (p.shape[1], p.shape[0]) != (nw, nh):
                f = P.CATMULLROM if nw > p.shape[1] or nh > p.shape[0] else P.TRIANGLE
                p = ctx.resize_rgba8(np.ascontiguousarray(p), nw, nh, f)
                resized += 1
        assert resized == 2
        left, top = (w - W) // 2, (h - H) // 2
        out.append(to_model_input(np.ascontiguousarray(p[None, top:top + H, left:left + W])))
    return out


@pytest.mark.parametrize("pinned", [(), (0, 1, 2, 3), (1,), (0, 2)])
def test_da3_batches(ctx, pinned):
    photos = _photos(DA3_SIZES, pinned)
    want = _da3_one_by_one(ctx, photos)
    for _ in range(2):
        img, fg = _da3(ctx, photos)
        for k in range(len(photos)):
            assert np.array_equal(img[k], want[k][0][0]), k
            assert np.array_equal(fg[k].astype(bool), want[k][1][0]), k


def test_host_pixels_are_read_on_return(ctx):
    """Page-locked photos, below and above the ring's threshold, overwritten as soon as the call returns."""
    for sizes in (DA3_SIZES[:2], [(300, 260), (280, 300)]):
        photos = _photos(sizes, range(len(sizes)))
        want = _da3(ctx, photos)
        W, H = splathip.da3_model_inputs_size([(p.shape[1], p.shape[0]) for p in photos])
        img = torch.zeros(len(photos), 3, H, W, device="cuda")
        torch.cuda.synchronize()
        ctx.da3_model_inputs_device(photos, img.data_ptr())
        for p in photos:
            p[:] = 255
        ctx.synchronize()
        assert np.array_equal(img.cpu().numpy(), want[0])


def test_one_cpu(ctx):
    """With a single CPU to run on, pageable photos go without the ring: the same bytes."""
    photos = _photos(DA3_SIZES)
    want = _da3(ctx, photos)
    cpus = os.sched_getaffinity(0)
    os.sched_setaffinity(0, {min(cpus)})
    try:
        got = _da3(ctx, photos)
    finally:
        os.sched_setaffinity(0, cpus)
    assert np.array_equal(got[0], want[0]) and np.array_equal(got[1], want[1])


def test_two_threads_and_a_busy_stream(ctx):
    """Two contexts on two threads, each with a ring of its own, behind attention launches still running on
    their streams."""
    import threading
    photos = [_photos(DA3_SIZES), _photos(DA3_SIZES[::-1])]
    want = [_da3(ctx, p) for p in photos]
    L, heads = 6000, 6
    qkv = torch.randn(L, 3 * heads * 64, device="cuda")
    got, errors = [None, None], []

    def run(k):
        try:
            other = splathip.Context(0)
            W, H = splathip.da3_model_inputs_size([(p.shape[1], p.shape[0]) for p in photos[k]])
            img = torch.zeros(len(photos[k]), 3, H, W, device="cuda")
            out = torch.empty(L, heads * 64, device="cuda")
            torch.cuda.synchronize()
            for _ in range(3):
                for _ in range(20):
                    other.kernel_attention(splathip.F32, qkv.data_ptr(), out.data_ptr(), 1, L, heads)
                other.da3_model_inputs_device(photos[k], img.data_ptr())
                other.synchronize()
                assert np.array_equal(img.cpu().numpy(), want[k][0])
            got[k] = True
            other.close()
        except Exception as e:   # shown by the main thread
            errors.append(e)

    threads = [threading.Thread(target=run, args=(k,)) for k in (0, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(timeout=60)
    assert not errors and got == [True, True]
