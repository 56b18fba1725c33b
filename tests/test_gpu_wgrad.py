"""GPU: the weight gradient's strips and chunks, and launches over images.

Bar: dW and db against float64 sums of the same BF16 products. An FP32 sum of
m products in chunks of any order is off by at most about sqrt(m) roundings of
its size, so 4e-5 * sqrt(pixels) as for the other backward tests (products are
of unit normals). Sizes: widths and heights around the 8 x 4 strips, one strip
and several tiles of 8, strips of several images in one tile, channel counts
around the 32 input and 32 / 64 output channel blocks.
"""
import numpy as np
import pytest

from oracle import denoiser_ref as D
from vulkanhybridraytracer_amd import denoise

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,h,w,cin,cout", [(1, 1, 1, 16, 16), (1, 4, 8, 32, 32), (1, 5, 9, 16, 48), (3, 3, 7, 48, 64),
                                            (5, 4, 8, 32, 16), (1, 37, 65, 32, 32), (1, 8, 80, 144, 32),
                                            (2, 6, 24, 16, 80), (1, 64, 72, 64, 64)])
def test_weight_gradient_edges(gpu_ctx, n, h, w, cin, cout):
    print("weight gradient", n, h, w, cin, cout, flush=True)
    r = np.random.default_rng(cin * 13 + cout + w)
    x = denoise.to_bf16_bits(r.normal(size=(n, h, w, cin)))
    dy = denoise.to_bf16_bits(r.normal(size=(n, h, w, cout)))
    wt = r.normal(size=(cout, 3, 3, cin)).astype(np.float32)
    _, dw, db = denoise.conv3x3_backward(gpu_ctx, x, dy, wt)
    val = lambda b: denoise.from_bf16_bits(b).astype(np.float64)  # noqa: E731
    _, rdw, rdb = D.conv3x3_backward(val(x), wt.astype(np.float64), val(dy))
    bound = 4e-5 * np.sqrt(n * h * w)
    assert np.all(np.abs(dw - rdw) <= bound + 1e-6 * np.abs(rdw))
    assert np.all(np.abs(db - rdb) <= bound + 1e-6 * np.abs(rdb))


@pytest.mark.parametrize("count", [1, 16, 17])
def test_gradients_of_repeated_images(gpu_ctx, count):
    """`count` copies of one image (more than one launch takes from 17 on): the
    mean loss and gradient are the single image's"""
    from vulkanhybridraytracer_amd import hr
    r = np.random.default_rng(4)
    h = w = 32
    g = hr.GBuffer(gpu_ctx, w, h)
    planes = {k: r.uniform(0.1, 1.0, size=(h, w, 4)).astype(np.float32)
              for k in ("position", "normal", "albedo", "material", "emissive")}
    g.upload(planes)
    noisy, target = gpu_ctx.alloc(w * h * 16), gpu_ctx.alloc(w * h * 16)
    noisy.upload(r.uniform(0, 2, size=(h, w, 4)).astype(np.float32))
    target.upload(r.uniform(0, 2, size=(h, w, 4)).astype(np.float32))
    dn = denoise.Denoiser(gpu_ctx, seed=5)
    im = denoise.Denoiser.image(g, noisy.ptr, target.ptr, None, (0.0, 0.0, 0.0))
    l1, g1 = dn.gradients([im])
    ln, gn = dn.gradients([im] * count)
    assert abs(ln - l1) <= 1e-6 * l1
    # each image's gradient carries the scale 1 / count through BF16 roundings
    assert np.linalg.norm(gn - g1) <= 2.0 ** -6 * np.linalg.norm(g1)
    dn.close()


@pytest.mark.parametrize("count", [1, 16, 17, 33])
def test_gradients_of_several_images(gpu_ctx, count):
    """`count` different images (more than one launch takes from 17 on): the mean
    loss and gradient are those of the single images"""
    from vulkanhybridraytracer_amd import hr
    r = np.random.default_rng(4)
    h = w = 32
    dn = denoise.Denoiser(gpu_ctx, seed=5)
    keep, images, losses, grads = [], [], [], []
    for k in range(count):
        g = hr.GBuffer(gpu_ctx, w, h)
        planes = {k2: r.uniform(0.1, 1.0, size=(h, w, 4)).astype(np.float32)
                  for k2 in ("position", "normal", "albedo", "material", "emissive")}
        g.upload(planes)
        noisy, target = gpu_ctx.alloc(w * h * 16), gpu_ctx.alloc(w * h * 16)
        noisy.upload(r.uniform(0, 0.5 + 0.2 * k, size=(h, w, 4)).astype(np.float32))
        target.upload(r.uniform(0, 2, size=(h, w, 4)).astype(np.float32))
        keep.append((g, noisy, target))
        images.append(denoise.Denoiser.image(g, noisy.ptr, target.ptr, None, (0.0, 0.0, 0.0)))
        loss, grad = dn.gradients(images[-1:])
        losses.append(loss)
        grads.append(grad.astype(np.float64))
    ln, gn = dn.gradients(images)
    mean, size = np.mean(grads, axis=0), np.mean([np.linalg.norm(g) for g in grads])
    assert abs(ln - np.mean(losses)) <= 1e-6 * ln
    # each image's gradient carries the scale 1 / count through BF16 roundings
    tol = 2.0 ** -6 * size
    assert np.linalg.norm(gn - mean) <= tol
    if count > 1:
        # the loss shows an image taken twice for another, both show one taken for all
        assert abs(np.mean(losses[:1] + losses[:-1]) - np.mean(losses)) > 1e-4 * ln
        assert np.linalg.norm(grads[0] - mean) > 4 * tol
    dn.close()
