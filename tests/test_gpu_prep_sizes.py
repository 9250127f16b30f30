"""Particle preparation at box sizes on both sides of its compile-time transforms and of the 64 positions
that a wavefront of the edge selection takes at a time: images prepared with shifts, against the
oracle, with the bound of test_gpu_prep.py (2e-5 of the largest component)."""
import numpy as np
import pytest

import prep_oracle as P
from gpu_helpers import say
from test_gpu_prep import _check, _handle, _particles

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,M", [(32, 32), (66, 66), (130, 66), (128, 128), (130, 130), (182, 154), (256, 200)])
def test_prep_box_sizes(B, M):
    say(f"prep parity: box {B}, boxmatch {M}")
    rng = np.random.default_rng(B + 1000 * M)
    imgs = _particles(rng, 3, B)
    shifts = rng.uniform(-4, 4, (3, 2)).astype(np.float32)
    shifts[1] = 0.0
    msk = 0.4 * M
    lib = _handle(M)
    got = lib.prep_imgs(imgs, shifts, box=B, msk=msk)
    lib.kill()
    _check(got, imgs, shifts, P.PrepCfg(box=B, boxmatch=M, msk=msk), None)


def test_inner_mask_starts_at_the_rounded_root():
    """Pixels at distance sqrt(N) and an inner edge that starts at exactly that FP32 number: their weight
    is 1 with the correctly rounded root, and about 1/2 with one that is an ulp too small (the edge is
    two ulps wide)."""
    B = 64
    rng = np.random.default_rng(5)
    imgs = _particles(rng, 1, B)
    shifts = np.zeros((1, 2), np.float32)
    lib = _handle(B)
    roots = sorted({x * x + y * y for x in range(1, 20) for y in range(x + 1) if 16 < x * x + y * y < 400})
    for N in roots[::3]:
        inner = np.sqrt(np.float32(N))
        width = np.float32(2) * np.spacing(inner)
        say(f"inner mask radius sqrt({N})")
        got = lib.prep_imgs(imgs, shifts, box=B, msk=24.0, inner=float(inner), width=float(width))
        _check(got, imgs, shifts, P.PrepCfg(box=B, boxmatch=B, msk=24.0, inner=float(inner), width=float(width)), None)
    lib.kill()
