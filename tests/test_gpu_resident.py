"""Which solves run in launches whose blocks wait for each other: the results
are the same either way, so the context's report tells."""
import numpy as np
import pytest
import torch

import damascene_amd as dm

pytestmark = pytest.mark.gpu

ALWAYS = 1 << 16  # polls that never run out on a card of one's own


@pytest.fixture
def own():
    c = dm.Context(0)
    yield c
    c.synchronize()
    c.close()


def solve(c, w, h, precision, nvec=5):
    y, x = np.mgrid[:h, :w]
    cell = (x * 7 // w + 2 * (y * 5 // h)) % 4
    pb = (0.4 * ((np.diff(cell, axis=1, append=cell[:, -1:]) != 0) | (np.diff(cell, axis=0, append=cell[-1:]) != 0))
          + 0.02 * np.random.RandomState(w).rand(h, w)).astype(np.float32)
    before = c.resident_report()
    vals, vecs, it = c.generalized_eigensolve(w, h, c.intervene(c.upload(pb)), nvec=nvec, tol=1e-2,
                                              precision=precision)
    after = c.resident_report()
    return (vals.tobytes(), vecs.cpu().numpy().tobytes(), it), tuple(b - a for a, b in zip(before, after))


# the sizes at which the plain steps run in one launch (up to 262,144 pixels
# on 256 compute units), and the block filter (tiles of 8 and of 12 units)
SERVED = [(32, 32, dm.PREC_FP32), (230, 57, dm.PREC_FP32), (481, 321, dm.PREC_FP32), (512, 512, dm.PREC_FP32),
          (320, 240, dm.PREC_MIXED), (481, 321, dm.PREC_MIXED), (512, 384, dm.PREC_MIXED)]


@pytest.mark.parametrize("w,h,precision", SERVED)
def test_served_sizes_take_the_launch(own, w, h, precision):
    print(f"case: resident {w}x{h} precision {precision}", flush=True)
    with dm.tuned(resident_polls=ALWAYS):
        got, (done, stalled) = solve(own, w, h, precision)
    assert done > 0 and stalled == 0
    with dm.tuned(resident_polls=0):
        ref, counts = solve(own, w, h, precision)
    assert counts == (0, 0) and got == ref
    assert got[2] > 0


# too large for one block per compute unit, small images of the block filter
@pytest.mark.parametrize("w,h,precision", [(520, 512, dm.PREC_FP32), (160, 120, dm.PREC_MIXED),
                                           (640, 480, dm.PREC_MIXED)])
def test_other_sizes_do_not(own, w, h, precision):
    print(f"case: not resident {w}x{h} precision {precision}", flush=True)
    with dm.tuned(resident_polls=ALWAYS):
        assert solve(own, w, h, precision)[1] == (0, 0)


# one poll allowed: the launch gives up, the host does its work again, and the
# next solve with more polls takes the launch again
@pytest.mark.parametrize("w,h,precision", [(230, 57, dm.PREC_FP32), (320, 240, dm.PREC_MIXED),
                                           (481, 321, dm.PREC_MIXED)])
def test_given_up_and_taken_again(own, w, h, precision):
    print(f"case: given up {w}x{h} precision {precision}", flush=True)
    with dm.tuned(resident_polls=1):
        first, counts = solve(own, w, h, precision)
    assert sum(counts) > 0
    with dm.tuned(resident_polls=ALWAYS):
        second, (done, stalled) = solve(own, w, h, precision)
    assert done > 0 and stalled == 0 and first == second


# a batch: the lanes' launches are in the report, and one lane at a time has them
def test_batch_report(own):
    print("case: resident launches of a batch", flush=True)
    images = [own.upload(dm.generate_image(64 + 8 * i, 48, 6, 77 + i)) for i in range(4)]
    with dm.tuned(resident_polls=ALWAYS):
        out = own.gpb_batch(images, precision=dm.PREC_FP32)
    torch.cuda.synchronize()
    done, stalled = own.resident_report()
    assert done > 0 and stalled == 0 and len(out) == 4
