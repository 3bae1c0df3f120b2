"""Which solves run in launches whose blocks wait for each other: the results
are the same either way, so the context's report tells."""
import ctypes

import numpy as np
import pytest
import torch

import damascene_amd as dm
from damascene_amd._lib import check, lib

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


# a device that stays busy: after a launch has given up the next solves do
# without, one, then two
@pytest.mark.parametrize("w,h,precision", [(230, 57, dm.PREC_FP32), (320, 240, dm.PREC_MIXED)])
def test_given_up_is_remembered(own, w, h, precision):
    print(f"case: remembered {w}x{h} precision {precision}", flush=True)
    with dm.tuned(resident_polls=1):
        tries = [solve(own, w, h, precision) for _ in range(6)]
        print([t[1] for t in tries], flush=True)
    assert all(t[0] == tries[0][0] for t in tries)
    stalled = [t[1][1] for t in tries]
    assert precision == dm.PREC_MIXED or sum(stalled) > 0  # a thousand waits or more of one poll each
    for i, t in enumerate(tries[:-1]):
        if t[1][1]:
            assert tries[i + 1][1] == (0, 0)


# a batch: the lanes' launches are in the report, and one lane at a time has them
def test_batch_report(own):
    print("case: resident launches of a batch", flush=True)
    images = [own.upload(dm.generate_image(64 + 8 * i, 48, 6, 77 + i)) for i in range(4)]
    with dm.tuned(resident_polls=ALWAYS):
        out = own.gpb_batch(images, precision=dm.PREC_FP32)
    torch.cuda.synchronize()
    done, stalled = own.resident_report()
    assert done > 0 and stalled == 0 and len(out) == 4


@pytest.fixture
def untuned():
    check(lib().dmsc_autotune_clear())
    yield
    check(lib().dmsc_autotune_clear())


# a tuned size keeps the launch, whichever of the two-kernel shapes was the
# faster one, and with it the results
@pytest.mark.parametrize("w,h", [(32, 32), (64, 48), (160, 120), (230, 57), (481, 321)])
def test_tuned_plain_size_keeps_the_launch(own, untuned, w, h):
    with dm.tuned(resident_polls=ALWAYS):
        before, _ = solve(own, w, h, dm.PREC_FP32)
        m = own.intervene(torch.rand(h, w, device="cuda"))
        best, trials = own.autotune_eigensolver(w, h, m, precision=dm.PREC_FP32, steps=200)
        print(f"case: tuned {w}x{h}: best {best}", flush=True)
        after, (done, stalled) = solve(own, w, h, dm.PREC_FP32)
    assert done > 0 and stalled == 0 and after == before


def product_us(c, w, h, m, products=100):
    ms = ctypes.c_float()
    check(lib().dmsc_chebyshev_time_products(c.handle, w, h, m.data_ptr(), m.shape[1], products, ctypes.byref(ms)))
    return ms.value * 1e3


# the block filter's trials decide between the launch and the fastest tile: at
# wide tiles with few columns in use the tile may win
@pytest.mark.parametrize("w,h", [(320, 240), (481, 321), (33, 2100), (64, 1200)])
def test_tuned_filter_takes_the_faster_form(own, untuned, w, h):
    with dm.tuned(resident_polls=ALWAYS):
        before, _ = solve(own, w, h, dm.PREC_MIXED)
        m = own.intervene(torch.rand(h, w, device="cuda"))
        own.convert_matrix(w, h, m)
        count = own.resident_report()[0]
        launch = min(product_us(own, w, h, m) for _ in range(3))
        served = own.resident_report()[0] > count
        best, us = own.autotune_chebyshev(w, h, m, products=100)
        after, (done, stalled) = solve(own, w, h, dm.PREC_MIXED)
    print(f"case: filter {w}x{h}: launch {launch:.1f} us ({served}), tile {best} {us[best]:.1f} us, taken {done}",
          flush=True)
    assert served and stalled == 0 and after == before
    if launch < 0.8 * us[best]:
        assert done > 0
    if us[best] < 0.8 * launch:
        assert done == 0


# the measuring entry points run what a solve of the size runs
def test_timed_steps_are_the_solves(own, untuned):
    print("case: timed steps", flush=True)
    w, h = 481, 321
    ms = ctypes.c_float()
    for polls, launches in ((ALWAYS, True), (0, False)):
        with dm.tuned(resident_polls=polls):
            a = own.resident_report()[0]
            m = own.intervene(torch.rand(h, w, device="cuda"))
            check(lib().dmsc_lanczos_time_steps(own.handle, w, h, m.data_ptr(), m.shape[1], dm.PREC_FP32, 200,
                                                ctypes.byref(ms)))
            b = own.resident_report()[0]
            product_us(own, w, h, m)
            c = own.resident_report()[0]
        assert ms.value > 0 and (b > a) == launches and (c > b) == launches
