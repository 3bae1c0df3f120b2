"""Kernels at the sizes where their tiles, chunks and dispatch rules end,
against the CPU oracle (bit for bit) or an FP64 reference."""
import ctypes

import numpy as np
import pytest
import torch

import damascene_amd as dm
from damascene_amd import autograd as AG
from damascene_amd._lib import check, lib
from oracle import grad_ref as G
from oracle import pyoracle as O

pytestmark = pytest.mark.gpu


def host(t):
    return t.cpu().numpy()


def bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


# spectral Pb: 64 x 4 pixel blocks, eight vectors staged at a time, taken in pairs
@pytest.mark.parametrize("w,h,nvec", [(32, 32, 2), (64, 36, 9), (65, 37, 10), (129, 33, 17), (33, 41, 32)])
def test_spectral_pb_tiles(ctx, w, h, nvec):
    print(f"case: spectral Pb {w}x{h}, {nvec} vectors", flush=True)
    r = np.random.RandomState(w + nvec)
    vecs = r.rand(nvec, h, w).astype(np.float32)
    vals = np.sort(r.rand(nvec)).astype(np.float32) + 1e-4
    got = host(ctx.spectral_pb(vals, ctx.upload(vecs)))[:, :w * h]
    assert np.array_equal(bits(got), bits(O.spectral_pb(vals, vecs, w, h).reshape(8, -1)))


# the differentiable pair: the same blocks forward, 32 x 8 pixel blocks and
# eight vectors a chunk in the eigenvector gradient
@pytest.mark.parametrize("w,h,nvec", [(32, 32, 2), (65, 37, 9), (64, 40, 10), (97, 33, 16)])
def test_spb_combine_tiles(ctx, w, h, nvec):
    print(f"case: spectral Pb + combine gradients {w}x{h}, {nvec} vectors", flush=True)
    r = np.random.RandomState(7 * w + nvec)
    n = w * h
    cues = [r.rand(24, n).astype(np.float32) for _ in range(4)]
    vecs = r.rand(nvec, h, w).astype(np.float32)
    params = np.concatenate([r.rand(12) * 0.02, [0.0139], r.rand(nvec) * 3 + 1]).astype(np.float32)
    grad = r.randn(h, w).astype(np.float32)
    op = AG.SpbCombine(ctx, w, h, [ctx.upload(c) for c in cues])
    p = ctx.upload(params).requires_grad_(True)
    v = ctx.upload(vecs).requires_grad_(True)
    pre = op(p, v)
    pre.backward(ctx.upload(grad))
    C = G.cue_planes(*cues, w, h)
    p64 = torch.as_tensor(params, dtype=torch.float64).requires_grad_(True)
    v64 = torch.as_tensor(vecs, dtype=torch.float64).requires_grad_(True)
    all64, R64 = G.parts64(p64, v64, C, w, h)
    (all64.max(0).values * torch.as_tensor(grad, dtype=torch.float64)).sum().backward()
    # FP32: a response is a chain of 49 fused multiply-adds of values below 1
    # with weights of unit L1 norm (error below 49 * 2^-24 = 2.9e-6), a plane
    # sums 12 + nvec of them
    top = all64.detach().max(0).values
    assert float((pre.detach().cpu().double() - top).abs().max()) < 1e-5 * float(all64.detach().abs().max())
    # the gradients agree where FP32 cannot route them elsewhere: no near-tie
    # of the maximising orientation or of a response's sign in the pixel's
    # 7 x 7 window (bounds as in test_backward_against_fp64)
    gv, gv64 = host(v.grad), v64.grad.numpy()
    s = np.sort(all64.detach().numpy(), axis=0)[-2:]
    tie = s[1] - s[0] < 1e-5 * s.max()
    ostar = all64.detach().numpy().argmax(axis=0)
    rstar = np.take_along_axis(np.abs(R64.detach().numpy()), ostar[None, None], axis=1)[:, 0]
    for i in range(1, nvec):
        amb = tie | (rstar[i - 1] < 1e-5)
        near = np.zeros_like(amb)
        for dy in range(-3, 4):
            for dx in range(-3, 4):
                near |= np.roll(np.roll(amb, dy, 0), dx, 1)
        assert np.abs(gv[i] - gv64[i])[~near].max() < 1e-4 * np.abs(gv64).max(), f"vector {i}"
    assert np.all(gv[0] == 0)
    # parameters: FP64 block sums of FP32 terms; an ambiguous pixel may move
    # its own term
    gp, gp64 = host(p.grad), p64.grad.numpy()
    assert np.abs(gp - gp64).max() < (1e-5 + 2.0 * tie.sum() / n) * np.abs(gp64).max()
    assert gp[13] == 0


# integral images: strips of 64 columns and bands of 16 rows of the rotated
# frames (whose sides these sizes put on and off those multiples), and frames
# wider than 2,048 columns
@pytest.mark.parametrize("w,h,ntex", [(32, 32, 32), (68, 36, 64), (69, 133, 32), (2200, 40, 32), (40, 2100, 64)])
def test_integral_strips(ctx, w, h, ntex):
    print(f"case: integral strips {w}x{h}, {ntex} textons", flush=True)
    r = np.random.RandomState(w + h)
    L, a, b = (ctx.upload(r.rand(h, w).astype(np.float32)) for _ in range(3))
    tex = ctx.upload(r.randint(0, ntex, (h, w)).astype(np.int32))
    choice = dm.TEXTON64 if ntex == 64 else dm.TEXTON32
    raws = []
    for one_write in (0, 1):
        with dm.tuned(integral_pass=one_write):
            raws.append(host(ctx.local_cues(L, a, b, tex, raw=True, texton_choice=choice)[1]))
    assert np.array_equal(bits(raws[0]), bits(raws[1]))


# gradients in 16 x 16 patches (32 textons and the L/a/b bins) and 16 x 8 ones
# (64 textons), smoothing in tiles of 128 x 32 outputs: partial tiles on both
# sides, against the oracle
@pytest.mark.parametrize("w,h,ntex", [(32, 33, 32), (129, 47, 32), (127, 65, 64), (144, 64, 64)])
def test_local_cues_tiles(ctx, w, h, ntex):
    print(f"case: local cues {w}x{h}, {ntex} textons", flush=True)
    r = np.random.RandomState(3 * w + h)
    L, a, b = (np.clip(r.rand(h, w) * 1.1 - 0.05, 0, 1).astype(np.float32) for _ in range(3))
    tex = r.randint(0, ntex, (h, w)).astype(np.int32)
    tex[h // 3:, w // 2:] = 1  # flat regions: empty bins on both sides of a split
    a[:, w // 2:] = 0.5
    got = ctx.local_cues(*[ctx.upload(v) for v in (L, a, b)], ctx.upload(tex),
                         texton_choice=dm.TEXTON64 if ntex == 64 else dm.TEXTON32)
    for c, ref in zip(got, O.local_cues(L, a, b, tex, ntex=ntex)):
        assert np.array_equal(bits(host(c)), bits(np.asarray(ref).reshape(24, -1)[:, :w * h]))


# k-means: 256-pixel chunks, up to 768 looping blocks, 32 clusters per pass of
# the matrix cores; ties and empty clusters
@pytest.mark.parametrize("w,h,k", [(7, 5, 32), (16, 16, 64), (257, 3, 32), (515, 397, 64), (900, 700, 32)])
def test_kmeans_chunks(ctx, w, h, k):
    print(f"case: k-means {w}x{h}, {k} clusters", flush=True)
    r = np.random.RandomState(w + k)
    resp = (r.randn(34, h, w) * 0.1).astype(np.float32)
    resp[:, : h // 2, : w // 3] = 0.0  # equal pixels: equal distances
    resp[33] = 0.0
    labels, it = ctx.kmeans(ctx.upload(resp), k=k)
    ref, rit = O.kmeans(resp, k=k)
    assert it == rit
    np.testing.assert_array_equal(host(labels), ref)
    # a pixel whose squared distance to every centroid passes 1e7 gets no label
    resp[5, h - 1, w - 1] = 30000.0 if w * h > 1000 else 0.0
    far, _ = ctx.kmeans(ctx.upload(resp), k=k, max_iter=1)
    assert int((far < 0).sum()) == (1 if w * h > 1000 else 0) and (w * h <= 1000 or far[h - 1, w - 1] == -1)


# filter bank: blocks of 64 x 4 pixels (one row per wave), and of 64 x 8 from
# 2,048 blocks on
@pytest.mark.parametrize("w,h", [(1, 1), (64, 4), (65, 9), (130, 7), (1025, 481)])
def test_texton_bank_tiles(ctx, w, h):
    print(f"case: filter bank {w}x{h}", flush=True)
    grey = np.random.RandomState(w + h).rand(h, w).astype(np.float32)
    assert np.array_equal(bits(host(ctx.texton_responses(ctx.upload(grey)))), bits(O.texton_responses(grey)))


# affinities: 64 x 4 pixel blocks; waves without a clipped window within reach
# take the compiled walks, the others the table (another one below 11 pixels a
# side); then L_sym
@pytest.mark.parametrize("w,h", [(6, 6), (7, 10), (11, 11), (10, 40), (23, 21), (84, 24), (150, 45)])
def test_affinity_windows(ctx, w, h):
    print(f"case: affinity {w}x{h}", flush=True)
    r = np.random.RandomState(w * h)
    pb = np.where(r.rand(h, w) < 0.4, r.rand(h, w), 0.0).astype(np.float32)
    pb[r.rand(h, w) < 0.05] = -0.3  # below 0: as nothing crossed
    m = ctx.intervene(ctx.upload(pb))
    ref = O.intervene(pb)
    n = w * h
    got = host(m)
    assert np.array_equal(bits(got[:, :n]), bits(np.asarray(ref).reshape(81, -1)[:, :n]))
    assert np.all(got[:, n:] == 0)
    d, rs = ctx.convert_matrix(w, h, m)
    d64 = np.zeros(n)
    for k, (dy, dx) in enumerate((y, x) for y in range(-5, 6) for x in range(-5, 6) if y * y + x * x <= 25):
        col = np.arange(n) + dy * w + dx
        d64 += np.where((col >= 0) & (col < n), got[k, :n], 0.0)
    assert np.allclose(host(d).ravel(), d64, rtol=81 * 2.0 ** -24, atol=0)
    assert np.allclose(host(rs).ravel(), 1 / np.sqrt(d64), rtol=82 * 2.0 ** -24, atol=0)
    L = host(m)[:, :n]
    assert np.allclose(L[40], (d64 - got[40, :n]) / d64, rtol=0, atol=82 * 2.0 ** -24)


# plain Lanczos steps in one launch: 1,024 rows per block, partial sums per 256
# rows; with one poll allowed the launch gives up and two kernels per step run
@pytest.mark.parametrize("w,h", [(32, 32), (41, 25), (64, 48), (97, 83), (230, 57)])
def test_resident_lanczos_steps(ctx, w, h):
    print(f"case: plain Lanczos {w}x{h}", flush=True)
    y, x = np.mgrid[:h, :w]
    cell = (x // 13 + 2 * (y // 11)) % 4
    pb = (0.4 * ((np.diff(cell, axis=1, append=cell[:, -1:]) != 0) | (np.diff(cell, axis=0, append=cell[-1:]) != 0))
          + 0.02 * np.random.RandomState(w).rand(h, w)).astype(np.float32)
    out = []
    for polls in (0, 1 << 16, 1):
        with dm.tuned(resident_polls=polls, lanczos_max_iter=1500):
            try:
                vals, vecs, it = ctx.generalized_eigensolve(w, h, ctx.intervene(ctx.upload(pb)), nvec=5)
                out.append((bits(vals), bits(host(vecs)), it))
            except dm.DmscError as e:
                out.append(str(e))
    for got in out[1:]:
        assert type(got) is type(out[0])
        if isinstance(got, str):
            assert got == out[0]
        else:
            assert got[2] == out[0][2]
            np.testing.assert_array_equal(got[0], out[0][0])
            np.testing.assert_array_equal(got[1], out[0][1])
    assert not isinstance(out[0], str)


# block filter in one launch: tiles of 32 x 16 and 32 x 24 pixels by image size,
# matrices that couple the ends of image rows, and the restart after a stall
@pytest.mark.parametrize("w,h", [(31, 2100), (40, 1031), (1025, 64), (261, 257), (330, 390), (500, 375)])
def test_resident_block_filter(ctx, w, h):
    print(f"case: block filter {w}x{h}", flush=True)
    r = np.random.RandomState(w)
    n = w * h
    y, x = np.mgrid[:h, :w]
    cell = ((3 * x // w) + 3 * (2 * y // h)).ravel()
    m = np.zeros((81, dm.pitch_in_floats(n)), np.float32)
    for k, (dy, dx) in enumerate((y, x) for y in range(-5, 6) for x in range(-5, 6) if y * y + x * x <= 25):
        off = dy * w + dx
        if off >= 0:
            v = np.zeros(n, np.float32)
            v[:n - off] = np.where(cell[:n - off] == cell[off:], 1.0, 0.02) * (0.9 + 0.1 * r.rand(n - off))
            m[k, :n] = v
            m[80 - k, off:n] = v[:n - off]
    out = []
    for polls in (0, 1 << 14, 1):
        with dm.tuned(resident_polls=polls):
            vals, vecs, products = ctx.generalized_eigensolve(w, h, ctx.upload(m), nvec=4, tol=1e-2,
                                                              precision=dm.PREC_MIXED)
            out.append((bits(vals), bits(host(vecs)), products))
    for got in out[1:]:
        assert got[2] == out[0][2]
        np.testing.assert_array_equal(got[0], out[0][0])
        np.testing.assert_array_equal(got[1], out[0][1])


# a context's first affinities inside a captured graph, replayed on new inputs
@pytest.mark.parametrize("w,h", [(9, 12), (70, 45)])
def test_affinities_in_a_graph(w, h):
    print(f"case: captured affinities {w}x{h}", flush=True)
    s = torch.cuda.Stream()
    c = dm.Context(stream=s)
    pb = torch.zeros(h, w, device="cuda")
    g = torch.cuda.CUDAGraph()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(g, stream=s):
        m = c.intervene(pb)
    for seed in range(3):
        pb.copy_(torch.from_numpy(np.random.RandomState(seed).rand(h, w).astype(np.float32)))
        torch.cuda.synchronize()
        g.replay()
        eager = c.intervene(pb)
        torch.cuda.synchronize()
        np.testing.assert_array_equal(bits(host(m)), bits(host(eager)))
    c.close()


# thinning: windows of 64 x 64 pixels for 32 x 32, two iterations per launch
@pytest.mark.parametrize("w,h,fill", [(6, 6, 1.0), (32, 33, 1.0), (65, 40, 0.6), (130, 97, 0.85), (96, 128, 1.0)])
def test_thinning_windows(ctx, w, h, fill):
    print(f"case: thinning {w}x{h}, {fill}", flush=True)
    r = np.random.RandomState(w)
    nm = (r.rand(h, w) < fill).astype(np.float32)  # up to a solid block: many iterations
    g = (0.1 + 0.9 * r.rand(h, w)).astype(np.float32)
    got, thin, it = ctx.postprocess(ctx.upload(g), ctx.upload(nm))
    rg, rthin, rit = O.postprocess(g, nm)
    assert it == rit
    assert np.array_equal(host(thin) == host(thin).min(), rthin == rthin.min())
    np.testing.assert_allclose(host(thin), rthin, rtol=0, atol=1e-6)
    np.testing.assert_allclose(host(got), rg, rtol=0, atol=1e-6)


# a context made while another stream is captured in the global mode (as
# torch captures), and used once the capture has ended
def test_context_made_during_a_capture(ctx):
    print("case: context made during a capture", flush=True)
    other = torch.cuda.Stream()
    s = torch.cuda.Stream()
    x = torch.zeros(1000, device="cuda")
    pb = torch.from_numpy(np.random.RandomState(5).rand(40, 33).astype(np.float32)).cuda()
    g = torch.cuda.CUDAGraph()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(g, stream=s):
        x.add_(1.0)
        c = dm.Context(stream=other)
        x.add_(1.0)
    for turn in range(1, 4):
        g.replay()
        torch.cuda.synchronize()
        assert float(x.sum()) == 2000.0 * turn
        m = c.intervene(pb)
        c.synchronize()
        np.testing.assert_array_equal(bits(host(m)), bits(host(ctx.intervene(pb))))
    c.close()


# matrices whose rows are padded: up to 4,096 columns past the image cleared by
# its own blocks, more by a launch of their own
@pytest.mark.parametrize("w,h,pad", [(6, 6, 4), (33, 21, 4096), (33, 21, 4100), (640, 480, 307200)])
def test_affinity_padding(ctx, w, h, pad):
    n = w * h
    pitch = n + pad
    print(f"case: affinity {w}x{h}, pitch {pitch}", flush=True)
    pb = ctx.upload(np.random.RandomState(w).rand(h, w).astype(np.float32))
    ref = ctx.intervene(pb)

    def call(m):
        check(lib().dmsc_intervene(ctx.handle, w, h, pb.data_ptr(), m.data_ptr(), m.shape[1], 0.1))

    m = torch.full((81, pitch), 7.0, device="cuda")
    call(m)
    assert torch.equal(m[:, :n], ref[:, :n]) and not bool(m[:, n:].any())

    def us(m, reps=10):
        call(m)
        e = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        e[0].record()
        for _ in range(reps):
            call(m)
        e[1].record()
        torch.cuda.synchronize()
        return e[0].elapsed_time(e[1]) / reps * 1e3

    if n > 100000:
        tight, wide = us(torch.empty_like(ref)), us(m)
        print(f"{tight:.0f} us at pitch {ref.shape[1]}, {wide:.0f} us at {pitch}", flush=True)
        # twice the bytes written; ten times leaves room for any launch effect
        assert wide < 10 * tight


# both precisions take exact distances: the same labels, nothing recomputed
@pytest.mark.parametrize("k", [32, 64])
def test_kmeans_recomputes_nothing(ctx, k):
    print(f"case: k-means re-checks, {k} clusters", flush=True)
    resp = ctx.upload((np.random.RandomState(k).randn(34, 61, 83) * 0.1).astype(np.float32))
    out = []
    for precision in (dm.PREC_FP32, dm.PREC_MIXED):
        labels, it = ctx.kmeans(resp, k=k, precision=precision)
        n = ctypes.c_int(-1)
        check(lib().dmsc_kmeans_rechecks(ctx.handle, ctypes.byref(n)))
        assert n.value == 0
        out.append((host(labels).tobytes(), it))
    assert out[0] == out[1]
