"""srx_draw_noalloc (every scratch buffer in one fixed per-GPU region, no allocation) through the
C ABI: byte for byte what srx_draw produces, on two calls in a row, the second smaller; a draw
that does not fit is refused without touching the targets."""
import numpy as np
import pytest

from salviarenderer_amd import api as A
from salviarenderer_amd import scenes as S

from helpers import Target, draw_colored

pytestmark = pytest.mark.gpu


def frame(lib, noalloc, **kw):
    r = lib.renderer()
    f = S.setup_plain(r, **kw)
    f.draw = (lambda: r.draw_noalloc(0, f.n_tris)) if noalloc else f.draw
    f.render()
    r.flush()
    out = {"color": f.color.read().copy(), "ds": f.ds.read().copy()}
    if f.resolved is not None:
        out["resolved"] = f.resolved.read().copy()
    return r, f, out


def same(a, b):
    for k in b:
        d = int((a[k] != b[k]).sum())
        assert d == 0, f"{k} differs in {d} bytes"


def test_noalloc_equals_draw_twice_second_smaller(hip_lib):
    big = dict(width=512, height=512, n_tris=2000)
    small = dict(width=256, height=192, n_tris=600, samples=4, seed=7)
    want_big = frame(hip_lib, False, **big)[2]
    want_small = frame(hip_lib, False, **small)[2]
    # one renderer per scene, calls back to back on the same GPU region
    got_big = frame(hip_lib, True, **big)[2]
    got_small = frame(hip_lib, True, **small)[2]
    same(got_big, want_big)
    same(got_small, want_small)
    # and on one renderer: the region keeps the last call's contents, the next call must not care
    r = hip_lib.renderer()
    f1 = S.setup_plain(r, **big)
    r.clear_color(f1.color, (0.0, 0.0, 0.0, 0.0))
    r.clear_depth_stencil(f1.ds, A.CLEAR_DEPTH | A.CLEAR_STENCIL, 1.0, 0)
    r.draw_noalloc(0, f1.n_tris)
    r.flush()
    same({"color": f1.color.read(), "ds": f1.ds.read()}, want_big)


def test_noalloc_refuses_what_does_not_fit(hip_lib):
    r = hip_lib.renderer()
    f = S.setup_plain(r, width=1024, height=1024, n_tris=400_000)
    r.clear_color(f.color, (0.25, 0.5, 0.75, 1.0))
    r.clear_depth_stencil(f.ds, A.CLEAR_DEPTH | A.CLEAR_STENCIL, 1.0, 0)
    r.flush()
    before = (f.color.read().copy(), f.ds.read().copy())
    with pytest.raises(A.SrxError) as e:
        r.draw_noalloc(0, f.n_tris)
    assert e.value.code == A.OUT_OF_MEMORY
    r.flush()
    assert np.array_equal(f.color.read(), before[0]) and np.array_equal(f.ds.read(), before[1])
    # the renderer keeps working, with and without the region
    small = S.setup_plain(r, width=128, height=128, n_tris=64)
    small.draw = lambda: r.draw_noalloc(0, small.n_tris)
    small.render()
    r.flush()
    got = small.color.read().copy()
    small.draw = lambda: r.draw(0, small.n_tris)
    small.render()
    r.flush()
    assert np.array_equal(got, small.color.read())


def test_noalloc_blends_on_a_large_target(hip_lib):
    """60,000 blended triangles on 262,144 GPU tiles take 52 of the region's 64 MiB: what a tile takes besides
    the triangles' 800 bytes has to stay below 40."""
    n, side = 60_000, 8191
    rng = np.random.default_rng(2)
    pos = np.concatenate([rng.uniform(-1, 1, (n, 1, 2)) + rng.uniform(-1e-3, 1e-3, (n, 3, 2)), rng.uniform(0.1, 0.9, (n, 3, 1)),
                          np.ones((n, 3, 1))], -1)
    col = rng.uniform(0.2, 1, (3 * n, 4))
    out = []
    for noalloc in (True, False):
        r = hip_lib.renderer()
        if noalloc:
            r.draw = r.draw_noalloc
        t = Target(r, side, side)
        t.clear((0.1, 0.2, 0.3, 0.4))
        keep = draw_colored(r, pos.reshape(-1, 4), col, blend=A.BLEND_ON)
        out.append(t.color.read().copy())
        del keep
    assert np.array_equal(*out) and len(np.unique(out[0][::7, ::7].reshape(-1, 4), axis=0)) > 1


@pytest.mark.parametrize("blend", [A.BLEND_OFF, A.BLEND_ON], ids=["opaque", "blend"])
@pytest.mark.parametrize("n,side", [(5000, 40), (200, 300)], ids=["long_lists", "spread"])
def test_noalloc_long_lists_and_blending(hip_lib, n, side, blend):
    """Lists that are split (opaque) or sorted in several partitions (blended), and ordinary ones."""
    rng = np.random.default_rng(n)
    pos = np.concatenate([rng.uniform(-0.6, 0.6, (n, 1, 2)) + rng.uniform(-0.3, 0.3, (n, 3, 2)), rng.uniform(0.1, 0.9, (n, 3, 1)),
                          np.ones((n, 3, 1))], -1).reshape(-1, 4)
    col = rng.uniform(0.0, 1, (3 * n, 4))
    for samples in (1, 4):
        out = []
        for noalloc in (True, False):
            r = hip_lib.renderer()
            if noalloc:
                r.draw = r.draw_noalloc
            t = Target(r, side, side, samples)
            t.clear((0.1, 0.2, 0.3, 0.4))
            keep = draw_colored(r, pos, col, blend=blend)
            out.append({"color": t.color.read().copy(), "ds": t.ds.read().copy()})
            del keep
        same(*out)
