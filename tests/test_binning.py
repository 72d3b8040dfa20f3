"""Binning of single draws at the sizes where it can go wrong, on the HIP library against the oracle, byte
for byte: primitive counts around the 256 of a workgroup, triangles from far below a pixel to beyond
the target in one draw (emitted by the lane that set them up or spread over the workgroup), record
lists that fill a tile's LDS sort or need several windows of it, and first draws whose records
outgrow the buffers."""
import numpy as np
import pytest

from salviarenderer_amd import api as A

from helpers import Target, draw_colored, screen_to_clip


def mixed(n, w, h, seed):
    """n triangles with centres over (and beyond) the target and sizes log-uniform from 0.01 pixels to twice it."""
    rng = np.random.default_rng(seed)
    c = rng.uniform(-0.1, 1.1, (n, 1, 2)) * (w, h)
    xy = c + rng.normal(0, 1, (n, 3, 2)) * np.exp(rng.uniform(np.log(0.01), np.log(2.0 * max(w, h)), (n, 1, 1)))
    x, y = screen_to_clip(xy[..., 0], xy[..., 1], w, h)
    pos = np.stack([x, y, rng.uniform(0.05, 0.95, (n, 3)), np.ones((n, 3))], -1).reshape(-1, 4)
    return pos, rng.uniform(0, 1, (3 * n, 4))


def render(lib, tris, w, h, samples, blend, draws=1):
    r = lib.renderer()
    t = Target(r, w, h, samples)
    t.clear((0.1, 0.2, 0.3, 0.4))
    keep = [draw_colored(r, *tris, blend=blend) for _ in range(draws)]
    out = t.color.read().copy(), t.ds.read().copy()
    del keep
    return out


def same(hip_lib, cpu_lib, *args, **kw):
    h, c = render(hip_lib, *args, **kw), render(cpu_lib, *args, **kw)
    assert np.array_equal(h[1], c[1]) and np.array_equal(h[0], c[0])


@pytest.mark.gpu
@pytest.mark.parametrize("blend", [A.BLEND_OFF, A.BLEND_ON], ids=["opaque", "blend"])
@pytest.mark.parametrize("n", [1, 3, 255, 256, 257, 1025])
def test_mixed_sizes(hip_lib, cpu_lib, n, blend):
    for w, h, samples in ((333, 130, 1), (64, 64, 2), (1030, 517, 4)):
        same(hip_lib, cpu_lib, mixed(n, w, h, 50 + n), w, h, samples, blend)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2047, 2048, 2049, 7000])
def test_long_lists(hip_lib, cpu_lib, n):
    """Every triangle lies on the same few tiles."""
    rng = np.random.default_rng(n)
    pos = np.concatenate([rng.uniform(-1.5, 1.5, (3 * n, 2)), rng.uniform(0.05, 0.95, (3 * n, 1)), np.ones((3 * n, 1))], 1)
    for blend in (A.BLEND_OFF, A.BLEND_ON):
        same(hip_lib, cpu_lib, (pos, rng.uniform(0, 1, (3 * n, 4))), 20, 18, 1, blend)


@pytest.mark.gpu
@pytest.mark.parametrize("ids", ["dense", "clusters", "sparse", "few_high"])
def test_long_lists_in_primitive_order(hip_lib, cpu_lib, ids):
    """Blended lists of 2,100 to 30,000 records on the same four tiles, their primitives consecutive, in clusters far
    apart, spread over many that draw nothing, or all near the end (their leading bits agree)."""
    n = {"dense": 30000, "clusters": 400000, "sparse": 400000, "few_high": 300001}[ids]
    on = np.zeros(n, bool)
    if ids == "dense":
        on[:] = True
    elif ids == "clusters":
        on[:3000] = on[131072 - 1500: 131072 + 1500] = on[-2500:] = True
    elif ids == "sparse":
        on[::37] = True
    else:
        on[-2100:] = True
    rng = np.random.default_rng(n)
    pos = np.zeros((n, 3, 4), np.float32)  # off: no area
    pos[..., 3] = 1
    pos[on, :, :2] = rng.uniform(-1.5, 1.5, (on.sum(), 3, 2))
    pos[on, :, 2] = rng.uniform(0.05, 0.95, (on.sum(), 3))
    col = rng.uniform(0, 1, (3 * n, 4)).astype(np.float32) * (1, 1, 1, 1e-3)  # so faint that every layer tells
    out = []
    for lib in (hip_lib, cpu_lib):
        r = lib.renderer()
        t = Target(r, 20, 18, 1, A.PF_RGBA32F)
        t.clear((0.1, 0.2, 0.3, 0.4))
        keep = draw_colored(r, pos.reshape(-1, 4), col, blend=A.BLEND_ON, depth_func=A.CMP_ALWAYS)
        out.append(t.color.read().copy())
        del keep
    assert np.array_equal(*out)

@pytest.mark.gpu
@pytest.mark.parametrize("blend", [A.BLEND_OFF, A.BLEND_ON], ids=["opaque", "blend"])
def test_records_outgrow_the_buffers(hip_lib, cpu_lib, blend):
    """The first draw of a renderer emits more records than its buffers hold and is repeated; the second fits."""
    rng = np.random.default_rng(3)
    n = 700
    pos = np.concatenate([rng.uniform(-1, 1, (3 * n, 2)), rng.uniform(0.05, 0.95, (3 * n, 1)), np.ones((3 * n, 1))], 1)
    for draws in (1, 2):
        same(hip_lib, cpu_lib, (pos, rng.uniform(0, 1, (3 * n, 4))), 512, 512, 1, blend, draws=draws)


@pytest.mark.gpu
@pytest.mark.parametrize("samples", [1, 4])
@pytest.mark.parametrize("n", [63, 64, 65, 1023, 1025, 2049, 5000])
def test_split_and_culled_tiles(hip_lib, cpu_lib, n, samples):
    """Opaque lists around the lengths where a tile is split and where depth culling begins, of triangles over
    several tiles and of triangles inside one, for every depth order and for a depth-only pass."""
    rng = np.random.default_rng(n)
    w, h = 40, 24
    for size in (2.0, 0.05):
        c = rng.uniform(-0.7, 0.7, (n, 1, 2)) if size > 1 else rng.uniform(0.05, 0.55, (n, 1, 2)) * (1, -1)
        xy = c + rng.uniform(-1, 1, (n, 3, 2)) * size
        pos = np.concatenate([xy, rng.uniform(0.02, 0.98, (n, 3, 1)), np.ones((n, 3, 1))], -1).reshape(-1, 4)
        col = rng.uniform(0, 1, (3 * n, 4))
        for func, depth in ((A.CMP_LESS, 1.0), (A.CMP_GREATER_EQUAL, 0.0), (A.CMP_LESS_EQUAL, 0.5)):
            out = []
            for lib in (hip_lib, cpu_lib):
                r = lib.renderer()
                t = Target(r, w, h, samples)
                t.clear((0.1, 0.2, 0.3, 0.4), depth)
                keep = [draw_colored(r, pos, col, depth_func=func)]
                r.set_render_targets([], t.ds)  # the same triangles nearer: depth only
                keep.append(draw_colored(r, pos * (1, 1, 0.9, 1), col, depth_func=func))
                out.append((t.color.read().copy(), t.ds.read().copy()))
                del keep
            assert np.array_equal(out[0][1], out[1][1]) and np.array_equal(out[0][0], out[1][0]), (size, func)


@pytest.mark.gpu
@pytest.mark.parametrize("blend", [A.BLEND_OFF, A.BLEND_ON], ids=["opaque", "blend"])
def test_more_records_than_32_bits_count(hip_lib, blend):
    """16,400 triangles over each of 262,144 GPU tiles are 4,299,161,600 records: the draw is refused, its targets
    keep what they held, and the renderer draws on."""
    n, side = 16400, 8191
    r = hip_lib.renderer()
    t = Target(r, side, side)
    t.clear((0.2, 0.4, 0.6, 0.8))
    pos = np.tile(np.array([[-1, -1, 0.5, 1], [3, -1, 0.5, 1], [-1, 3, 0.5, 1]], np.float32), (n, 1))
    col = np.ones((3 * n, 4), np.float32)
    with pytest.raises(A.SrxError) as e:
        draw_colored(r, pos, col, blend=blend)
    assert e.value.code == A.OUT_OF_MEMORY
    assert (t.color.read().reshape(-1, 4) == (51, 102, 153, 204)).all()
    small = [Target(r, 40, 30)]
    small[0].clear()
    keep = draw_colored(r, pos[:3], col[:3], blend=blend)
    assert (small[0].color.read() == 255).all()
    del keep
