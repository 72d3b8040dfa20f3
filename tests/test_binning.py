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


def stack(n, seed, clipped=False):
    """n triangles over the whole target (and well beyond), at random depths; clipped: some cross the near plane."""
    rng = np.random.default_rng(seed)
    xy = np.array([[-1, -1], [3, -1], [-1, 3]]) * rng.uniform(1, 1.3, (n, 1, 2))
    z = rng.uniform(0.05, 0.95, (n, 3, 1))
    if clipped:
        z[::3, 0] = -0.2
    pos = np.concatenate([xy, z, np.ones((n, 3, 1))], -1).reshape(-1, 4)
    return pos, rng.uniform(0, 1, (3 * n, 4))


# on 36 GPU tiles with room for 65,536 records at first, in buffers of 98,304: the lists alone are formed again
# (79,200 records), or the records are emitted again into larger buffers (108,000)
GROWTH = pytest.mark.parametrize("n", [2200, 3000], ids=["requeued", "emitted_again"])


@pytest.mark.gpu
@GROWTH
@pytest.mark.parametrize("blend", [A.BLEND_OFF, A.BLEND_ON], ids=["opaque", "blend"])
def test_growth_with_split_tiles(hip_lib, cpu_lib, n, blend):
    """Every tile's list is long enough to be split."""
    for samples in (1, 2):
        same(hip_lib, cpu_lib, stack(n, n), 96, 96, samples, blend)


@pytest.mark.gpu
@GROWTH
@pytest.mark.parametrize("blend", [A.BLEND_OFF, A.BLEND_ON], ids=["opaque", "blend"])
def test_growth_under_queries(hip_lib, cpu_lib, n, blend):
    """The repeat counts no primitive, clipped or not, and no pixel a second time."""
    out = []
    for lib in (hip_lib, cpu_lib):
        r = lib.renderer()
        t = Target(r, 96, 96)
        t.clear()
        q, qi = r.create_query(A.QUERY_PIPELINE_STATISTICS), r.create_query(A.QUERY_INTERNAL_STATISTICS)
        r.begin(q)
        r.begin(qi)
        keep = draw_colored(r, *stack(n, n, clipped=True), blend=blend)
        r.end(q)
        r.end(qi)
        st, sti = r.get_data(q)[1], r.get_data(qi)[1]
        out.append([st.ia_primitives, st.cinvocations, st.cprimitives, st.ps_invocations, sti.backend_input_pixels,
                    t.color.read().tobytes(), t.ds.read().tobytes()])
        del keep
    assert out[0] == out[1] and out[0][2] > 0


@pytest.mark.gpu
@GROWTH
@pytest.mark.parametrize("blend", [A.BLEND_OFF, A.BLEND_ON], ids=["opaque", "blend"])
def test_growth_with_a_sasl_shader(hip_lib, cpu_lib, n, blend):
    out = []
    for lib in (hip_lib, cpu_lib):
        r = lib.renderer()
        t = Target(r, 96, 96)
        t.clear((0.1, 0.2, 0.3, 0.4))
        code = lib.compile_shader("float4 half_main(float4 c : TEXCOORD0) : COLOR { return c * 0.5f; }")
        r.set_pixel_shader_code(code)
        keep = draw_colored(r, *stack(n, n + 1), blend=blend)
        out.append((t.color.read().copy(), t.ds.read().copy()))
        del keep, code
    assert np.array_equal(out[0][1], out[1][1]) and np.array_equal(out[0][0], out[1][0])


@pytest.mark.gpu
def test_frames_of_large_and_small_draws(hip_lib, cpu_lib):
    """Draws of 3,000 large triangles and then more, smaller ones than the estimate remembers, three
    frames: the buffers are the last large draw's while the small ones draw, and the other way round."""
    big, small, tiny = stack(3000, 1), mixed(1500, 96, 96, 2), mixed(3, 96, 96, 3)
    out = []
    for lib in (hip_lib, cpu_lib):
        r = lib.renderer()
        t = Target(r, 96, 96, 2)
        images = []
        for k in range(3):
            t.clear((0.1, 0.2, 0.3, 0.4))
            keep = [draw_colored(r, *big)]
            keep += [draw_colored(r, *d, blend=b) for d in (small, tiny) for b in (A.BLEND_ON, A.BLEND_OFF) for _ in range(3 + k)]
            images.append((t.color.read().copy(), t.ds.read().copy()))
            del keep
        out.append(images)
    for h, c in zip(*out):
        assert np.array_equal(h[1], c[1]) and np.array_equal(h[0], c[0])


@pytest.mark.gpu
def test_draws_that_are_not_waited_for(hip_lib, cpu_lib):
    """40 small draws in a row, issued without a wait, each with another texture and every third with another filter:
    the sampler table's staging is written again only when the last copy of it has run."""
    out = []
    for lib in (hip_lib, cpu_lib):
        r = lib.renderer()
        t = Target(r, 64, 64)
        t.clear()
        rng = np.random.default_rng(4)
        v = np.zeros((120, 8), np.float32)
        v[:, 0:2] = rng.uniform(-1, 1, (120, 2))
        v[:, 2] = rng.uniform(0.1, 0.9, 120)
        v[:, 5] = 1
        v[:, 6:8] = rng.uniform(0, 2, (120, 2))
        vb = r.create_buffer_from(v)
        layout = r.create_input_layout([("POSITION", 0, A.FMT_R32G32B32_FLOAT, 0, 0), ("NORMAL", 0, A.FMT_R32G32B32_FLOAT, 0, 12),
                                        ("TEXCOORD", 0, A.FMT_R32G32_FLOAT, 0, 24)], A.VS_WVP_NORMAL_UV)
        r.set_input_layout(layout)
        r.set_primitive_topology(A.TOPOLOGY_TRIANGLE_LIST)
        r.set_vertex_shader(A.VS_WVP_NORMAL_UV, np.eye(4, dtype=np.float32).ravel())
        r.set_pixel_shader(A.PS_LAMBERT_TEX, np.array([0.0, 0.3, 0.9, 0.0], np.float32))
        rd = A.default_raster_desc(lib)
        rd.cull_mode = A.CULL_NONE
        rs = r.create_raster_state(rd)
        r.set_rasterizer_state(rs)
        dss = r.create_depth_stencil_state(A.default_depth_stencil_desc(lib))
        r.set_depth_stencil_state(dss, 0)
        samplers = []
        for k in range(40):
            tex = r.create_tex2d(8, 8, 1, A.PF_RGBA8)
            tex.surface(0).write(rng.integers(0, 256, (8, 8, 4), dtype=np.uint8))
            tex.gen_mipmap(A.FILTER_LINEAR, True)
            sd = A.default_sampler_desc(lib)
            sd.min_filter = sd.mag_filter = A.FILTER_POINT if k % 3 == 0 else A.FILTER_LINEAR
            samplers.append((r.create_sampler(sd, tex), tex))
        r.flush()
        for k, (s, _) in enumerate(samplers):
            r.set_ps_sampler(0, s)
            r.set_blend_shader(A.BLEND_ON if k % 5 == 0 else A.BLEND_OFF)
            r.set_vertex_buffers(0, [vb], [32], [96 * k])
            r.draw(0, 1)
        r.flush()
        out.append((t.color.read().copy(), t.ds.read().copy()))
    assert np.array_equal(out[0][1], out[1][1]) and np.array_equal(out[0][0], out[1][0])
