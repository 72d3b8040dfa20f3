"""Texture samples of RGBA8 wrap/linear samplers on the HIP library against the oracle, byte for byte, where
the inline taps begin and end: sides that are and are not powers of two, one texel and 4096, levels of a
non-square chain, magnification and up to 16 probes, and coordinates below zero and past the range that
the taps take."""
import numpy as np
import pytest

from salviarenderer_amd import api as A

from helpers import Target


LAMBERT = (A.VS_WVP_NORMAL_UV, np.eye(4, dtype=np.float32).ravel(),
           A.PS_LAMBERT_TEX, np.array([0.0, 0.3, 0.9, 0.0], np.float32))


def render(lib, tw, th, mip, aniso, offset, scale, blend, samples, shaders=LAMBERT):
    vs, vs_consts, ps, ps_consts = shaders
    r = lib.renderer()
    t = Target(r, 150, 90, samples)
    t.clear((0.1, 0.2, 0.3, 0.4))
    rng = np.random.default_rng(tw * 7 + th)
    n = 24
    v = np.zeros((3 * n, 8), np.float32)
    v[:, 0:2] = rng.uniform(-1.3, 1.3, (3 * n, 2))
    v[:, 2] = rng.uniform(0.1, 0.9, 3 * n)
    v[:, 3:6] = (0.2, 0.1, 1.0)
    v[:, 6:8] = offset + rng.uniform(-1, 1, (3 * n, 2)) * (scale, scale * 0.2)
    vb = r.create_buffer_from(v)
    layout = r.create_input_layout([("POSITION", 0, A.FMT_R32G32B32_FLOAT, 0, 0),
                                    ("NORMAL", 0, A.FMT_R32G32B32_FLOAT, 0, 12),
                                    ("TEXCOORD", 0, A.FMT_R32G32_FLOAT, 0, 24)], vs)
    r.set_input_layout(layout)
    r.set_vertex_buffers(0, [vb], [32])
    r.set_primitive_topology(A.TOPOLOGY_TRIANGLE_LIST)
    r.set_vertex_shader(vs, vs_consts)
    r.set_pixel_shader(ps, ps_consts)
    tex = r.create_tex2d(tw, th, 1, A.PF_RGBA8)
    tex.surface(0).write(rng.integers(0, 256, (th, tw, 4), dtype=np.uint8))
    tex.gen_mipmap(A.FILTER_LINEAR, True)
    sd = A.default_sampler_desc(lib)
    sd.min_filter = sd.mag_filter = A.FILTER_LINEAR
    sd.mip_filter = mip
    sd.max_anisotropy = aniso
    samp = r.create_sampler(sd, tex)
    r.set_ps_sampler(0, samp)
    r.set_blend_shader(blend)
    rd = A.default_raster_desc(lib)
    rd.cull_mode = A.CULL_NONE
    rs = r.create_raster_state(rd)
    r.set_rasterizer_state(rs)
    dss = r.create_depth_stencil_state(A.default_depth_stencil_desc(lib))
    r.set_depth_stencil_state(dss, 0)
    r.draw(0, n)
    r.flush()
    return t.color.read().copy()


@pytest.mark.gpu
@pytest.mark.parametrize("blend", [A.BLEND_OFF, A.BLEND_ON], ids=["opaque", "blend"])
@pytest.mark.parametrize("mip,aniso", [(A.FILTER_LINEAR, 1), (A.FILTER_ANISOTROPIC, 3), (A.FILTER_ANISOTROPIC, 16)],
                         ids=["trilinear", "aniso3", "aniso16"])
@pytest.mark.parametrize("tw,th", [(1, 1), (2, 64), (64, 64), (48, 64), (61, 37), (4096, 8)])
def test_taps(hip_lib, cpu_lib, tw, th, mip, aniso, blend):
    for offset, scale, samples in ((0, 0.02, 1), (0, 1.0, 4), (-3, 40.0, 2), (65535.5, 4.0, 1), (-65536, 6.0, 4), (1e9, 1e9, 1)):
        args = tw, th, mip, aniso, offset, scale, blend, samples
        assert np.array_equal(render(hip_lib, *args), render(cpu_lib, *args)), args


@pytest.mark.gpu
@pytest.mark.parametrize("blend", [A.BLEND_OFF, A.BLEND_ON], ids=["opaque", "blend"])
@pytest.mark.parametrize("ps", [A.PS_LAMBERT_TEX, A.PS_TEX_CPP, A.PS_BOX, A.PS_CUP], ids=["lambert", "tex", "box", "cup"])
def test_taps_of_four_attributes(hip_lib, cpu_lib, ps, blend):
    """The shaders' samples behind a vertex shader of four attributes, where only PS_CUP's are inline."""
    vs_consts = np.concatenate([np.eye(4).ravel(), (0, 0, -1, 1), (1, 1, -1, 1)]).astype(np.float32)
    ps_consts = {A.PS_LAMBERT_TEX: LAMBERT[3], A.PS_CUP: np.linspace(0.1, 0.9, 12, dtype=np.float32)}.get(ps)
    for (mip, aniso), (tw, th), samples in (((A.FILTER_LINEAR, 1), (64, 32), 1), ((A.FILTER_ANISOTROPIC, 8), (64, 64), 4),
                                            ((A.FILTER_LINEAR, 1), (48, 20), 2), ((A.FILTER_ANISOTROPIC, 8), (61, 37), 1)):
        args = tw, th, mip, aniso, 0, 1.0, blend, samples, (A.VS_CUP, vs_consts, ps, ps_consts)
        assert np.array_equal(render(hip_lib, *args), render(cpu_lib, *args)), args[:4]
