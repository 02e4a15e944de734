"""Brute-force RSM reference (bruteforcersm.frag) on the GPU against the
oracle, and the end-to-end error of the cache path against it.

Tolerance: relative L2 1e-4 over the image (the device uses hardware
reciprocal square root / reciprocal and exp2 / log2 for pow, the oracle libm;
sums run in different VAL orders).
"""
import numpy as np
import pytest
import torch

from canon import rel_l2
from conftest import announce, frame_inputs

pytestmark = pytest.mark.gpu


def _setup(fi):
    from dynamicradiancevolume_amd.pipeline import DeviceFrame, Renderer

    r = Renderer(fi.workload.config())
    df = DeviceFrame(fi)
    r.set_frame(fi.frame())
    return r, df


@pytest.mark.parametrize("diffuse_only", [True, False])
def test_bruteforce_cornell_matches_oracle(diffuse_only):
    from oracle import orc

    fi = frame_inputs("cornell_256")
    announce(f"brute force cornell diffuse_only={diffuse_only}")
    r, df = _setup(fi)
    W, H = fi.workload.width, fi.workload.height
    rng = np.random.default_rng(4)
    rm = rng.integers(80, 256, (H, W, 2)).astype(np.uint8)
    rm[..., 1] = rng.integers(0, 256, (H, W))
    rm_dev = torch.from_numpy(rm).cuda() if not diffuse_only else None
    out = torch.zeros((H, W, 3), device="cuda")
    r.bruteforce_rsm(df.gbuffer(), df.rsm(), fi.light, out, diffuse_only, rm_dev)
    got = out.cpu().numpy().reshape(-1, 3)
    ref = orc.bruteforce_rsm(fi, diffuse_only, rm if not diffuse_only else None)
    assert rel_l2(got, ref) <= 1e-4
    # accumulate adds a second light's worth
    r.bruteforce_rsm(df.gbuffer(), df.rsm(), fi.light, out, diffuse_only, rm_dev, accumulate=True)
    assert rel_l2(out.cpu().numpy().reshape(-1, 3), 2 * ref) <= 1e-4


def test_bruteforce_boxes_subset_matches_oracle():
    from oracle import orc

    fi = frame_inputs("boxes_1080p")
    announce("brute force boxes_1080p (pixel subset)")
    r, df = _setup(fi)
    W, H = fi.workload.width, fi.workload.height
    out = torch.zeros((H, W, 3), device="cuda")
    r.bruteforce_rsm(df.gbuffer(), df.rsm(), fi.light, out, True)
    px = np.random.default_rng(7).choice(W * H, 3000, replace=False).astype(np.uint32)
    got = out.cpu().numpy().reshape(-1, 3)[px]
    ref = orc.bruteforce_rsm(fi, True, None, px)
    assert rel_l2(got, ref) <= 1e-4


@pytest.mark.parametrize("diffuse_only", [True, False])
@pytest.mark.parametrize("width,height,read,wide", [(9, 7, 8, 0), (250, 131, 16, 1), (65, 63, 1, 0), (8, 8, 2, 0)])
def test_bruteforce_tile_and_group_edges_match_oracle(width, height, read, wide, diffuse_only):
    """Pixel tiles cut by the window's edge, VAL counts from one (fewer than a
    group of four) to 2:1, every wave's share of the groups empty or not."""
    from dataclasses import replace

    from dynamicradiancevolume_amd import workloads as W
    from oracle import orc

    light = replace(W.BOXES_1080P.light, rsm_resolution=read, rsm_read_lod=0, rsm_wide=wide, indirect_shadow_lod=0)
    fi = frame_inputs("boxes_1080p", n_objects=60, tess=3, width=width, height=height, light=light)
    announce(f"brute force {width}x{height}, read level {read}, wide {wide}, diffuse_only={diffuse_only}")
    r, df = _setup(fi)
    out = torch.full((height, width, 3), 7.0, device="cuda")
    rm = None if diffuse_only else df.groughmetal
    r.bruteforce_rsm(df.gbuffer(), df.rsm(), fi.light, out, diffuse_only, rm)
    got = out.cpu().numpy().reshape(-1, 3)
    ref = orc.bruteforce_rsm(fi, diffuse_only, None if diffuse_only else fi.groughmetal)
    assert np.linalg.norm(ref) > 0 and rel_l2(got, ref) <= 1e-4
    assert np.all(got[fi.depth.reshape(-1) < 1e-5] == 0)


def _odd_frame(kind):
    """cornell_256 in a small window with VALs or pixels that leave the range
    of a float, or of the reciprocal of a fourth power of a distance."""
    from dataclasses import replace

    from dynamicradiancevolume_amd.workloads import CORNELL_256

    fi = frame_inputs("cornell_256", width=96, height=64,
                      light=replace(CORNELL_256.light, rsm_resolution=16, indirect_shadow_lod=0))
    flux, nrm, dls = (a.copy() for a in fi.read_level)
    if kind == "dark inf depth":  # one texel in each 2x2 square, three lit neighbours
        dls[::2, ::2] = np.float16(np.inf).view(dls.dtype)
        flux[::2, ::2] = 0
    elif kind == "lit inf depth":
        dls[5, 6] = np.float16(np.inf).view(dls.dtype)
    elif kind == "nan depth":
        dls[5, 6] = np.float16(np.nan).view(dls.dtype)
        flux[5, 6] = 0
    elif kind == "inf flux":
        flux[5, 6] = np.float16(np.inf).view(flux.dtype)
    elif kind == "far pixels":
        m = np.asarray(fi.inv_view_proj, np.float32).reshape(4, 4).copy()
        m[:3] *= 1e10
        fi = replace(fi, inv_view_proj=m.reshape(np.shape(fi.inv_view_proj)))
    return replace(fi, rsm_levels=[(flux, nrm, dls)] + list(fi.rsm_levels[1:]))


# An infinite distance gives no light (1 / (inf + inf)), a NaN one or infinite
# flux times a cosine of zero a NaN, as in the shader; a pixel 1e10 away gets
# light of 1e-20 of a near one's.  Masks may differ where a cosine is zero to
# rounding: in 1 of 1000 pixels.
@pytest.mark.parametrize("diffuse_only", [True, False])
@pytest.mark.parametrize("kind", ["dark inf depth", "lit inf depth", "nan depth", "inf flux", "far pixels"])
def test_bruteforce_beyond_the_range_matches_oracle(kind, diffuse_only):
    from oracle import orc

    fi = _odd_frame(kind)
    announce(f"brute force {kind}, diffuse_only={diffuse_only}")
    r, df = _setup(fi)
    r.bruteforce_rsm(df.gbuffer(), df.rsm(), fi.light, df.out, diffuse_only, None if diffuse_only else df.groughmetal)
    got = df.out.cpu().numpy().reshape(-1, 3)
    ref = orc.bruteforce_rsm(fi, diffuse_only, None if diffuse_only else fi.groughmetal)
    same = np.isfinite(got) == np.isfinite(ref)
    assert same.mean() >= 0.999, same.mean()
    ok = np.isfinite(got) & np.isfinite(ref)
    if kind in ("nan depth", "inf flux"):
        assert not ok[fi.depth.reshape(-1) >= 1e-5].all()
    else:
        assert ok.all() and np.abs(ref).max() > 0
    assert rel_l2(got[ok], ref[ok]) <= 1e-4


@pytest.mark.parametrize("sh_bands", [1, 2])
def test_cache_path_vs_bruteforce_end_to_end(sh_bands):
    """The unshadowed cache path (SH interpolation of the diffuse irradiance)
    against the per-pixel ground truth: the method's own approximation error
    (cache spacing + SH truncation), measured, with a loose bound."""
    fi = frame_inputs("cornell_256")
    announce(f"cache path vs brute force, end to end, SH{sh_bands}")
    from dynamicradiancevolume_amd.pipeline import DeviceFrame, Renderer

    r = Renderer(fi.workload.with_(indirect_shadow=0, sh_bands=sh_bands).config())
    df = DeviceFrame(fi)
    r.render_frame(df)
    cache_rgb = df.out.clone()
    bf = torch.zeros_like(cache_rgb)
    r.bruteforce_rsm(df.gbuffer(), df.rsm(), fi.light, bf, True)
    lit = torch.from_numpy(fi.depth >= 1e-5).cuda()
    err = rel_l2(cache_rgb[lit].cpu().numpy(), bf[lit].cpu().numpy())
    print(f"[measure] cornell_256 SH{sh_bands} unshadowed cache path vs brute force: rel L2 {err:.4f}")
    assert err <= 0.5
