"""Inputs rendered on the device (G-buffer fill, RSM fill and mip chain)
against the host producer in csrc/inputs (the same raster rules), and a
frame lit from device-rendered inputs against the same frame from host
inputs.

Depth, coverage, flux and depth/depth^2 are bit-identical (the same FP64
raster and FP32 shading in the same order).  Packed normals use atan2 (and,
in the mip chain, sin / cos of the unpacked angle), whose last-ulp results
differ between the host and device math libraries: a value may land on the
other side of an integer truncation, so a few normals may differ by one
unit; the same holds for sRGB albedo through pow.
"""
import numpy as np
import pytest
import torch

from canon import rel_l2
from conftest import announce, frame_inputs

pytestmark = pytest.mark.gpu


def _device(fi):
    from dynamicradiancevolume_amd.pipeline import DeviceFrame

    return DeviceFrame(fi)


def _renderer(fi):
    from dynamicradiancevolume_amd.pipeline import Renderer

    return Renderer(fi.workload.config())


def _off_by_one(a, b, max_frac, max_units=1):
    d = np.abs(a.astype(np.int64) - b.astype(np.int64))
    assert d.max() <= max_units, d.max()
    assert (d > 0).mean() <= max_frac, (d > 0).mean()


def _normals_close(a, b, max_frac, max_units):
    # packed (angle, z): the angle wraps at +-pi (32767 and -32768 are neighbours)
    d = a.astype(np.int64) - b.astype(np.int64)
    d[..., 0] = (d[..., 0] + 32768) % 65536 - 32768
    d = np.abs(d)
    assert d.max() <= max_units, d.max()
    assert (d > 0).sum() <= max(2, max_frac * d.size), (d > 0).sum()


@pytest.mark.parametrize("name", ["cornell_256", "boxes_1080p"])
def test_gbuffer_matches_host_producer(name):
    fi = frame_inputs(name)
    announce(f"device G-buffer {name}")
    r = _renderer(fi)
    df = _device(fi)
    r.render_gbuffer(df.scene(), fi.view_proj)
    depth, nrm, alb = r.read_gbuffer()
    np.testing.assert_array_equal(depth.view(np.uint32), fi.depth.view(np.uint32))
    _normals_close(nrm, fi.gnormal, 1e-4, 1)
    _off_by_one(alb, fi.galbedo, 1e-4)


@pytest.mark.parametrize("name", ["cornell_256", "boxes_1080p"])
def test_rsm_chain_matches_host_producer(name):
    fi = frame_inputs(name)
    announce(f"device RSM {name}")
    r = _renderer(fi)
    df = _device(fi)
    r.render_rsm(df.scene(), fi.light)
    res = int(fi.light.rsm_render_resolution)
    for level, (flux, nrm, dls) in enumerate(fi.rsm_levels):
        gf, gn, gd = r.read_rsm(level, res)
        # Flux and depth/depth^2 (and their 2x2 sums and means) are exact.
        np.testing.assert_array_equal(gf, flux)
        np.testing.assert_array_equal(gd, dls)
        # A mip normal is the repacked mean of four unpacked children, so
        # last-ulp sin / cos / atan2 differences reach it more often (0.3 %
        # of the 128^2 level of boxes_1080p) and compound over levels.
        if level == 0:
            _normals_close(gn, nrm, 1e-4, 1)
        else:
            _normals_close(gn, nrm, 2e-2, 4)


# Less than, just, and more than the five levels of one launch; three launches.
@pytest.mark.parametrize("res", [8, 16, 32, 128, 2048])
def test_rsm_mip_launches_match_host_producer(res):
    from dataclasses import replace

    from dynamicradiancevolume_amd.workloads import CORNELL_256

    fi = frame_inputs("cornell_256", light=replace(CORNELL_256.light, rsm_resolution=res))
    announce(f"device RSM mips {res}")
    cfg = fi.workload.config()
    from dynamicradiancevolume_amd.pipeline import Renderer

    r = Renderer(cfg)
    df = _device(fi)
    r.render_rsm(df.scene(), fi.light)
    assert len(fi.rsm_levels) == res.bit_length()
    for level, (flux, nrm, dls) in enumerate(fi.rsm_levels):
        gf, gn, gd = r.read_rsm(level, res)
        np.testing.assert_array_equal(gf, flux)
        np.testing.assert_array_equal(gd, dls)
        _normals_close(gn, nrm, *((1e-4, 1) if level == 0 else (2e-2, 4)))


def test_frame_from_device_inputs_matches_host_inputs():
    from dynamicradiancevolume_amd.pipeline import entries_sh

    fi = frame_inputs("cornell_256")
    announce("frame from device-rendered inputs")
    df = _device(fi)
    r = _renderer(fi)
    r.render_frame(df)
    _, live = r.cache_count()
    e0 = r.read_caches(live)
    out0 = df.out.clone()
    # the same frame with both inputs rendered on the device
    r2 = _renderer(fi)
    w = fi.workload
    r2.set_frame(fi.frame())
    r2.update_volume(w.eye, fi.bbox[:3], fi.bbox[3:])
    r2.voxelize_scene(df.positions, len(fi.positions), adaption_factor=w.adaption_factor)
    gb = r2.render_gbuffer(df.scene(), fi.view_proj)
    rsm = r2.render_rsm(df.scene(), fi.light)
    r2.allocate_caches(gb)
    r2.light_caches_rsm(rsm, fi.light)
    out1 = torch.zeros_like(df.out)
    r2.apply_caches(gb, out1)
    _, live2 = r2.cache_count()
    e1 = r2.read_caches(live2)
    assert live2 == live
    o0 = np.lexsort(e0[:, :3].view(np.uint32).T)
    o1 = np.lexsort(e1[:, :3].view(np.uint32).T)
    np.testing.assert_array_equal(e0[o0, :3], e1[o1, :3])
    assert rel_l2(entries_sh(e1[o1], w.sh_bands), entries_sh(e0[o0], w.sh_bands)) <= 1e-4
    assert rel_l2(out1.cpu().numpy(), out0.cpu().numpy()) <= 1e-4


def _raster_scene(kind, n, w, h):
    """Triangles [n, 3, 3] under clip = (x, y, 0.5, z): near plane at z = 0.5,
    pixel (x / z + 1) / 2 * w."""
    rng = np.random.default_rng(n * 7919 + w)
    size = {"mesh": 0.05, "near": 1.5, "wide": 0.5, "ties": 0.3}[kind]
    z = rng.uniform(0.6, 20.0, (n, 1))
    if kind == "near":
        z = rng.uniform(-1.0, 2.5, (n, 3))  # vertices before, on and behind the near plane
        z[::7, 0] = 0.5
    pos = np.empty((n, 3, 3))
    pos[:, :, :2] = rng.uniform(-1.2, 1.2, (n, 1, 2)) + rng.uniform(-size, size, (n, 3, 2))
    pos[:, :, 2] = z if kind == "near" else z + rng.uniform(0, 0.3, (n, 3))
    pos[:, :, :2] *= np.maximum(pos[:, :, 2:], 0.25)
    if kind == "ties":  # equal depths: the lowest index wins
        pos[n // 2:] = pos[:n - n // 2][::-1]
    pos[1] = pos[1, 0]  # no area
    return np.ascontiguousarray(pos.astype(np.float32))


# Windows on both sides of the tiled raster's least (384 tiles of 16x16), whole
# and ragged tiles; triangles below and above the sizes at which one thread, a
# wave or the workgroup takes them (24 and 4096 pixels) and past the 64 tiles
# that the lists take; 6000 of some 23 tiles exceed the lists' capacity
# (4 n + 65536 pairs).
@pytest.mark.parametrize("kind,n,w,h", [
    ("mesh", 1, 512, 256), ("mesh", 4000, 401, 300), ("mesh", 4000, 100, 37), ("near", 700, 401, 300),
    ("near", 300, 130, 130), ("wide", 2, 1025, 481), ("wide", 6000, 400, 300), ("wide", 900, 255, 255),
    ("ties", 1025, 512, 192), ("ties", 1025, 64, 64),
])
def test_raster_paths_match_host_producer(kind, n, w, h):
    from dynamicradiancevolume_amd import _abi
    from dynamicradiancevolume_amd.pipeline import Renderer

    announce(f"raster {kind} {n} {w}x{h}")
    pos = _raster_scene(kind, max(n, 2), w, h)[:n]
    # The colour is the index, at the centres of the 8-bit sRGB steps.
    code = np.stack([np.arange(n) % 251 + 1, np.arange(n) // 251 % 251 + 1, np.full(n, 7)], 1) / 255.0
    albedo = np.where(code <= 0.04045, code / 12.92, ((code + 0.055) / 1.055) ** 2.4).astype(np.float32)
    normals = np.tile(np.float32([0.0, 0.0, 1.0]), (n, 1))
    vp = np.float32([1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 0, 0.5, 0, 0, 1, 0])
    depth = np.empty((h, w), np.float32)
    gn = np.empty((h, w, 2), np.int16)
    ga = np.empty((h, w, 3), np.uint8)
    _abi.load_inputs().drvin_raster_gbuffer(pos.ctypes.data, albedo.ctypes.data, normals.ctypes.data, n,
                                            vp.ctypes.data, w, h, depth.ctypes.data, gn.ctypes.data, ga.ctypes.data,
                                            0)
    cfg = frame_inputs("cornell_256").workload.config()
    cfg.width, cfg.height = w, h
    r = Renderer(cfg)
    dev = [torch.from_numpy(x).cuda() for x in (pos, albedo, normals)]
    scene = _abi.DrvScene(*(x.data_ptr() for x in dev), n)
    for _ in range(2):
        r.render_gbuffer(scene, vp)
        got = r.read_gbuffer()
        np.testing.assert_array_equal(got[0].view(np.uint32), depth.view(np.uint32))
        np.testing.assert_array_equal(got[2], ga)


# Triangles past the room of the tiled raster: 90000 of some 55 tiles (more pairs
# than 4 n + 2^22), 40000 of more than 64 tiles at 3840x2160 (33140 records that
# all tiles look at), and 70000 cut by the near plane (65536 records of pieces).
# The first of each kind find room, the others are drawn before the tiles; equal
# depths of both halves go to the lowest index.
@pytest.mark.parametrize("kind,n,w,h", [("lists", 90000, 800, 600), ("wide", 40000, 3840, 2160), ("cut", 70000, 400, 300)])
def test_raster_of_triangles_without_room_matches_host_producer(kind, n, w, h):
    from dynamicradiancevolume_amd import _abi
    from dynamicradiancevolume_amd.pipeline import Renderer

    announce(f"raster without room {kind} {n} {w}x{h}")
    rng = np.random.default_rng(n)
    side = {"lists": 106, "wide": 160, "cut": 6}[kind]  # pixels of a triangle's box
    pos = np.empty((n, 3, 3))
    corner = rng.uniform(-1.0, 0.9, (n, 1, 2))
    pos[:, :, :2] = corner + np.float64([[0, 0], [2, 0], [0, 2]]) * side / [w, h]
    pos[:, :, 2] = rng.uniform(0.6, 20.0, (n, 1)) + rng.uniform(0.0, 0.3, (n, 3))
    if kind == "cut":
        pos[:, :, 2] = [0.55, 0.53, 0.45]  # one vertex behind z = 0.5
        pos[::2, 1, 2] = 0.46  # or two
    pos[n // 2:] = pos[:n - n // 2][::-1]
    pos[:, :, :2] *= pos[:, :, 2:]
    pos = np.ascontiguousarray(pos.astype(np.float32))
    i = np.arange(n)
    code = np.stack([i % 251 + 1, i // 251 % 251 + 1, i // 63001 + 7], 1) / 255.0  # as above
    albedo = np.where(code <= 0.04045, code / 12.92, ((code + 0.055) / 1.055) ** 2.4).astype(np.float32)
    normals = np.tile(np.float32([0.0, 0.0, 1.0]), (n, 1))
    vp = np.float32([1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 0, 0.5, 0, 0, 1, 0])
    depth = np.empty((h, w), np.float32)
    gn = np.empty((h, w, 2), np.int16)
    ga = np.empty((h, w, 3), np.uint8)
    _abi.load_inputs().drvin_raster_gbuffer(pos.ctypes.data, albedo.ctypes.data, normals.ctypes.data, n,
                                            vp.ctypes.data, w, h, depth.ctypes.data, gn.ctypes.data, ga.ctypes.data,
                                            0)
    cfg = frame_inputs("cornell_256").workload.config()
    cfg.width, cfg.height = w, h
    r = Renderer(cfg)
    dev = [torch.from_numpy(x).cuda() for x in (pos, albedo, normals)]
    scene = _abi.DrvScene(*(x.data_ptr() for x in dev), n)
    for _ in range(2):
        r.render_gbuffer(scene, vp)
        got = r.read_gbuffer()
        np.testing.assert_array_equal(got[0].view(np.uint32), depth.view(np.uint32))
        np.testing.assert_array_equal(got[2], ga)
