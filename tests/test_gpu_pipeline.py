"""Parity of the HIP pipeline (through the C ABI) against the CPU oracle.

Integer work (allocation: claimed cells and positions; voxels and mips) must
be bit-exact.  Floating-point results (SH coefficients, visibility, the apply
output) must be within relative L2 1e-4 of the FP32 oracle on the same inputs.
"""
import numpy as np
import pytest
import torch

from canon import canonical, rel_l2
from conftest import announce, frame_inputs

pytestmark = pytest.mark.gpu

SH_TOL = 1e-4      # relative L2 of SH coefficients vs the FP32 oracle
RGB_TOL = 1e-4     # relative L2 of the apply output
VIS_TOL = 1e-4     # max |visibility difference|


def _orc():
    from oracle import orc

    return orc


def _renderer(fi, **overrides):
    from dynamicradiancevolume_amd.pipeline import Renderer

    cfg = fi.workload.with_(**overrides).config() if overrides else fi.workload.config()
    return Renderer(cfg)


def _device(fi):
    from dynamicradiancevolume_amd.pipeline import DeviceFrame

    return DeviceFrame(fi)


def _assert_alloc_equal(r, fi, cfg, orc, capacity=None):
    vol = orc.update_volume(cfg, fi.workload.eye, fi.bbox[:3], fi.bbox[3:])
    count, cav, entries = orc.allocate(cfg, vol, fi.frame(), fi.depth)
    demanded, live = r.cache_count()
    assert demanded == count
    assert live == min(count, cfg.max_caches)
    g_entries = r.read_caches(live)
    g_cav = r.read_cav()
    cap = cfg.max_caches if capacity is None else capacity
    gc, gp, gph, gok = canonical(demanded, g_cav, g_entries, cap)
    oc, op, oph, ook = canonical(count, cav, entries, cap)
    assert gok and ook
    np.testing.assert_array_equal(gc, oc)
    if cap >= count:
        np.testing.assert_array_equal(gp, op)
        assert gph == oph
    return vol, count, cav, entries, g_entries, g_cav


@pytest.mark.parametrize("name", ["cornell_256", "boxes_1080p", "boxes_1080p_dense"])
def test_volume_ubo_matches_oracle(name):
    orc = _orc()
    fi = frame_inputs(name)
    announce(f"volume ubo {name}")
    r = _renderer(fi)
    cfg = fi.workload.config()
    r.update_volume(fi.workload.eye, fi.bbox[:3], fi.bbox[3:])
    v = r.volume()
    o = orc.update_volume(cfg, fi.workload.eye, fi.bbox[:3], fi.bbox[3:])
    assert bytes(v) == bytes(o)


@pytest.mark.parametrize("name", ["cornell_256", "boxes_1080p", "boxes_1080p_dense"])
def test_allocation_bit_exact(name):
    orc = _orc()
    fi = frame_inputs(name)
    df = _device(fi)
    announce(f"allocate {name}")
    r = _renderer(fi)
    r.set_frame(fi.frame())
    r.update_volume(fi.workload.eye, fi.bbox[:3], fi.bbox[3:])
    r.allocate_caches(df.gbuffer())
    _assert_alloc_equal(r, fi, fi.workload.config(), orc)


@pytest.mark.parametrize(
    "overrides",
    [
        dict(width=250, height=131),               # ragged tiles
        dict(transition_size=0.0),                 # no transition list
        dict(cav_cascades=1),                      # single cascade: clamped cells + phantoms
        dict(cav_cascades=2, cav_resolution=16),
        dict(cav_cascades=2, cav_resolution=20),   # bricks, 5^3 of them (not a power of two)
        dict(cav_cascades=3, cav_resolution=18),   # R % 4 != 0: rows of x, one cell per lane
    ],
)
def test_allocation_variants(overrides):
    orc = _orc()
    fi = frame_inputs("cornell_256", **{k: v for k, v in overrides.items() if k in ("width", "height")})
    cfg = fi.workload.with_(**overrides).config()
    df = _device(fi)
    announce(f"allocate cornell {overrides}")
    r = _renderer(fi, **overrides)
    r.set_frame(fi.frame())
    r.update_volume(fi.workload.eye, fi.bbox[:3], fi.bbox[3:])
    r.allocate_caches(df.gbuffer())
    _assert_alloc_equal(r, fi, cfg, orc)


# Blocks of 64 cells: fewer cells than one, bricks in Morton and in row order,
# rows that end inside a block, cascades that start inside one, and chunks of
# more blocks than a workgroup looks at together (1024; 240^3 x 4 has 844).
@pytest.mark.parametrize("cav,cascades", [(2, 1), (3, 4), (5, 3), (12, 4), (33, 4), (50, 2), (64, 3), (96, 4), (270, 4)])
def test_allocation_block_sizes(cav, cascades):
    orc = _orc()
    fi = frame_inputs("cornell_256")
    over = dict(cav_resolution=cav, cav_cascades=cascades, cascade0_world_size=0.6)
    cfg = fi.workload.with_(**over).config()
    df = _device(fi)
    announce(f"allocate {cav}^3 x {cascades}")
    r = _renderer(fi, **over)
    r.set_frame(fi.frame())
    r.update_volume(fi.workload.eye, fi.bbox[:3], fi.bbox[3:])
    for _ in range(2):  # the second call starts from the first one's flags and claims
        r.allocate_caches(df.gbuffer())
        _assert_alloc_equal(r, fi, cfg, orc)


def test_allocation_overflow_counts_and_clamps():
    """Capacity below the live count: demanded count is still exact, only
    `capacity` caches are stored, the claimed cell set is unchanged and apply
    reads caches past the capacity as zero."""
    orc = _orc()
    fi = frame_inputs("cornell_256")
    full = fi.workload.config()
    vol = orc.update_volume(full, fi.workload.eye, fi.bbox[:3], fi.bbox[3:])
    count, _, _ = orc.allocate(full, vol, fi.frame(), fi.depth)
    cap = count // 3
    cfg = fi.workload.with_(max_caches=cap).config()
    df = _device(fi)
    announce(f"overflow cap={cap} count={count}")
    r = _renderer(fi, max_caches=cap)
    r.set_frame(fi.frame())
    r.update_volume(fi.workload.eye, fi.bbox[:3], fi.bbox[3:])
    r.allocate_caches(df.gbuffer())
    demanded, live = r.cache_count()
    assert demanded == count and live == cap
    g_entries = r.read_caches(live)
    g_cav = r.read_cav()
    gc, gp, _, gok = canonical(demanded, g_cav, g_entries, cap)
    _, ocav, oentries = orc.allocate(full, vol, fi.frame(), fi.depth)
    oc, op, _, _ = canonical(count, ocav, oentries, count)
    assert gok
    np.testing.assert_array_equal(gc, oc)
    stored = gp[:, 0] != 0xFFFFFFFF
    assert stored.sum() <= cap
    np.testing.assert_array_equal(gp[stored], op[stored])
    # gather + apply still run; apply must match the oracle on the same state
    r.light_caches_rsm(df.rsm(), fi.light)
    r.apply_caches(df.gbuffer(), df.out)
    torch.cuda.synchronize()
    g_entries = r.read_caches(live)
    shc = orc.sh_constants()
    ref = orc.apply(cfg, vol, fi.frame(), shc, fi, g_cav, g_entries, live)
    assert rel_l2(df.out.cpu().numpy(), ref) < RGB_TOL


# Waves with cells at the volume's faces (a cascade that ends inside the view;
# one cell, whose pairs lie outside), three and more caches at a corner (fine
# cells), windows that end inside a wave's 8x8 pixels.
@pytest.mark.parametrize("cav,cascades,size,width,height,sh", [
    (1, 1, 12.0, 64, 48, 2), (1, 2, 8.0, 33, 17, 1), (4, 1, 9.0, 67, 41, 2), (16, 1, 8.0, 129, 70, 1),
    (64, 1, 10.0, 120, 64, 2), (120, 4, 1.0, 71, 9, 2),
])
def test_apply_cell_edges_match_oracle(cav, cascades, size, width, height, sh):
    orc = _orc()
    fi = frame_inputs("cornell_256", width=width, height=height)
    over = dict(cav_resolution=cav, cav_cascades=cascades, cascade0_world_size=size, sh_bands=sh)
    w = fi.workload.with_(**over)
    df = _device(fi)
    announce(f"apply {over} {width}x{height}")
    r = _renderer(fi, **over)
    r.set_frame(fi.frame())
    r.update_volume(w.eye, fi.bbox[:3], fi.bbox[3:])
    r.voxelize_scene(df.positions, len(fi.positions))
    r.allocate_caches(df.gbuffer())
    r.light_caches_rsm(df.rsm(), fi.light)
    r.apply_caches(df.gbuffer(), df.out)
    _, live = r.cache_count()
    vol = orc.update_volume(w.config(), w.eye, fi.bbox[:3], fi.bbox[3:])
    ref = orc.apply(w.config(), vol, fi.frame(), orc.sh_constants(), fi, r.read_cav(), r.read_caches(live), live)
    out = df.out.cpu().numpy()
    if cav == 1:  # the one cell's corners lie outside the volume: no pixel finds a cache but its own cell's
        assert np.abs(out - ref).max() <= RGB_TOL * max(1.0, np.abs(ref).max())
    else:
        assert np.abs(ref).max() > 0.0
        assert rel_l2(out, ref) < RGB_TOL


def test_cascades_of_unrelated_cell_sizes_match_oracle():
    """Four cascades whose cell sizes are neither powers of two nor multiples
    of each other, all of them in a tile's view: every pixel looks its own
    cascade up, in the allocation and in the apply."""
    orc = _orc()
    fi = frame_inputs("cornell_256", width=160, height=96)
    over = dict(cav_resolution=24, cav_cascades=4, cascade0_world_size=1.0, sh_bands=2)
    w = fi.workload.with_(**over)
    cfg = w.config()
    df = _device(fi)
    announce("cascades of unrelated cell sizes")
    r = _renderer(fi, **over)
    r.set_frame(fi.frame())
    r.update_volume(w.eye, fi.bbox[:3], fi.bbox[3:])
    v = r.volume()
    for c, half in enumerate((0.9, 2.3, 5.3, 9.7)):
        k = v.cascades[c]
        for i in range(3):
            k.min[i], k.max[i] = w.eye[i] - half, w.eye[i] + half
            k.decision_min[i], k.decision_max[i] = w.eye[i] - 0.8 * half, w.eye[i] + 0.8 * half
        k.world_voxel_size = 2.0 * half / 24
    r.set_volume(v)
    r.voxelize_scene(df.positions, len(fi.positions))
    r.allocate_caches(df.gbuffer())
    count, cav, entries = orc.allocate(cfg, v, fi.frame(), fi.depth)
    demanded, live = r.cache_count()
    assert demanded == count
    got, want = (canonical(count, *x, cfg.max_caches) for x in ((r.read_cav(), r.read_caches(live)), (cav, entries)))
    assert got[3] and want[3] and got[2] == want[2]
    np.testing.assert_array_equal(got[0], want[0])
    np.testing.assert_array_equal(got[1], want[1])
    r.light_caches_rsm(df.rsm(), fi.light)
    r.apply_caches(df.gbuffer(), df.out)
    ref = orc.apply(cfg, v, fi.frame(), orc.sh_constants(), fi, r.read_cav(), r.read_caches(live), live)
    assert np.abs(ref).max() > 0.0
    assert rel_l2(df.out.cpu().numpy(), ref) < RGB_TOL


# Pixels that unproject to cells past the 32-bit range along one axis, the
# others inside the volume, and to infinity: no cache is there to light them.
@pytest.mark.parametrize("cascades", [1, 4])
@pytest.mark.parametrize("far", ["x", "y", "z", "inf"])
def test_apply_of_pixels_beyond_the_integer_range_finds_no_cache(far, cascades):
    fi = frame_inputs("cornell_256", width=64, height=48)
    over = dict(cav_cascades=cascades, cascade0_world_size=8.0)
    w = fi.workload.with_(**over)
    df = _device(fi)
    announce(f"apply far along {far}, {cascades} cascades")
    r = _renderer(fi, **over)
    r.set_frame(fi.frame())
    r.update_volume(w.eye, fi.bbox[:3], fi.bbox[3:])
    r.voxelize_scene(df.positions, len(fi.positions))
    r.allocate_caches(df.gbuffer())
    r.light_caches_rsm(df.rsm(), fi.light)
    frame = fi.frame()
    rows = [[0.01, 0.01, 0.0, e] for e in w.eye] + [[0.0, 0.0, 0.0, 0.0 if far == "inf" else 1.0]]
    if far != "inf":
        rows["xyz".index(far)] = [1e30, 1e25, 0.0, 0.0]
    frame.inverse_view_projection[:] = [v for row in rows for v in row]
    r.set_frame(frame)
    df.out.fill_(7.0)
    r.apply_caches(df.gbuffer(), df.out)
    assert not df.out.cpu().numpy().any()
    r.set_frame(fi.frame())
    r.apply_caches(df.gbuffer(), df.out)
    assert df.out.cpu().numpy().any()


def test_allocation_reuses_address_volume_across_frames():
    """A renderer that allocates frame A, then frame B (a G-buffer with its
    upper half cleared and its lower half shifted), then A again holds the
    same claimed cells, positions, phantoms and counts as fresh renderers on
    B and on A: no claim of an earlier frame survives into the next."""
    from dataclasses import replace

    orc = _orc()
    fi = frame_inputs("cornell_256")
    cfg = fi.workload.config()
    h, w = cfg.height, cfg.width
    depth_b = fi.depth.reshape(h, w).copy()
    depth_b[: h // 2] = 0.0
    depth_b[h // 2:] = np.roll(depth_b[h // 2:], 7, axis=1)
    fi_b = replace(fi, depth=depth_b.reshape(fi.depth.shape))
    announce("allocate A, B, A on one renderer")
    r = _renderer(fi)
    r.set_frame(fi.frame())
    r.update_volume(fi.workload.eye, fi.bbox[:3], fi.bbox[3:])
    counts = []
    for f in (fi, fi_b, fi):
        df = _device(f)
        r.allocate_caches(df.gbuffer())
        torch.cuda.synchronize()
        _assert_alloc_equal(r, f, cfg, orc)
        counts.append(r.cache_count()[0])
    assert counts[1] < counts[0] == counts[2]  # B claims a different, smaller set
    r.close()


def test_allocation_empty_gbuffer():
    fi = frame_inputs("cornell_256")
    df = _device(fi)
    df.depth.zero_()
    announce("allocate empty gbuffer")
    r = _renderer(fi)
    r.set_frame(fi.frame())
    r.update_volume(fi.workload.eye, fi.bbox[:3], fi.bbox[3:])
    r.voxelize_scene(df.positions, len(fi.positions))
    r.allocate_caches(df.gbuffer())
    assert r.cache_count() == (0, 0)
    r.light_caches_rsm(df.rsm(), fi.light)
    df.out.fill_(7.0)
    r.apply_caches(df.gbuffer(), df.out)
    torch.cuda.synchronize()
    assert float(df.out.abs().max()) == 0.0
    assert not r.read_cav().any()


@pytest.mark.parametrize("name,adapt", [("cornell_256", 1.0), ("boxes_1080p", 1.0)])
def test_voxelization_bit_exact(name, adapt):
    orc = _orc()
    fi = frame_inputs(name)
    w = fi.workload
    df = _device(fi)
    announce(f"voxelize {name}")
    r = _renderer(fi)
    r.update_volume(w.eye, fi.bbox[:3], fi.bbox[3:])
    r.voxelize_scene(df.positions, len(fi.positions), adaption_factor=adapt)
    vol = orc.update_volume(w.config(), w.eye, fi.bbox[:3], fi.bbox[3:])
    target, mips = orc.voxelize(w.voxel_resolution, vol, fi.positions, adaption_factor=adapt)
    np.testing.assert_array_equal(r.read_voxels(-1), target)
    level = 0
    while (w.voxel_resolution >> level) >= 1:
        np.testing.assert_array_equal(r.read_voxels(level), orc.mip_level(mips, w.voxel_resolution, level),
                                      err_msg=f"mip level {level}")
        level += 1


# Volumes without a whole 16^3 brick, of one brick and of slabs of one, two and
# four bricks; one triangle (32 lanes share it), the smallest scene and one past
# the last that shares lanes (2^19 of them); a blend over old voxels.
@pytest.mark.parametrize("res,n_tri", [(2, 36), (8, 36), (16, 1), (32, 2176), (64, 8191), (128, 262145), (256, 2176)])
def test_voxelization_sizes_bit_exact(res, n_tri):
    orc = _orc()
    fi = frame_inputs("cornell_256")
    announce(f"voxelize {res} {n_tri}")
    rng = np.random.default_rng(res)
    src = fi.positions[np.arange(n_tri) % len(fi.positions)].reshape(n_tri, 3, 3)
    centre = src.mean(1, keepdims=True)
    # copies of the scene's triangles, smaller and moved beyond the first round
    k = (np.arange(n_tri) >= len(fi.positions))[:, None, None]
    pos = np.where(k, centre + 0.3 * (src - centre) + rng.uniform(-0.3, 0.3, (n_tri, 1, 3)), src)
    pos = np.ascontiguousarray(pos.reshape(n_tri, 9).astype(np.float32))
    moved = pos.copy()
    moved[:, 1::3] += 0.4
    r = _renderer(fi, voxel_resolution=res)
    w = fi.workload.with_(voxel_resolution=res)
    r.update_volume(w.eye, fi.bbox[:3], fi.bbox[3:])
    vol = orc.update_volume(w.config(), w.eye, fi.bbox[:3], fi.bbox[3:])
    mips = None
    for p, adapt in ((pos, 1.0), (moved, 0.3), (pos, 0.6)):
        dev = torch.from_numpy(p).cuda()
        r.voxelize_scene(dev, n_tri, adaption_factor=adapt)
        target, mips = orc.voxelize(res, vol, p, adaption_factor=adapt, previous=mips)
        np.testing.assert_array_equal(r.read_voxels(-1), target)
        for level in range(res.bit_length()):
            np.testing.assert_array_equal(r.read_voxels(level), orc.mip_level(mips, res, level),
                                          err_msg=f"mip level {level}")


@pytest.mark.parametrize("res", [16, 32, 256])
def test_gather_voxel_sizes_match_oracle(res):
    announce(f"gather voxels {res}")
    _gather_case("cornell_256", voxel_resolution=res)


def test_voxel_blend_partial_adaption():
    """Two frames: the second voxelizes a moved scene with AdaptionFactor 0.25,
    so texels move a quarter step towards the new target."""
    orc = _orc()
    fi = frame_inputs("cornell_256")
    w = fi.workload
    df = _device(fi)
    moved = fi.positions.copy()
    moved[:, 0::3] += 0.7
    moved_dev = torch.from_numpy(moved).cuda()
    world = (1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1, 0, 0, 0, 0, 1)
    announce("voxel blend 0.25")
    r = _renderer(fi)
    r.update_volume(w.eye, fi.bbox[:3], fi.bbox[3:])
    r.voxelize_scene(df.positions, len(fi.positions), adaption_factor=1.0)
    r.voxelize_scene(moved_dev, len(moved), world=world, adaption_factor=0.25)
    vol = orc.update_volume(w.config(), w.eye, fi.bbox[:3], fi.bbox[3:])
    _, mips = orc.voxelize(w.voxel_resolution, vol, fi.positions, adaption_factor=1.0)
    _, mips2 = orc.voxelize(w.voxel_resolution, vol, moved, adaption_factor=0.25, previous=mips)
    for level in range(3):
        np.testing.assert_array_equal(r.read_voxels(level), orc.mip_level(mips2, w.voxel_resolution, level))


@pytest.mark.parametrize("overlap", [False, True])
def test_voxelization_order_on_the_stream(overlap):
    """A whole frame, then the scene moved and voxelized again.  Without the
    voxel overlap the move is written on the stream after the frame and the
    voxelization sees it; with the overlap on (drv_set_voxel_overlap) the
    moved geometry is written before the frame's light pass, as the contract
    asks.  Either way the second voxelization equals the oracle's for the
    moved scene, and the frame after it lights the caches as a renderer
    without the overlap does."""
    orc = _orc()
    fi = frame_inputs("cornell_256")
    w = fi.workload
    df = _device(fi)
    moved = fi.positions.copy()
    moved[:, 0::3] += 0.7
    announce(f"voxelization order, overlap {overlap}")
    r = _renderer(fi)
    r.set_voxel_overlap(overlap)
    geometry = df.positions.clone()
    moved_dev = torch.from_numpy(moved).cuda()
    if overlap:
        # written before the frame's light pass
        geometry2 = moved_dev
        r.render_frame(df)
    else:
        geometry2 = geometry
        r.render_frame(df)
        geometry.copy_(moved_dev)  # on the renderer's stream, after the frame
    r.update_volume(w.eye, fi.bbox[:3], fi.bbox[3:])
    r.voxelize_scene(geometry2, len(moved), adaption_factor=1.0)
    vol = orc.update_volume(w.config(), w.eye, fi.bbox[:3], fi.bbox[3:])
    target, mips = orc.voxelize(w.voxel_resolution, vol, moved, adaption_factor=1.0)
    np.testing.assert_array_equal(r.read_voxels(-1), target)
    for level in range(3):
        np.testing.assert_array_equal(r.read_voxels(level), orc.mip_level(mips, w.voxel_resolution, level))
    # the next frame (its voxelization overlapping this one's tail when on)
    # against a renderer that never overlaps
    ref = _renderer(fi)
    for rr in (r, ref):
        rr.render_frame(df)
        rr.render_frame(df)
    torch.cuda.synchronize()
    live = r.cache_count()[1]
    assert live == ref.cache_count()[1]
    np.testing.assert_array_equal(r.read_caches(live), ref.read_caches(live))


def _gather_case(name, n_sub=None, **overrides):
    orc = _orc()
    fi = frame_inputs(name)
    w = fi.workload.with_(**overrides) if overrides else fi.workload
    cfg = w.config()
    df = _device(fi)
    r = _renderer(fi, **overrides)
    r.set_frame(fi.frame())
    r.update_volume(w.eye, fi.bbox[:3], fi.bbox[3:])
    r.voxelize_scene(df.positions, len(fi.positions), adaption_factor=w.adaption_factor)
    r.allocate_caches(df.gbuffer())
    _, live = r.cache_count()
    before = r.read_caches(live)
    r.light_caches_rsm(df.rsm(), fi.light)
    after = r.read_caches(live)
    vol = orc.update_volume(cfg, w.eye, fi.bbox[:3], fi.bbox[3:])
    _, mips = orc.voxelize(w.voxel_resolution, vol, fi.positions, adaption_factor=w.adaption_factor)
    ids = np.arange(live, dtype=np.uint32) if n_sub is None else np.linspace(0, live - 1, n_sub).astype(np.uint32)
    ref = before.copy()
    vis, _ = orc.gather_f32(cfg, vol, orc.sh_constants(), fi.light, fi, mips, ref, ids=ids,
                            want_visibility=bool(cfg.indirect_shadow))
    from dynamicradiancevolume_amd.pipeline import entries_sh

    g = entries_sh(after[ids], cfg.sh_bands)
    o = entries_sh(ref[ids], cfg.sh_bands)
    np.testing.assert_array_equal(after[ids, :3], before[ids, :3])
    err = rel_l2(g, o)
    assert err < SH_TOL, f"SH relative L2 {err:.3e}"
    if cfg.indirect_shadow:
        nb = vis.shape[1]
        gvis = r.read_visibility(live, nb)[ids]
        assert np.abs(gvis - vis).max() < VIS_TOL
        # A ray stopped at transmittance <= 2^-20 returns exactly 0; the
        # oracle marches on, and its visibility there is at most 2^-20 up to
        # the FP32 rounding of 1 - occlusion near 1 (a few ulp of 1 per step).
        zero = gvis == 0.0
        assert zero.any() and (vis[zero] <= 2.0 ** -20 + 2e-6).all(), float(vis[zero].max())
    return r, df, fi, cfg, vol, live


def test_gather_cornell_sh1_shadowed():
    announce("gather cornell sh1 shadow")
    _gather_case("cornell_256")


def test_gather_cornell_sh2_shadowed():
    announce("gather cornell sh2 shadow")
    _gather_case("cornell_256", sh_bands=2)


def test_gather_cornell_unshadowed():
    announce("gather cornell no shadow")
    _gather_case("cornell_256", indirect_shadow=0, sh_bands=2)


@pytest.mark.parametrize("read,lod,wide,sh_bands", [(8, 0, 0, 2), (16, 0, 1, 1), (32, 1, 0, 2), (32, 4, 0, 1)])
def test_gather_shadow_block_sizes_match_oracle(read, lod, wide, sh_bands):
    """Blocks of one VPL (each with its own visibility), of exactly one group
    of four, and of more VPLs than a wave has lanes; alone and as the view of
    a batch's queued gather, whose blocks differ from its neighbour's."""
    from dynamicradiancevolume_amd import workloads as W
    from dynamicradiancevolume_amd.pipeline import Batch, DeviceFrame, Renderer, entries_sh

    orc = _orc()
    c = W.CORNELL_256.with_(sh_bands=sh_bands, width=96, height=64, max_caches=8192)
    light = W.replace(c.light, rsm_resolution=read, rsm_read_lod=0, rsm_wide=wide, indirect_shadow_lod=lod)
    frames = [W.make_inputs(c.with_(light=light)), W.make_inputs(c)]
    announce(f"gather read level {read}, wide {wide}, shadow LOD {lod}, SH{sh_bands}")
    dfs = [DeviceFrame(fi) for fi in frames]
    alone, view, other = (Renderer(c.config()) for _ in range(3))
    alone.render_frame(dfs[0])
    batch = Batch([view, other])
    batch.set_tuning(-2, 1024)
    batch.render_frame(dfs)
    fi, cfg = frames[0], c.config()
    vol = orc.update_volume(cfg, c.eye, fi.bbox[:3], fi.bbox[3:])
    _, mips = orc.voxelize(c.voxel_resolution, vol, fi.positions, adaption_factor=1.0)
    for r in (alone, view):
        _, live = r.cache_count()
        got = r.read_caches(live)
        ref = got.copy()
        ref[:, 4:] = 0.0
        orc.gather_f32(cfg, vol, orc.sh_constants(), fi.light, fi, mips, ref, n=live)
        err = rel_l2(entries_sh(got, sh_bands), entries_sh(ref, sh_bands))
        assert err < SH_TOL, f"SH relative L2 {err:.3e}"
    batch.close()


def _with_odd_vpl(fi, kind, x=3, y=5):
    """`fi` whose VPL at texel (x, y) of the read level is turned away from the
    scene and has infinite flux or lies at infinity."""
    from dataclasses import replace

    flux, nrm, dls = (a.copy() for a in fi.read_level)
    nrm[y, x] = (-16384, 0)  # (0, -1, 0): down, on a floor lit from above
    if kind == "flux":
        flux[y, x] = np.float16(np.inf).view(flux.dtype)
    else:
        dls[y, x] = np.float16(np.inf).view(dls.dtype)
    lod = fi.workload.light.rsm_read_lod
    return replace(fi, rsm_levels=list(fi.rsm_levels[:lod]) + [(flux, nrm, dls)] + list(fi.rsm_levels[lod + 1:]))


# Infinite flux times a cosine of zero, and an infinite direction, are NaN in the
# shader's sums: for every cache without shadows, and for the caches of a wave
# (64 in a row) of which one sees the VPL's shadow block.
@pytest.mark.parametrize("kind,read,lod,shadow", [("flux", 16, 0, 0), ("depth", 16, 0, 0), ("flux", 16, 0, 1),
                                                  ("flux", 32, 1, 1), ("flux", 32, 2, 1)])
def test_gather_of_odd_vpls_reaches_every_cache(kind, read, lod, shadow):
    from dynamicradiancevolume_amd import workloads as W
    from dynamicradiancevolume_amd.pipeline import entries_sh

    c = W.CORNELL_256
    light = W.replace(c.light, rsm_resolution=read, rsm_read_lod=0, indirect_shadow_lod=lod)
    w = c.with_(width=96, height=64, max_caches=16384, light=light, indirect_shadow=shadow, cav_resolution=48)
    fi = _with_odd_vpl(W.make_inputs(w), kind)
    announce(f"gather odd {kind} read {read} lod {lod} shadow {shadow}")
    r, df = _renderer(fi), _device(fi)
    r.render_frame(df)
    _, live = r.cache_count()
    finite = np.isfinite(entries_sh(r.read_caches(live), w.sh_bands)).reshape(live, -1).all(1)
    if shadow:
        block = sum(((3 >> lod) >> b & 1) << 2 * b | ((5 >> lod) >> b & 1) << 2 * b + 1 for b in range(8))
        seen = r.read_visibility(live, read * read >> 2 * lod)[:, block] != 0.0
        tiles = np.arange(live) // 64
        want = ~np.isin(tiles, tiles[seen])
        assert seen.any()
    else:
        want = np.zeros(live, bool)
    np.testing.assert_array_equal(finite, want)


def test_gather_boxes_all_caches():
    """Every cache of the 1080p frame (6.5M cone traces) against the oracle."""
    announce("gather boxes_1080p, all caches")
    _gather_case("boxes_1080p")


def test_gather_cornell_wide_rsm():
    """The 2:1 RSM extension: a 64 x 32 read level (2048 VPLs, 16 x 8 shadow
    blocks) against the oracle."""
    from dynamicradiancevolume_amd import workloads as W

    announce("gather cornell 2:1 RSM (64 x 32)")
    fi = frame_inputs("cornell_256", light=W.replace(W.CORNELL_256.light, rsm_wide=1))
    assert (fi.read_resolution, fi.read_height) == (64, 32)
    _gather_case("cornell_256", light=W.replace(W.CORNELL_256.light, rsm_wide=1))


def test_gather_boxes_32768_vpls_subset():
    """The 2:1 RSM extension at 32768 VPLs (512 x 256 rendered, 256 x 128
    read) on the 1080p frame: a spread subset of the caches against the oracle."""
    from dynamicradiancevolume_amd import workloads as W

    light = W.replace(W.BOXES_1080P.light, rsm_resolution=512, rsm_wide=1)
    announce("gather boxes_1080p 32768 VPLs (2:1 RSM) subset")
    fi = frame_inputs("boxes_1080p", light=light)
    assert fi.n_vpl == 32768 and fi.read_height == 128
    _gather_case("boxes_1080p", n_sub=256, light=light)


def test_gather_boxes_dense_subset():
    """The ~60k-cache frame: a spread subset of its caches against the oracle."""
    announce("gather boxes_1080p_dense subset")
    r, df, fi, cfg, vol, live = _gather_case("boxes_1080p_dense", n_sub=4096)
    assert live > 50000


def test_gather_two_lights_accumulate():
    """LightCachesRSM runs once per light and accumulates (renderer.cpp:924-932)."""
    orc = _orc()
    announce("gather two lights")
    r, df, fi, cfg, vol, live = _gather_case("cornell_256")
    once = r.read_caches(live)
    r.light_caches_rsm(df.rsm(), fi.light)
    twice = r.read_caches(live)
    from dynamicradiancevolume_amd.pipeline import entries_sh

    assert rel_l2(entries_sh(twice, 1), 2.0 * entries_sh(once, 1)) < SH_TOL


@pytest.mark.parametrize("name", ["cornell_256", "boxes_1080p", "boxes_1080p_dense"])
def test_full_frame_matches_oracle(name):
    """Voxelize -> allocate -> gather -> apply on the GPU against the whole
    oracle frame (cells matched canonically, SH by cell, RGB per pixel)."""
    orc = _orc()
    fi = frame_inputs(name)
    w = fi.workload
    cfg = w.config()
    df = _device(fi)
    announce(f"full frame {name}")
    r = _renderer(fi)
    r.render_frame(df)
    torch.cuda.synchronize()
    demanded, live = r.cache_count()
    g_entries = r.read_caches(live)
    g_cav = r.read_cav()
    vol = orc.update_volume(cfg, w.eye, fi.bbox[:3], fi.bbox[3:])
    count, o_cav, o_entries = orc.allocate(cfg, vol, fi.frame(), fi.depth)
    assert demanded == count
    gc, gp, _, _ = canonical(demanded, g_cav, g_entries, cfg.max_caches)
    oc, op, _, _ = canonical(count, o_cav, o_entries, cfg.max_caches)
    np.testing.assert_array_equal(gc, oc)
    np.testing.assert_array_equal(gp, op)
    # Oracle apply over the GPU's caches: checks apply exactly
    shc = orc.sh_constants()
    ref = orc.apply(cfg, vol, fi.frame(), shc, fi, g_cav, g_entries, live)
    got = df.out.cpu().numpy()
    assert rel_l2(got, ref) < RGB_TOL
    if name == "cornell_256":
        # and the independent oracle frame end to end
        ro = orc.run_frame(fi)
        from dynamicradiancevolume_amd.pipeline import entries_sh

        gsh = entries_sh(g_entries[(g_cav.reshape(-1)[gc] - 1)], cfg.sh_bands)
        osh = entries_sh(ro["entries"][(ro["cav"].reshape(-1)[oc] - 1)], cfg.sh_bands)
        assert rel_l2(gsh, osh) < SH_TOL
        assert rel_l2(got, ro["rgb"]) < RGB_TOL


@pytest.mark.parametrize("tuning", [
    dict(visibility_kernel=0, blocks_per_item=8),
    dict(visibility_kernel=0, blocks_per_item=2),
    dict(visibility_kernel=0, waves_per_cu=64),
    dict(visibility_kernel=0, waves_per_cu=1024),
    dict(visibility_kernel=1, blocks_per_item=8),
    dict(visibility_kernel=1, blocks_per_item=1, waves_per_cu=8),
    dict(visibility_kernel=1, blocks_per_item=32, gather_max_splits=128, waves_per_cu=64),
    dict(visibility_kernel=0, blocks_per_item=3, gather_max_splits=1, waves_per_cu=4),
    dict(visibility_kernel=0, steps_per_batch=4),
    dict(visibility_kernel=0, steps_per_batch=2),
    dict(visibility_kernel=0, steps_per_batch=1, blocks_per_item=7),
    dict(visibility_kernel=1, steps_per_batch=3, refill_min_lanes=1),
    dict(visibility_kernel=0, steps_per_batch=8, blocks_per_item=5),
])
def test_tuning_variants_agree(tuning):
    """Every launch shape traces the same rays: visibility is bit-identical to
    the default's (up to the early-exit granularity when the steps per batch
    change); SH differ only by the split summation order."""
    from canon import rel_l2

    fi = frame_inputs("boxes_1080p")
    df = _device(fi)
    announce(f"tuning variant {tuning}")
    res = []
    for t in ({}, tuning):
        r = _renderer(fi)
        if t:
            r.set_tuning(**t)
        r.render_frame(df)
        _, live = r.cache_count()
        e = r.read_caches(live)
        nb = fi.n_vpl // int(fi.light.indirect_shadow_sample_interval)
        order = np.lexsort(e[:, :3].view(np.uint32).T)
        vis = r.read_visibility(live, nb)
        res.append((e[order], vis[order]))
        r.close()
    (e0, v0), (e1, v1) = res
    np.testing.assert_array_equal(e0[:, :3], e1[:, :3])
    if tuning.get("steps_per_batch", 1) == 1:
        np.testing.assert_array_equal(v0, v1)
    else:
        # A ray stops at the first batch boundary after its transmittance
        # drops below 2^-20, so the visibility of opaque rays may differ by
        # less than that.
        assert np.abs(v0 - v1).max() <= 2.0 ** -19
    assert rel_l2(e1[:, 4:], e0[:, 4:]) <= 1e-5


@pytest.mark.parametrize("res", [128, 256])
def test_planned_trace_index_paths_agree_with_per_lane_tracer(res):
    """The planned cone trace forms corner-record indices in FP32 while every
    level has fewer than 2^24 records (voxel grids up to 128^3) and in
    integers beyond; either way its visibility equals the per-lane tracer's
    (the lane pool at one step per batch) bit for bit."""
    fi = frame_inputs("cornell_256")
    df = _device(fi)
    announce(f"planned trace index path at {res}^3 voxels vs per-lane tracer")
    vis = []
    for tuning in ({}, dict(visibility_kernel=1, steps_per_batch=1)):
        r = _renderer(fi, voxel_resolution=res)
        if tuning:
            r.set_tuning(**tuning)
        r.render_frame(df)
        _, live = r.cache_count()
        nb = fi.n_vpl // int(fi.light.indirect_shadow_sample_interval)
        vis.append(r.read_visibility(live, nb))
        r.close()
    assert (vis[0] > 0).any() and (vis[0] < 1).any()
    np.testing.assert_array_equal(vis[0], vis[1])


def test_stage_times_after_late_profiling():
    """Turning profiling on after unprofiled frames: querying stages that were
    never timed reports 0 and leaves no error for the next call."""
    fi = frame_inputs("cornell_256")
    df = _device(fi)
    announce("stage times after late profiling")
    r = _renderer(fi)
    r.render_frame(df)
    r.set_profiling(True)
    r.light_caches_rsm(df.rsm(), fi.light)
    t = r.stage_times()
    assert t["voxelize_ms"] == 0.0 and t["light_caches_ms"] > 0.0
    r.light_caches_rsm(df.rsm(), fi.light)
    r.apply_caches(df.gbuffer(), df.out)
    assert r.stage_times()["apply_ms"] > 0.0
