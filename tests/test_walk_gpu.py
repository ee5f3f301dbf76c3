"""The whole-ray walk's launch paths against the oracle at their edges: node
forms and depths of the path stack, ray counts around a wave, finite and
non-finite rays in one wave, level-of-detail cut-offs, trees at the end of
the 32-bit byte addresses. Bit-exact."""
import os

import numpy as np
import pytest

import oracle_py as orc
from test_format import relocated
from walk_trees import mixed_tree

pytestmark = pytest.mark.gpu


def _same(mine, ref, what):
    for k in ("hit", "normal", "leaf"):
        assert np.array_equal(mine[k], ref[k]), (what, k)
    assert np.array_equal(mine["t"].view(np.uint32), ref["t"].view(np.uint32)), what


def _rays(n, seed):
    rng = np.random.default_rng(seed)
    o = rng.uniform(0.6, 2.4, (n, 3)).astype(np.float32)
    d = (rng.uniform(1.1, 1.9, (n, 3)) - o).astype(np.float32)
    return o, d, rng


@pytest.mark.parametrize("levels,loose", [(n, False) for n in (1, 2, 3, 9, 10, 13, 14, 22, 23)] + [(3, True), (10, True)])
def test_mixed_trees_match_oracle(svo, levels, loose):
    words = mixed_tree(levels, levels, loose=loose)
    tree = svo.VoxelOctree.from_words(words, np.full(3, 0.5, np.float32))
    print(f"[gpu] walk: mixed tree of {levels} levels, {len(words)} words", flush=True)
    for n in (1, 63, 64, 65, 1000):
        o, d, rng = _rays(n, 100 * levels + n)
        _same(tree.raymarch_batch(o, d, 0.0), orc.raymarch(words, o, d, 0.0), ("no cut-off", n))
        rs = rng.uniform(0.0, 0.1, n).astype(np.float32)
        _same(tree.raymarch_batch(o, d, rs), orc.raymarch(words, o, d, rs), ("cut-off", n))
        # non-finite and extreme rays between ordinary ones
        d[::7, 0] = np.inf
        d[::5, 1] = 0.0
        o[::9, 2] = 3e30
        d[1::11] *= np.float32(1e-30)
        _same(tree.raymarch_batch(o, d, rs), orc.raymarch(words, o, d, rs), ("mixed rays", n))
    cam = tree.orbit_camera(25.0, 40.0, 1.0)
    tf, pos = np.frombuffer(cam.tform, np.float32), np.frombuffer(cam.pos, np.float32)
    w, h = 93, 61
    ref = orc.raymarch(words, pos[None, :], orc.primary_dirs(tf, w, h), 0.0)
    _same(tree.render_primary(cam, w, h), ref, "primary")
    rgba, depth = tree.render_frame(cam, 96, 64, 16, 1)
    ref_rgba, ref_depth = orc.render_frame(words, tf, np.full(3, 0.5, np.float32), 96, 64, 16, 1)
    assert np.array_equal(rgba, ref_rgba) and np.array_equal(depth.view(np.uint32), ref_depth.view(np.uint32))


@pytest.mark.parametrize("short", [1, 0])
def test_trees_at_the_end_of_32_bit_addresses(svo, golden, short):
    """The dragon moved to the end of an array of 2^30 - short words: the last
    size whose byte addresses fit 32 bits, and the first that takes 64."""
    c, w = orc.read_oct(os.path.join(golden, "dragon.oct"))
    base = (1 << 30) - short - len(w)
    print(f"[gpu] walk: dragon at word {base}", flush=True)
    big = svo.VoxelOctree.from_words(relocated(w, base), c)
    assert big.word_count() == (1 << 30) - short
    small = svo.VoxelOctree(os.path.join(golden, "dragon.oct"))
    o, d, rng = _rays(5000, 3)
    for rs in (0.0, rng.uniform(0.0, 0.05, 5000).astype(np.float32)):
        mine, ref = big.raymarch_batch(o, d, rs), small.raymarch_batch(o, d, rs)
        ref["leaf"] = np.where(ref["hit"] == 1, ref["leaf"] + np.uint64(base), ref["leaf"])
        assert (ref["hit"] == 1).sum() > 10
        _same(mine, ref, "rays")


@pytest.mark.parametrize("tiles", [1, 127, 128, 129, 255, 256, 383])
def test_every_tile_runs_once_around_the_run_length(svo, golden, tiles):
    """Tile counts around a full round of the XCD runs (128): the plain, the
    planned (first and second launch) and the batched launch equal the oracle."""
    import torch
    tree = svo.VoxelOctree(os.path.join(golden, "dragon.oct"))
    w, h = 8 * tiles, 8
    cam = tree.orbit_camera(10.0, 30.0, 1.0)
    tf, pos = np.frombuffer(cam.tform, np.float32), np.frombuffer(cam.pos, np.float32)
    ref = orc.raymarch(tree.words(), pos[None, :], orc.primary_dirs(tf, w, h), 0.0)
    _same(tree.render_primary(cam, w, h), ref, "plain")
    out = {k: torch.full((w * h,), 7, dtype=dt, device="cuda")
           for k, dt in (("hit", torch.uint8), ("normal", torch.int32), ("t", torch.float32), ("leaf", torch.int64))}
    ptr = {k: v.data_ptr() for k, v in out.items()}

    def got():
        torch.cuda.synchronize()
        r = {"hit": out["hit"].cpu().numpy(), "normal": out["normal"].cpu().numpy().view(np.uint32),
             "t": out["t"].cpu().numpy(), "leaf": out["leaf"].cpu().numpy().view(np.uint64)}
        for v in out.values():
            v.fill_(7)
        torch.cuda.synchronize()
        return r

    plan = svo.svo.TilePlan(w, h)
    for k in range(3):
        plan.render_device(tree, cam, ptr["hit"], ptr["normal"], ptr["t"], ptr["leaf"])
        _same(got(), ref, ("planned", k))
    ren = svo.svo.Renderer(2)
    ren.render_device([ren.view(tree, cam, w, h, **ptr)])
    _same(got(), ref, "batch")


def test_device_arrays_have_a_word_to_spare(svo, golden):
    """The walk reads the word after a two-word slot's descriptor: the device
    arrays of built trees and of trees from words are longer than the trees."""
    import ctypes
    import torch
    assert torch.cuda.is_available()
    hip = ctypes.CDLL("libamdhip64.so.7")  # the runtime in use, by its soname
    vol = np.random.default_rng(2).integers(1, 2**32, (40, 40, 40), dtype=np.uint32)
    built = svo.VoxelOctree.build_from_grid(vol)
    for what, tree in (("built", built), ("from words", svo.VoxelOctree.from_words(built.words(), built.center()))):
        base, size = ctypes.c_void_p(), ctypes.c_size_t()
        assert hip.hipMemGetAddressRange(ctypes.byref(base), ctypes.byref(size), ctypes.c_void_p(tree.upload())) == 0
        assert size.value >= 4 * (tree.word_count() + 1), what


def _device_outputs(n):
    import torch
    return {k: torch.full((n,), 7, dtype=dt, device="cuda")
            for k, dt in (("hit", torch.uint8), ("normal", torch.int32), ("t", torch.float32), ("leaf", torch.int64))}


def _fetch(out):
    """The outputs on the host; filled again for the next launch."""
    import torch
    torch.cuda.synchronize()
    r = {"hit": out["hit"].cpu().numpy(), "normal": out["normal"].cpu().numpy().view(np.uint32), "t": out["t"].cpu().numpy(),
         "leaf": out["leaf"].cpu().numpy().view(np.uint64)}
    for v in out.values():
        v.fill_(7)
    torch.cuda.synchronize()
    return r


@pytest.mark.parametrize("levels", [3, 10])
def test_wide_walk_through_plans_shadows_and_mixed_batches(svo, levels):
    """The 64-bit walk (a loose tree's) in the planned primary, shadow, frame and
    batch launches; in a batch it carries a tight tree's views along. Plans run
    three times: raster order, then filed orders."""
    import torch
    loose, tight = mixed_tree(levels, levels, loose=True), mixed_tree(levels, levels)
    centre = np.full(3, 0.5, np.float32)
    trees = {"loose": svo.VoxelOctree.from_words(loose, centre), "tight": svo.VoxelOctree.from_words(tight, centre)}
    words = {"loose": loose, "tight": tight}
    w, h, eps = 203, 131, 0.01
    light = np.array([0.3, 0.8, 0.2], np.float32)
    tree = trees["loose"]
    cam = tree.orbit_camera(25.0, 40.0, 1.0)
    tf, pos = np.frombuffer(cam.tform, np.float32), np.frombuffer(cam.pos, np.float32)
    dirs = orc.primary_dirs(tf, w, h)
    prim = {k: orc.raymarch(v, pos[None, :], dirs, 0.0) for k, v in words.items()}
    cut = {k: orc.raymarch(v, pos[None, :], dirs, 0.02) for k, v in words.items()}
    hit = prim["loose"]["hit"] == 1
    assert hit.mean() > 0.3 and (levels == 3 or (cut["loose"]["hit"] == 2).any())
    o = (pos[None, :] + dirs[hit] * (prim["loose"]["t"][hit] - np.float32(eps))[:, None]).astype(np.float32)
    shadow = np.zeros(w * h, np.uint8)
    shadow[hit] = orc.raymarch(loose, o, np.broadcast_to(light, o.shape).copy(), 0.0)["hit"] != 0
    assert 0.1 < shadow[hit].mean() < 0.9
    print(f"[gpu] wide walk: {levels} levels, planned primary", flush=True)
    out = _device_outputs(w * h)
    p = {k: v.data_ptr() for k, v in out.items()}
    plan = svo.svo.TilePlan(w, h)
    for k in range(3):
        plan.render_device(tree, cam, p["hit"], p["normal"], p["t"], p["leaf"])
        _same(_fetch(out), prim["loose"], ("planned", k))
    print("[gpu] wide walk: shadows", flush=True)
    sh = torch.full((w * h,), 7, dtype=torch.uint8, device="cuda")
    splan = svo.svo.TilePlan(w, h)
    for k, pl in enumerate((None, splan, splan, splan)):
        tree.render_shadow_device(cam, w, h, light, eps, p["hit"], p["t"], sh.data_ptr(), p["normal"], p["leaf"], plan=pl)
        _same(_fetch(out), prim["loose"], ("shadow primary", k))
        assert np.array_equal(sh.cpu().numpy(), shadow), ("shadow", k)
        sh.fill_(7)
    print("[gpu] wide walk: frames", flush=True)
    fw, fh = 208, 128
    ref_rgba, ref_depth = orc.render_frame(loose, tf, centre, fw, fh, 16, 1)
    rgba = torch.zeros(fw * fh, dtype=torch.int32, device="cuda")
    depth = torch.zeros(svo.svo.frame_depth_count(fw, fh, 16), dtype=torch.float32, device="cuda")
    fplan = svo.svo.TilePlan.for_frame(fw, fh, 16)
    for k, pl in enumerate((None, fplan, fplan, fplan)):
        tree.render_frame_device(cam, fw, fh, rgba.data_ptr(), depth.data_ptr(), 16, 1, plan=pl)
        torch.cuda.synchronize()
        assert np.array_equal(rgba.cpu().numpy().view(np.uint32).reshape(-1), np.asarray(ref_rgba).reshape(-1)), k
        assert np.array_equal(depth.cpu().numpy().view(np.uint32), np.asarray(ref_depth).reshape(-1).view(np.uint32)), k
        rgba.zero_()
        depth.zero_()
    print("[gpu] wide walk: batches", flush=True)
    ren = svo.svo.Renderer(4)
    for scales in ((0.0, 0.0), (0.0, 0.02), (0.02, 0.0)):
        outs = [_device_outputs(w * h) for _ in range(2)]
        views = [ren.view(trees[n], cam, w, h, ray_scale=rs, **{k: v.data_ptr() for k, v in out.items()})
                 for n, rs, out in zip(("loose", "tight"), scales, outs)]
        refs = [(cut if rs else prim)[n] for n, rs in zip(("loose", "tight"), scales)]
        bplan = svo.svo.TilePlan.for_batch(views)
        for k, opts in enumerate(({}, {"form": svo.svo.BATCH_PERSISTENT}, {"plan": bplan}, {"plan": bplan}, {"plan": bplan})):
            ren.render_device(views, **opts)
            for out, ref in zip(outs, refs):
                _same(_fetch(out), ref, ("batch", scales, k))
