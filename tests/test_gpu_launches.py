"""What a launch may not depend on: capacities, kernel variants, what other calls of the context ran before it or run
beside it."""
import numpy as np
import pytest

from neraulgraphics_amd import _lib, workloads
from neraulgraphics_amd.batch import BatchRenderer
from neraulgraphics_amd.geometry import Instance, Light, Material, Mesh, make_grid, make_icosphere

pytestmark = pytest.mark.gpu


def _say(*a):
    print(*a, flush=True)


def _eyes(n, z=0.0):
    c = np.tile(np.eye(3, 4, dtype=np.float32), (n, 1, 1))
    c[:, 2, 3] = z
    return c.reshape(n, 12)


@pytest.mark.parametrize("subdivisions,grid,lane_min", [(3, (38, 20), 1400), (5, (200, 75), 25000)],
                         ids=["with octant copies", "without"])
def test_packets_that_give_many_subtrees_under_a_lowered_share_capacity(gpu, subdivisions, grid, lane_min):
    """A mesh below lane_min_triangles is walked as a packet, which gives subtrees that few rays enter to the shared
    per-lane walk: up to 128 at once, whatever the capacity of its stack. Cut to 1, 3 and 100 entries, images are those of
    the default capacity."""
    _say(f"share capacity against a packet's subtrees: {subdivisions} subdivisions")
    worlds = 40
    r = BatchRenderer(64, 64, worlds, meshes=[make_icosphere(1.0, subdivisions), make_grid(*grid, 1.0, 1.0, 0.1, seed=3)],
                      instances=[Instance(0)] * 6 + [Instance(1)])
    rng = np.random.default_rng(5)
    m = np.tile(np.eye(3, 4, dtype=np.float32), (worlds, 7, 1, 1))
    m[..., :3] *= rng.uniform(0.4, 1.2, size=(worlds, 7, 1, 1)).astype(np.float32)
    m[..., 3] = rng.uniform(-2, 2, size=(worlds, 7, 3)) - [0, 0, 5]
    r.set_instance_transforms(m)
    r.set_trace_config(lane_min_triangles=lane_min)
    want = r.render(_eyes(worlds), 1.0, depth=True, object_ids=True, normals=True)
    assert np.isfinite(want["depth"]).mean() > 0.2
    for entries in (1, 3, 100):
        _lib.check(r._lib.ngx_debug_set_share_capacity(r._h, entries))
        got = r.render(_eyes(worlds), 1.0, depth=True, object_ids=True, normals=True)
        r.synchronize()
        # the same triangles tested in another order: equal but for rays through a shared edge, 1 in 10^6
        off = {k: int(np.sum(np.asarray(got[k]) != np.asarray(want[k]))) for k in want}
        _say(f"{entries} entries: values that differ {off}")
        assert off["depth"] <= 4 and off["object_ids"] <= 4 and off["normals"] <= 12, (entries, off)


def test_frames_on_several_streams_wait_for_each_other(gpu):
    """Frames of one context share their tile counters, view tables and hit records: a frame on another stream than the last
    starts after it, so frames queued on three streams at once with no order between them, and those queued after them, are
    the ones drawn alone. The same where the launches are not persistent, which share nothing."""
    import torch
    _say("frames on three streams")
    worlds = 600
    rng = np.random.default_rng(6)
    r = BatchRenderer(64, 64, worlds, meshes=[make_icosphere(1.0, 2)], instances=[Instance(0)] * 6,
                      lights=[Light((5.0, 12.0, 6.0), intensity=1.0, radius=0.5)])
    m = np.tile(np.eye(3, 4, dtype=np.float32), (worlds, 6, 1, 1))
    m[..., 3] = rng.uniform(-3, 3, size=(worlds, 6, 3)) - [0, 0, 6]
    r.set_instance_transforms(torch.from_numpy(m).cuda())
    cams = [torch.from_numpy(_eyes(worlds, z)).cuda() for z in (0.0, 0.4, 0.8)]
    outputs = [dict(depth=True), dict(normals=True), dict(rgb=True)]  # buffers of their own
    for persistent in (True, False):
        r.set_trace_config(persistent=persistent)
        want = []
        for k in range(3):
            want.append({n: v.clone() for n, v in r.render(cams[k], 1.0, zero_copy=True, **outputs[k]).items()})
            torch.cuda.synchronize()
        assert torch.isfinite(want[0]["depth"]).sum() > 1000
        streams = [torch.cuda.Stream() for _ in range(3)]
        for order in rng.integers(0, 3, size=(12, 5)):
            got = {}
            for k in order:
                with torch.cuda.stream(streams[k]):
                    got[int(k)] = r.render(cams[k], 1.0, zero_copy=True, **outputs[k])
            torch.cuda.synchronize()
            assert r.last_kernel_ms > 0
            for k, out in got.items():
                for n, v in want[k].items():
                    assert torch.equal(out[n], v), (persistent, list(order), k, n)


def _two_sheets(n=20):
    """Two triangulations of one flat square, each with normals of its own: a ray meets both at next to the same distance,
    so which it keeps shows in the picture."""
    def sheet(shift, normal):
        x = np.linspace(-1.0, 1.0, n + 1, dtype=np.float32)
        x[1:-1] += shift / n
        g = np.stack(np.meshgrid(x, x, indexing="ij"), axis=-1).reshape(-1, 2)
        v = np.concatenate([g, np.zeros((len(g), 1), np.float32)], axis=1)
        i = np.arange((n + 1) * (n + 1)).reshape(n + 1, n + 1)
        a, b, c, d = i[:-1, :-1].ravel(), i[1:, :-1].ravel(), i[1:, 1:].ravel(), i[:-1, 1:].ravel()
        t = np.concatenate([np.stack([a, b, c], 1), np.stack([a, c, d], 1)])
        return v, t, np.tile(np.float32(normal) / np.linalg.norm(normal), (len(v), 1))
    v0, t0, n0 = sheet(0.0, [0.6, 0.0, 0.8])
    v1, t1, n1 = sheet(0.9, [0.0, -0.6, 0.8])
    return Mesh(np.concatenate([v0, v1]).astype(np.float32), np.concatenate([t0, t1 + len(v0)]).astype(np.uint32),
                np.concatenate([n0, n1]).astype(np.float32))


def test_small_pictures_do_not_depend_on_the_kernel_variant_or_the_launch(gpu):
    """A picture of few rays draws its paths with a walk of its own. Where a ray meets two surfaces at once the walk decides
    which it keeps, so the variant that is asked for and the kind of launch must not change the walk: the same bytes."""
    _say("small pictures of mirrors with every RGB variant, persistent and not")
    r = BatchRenderer(48, 40, 2, meshes=[_two_sheets()], lights=[Light((5.0, 12.0, 6.0), intensity=1.0, radius=0.5)],
                      instances=[Instance(0, material=Material((0.8, 0.4, 0.3), 0.9, 0.2, 0.3, 40.0))] * 5)
    rng = np.random.default_rng(8)
    q = np.linalg.qr(rng.normal(size=(2, 5, 3, 3)))[0]
    m = np.concatenate([q * 1.5, rng.uniform(-1.5, 1.5, size=(2, 5, 3, 1)) - np.float32([[0], [0], [5]])], axis=-1)
    r.set_instance_transforms(m.astype(np.float32))
    pictures = {}
    for blocks in (0, 4, 5, 6, 7):
        for persistent in (True, False):
            r.set_trace_config(rgb_blocks=blocks, persistent=persistent)
            pictures[blocks, persistent] = np.array(r.render(_eyes(2), 1.0, 2, rgb=True)["rgb"])
    base = pictures[0, True]
    assert len(np.unique(base.reshape(-1, 3), axis=0)) > 100
    for k, v in pictures.items():
        assert np.array_equal(v, base), k


def test_range_gradients_of_fewer_rays_under_capture(gpu):
    """A scan's gradient splits few rays over more workgroups than many, each with its own partial sums: their memory, once
    made for a call, holds every smaller one, so that it can be captured into a graph."""
    import torch
    _say("range gradient of 131,072 rays eagerly, then of fewer under capture")
    cfg = workloads.make("posed_bodies", worlds=1)
    r = workloads.make_renderer(cfg)
    poses = torch.from_numpy(np.ascontiguousarray(cfg["body_poses"])).cuda()
    rng = np.random.default_rng(4)
    rays = 131072
    d = torch.from_numpy((rng.normal(size=(1, rays, 3)) * [0.3, 0.3, 1.0] - [0, 0, 3]).astype(np.float32)).cuda()
    o = torch.from_numpy(np.broadcast_to(cfg["cameras"].reshape(1, 1, 3, 4)[..., 3], (1, rays, 3)).astype(np.float32)).cuda()
    dist = r.cast_rays(o, d, 50.0)["distance"].clone()
    g = torch.from_numpy(rng.normal(size=(1, rays)).astype(np.float32)).cuda()
    assert torch.isfinite(dist).float().mean() > 0.01
    r.pose_backward_range(poses, o, d, 50.0, dist, g)
    torch.cuda.synchronize()
    few = {n: [a[:, :n].contiguous() for a in (o, d, dist, g)] for n in (65536, 20000, 4096)}
    for n, (fo, fd, fdist, fg) in few.items():
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got = r.pose_backward_range(poses, fo, fd, 50.0, fdist, fg)
        graph.replay()
        torch.cuda.synchronize()
        want = r.pose_backward_range(poses, fo, fd, 50.0, fdist, fg)
        assert torch.equal(got, want) and want.abs().sum() > 0, n


def _last_launch(r):
    """(rays a wavefront took in the last launch, whether the last render had view tables)"""
    import ctypes
    rays, tables = ctypes.c_int32(-1), ctypes.c_int32(-1)
    _lib.check(r._lib.ngx_debug_last_launch(r._h, ctypes.byref(rays), ctypes.byref(tables)))
    return rays.value, bool(tables.value)


def _wave_rays(rays, shown=False, paths=1):
    """The rays a wavefront takes, by the limits the launches choose by: up to 131,072 rays, or 65,536 where the triangle
    shows, over the segments and samples of a path; few enough for two wavefronts of 64 a compute unit or not."""
    import torch
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    if rays > (65536 if shown else 131072) // paths:
        return 64
    few = (rays + 63) // 64 <= 2 * cus
    return (4 if few else 8) if paths > 1 else (8 if few else 16)


MIRRORS = dict(lights=[Light((5.0, 12.0, 6.0), intensity=1.0, radius=0.5)])


def _mirror_worlds(full, n, reflectivity):
    instances = [Instance(i.mesh, i.transform, Material((0.8, 0.5, 0.3), 0.9, 0.2, reflectivity, 40.0)) for i in full["instances"]]
    r = BatchRenderer(64, 64, n, meshes=full["meshes"], instances=instances, **MIRRORS)
    r.bind_bodies(full["body_of_instance"], full["local_pose"], full["scale"], full["bodies"])
    r.set_body_poses(full["body_poses"][:n])
    return r


@pytest.fixture(scope="module")
def posed_1600(gpu):
    """1,600 worlds of posed bodies, every launch over them of full wavefronts, and what they look like."""
    import torch
    full = workloads.make("posed_bodies", worlds=1600)
    rng = np.random.default_rng(5)
    rays = 2000
    dirs = (rng.normal(size=(1600, rays, 3)) * [0.4, 0.4, 1.0] - [0, 0, 2]).astype(np.float32)
    origins = np.repeat(full["cameras"].reshape(-1, 3, 4)[:, None, :, 3], rays, axis=1).astype(np.float32)
    seeds = rng.normal(size=(1600, 64, 64)).astype(np.float32), rng.normal(size=(1600, rays)).astype(np.float32)

    def run(n, kind):
        up = lambda a: torch.from_numpy(np.ascontiguousarray(a[:n])).cuda()  # noqa: E731
        cams, poses = up(full["cameras"]), up(full["body_poses"])
        if kind in ("mirrors", "samples"):
            r = _mirror_worlds(full, n, 0.3 if kind == "mirrors" else 0.0)
            rgb = r.render(cams, full["fov"], 1 if kind == "mirrors" else 4, rgb=True, zero_copy=True)["rgb"]
            return {"rgb": rgb.cpu().numpy()}, _last_launch(r)[0]
        r = workloads.make_renderer(dict(full, worlds=n, cameras=full["cameras"][:n], body_poses=full["body_poses"][:n]))
        if kind in ("depth", "normals"):
            out = r.render(cams, full["fov"], depth=True, object_ids=True, normals=kind == "normals", zero_copy=True)
        elif kind == "depth gradient":
            depth = r.render(cams, full["fov"], depth=True, zero_copy=True)["depth"].clone()
            out = {"gradient": r.pose_backward_depth(poses, cams, full["fov"], depth, up(seeds[0]))}
        else:
            o, d = up(origins), up(dirs)
            out = r.cast_rays(o, d, 50.0)
            if kind == "range gradient":
                out = {"gradient": r.pose_backward_range(poses, o, d, 50.0, out["distance"].clone(), up(seeds[1]))}
        return {k: v.cpu().numpy() for k, v in out.items()}, _last_launch(r)[0]

    large = {}

    def both(n, kind):
        if kind not in large:
            large[kind], lanes = run(1600, kind)
            assert lanes == 64
        small, lanes = run(n, kind)
        return small, {k: v[:n] for k, v in large[kind].items()}, lanes

    return both


@pytest.mark.parametrize("kind,worlds", [("depth", (1, 8, 9, 31, 32, 33)), ("normals", (8, 9, 16, 17)), ("rays", (1, 16, 17, 32, 33)),
                                         ("mirrors", (1, 8, 9)), ("samples", (1, 4, 5)), ("depth gradient", (1, 8, 9, 32, 33)),
                                         ("range gradient", (1, 16, 17, 32, 33))])
def test_part_wavefronts_either_side_of_their_limits(posed_1600, kind, worlds):
    """Worlds drawn by launches of 4, 8, 16 and 64 rays a wavefront, on both sides of every limit between them, look as they
    do in a batch of full wavefronts: the same triangle tests in another order, equal but for ties, of which these meshes
    show next to none; gradients to the rounding of their sums of up to 4,096 terms in another grouping."""
    seen = set()
    for n in worlds:
        small, large, lanes = posed_1600(n, kind)
        _say(f"{kind}, {n} worlds: {lanes} rays a wavefront")
        rays = n * (2000 if kind in ("rays", "range gradient") else 4096)
        assert lanes == _wave_rays(rays, not kind.startswith("depth"), {"mirrors": 2, "samples": 4}.get(kind, 1)), (kind, n)
        seen.add(lanes)
        for k, v in small.items():
            assert v.shape == large[k].shape and np.abs(large[k]).sum() > 0, k
            if k == "gradient":
                assert np.abs(v - large[k]).max() <= 1e-4 * np.abs(large[k]).max(), (kind, n)
            else:
                assert np.mean(v != large[k]) < 1e-5, (kind, n, k)
    assert 64 in seen and len(seen) > 1, seen


def test_view_tables_are_made_where_they_should_be(gpu):
    """Launches of 4,096 tiles or more, of at most four instances and camera a tile, have their views laid out first, others
    do not, and the worlds both draw are the same: 64 rays a wavefront in both, so bit for bit."""
    _say("view tables or none")
    rng = np.random.default_rng(9)
    n = 5
    m = np.concatenate([np.linalg.qr(rng.normal(size=(4100, n, 3, 3)))[0] * rng.uniform(0.3, 1.2, size=(4100, n, 1, 1)),
                        rng.uniform(-3, 3, size=(4100, n, 3, 1)) - [[0], [0], [5]]], axis=-1).astype(np.float32)

    def run(worlds, instances=4, **config):
        r = BatchRenderer(8, 8, worlds, meshes=[make_icosphere(1.0, 2)], instances=[Instance(0)] * instances)
        r.set_trace_config(**config)
        r.set_instance_transforms(m[:worlds, :instances])
        out = r.render(_eyes(worlds), 1.0, depth=True, object_ids=True)
        return out, *_last_launch(r)

    many, lanes, tables = run(4100)
    assert tables and lanes == 64 and np.isfinite(many["depth"]).sum() > 1000
    few, lanes, tables = run(4090)
    assert not tables and lanes == 64
    loose, _, tables = run(4100, persistent=False)
    assert not tables
    assert not run(4100, 5)[2]
    for k, v in many.items():
        assert np.array_equal(few[k], v[:4090]) and np.array_equal(loose[k], v), k


@pytest.mark.parametrize("worlds", [1, 9, 16, 17, 32, 33])
def test_a_gradient_takes_its_rays_as_its_forward_did(gpu, worlds):
    """Which of two surfaces at one distance a ray keeps depends on the rays it is walked with: a depth image and its
    gradient's re-trace, a range query and its gradient's, take as many a wavefront, on either side of the limits."""
    import torch
    from neraulgraphics_amd.autograd import cast_range, render_depth
    cfg = workloads.make("posed_bodies", worlds=worlds)
    r = workloads.make_renderer(cfg)
    poses = torch.from_numpy(cfg["body_poses"]).cuda().requires_grad_()
    depth = render_depth(r, poses, torch.from_numpy(cfg["cameras"]).cuda(), cfg["fov"])
    forward = _last_launch(r)[0]
    torch.where(torch.isfinite(depth), depth, 0.0).sum().backward()
    _say(f"{worlds} worlds: {forward} rays a wavefront forward, {_last_launch(r)[0]} backward")
    assert _last_launch(r)[0] == forward
    d = torch.randn(worlds, 4096, 3, device="cuda", generator=torch.Generator("cuda").manual_seed(1)) * 0.3 - torch.tensor([0.0, 0.0, 1.0], device="cuda")
    o = torch.from_numpy(np.repeat(cfg["cameras"].reshape(worlds, 1, 3, 4)[..., 3], 4096, axis=1)).cuda()
    distance = cast_range(r, poses, o, d, 50.0)
    forward = _last_launch(r)[0]
    torch.where(torch.isfinite(distance), distance, 0.0).sum().backward()
    assert _last_launch(r)[0] == forward


def test_gradients_of_more_than_2_to_28_bodies(gpu):
    """1,048,577 worlds of 256 bodies, of which each world shows one: the gradient is taken, the shown bodies' is that of a
    batch of the first 154 worlds, and the others' is zero, the last world's among them."""
    import torch
    worlds, bodies, shown = (1 << 20) + 1, 256, 255
    _say(f"gradient of {worlds} worlds x {bodies} bodies")
    if torch.cuda.mem_get_info()[0] < 40 << 30:
        pytest.skip("needs 40 GB of device memory")

    def run(n):
        r = BatchRenderer(1, 1, n, meshes=[make_icosphere(1.0, 0)], instances=[Instance(0)])
        r.bind_bodies([shown], [[0, 0, 0, 0, 0, 0, 1]], [[1, 1, 1]], bodies)
        poses = torch.zeros(n, bodies, 7, device="cuda")
        poses[..., 6] = 1.0
        at = torch.arange(n, device="cuda")
        poses[:, shown, 0] = 0.1 + 0.01 * (at % 7)
        poses[:, shown, 1] = 0.2
        poses[:, shown, 2] = -4.0 - 0.01 * (at % 11)
        r.set_body_poses(poses)
        cams = torch.from_numpy(_eyes(1)).cuda().repeat(n, 1)
        depth = r.render(cams, 1.0, depth=True, zero_copy=True)["depth"].clone()
        assert bool(torch.isfinite(depth).all())
        return r.pose_backward_depth(poses, cams, 1.0, depth, torch.ones_like(depth))

    few, many = run(154), run(worlds)
    assert float(few[:, shown].abs().amin(dim=0).max()) > 0 and torch.equal(many[:154], few)
    assert torch.equal(many[-1, shown], few[(worlds - 1) % 77, shown])
    assert int(torch.count_nonzero(many[:, :shown])) == 0
    del few, many
    torch.cuda.empty_cache()
