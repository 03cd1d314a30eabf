"""The fog march and the level-set crossings over a slot map against the same queries through the
accessor, bit for bit, and the march's adjoint (2x2x2 blocks in LDS) against the FP64 oracle and across schedules and grid types.

A launch under graph capture takes no scratch and goes through the accessor, so a captured call is
the reference here; the march itself is compared with the FP64 oracle in test_gpu_parity.py.
Covered: every codec, active tiles, leaves and nodes under render-skip flags (which the map leaves to
the accessor), bboxes that start and end inside a leaf, steps that round off their slot, rays that
start inside, run along an axis or miss, and launches of one ray up to more tiles than take four lanes per ray.
"""
import gc

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(autouse=True)
def _no_collection_while_recording():
    """A DeviceGrid that the collector frees waits for the device, which ends a capture: collect before, not then."""
    gc.collect()
    gc.disable()
    yield
    gc.enable()


def _nvq():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import openvdb_amd
    return openvdb_amd


def _flagged(grid):
    """A copy whose every 7th leaf and 3rd lower node carries the render-skip flag."""
    g = grid.copy()
    off, count = 672 + np.frombuffer(g, np.int64, 4, 672), np.frombuffer(g, np.uint32, 3, 704)
    g[off[0] + 15 + 2144 * np.arange(0, count[0], 7)] |= 1
    g[off[1] + 24 + 33856 * np.arange(0, count[1], 3)] |= 1
    return g


def _host(nvq, name):
    if name == "fog_sphere":
        return nvq.tools.create_fog_volume_sphere(45.0, (3.0, -2.0, 5.0), 1.0, 3.0)
    if name == "tiles":
        return nvq.tools.create_fog_fbm([0, 0, 0, 95, 95, 95], seed=5, amplitude=8.0)
    fog = nvq.tools.create_fog_fbm([-41, -9, 16, 56, 70, 91], seed=9)
    return _flagged(fog) if name == "flagged" else fog


def _grid(nvq, host, codec):
    if codec == "onindex":
        ijk, values = nvq.tools.active_voxels(host)
        d, index = nvq.DeviceGrid.from_voxels(torch.from_numpy(ijk).cuda(), "OnIndex", return_index=True)
        channel = torch.zeros(d.value_count, device="cuda")
        channel[index] = torch.from_numpy(values).cuda()
        d.set_channel(channel)
        return d
    return nvq.DeviceGrid(host if codec == "float" else nvq.tools.quantize(host, codec, 1e-3))


def _rays(d, n):
    r = np.random.default_rng(n)
    lo, hi = np.array(d.index_bbox[:3], np.float64), np.array(d.index_bbox[3:], np.float64) + 1
    v = r.normal(size=(n, 3))
    eye = 0.5 * (lo + hi) + np.linalg.norm(hi - lo) * v / np.linalg.norm(v, axis=1, keepdims=True)
    aim = r.random((n, 3)) * (hi - lo) * 1.2 + lo - 0.1 * (hi - lo)
    k = n // 6
    eye[:k] = r.random((k, 3)) * (hi - lo) + lo
    dirs = aim - eye
    dirs[k:2 * k] = np.eye(3)[r.integers(0, 3, k)] * r.choice([-1.0, 1.0], (k, 1))
    eye[k:2 * k] = np.floor(aim[k:2 * k]) - 300.0 * dirs[k:2 * k]
    return (torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).cuda() for x in (eye, dirs))


@pytest.mark.parametrize("name,codec", [("fog", c) for c in ("float", "fp4", "fp8", "fp16", "fpn", "onindex")] +
                         [("tiles", "float"), ("tiles", "fp8"), ("fog_sphere", "float"), ("flagged", "float")])
def test_march_over_slots_equals_march_through_the_accessor(name, codec):
    nvq = _nvq()
    d = _grid(nvq, _host(nvq, name), codec)
    for n, dt in ((1, 0.5), (65, 0.37), (4097, 0.5), (4096, 1.9)):
        eye, dirs = _rays(d, n)
        L, T = nvq.ops.fog_march(d, eye, dirs, dt, 0.05)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            Lc, Tc = nvq.ops.fog_march(d, eye, dirs, dt, 0.05)
        for _ in range(2):
            Lc.fill_(-1.0)
            Tc.fill_(-1.0)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(L.view(torch.int32), Lc.view(torch.int32)), (n, dt)
            assert torch.equal(T.view(torch.int32), Tc.view(torch.int32)), (n, dt)
            L2, _ = nvq.ops.fog_march(d, eye, dirs, dt, 0.05)
            assert torch.equal(L, L2)
        if n > 64:
            assert float(L.max()) > 0.0


QUAD_RAYS = 64 * 8192  # the march takes four lanes per ray up to here, one lane from there on


@pytest.mark.parametrize("name,codec", [("fog", c) for c in ("float", "fp4", "fp8", "fp16", "fpn", "onindex")] +
                         [("tiles", "float"), ("flagged", "float")])
def test_one_lane_march_equals_four(name, codec):
    """Launches above that size, whole, against the same rays in launches below it (which the test above compares
    with the accessor): a linear batch with a ragged last tile and an image."""
    nvq = _nvq()
    d = _grid(nvq, _host(nvq, name), codec)
    n = QUAD_RAYS + 65
    eye, dirs = _rays(d, n)
    L, T = nvq.ops.fog_march(d, eye, dirs, 0.37, 0.05)
    parts = [nvq.ops.fog_march(d, e.contiguous(), x.contiguous(), 0.37, 0.05)
             for e, x in zip(eye.split(QUAD_RAYS // 2 + 7), dirs.split(QUAD_RAYS // 2 + 7))]
    for a, b in zip((L, T), zip(*parts)):
        assert torch.equal(a.view(torch.int32), torch.cat(b).view(torch.int32))
    assert int((L > 0.0).sum()) > n // 8
    first = nvq.ops.fog_march(d, eye[:4099].contiguous(), dirs[:4099].contiguous(), 0.37, 0.05)  # in image order
    assert torch.equal(L[:4099], first[0]) and torch.equal(T[:4099], first[1])
    w, h = 1021, 517  # 128 x 65 tiles
    eye, dirs = _image(d, w, h)
    L, T = nvq.ops.fog_march(d, eye, dirs, 0.5, 0.05, image_width=w)
    rows = 200 * w
    parts = [nvq.ops.fog_march(d, e.contiguous(), x.contiguous(), 0.5, 0.05, image_width=w)
             for e, x in zip(eye.split(rows), dirs.split(rows))]
    for a, b in zip((L, T), zip(*parts)):
        assert torch.equal(a.view(torch.int32), torch.cat(b).view(torch.int32))
    assert int((L > 0.0).sum()) > 1000


def _level_set(nvq, name):
    if name == "torus":
        return nvq.tools.create_level_set_torus(50.0, 14.0, (3.0, -2.0, 5.0), 0.5, 3.0)
    if name == "tiles":
        return _host(nvq, "tiles")  # active tiles: candidates outside leaves
    sphere = nvq.tools.create_level_set_sphere(37.0, (1.5, -2.0, 3.0), 1.0, 3.0)
    return _flagged(sphere) if name == "flagged" else sphere


@pytest.mark.parametrize("name,codec", [("sphere", c) for c in ("float", "fp4", "fp8", "fp16", "fpn")] +
                         [("torus", "float"), ("torus", "fpn"), ("tiles", "float"), ("flagged", "float")])
def test_crossing_over_slots_equals_crossing_through_the_accessor(name, codec):
    nvq = _nvq()
    d = _grid(nvq, _level_set(nvq, name), codec)
    for n, iso in ((1, 0.0), (65, 0.0), (20011, 0.0), (20011, 0.4), (4097, -0.7)):
        eye, dirs = _rays(d, n)
        eye *= d.voxel_size[0]
        got = nvq.ops.iso_crossing(d, eye, dirs, iso)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            want = nvq.ops.iso_crossing(d, eye, dirs, iso)
        for _ in range(2):
            for x in want:
                x.fill_(7)
            graph.replay()
            torch.cuda.synchronize()
            for a, b in zip(got, want):
                assert torch.equal(a.view(torch.uint8), b.view(torch.uint8)), (n, iso)
            nvq.ops.iso_crossing(d, eye, dirs, iso)
        if n > 4096 and iso == 0.0 and name != "tiles":
            assert int(got[0].sum()) > 1000


@pytest.fixture(scope="module")
def oracle():
    from pyoracle import Oracle
    return Oracle()


def _image(d, w, h):
    lo, hi = np.array(d.index_bbox[:3], np.float64), np.array(d.index_bbox[3:], np.float64) + 1
    eye = 0.5 * (lo + hi) + 1.1 * np.linalg.norm(hi - lo) * np.array([0.48, -0.36, 0.8])
    e, r = _nvq().tools.camera_rays(w, h, tuple(eye), tuple(0.5 * (lo + hi)), (0.0, 1.0, 0.0), 45.0)
    return torch.from_numpy(e).cuda(), torch.from_numpy(r).cuda()


@pytest.mark.parametrize("name,w,h", [("fog", 1, 1), ("fog", 40, 27), ("fog", 203, 161), ("tiles", 61, 50),
                                      ("fog_sphere", 61, 50), ("flagged", 61, 50)])
def test_adjoint_over_blocks(oracle, name, w, h):
    nvq = _nvq()
    host = _host(nvq, name)
    d = nvq.DeviceGrid(host)
    eye, dirs = _image(d, w, h)
    r = torch.Generator(device="cuda")
    r.manual_seed(w)
    gL, gT = (torch.randn(w * h, generator=r, device="cuda") for _ in range(2))
    gL[::7] = 0.0
    gT[::7] = 0.0  # rays without a gradient idle beside the others
    L, T = nvq.ops.fog_march(d, eye, dirs, 0.5, 0.05, image_width=w)
    acc = nvq.ops.fog_march_backward(d, eye, dirs, L, gL, T, gT, 0.5, 0.05, image_width=w)
    # integer sums: other wavefronts, other blocks in each cache, the same result
    order = torch.randperm(w * h, generator=r, device="cuda")
    mixed = [x[order].contiguous() for x in (eye, dirs, L, gL, T, gT)]
    assert torch.equal(acc, nvq.ops.fog_march_backward(d, *mixed, 0.5, 0.05))
    g = nvq.ops.fixed_to_float(acc).double().cpu().numpy()
    want = oracle.fog_march_adjoint(host, eye.cpu().numpy(), dirs.cpu().numpy(), 0.5, 0.05,
                                    gL.double().cpu().numpy(), gT.double().cpu().numpy())
    assert np.abs(g - want).max() <= 1e-4 * np.abs(want).max()  # the bound of the accessor adjoint's test
    if name == "fog":
        # the same voxels as an index grid: entry by entry the same integers
        ijk, values = nvq.tools.active_voxels(host)
        i, index = nvq.DeviceGrid.from_voxels(torch.from_numpy(ijk).cuda(), "OnIndex", return_index=True)
        channel = torch.zeros(i.value_count, device="cuda")
        channel[index] = torch.from_numpy(values).cuda()
        i.set_channel(channel)
        Li, Ti = nvq.ops.fog_march(i, eye, dirs, 0.5, 0.05, image_width=w)
        assert torch.equal(L, Li) and torch.equal(T, Ti)
        acci = nvq.ops.fog_march_backward(i, eye, dirs, L, gL, T, gT, 0.5, 0.05, image_width=w)
        mask = np.unpackbits(host[_leaf_bytes(host)].reshape(-1, 2144)[:, 16:80], axis=1, bitorder="little")
        on = torch.from_numpy(np.flatnonzero(mask.reshape(-1))).cuda()
        assert torch.equal(acc[on], acci[index])
        off = torch.from_numpy(np.flatnonzero(mask.reshape(-1) == 0)).cuda()
        if w > 1:
            assert int(acc[off].ne(0).sum()) > 0 and int(acci[0]) != 0  # the inactive voxels' sums


def _leaf_bytes(host):
    off, count = 672 + int(np.frombuffer(host, np.int64, 1, 672)[0]), int(np.frombuffer(host, np.uint32, 1, 704)[0])
    return slice(off, off + 2144 * count)


@pytest.mark.parametrize("name", ["fog", "tiles"])
def test_adjoint_of_rays_far_apart(name):
    """Wavefronts whose rays' first steps lie farther apart than they march side by side, and nearer: the order
    of the batch does not change the integers, and an image gives them too."""
    nvq = _nvq()
    d = _grid(nvq, _host(nvq, name), "float")
    lo, hi = np.array(d.index_bbox[:3], np.float64), np.array(d.index_bbox[3:], np.float64) + 1
    r = np.random.default_rng(6)
    v = r.normal(size=(4160, 3))
    far = r.choice([0.0, 0.7, 0.8, 2.0, 12.0], 4160)[:, None]  # times the diagonal: some inside the bbox
    eye = 0.5 * (lo + hi) + far * np.linalg.norm(hi - lo) * v / np.linalg.norm(v, axis=1, keepdims=True)
    aim = r.random((4160, 3)) * (hi - lo) + lo + 0.01
    eye, dirs = (torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).cuda() for x in (eye, aim - eye))
    gL, gT = (torch.from_numpy(r.normal(size=4160).astype(np.float32)).cuda() for _ in range(2))
    L, T = nvq.ops.fog_march(d, eye, dirs, 0.5, 0.05)
    want = nvq.ops.fog_march_backward(d, eye, dirs, L, gL, T, gT, 0.5, 0.05, image_width=65)  # no rule on spread
    assert int(want.ne(0).sum()) > 1000
    by_distance = torch.from_numpy(np.argsort(far[:, 0], kind="stable")).cuda()
    for order in (torch.arange(4160, device="cuda"), by_distance):
        x = [a[order].contiguous() for a in (eye, dirs, L, gL, T, gT)]
        assert torch.equal(want, nvq.ops.fog_march_backward(d, *x, 0.5, 0.05))


@pytest.mark.parametrize("codec", ["float", "fp8", "fpn"])
def test_multi_query_over_maps_equals_the_accessor_launch(codec):
    """nvq_multi_query (slot maps, tiles left open answered again) against nvq_multi_query_noalloc."""
    nvq = _nvq()
    hosts = [_level_set(nvq, "sphere"), _host(nvq, "fog"), _level_set(nvq, "torus"), _host(nvq, "tiles")]
    if codec != "float":
        hosts = [nvq.tools.quantize(h, codec, 1e-3) for h in hosts]
    else:
        hosts += [_flagged(hosts[0]), _flagged(hosts[1])]
    grids = [nvq.DeviceGrid(h) for h in hosts]
    for w, h in ((9, 7), (203, 121)):  # below and above the tile count that is ordered
        rays = [_image(d, w, h) for d in grids]
        eye, dirs = (torch.cat(x) for x in zip(*rays))
        offs = [w * h * j for j in range(len(grids) + 1)]
        for widths in ([w] * len(grids), [0] + [w] * (len(grids) - 1)):
            a = nvq.ops.multi_query(grids, eye, dirs, offs, widths, 0.5, 0.05)
            b = nvq.ops.multi_query(grids, eye, dirs, offs, widths, 0.5, 0.05, noalloc=True)
            for x, y in zip(a, b):
                assert torch.equal(x.view(torch.uint8), y.view(torch.uint8))
        assert int(a[0].sum()) > 0 and float(a[2].max()) > 0.0
