"""The fog march over a slot map against the same march through the accessor, bit for bit.

A launch under graph capture takes no scratch and goes through the accessor, so a captured call is
the reference here; the march itself is compared with the FP64 oracle in test_gpu_parity.py.
Covered: every codec, active tiles, leaves and nodes under render-skip flags (which the map leaves to
the accessor), bboxes that start and end inside a leaf, steps that round off their slot, rays that
start inside, run along an axis or miss, and launches of one ray up to several tiles.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


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
