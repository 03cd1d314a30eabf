"""Point queries below the binned threshold (staged lookups of the block around a query) and their
adjoint against the oracle, bit for bit: points on slot, node and root-tile boundaries, FD6 samples that
round into a farther cell, far outside the grid and at the ends of the integer range, and batches that
end inside a wavefront.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def grids():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import openvdb_amd as nvq
    torus = nvq.tools.create_level_set_torus(50.0, 14.0, (0.0, 0.0, 0.0), 1.0, 3.0)  # eight root tiles
    fog = nvq.tools.create_fog_fbm([4070, -30, 100, 4133, 33, 163], seed=5, amplitude=8.0)  # active tiles
    out = {"torus": torus, "fog": fog}
    for c in ("fp4", "fp8", "fp16", "fpn"):
        out["torus_" + c] = nvq.tools.quantize(torus, c, 1e-3)
    return nvq, out


def _points(d, n):
    r = np.random.default_rng(n)
    lo, hi = np.array(d.index_bbox[:3], np.float64), np.array(d.index_bbox[3:], np.float64) + 1
    p = (r.random((n, 3)) * (hi - lo + 20) + lo - 10).astype(np.float32)
    k = n // 8
    p[:k] = np.rint(p[:k] / 8) * 8 + r.integers(-2, 3, (k, 3))                   # around slot boundaries
    p[k:2 * k] = np.nextafter(np.rint(p[k:2 * k]), np.float32(0))                # p +- 1 rounds up a cell
    p[2 * k:3 * k] = r.choice([-4096.0, 0.0, 4096.0, 128.0], (k, 3)) + r.normal(0, 1.5, (k, 3))
    if n > 60:
        p[-1] = 1e9
        p[-2] = [-2.1e9, 0.5, 3.0]
        p[-3] = [16777216.0, 1.0, 1.0]
    return p


@pytest.mark.parametrize("name", ["torus", "fog", "torus_fp4", "torus_fp8", "torus_fp16", "torus_fpn"])
@pytest.mark.parametrize("n", [1, 65, 20011])
def test_staged_queries(oracle, grids, name, n):
    nvq, hosts = grids
    host = hosts[name]
    d = nvq.DeviceGrid(host)
    p = _points(d, n)
    for mode in (1, 2, 3):
        got = nvq.ops.sample(d, torch.from_numpy(p).cuda(), grad_mode=mode)
        for a, b in zip(got, oracle.sample(host, p, grad_mode=mode)):
            assert np.array_equal(a.cpu().numpy().view(np.uint32), np.ascontiguousarray(b).view(np.uint32)), mode


@pytest.mark.parametrize("n", [1, 65, 5003])
def test_staged_adjoint(oracle, grids, n):
    nvq, hosts = grids
    for name in ("torus", "fog"):
        d = nvq.DeviceGrid(hosts[name])
        p = _points(d, n)
        r = np.random.default_rng(7)
        gn, gv, gg = (r.normal(size=s).astype(np.float32) for s in ((n,), (n,), (n, 3)))
        gv[::3] = 0.0
        gg[::5] = 0.0
        x = torch.from_numpy(p).cuda()
        for mode in (1, 2, 3):
            acc = nvq.ops.sample_backward(d, x, *(torch.from_numpy(a).cuda() for a in (gn, gv, gg)), mode)
            want, over = oracle.sample_bwd_fixed(hosts[name], p, gn, gv, gg, mode, shift=40)
            assert not over
            assert np.array_equal(acc.cpu().numpy(), np.asarray(want).reshape(-1)), (name, mode)


def _off_block(d, n):
    """Points whose FD6 samples round out of their block: a coordinate just under a power of two or just under 0."""
    r = np.random.default_rng(n + 1)
    lo, hi = np.array(d.index_bbox[:3], np.float64), np.array(d.index_bbox[3:], np.float64) + 1
    p = (r.random((n, 3)) * (hi - lo + 8) + lo - 4).astype(np.float32)
    under = np.nextafter(np.float32([1, 2, 4, 8, 16, 32, 64]), np.float32(0))
    under = np.concatenate([under, np.float32([-1e-9, -3e-8, -1e-30]), np.nextafter(-under, np.float32(-1e9))])
    for a in range(3):
        k = slice(a * n // 4, (a + 1) * n // 4)  # whole wavefronts of them, on each axis
        p[k, a] = r.choice(under, len(p[k]))
    k = slice(3 * n // 4, 7 * n // 8)  # some lanes of a wavefront, any axes
    p[k] = np.where(r.random((len(p[k]), 3)) < 0.15, r.choice(under, (len(p[k]), 3)), p[k])
    return p


@pytest.mark.parametrize("name", ["torus", "fog_near", "torus_fp8", "torus_fpn", "far"])
@pytest.mark.parametrize("n", [5003, (1 << 20) + 37])
def test_queries_off_their_block(oracle, grids, name, n):
    """Staged (small) and binned (large) batches of them; `far` lies beyond 2^24, where p +- 1 can also land two
    cells away."""
    nvq, hosts = grids
    host = hosts.get(name)
    if name == "far":
        host = nvq.tools.create_level_set_sphere(60.0, (16777216.0 + 128.0, 0.0, 0.0), 1.0, 3.0)
    elif name == "fog_near":
        host = nvq.tools.create_fog_fbm([-40, -30, -20, 70, 64, 90], seed=5, amplitude=8.0)
    d = nvq.DeviceGrid(host)
    p = _off_block(d, n)
    if name == "far":
        p[:, 0] = 16777216.0 + 2.0 * np.random.default_rng(2).integers(30, 96, n)
    got = nvq.ops.sample(d, torch.from_numpy(p).cuda(), grad_mode=1)
    for a, b in zip(got, oracle.sample(host, p, grad_mode=1)):
        assert np.array_equal(a.cpu().numpy().view(np.uint32), np.ascontiguousarray(b).view(np.uint32))


def _far(nvq, x):
    """A grid around x = `x` whose voxels all differ: at 2^24 and beyond, p + 1 and p - 1 round to even voxels."""
    g = nvq.tools.create_level_set_sphere(60.0, (x + 128.0, 0.0, 0.0), 1.0, 3.0)
    off, count = 672 + int(np.frombuffer(g, np.int64, 1, 672)[0]), int(np.frombuffer(g, np.uint32, 1, 704)[0])
    leaves = g[off:off + 2144 * count].reshape(-1, 2144)
    leaves[:, 96:] = np.random.default_rng(8).normal(size=(count, 512)).astype(np.float32).view(np.uint8)
    return g


@pytest.mark.parametrize("x", [2.0 ** 23, 2.0 ** 24, 2.0 ** 25])
@pytest.mark.parametrize("n", [5003, (1 << 20) + 37])
def test_queries_beyond_the_exact_range(oracle, grids, x, n):
    nvq = grids[0]
    host = _far(nvq, x)
    d = nvq.DeviceGrid(host)
    r = np.random.default_rng(3)
    p = r.uniform([60, -64, -64], [196, 64, 64], (n, 3))
    p = (p + [x, 0.0, 0.0]).astype(np.float32)
    for mode in (1, 2, 3):
        got = nvq.ops.sample(d, torch.from_numpy(p).cuda(), grad_mode=mode)
        for a, b in zip(got, oracle.sample(host, p, grad_mode=mode)):
            assert np.array_equal(a.cpu().numpy().view(np.uint32), np.ascontiguousarray(b).view(np.uint32)), mode
    gn, gv, gg = (r.normal(size=s).astype(np.float32) for s in ((n,), (n,), (n, 3)))
    for mode in (1, 2, 3):
        acc = nvq.ops.sample_backward(d, torch.from_numpy(p).cuda(), *(torch.from_numpy(a).cuda() for a in (gn, gv, gg)), mode)
        want, over = oracle.sample_bwd_fixed(host, p, gn, gv, gg, mode, shift=40)
        assert not over
        assert np.array_equal(acc.cpu().numpy(), np.asarray(want).reshape(-1)), mode


@pytest.mark.parametrize("name", ["torus", "fog_near", "far"])
@pytest.mark.parametrize("n", [5003, (1 << 20) + 37])
def test_adjoint_off_their_block(oracle, grids, name, n):
    nvq, hosts = grids
    if name == "far":
        host = nvq.tools.create_level_set_sphere(60.0, (16777216.0 + 128.0, 0.0, 0.0), 1.0, 3.0)
    elif name == "fog_near":
        host = nvq.tools.create_fog_fbm([-40, -30, -20, 70, 64, 90], seed=5, amplitude=8.0)
    else:
        host = hosts[name]
    d = nvq.DeviceGrid(host)
    p = _off_block(d, n)
    if name == "far":
        p[:, 0] = 16777216.0 + 2.0 * np.random.default_rng(2).integers(30, 96, n)
    r = np.random.default_rng(n)
    gn, gv, gg = (r.normal(size=s).astype(np.float32) for s in ((n,), (n,), (n, 3)))
    gv[::3] = 0.0
    gn[::4] = 0.0
    gg[::5] = 0.0
    acc = nvq.ops.sample_backward(d, torch.from_numpy(p).cuda(), *(torch.from_numpy(a).cuda() for a in (gn, gv, gg)), 1)
    want, over = oracle.sample_bwd_fixed(host, p, gn, gv, gg, 1, shift=40)
    assert not over
    assert np.array_equal(acc.cpu().numpy(), np.asarray(want).reshape(-1))
