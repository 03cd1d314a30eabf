"""Which form a ray query takes where the size rules turn a slot map away, and that all forms give the same bits.

A grid's root bbox is stretched, so that the same leaves lie in a box of few slots (map), of more than 2^23
(a map for the march, none for the adjoint's block cache) or of more than 2^24 (no map).  The rays start inside
the smallest of these boxes, so that every form walks the same cells.
"""
import ctypes

import numpy as np
import pytest
from test_gpu_slots import _grid, _host, _level_set

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def nvq():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import openvdb_amd
    return openvdb_amd


def _launches(nvq, name, call):
    """call()'s result and how often the library recorded `name` in it."""
    lib, ms, n = nvq.lib(), ctypes.c_double(), ctypes.c_uint64()
    lib.nvq_profile_reset()
    lib.nvq_profile_enable(1)
    try:
        out = call()
        torch.cuda.synchronize()
    finally:
        lib.nvq_profile_enable(0)
    lib.nvq_profile_read(name.encode(), ctypes.byref(ms), ctypes.byref(n))
    return out, n.value


def _stretched(host, edge):
    """A copy whose root bbox reaches from -256 over `edge` voxels on every axis."""
    g = host.copy()
    root = 672 + int(np.frombuffer(g, np.int64, 4, 672)[3])
    g[root:root + 24] = np.array([-256] * 3 + [edge - 257] * 3, np.int32).view(np.uint8)
    return g


# slots per axis: edge / 8 + 3
EDGES = {"map": 512, "march only": 8 * 220, "none": 8 * 260}


def _rays(n, seed):
    r = np.random.default_rng(seed)
    eye, aim = r.uniform(-250.0, 250.0, (n, 3)), r.uniform(0.0, 80.0, (n, 3))
    eye[:n // 8] = r.uniform(0.0, 80.0, (n // 8, 3))  # inside the fog
    return (torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).cuda() for x in (eye, aim - eye))


def _forms(nvq, name):
    if name == "onindex":
        ijk, values = nvq.tools.active_voxels(_host(nvq, "fog"))
        d, index = nvq.DeviceGrid.from_voxels(torch.from_numpy(ijk).cuda(), "OnIndex", return_index=True)
        channel = torch.zeros(d.value_count, device="cuda")
        channel[index] = torch.from_numpy(values).cuda()
        host = d.download()
    else:
        host, channel = _host(nvq, name), None
    forms = {}
    for k, edge in EDGES.items():
        forms[k] = nvq.DeviceGrid(nvq.aligned_buffer(_stretched(host, edge)))
        if channel is not None:
            forms[k].set_channel(channel)
    return forms


@pytest.mark.parametrize("name", ["fog", "tiles", "flagged", "onindex"])
@pytest.mark.parametrize("n", [65, 50021])
def test_adjoint_is_the_same_in_every_form(nvq, name, n):
    forms = _forms(nvq, name)
    eye, dirs = _rays(n, n)
    r = torch.Generator(device="cuda")
    r.manual_seed(n)
    gL, gT = (torch.randn(n, generator=r, device="cuda") for _ in range(2))
    out = {}
    for k, d in forms.items():
        (L, T), maps = _launches(nvq, "slot_map", lambda: nvq.ops.fog_march(d, eye, dirs, 0.5, 0.05))
        assert maps == (1 if k == "map" or (k == "march only" and n > 50000) else 0)  # 256 slots per ray
        acc, maps = _launches(nvq, "slot_map", lambda: nvq.ops.fog_march_backward(d, eye, dirs, L, gL, T, gT, 0.5, 0.05))
        assert maps == (1 if k == "map" else 0), k
        out[k] = (L, T, acc)
    assert float(out["map"][0].max()) > 0.0 and int(out["map"][2].ne(0).sum()) > 1000
    for k in ("march only", "none"):
        for a, b in zip(out["map"], out[k]):
            assert torch.equal(a, b), k


def test_adjoint_of_few_rays(nvq):
    """Three rays through the accessor, four with the block cache: the fourth's gradients are zero."""
    d = nvq.DeviceGrid(_host(nvq, "fog"))
    eye, dirs = _rays(8, 2)  # the first inside the fog
    eye, dirs = eye[:4].contiguous(), dirs[:4].contiguous()
    gL = torch.tensor([1.0, -2.0, 0.5, 0.0], device="cuda")
    L, T = nvq.ops.fog_march(d, eye, dirs, 0.5, 0.05)
    out = []
    for n, maps in ((4, 1), (3, 0)):
        x = [a[:n].contiguous() for a in (eye, dirs, L, gL, T, gL)]
        acc, built = _launches(nvq, "slot_map", lambda: nvq.ops.fog_march_backward(d, *x, 0.5, 0.05))
        assert built == maps
        out.append(acc)
    assert torch.equal(*out) and int(out[0].ne(0).sum()) > 10


@pytest.mark.parametrize("rays,maps", [(63, 0), (64, 1), (4097, 1)])
def test_crossings_take_a_map_where_it_pays(nvq, rays, maps):
    """Around the number of rays from which a sphere's crossing takes a map; the smaller call is the larger one's
    first rays, through the accessor."""
    d = nvq.DeviceGrid(nvq.tools.create_level_set_sphere(37.0, (1.5, -2.0, 3.0), 1.0, 3.0))
    eye, dirs = _rays(rays, 5)
    got, built = _launches(nvq, "slot_map", lambda: nvq.ops.zero_crossing(d, eye, dirs))
    assert built == maps
    part, built = _launches(nvq, "slot_map", lambda: nvq.ops.zero_crossing(d, eye[:63].contiguous(), dirs[:63].contiguous()))
    assert built == 0
    for a, b in zip(got, part):
        assert torch.equal(a[:63].contiguous().view(torch.uint8), b.view(torch.uint8))


def _voxels(d, n, seed):
    """Inside leaves, on tiles and background in the bbox, on the table's rim, around it, far out, at the ends of
    the integer range; n not a multiple of a wavefront."""
    r = np.random.default_rng(seed)
    lo, hi = np.array(d.index_bbox[:3], np.int64), np.array(d.index_bbox[3:], np.int64) + 1
    ijk = r.integers(lo - 3, hi + 3, (n, 3))
    k = n // 16
    ijk[:k] = r.integers(lo - 40, hi + 40, (k, 3))
    ijk[k:2 * k] = r.integers(-2 ** 31, 2 ** 31, (k, 3))
    rim = np.stack([(lo >> 3 << 3) - 9, (lo >> 3 << 3) - 8, (hi >> 3 << 3) + 15, (hi >> 3 << 3) + 16, (hi >> 3 << 3) + 24])
    ijk[2 * k:3 * k] = np.where(r.random((k, 3)) < 0.5, rim[r.integers(0, 5, k)], ijk[2 * k:3 * k])
    ends = np.array([-2 ** 31, -2 ** 31 + 7, 2 ** 31 - 1, 2 ** 31 - 8, -1, 0])
    ijk[3 * k:3 * k + 512] = r.choice(ends, (512, 3))
    return np.ascontiguousarray(ijk.astype(np.int32))


@pytest.mark.parametrize("name,codec", [("fog", c) for c in ("float", "fp4", "fp8", "fp16", "fpn", "onindex")] +
                         [("tiles", "float"), ("tiles", "fp8"), ("flagged", "float"), ("sphere", "fp16")])
def test_large_value_batches_equal_small_ones(nvq, oracle, name, codec):
    """getValue through the slot table (from 2^22 voxels on, not FpN) against the same voxels in smaller batches
    through the tree, and against the oracle."""
    host = _level_set(nvq, name) if name == "sphere" else _host(nvq, name)
    d = _grid(nvq, host, codec)
    n = (1 << 22) + 37
    ijk = _voxels(d, n, 3)
    x = torch.from_numpy(ijk).cuda()
    got, maps = _launches(nvq, "slot_map", lambda: nvq.ops.get_value(d, x, want_dim=True))
    assert maps == (0 if codec == "fpn" else 1)
    pieces, maps = _launches(nvq, "slot_map", lambda: [nvq.ops.get_value(d, y.contiguous(), want_dim=True) for y in x.split(1 << 21)])
    assert maps == 0
    for a, b in zip(got, zip(*pieces)):
        assert torch.equal(a.view(torch.uint8), torch.cat(b).view(torch.uint8))
    if codec == "float":
        for a, b in zip(got, oracle.get_value(host, ijk[:300000])):
            assert np.array_equal(a[:300000].cpu().numpy().view(np.uint8), np.ascontiguousarray(b).view(np.uint8))
    assert 1000 < int(got[1].sum()) < n


def test_value_table_limits(nvq):
    """One voxel below the batch size, and a box of more slots than the table takes: through the tree."""
    d = nvq.DeviceGrid(_host(nvq, "fog"))
    x = torch.zeros(1 << 22, 3, dtype=torch.int32, device="cuda")
    assert _launches(nvq, "slot_map", lambda: nvq.ops.get_value(d, x[:-1]))[1] == 0
    assert _launches(nvq, "slot_map", lambda: nvq.ops.get_value(d, x))[1] == 1
    wide = nvq.DeviceGrid(nvq.aligned_buffer(_stretched(_host(nvq, "fog"), 8 * 78)))  # 81^3 slots
    assert _launches(nvq, "slot_map", lambda: nvq.ops.get_value(wide, x))[1] == 0
