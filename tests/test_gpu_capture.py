"""Ray queries recorded into a graph: on a stream without scratch, and on one whose scratch block a later call
replaces by a larger one.  Every replay against the eager call, bit for bit, with eager work between the replays."""
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

RAYS = (1 << 19) + 65  # 8194 tiles: the march takes them longest first, which needs scratch


@pytest.fixture(scope="module")
def scene():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import openvdb_amd as nvq
    fog = nvq.DeviceGrid(nvq.tools.create_fog_fbm([-41, -9, 16, 56, 70, 91], seed=9))
    ball = nvq.DeviceGrid(nvq.tools.create_level_set_sphere(37.0, (1.5, -2.0, 3.0), 1.0, 3.0))
    big = nvq.DeviceGrid(nvq.tools.create_level_set_torus(300.0, 80.0, (0.0, 0.0, 0.0), 1.0, 3.0))
    r = np.random.default_rng(4)
    eye = r.normal(size=(RAYS, 3))
    eye = 300.0 * eye / np.linalg.norm(eye, axis=1, keepdims=True)
    aim = r.uniform([-41, -9, 16], [56, 70, 91], (RAYS, 3))
    eye, dirs = (torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).cuda() for x in (eye, aim - eye))
    calls = {
        "march": lambda: nvq.ops.fog_march(fog, eye, dirs, 0.5, 0.05),
        "multi": lambda: nvq.ops.multi_query([fog, ball], eye, dirs, [0, RAYS // 2, RAYS], [0, 0], 0.5, 0.05),
        "iso": lambda: nvq.ops.render_iso_surface(ball, nvq.tools.iso_camera(ball_host(nvq), 333, 121)),
    }
    return nvq, big, eye, dirs, calls


def ball_host(nvq):
    return nvq.tools.create_level_set_sphere(37.0, (1.5, -2.0, 3.0), 1.0, 3.0)


def _replay(graph, out, want, eager):
    for _ in range(3):
        for x in out:
            x.fill_(7)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip(out, want):
            assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
        eager()


@pytest.mark.parametrize("name", ["march", "multi", "iso"])
def test_capture_on_a_stream_without_scratch(scene, name):
    call = scene[4][name]
    want = call()
    torch.cuda.synchronize()
    s, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        out = call()
    _replay(graph, out, want, call)


@pytest.mark.parametrize("name", ["march", "multi", "iso"])
def test_scratch_of_a_graph_outlives_larger_calls(scene, name):
    nvq, big, eye, dirs, calls = scene
    call = calls[name]
    s, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        want = call()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=s):
        out = call()
    points = torch.randn(1 << 20, 3, device="cuda") * 100.0

    def grow():  # a slot map of the torus, then 120 MB of sort buffers
        with torch.cuda.stream(s):
            nvq.ops.zero_crossing(big, eye, dirs)
            nvq.ops.sample(big, points)
        torch.cuda.synchronize()
    grow()
    _replay(graph, out, want, grow)
