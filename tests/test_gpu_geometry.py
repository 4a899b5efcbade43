"""The geometry kernel (normals, curls and records from the vertices) and its
checks, on meshes around its 256-triangle workgroups.  The arrays are FP64
values rounded once, so they match numpy's to one FP32 rounding."""
import ctypes
import threading

import numpy as np
import pytest
import torch

from neuralat_amd import _lib, mesh

pytestmark = pytest.mark.gpu


def _dev():
    return torch.device("cuda:0")


def _normals_curls(v, t):
    e = v[t].astype(np.float64)
    c = np.cross(e[:, 1] - e[:, 0], e[:, 2] - e[:, 0])
    J = np.linalg.norm(c, axis=1)
    curls = np.stack([e[:, 1] - e[:, 2], e[:, 2] - e[:, 0], e[:, 0] - e[:, 1]], 1) / J[:, None, None]
    return c / J[:, None], curls


@pytest.mark.parametrize("nt", [1, 255, 256, 257, 320])
def test_normals_and_curls(nt):
    from neuralat_amd.bem import Mesh

    v, t = mesh.icosphere(2, 0.1)
    v = mesh.sh_perturb(v, 4, 0.05, seed=nt).astype(np.float32)
    t = t[:nt]
    used, t = np.unique(t, return_inverse=True)
    v, t = v[used], t.reshape(-1, 3).astype(np.int32)
    print("geometry", nt, flush=True)
    m = Mesh(torch.tensor(v, device=_dev()), torch.tensor(t, device=_dev()))
    moved = (v * np.float32(1.7) + np.float32(0.3)).astype(np.float32)
    for x, source in ((v, None), (moved, "device"), (v, "host")):
        if source == "device":
            m.set_vertices(torch.tensor(x, device=_dev()))
        elif source == "host":
            _lib.check(_lib.load().bem_mesh_set_vertices(m.handle, x.ctypes.data, 0, ctypes.c_void_p(0)))
        n, c = (a.cpu().numpy() for a in m.normals_curls())
        rn, rc = _normals_curls(x, t)
        assert np.abs(n - rn).max() < 1.2e-7
        assert np.abs(c - rc).max() < 1.2e-7 * np.abs(rc).max()


def test_faults_are_reported_and_change_nothing():
    from neuralat_amd.bem import GeometrySet, Mesh

    v, t = mesh.icosphere(1, 0.1)
    v = v.astype(np.float32)
    nan, flat = v.copy(), v.copy()
    nan[7, 1] = np.nan
    flat[t[5, 1]] = flat[t[5, 0]]
    for bad, what in ((nan, "non-finite"), (flat, "zero area")):
        with pytest.raises(ValueError, match=what):
            Mesh(torch.tensor(bad, device=_dev()), torch.tensor(t, device=_dev()))
    m = Mesh(torch.tensor(v, device=_dev()), torch.tensor(t, device=_dev()))
    before = m.normals_curls()[0].clone()
    for bad, what in ((nan, "non-finite"), (flat, "zero area")):
        with pytest.raises(ValueError, match=what):
            m.set_vertices(torch.tensor(bad, device=_dev()))
        with pytest.raises(ValueError, match=f"sample 2: .*{what}"):
            GeometrySet(m, np.stack([v, v, bad, v]))
    assert torch.equal(before, m.normals_curls()[0])


def test_positions_outside_the_device_are_copied():
    """Positions that are not an allocation of the mesh's own GPU (here pinned host
    memory passed as device memory) are copied, not read in place."""
    from neuralat_amd.bem import Mesh

    v, t = mesh.icosphere(1, 0.1)
    v = v.astype(np.float32)
    m = Mesh(torch.tensor(v, device=_dev()), torch.tensor(t, device=_dev()))
    moved = torch.tensor(v * np.float32(1.3) + np.float32(0.1)).pin_memory()
    print("positions in pinned memory", flush=True)
    _lib.check(_lib.load().bem_mesh_set_vertices(m.handle, moved.data_ptr(), 1, ctypes.c_void_p(0)))
    n, c = (a.cpu().numpy() for a in m.normals_curls())
    rn, rc = _normals_curls(moved.numpy(), t)
    assert np.abs(n - rn).max() < 1.2e-7 and np.abs(c - rc).max() < 1.2e-7 * np.abs(rc).max()


def test_setup_does_not_wait_for_another_stream():
    """A geometry set created behind other work on its stream holds the pinned
    stage until its upload is done; a mesh created by another thread on another
    stream meanwhile stages elsewhere and finishes first."""
    from neuralat_amd.bem import GeometrySet, Mesh

    v, t = mesh.icosphere(2, 0.1)
    v = v.astype(np.float32)
    vt, tt = torch.tensor(v, device=_dev()), torch.tensor(t, device=_dev())
    base = Mesh(vt, tt)
    busy, other = torch.cuda.Stream(), torch.cuda.Stream()
    big = torch.randn(8192, 8192, device=_dev())
    kept = [big @ big]  # the library's own set-up and the allocation, done before
    torch.cuda.synchronize()
    print("set-up beside a busy stream", flush=True)

    def queue_and_create():
        with torch.cuda.stream(busy):
            for _ in range(60):  # 7 ms each
                torch.mm(big, big, out=kept[0])
            queued.set()
            kept.append(GeometrySet(base, np.stack([v, v * np.float32(1.1)])))

    queued = threading.Event()
    a = threading.Thread(target=queue_and_create)
    a.start()
    assert queued.wait(30)
    a.join(0.05)  # into the upload
    assert a.is_alive()
    with torch.cuda.stream(other):
        m = Mesh(vt, tt)
        first = a.is_alive()
    a.join()
    assert first, "the mesh waited for the other thread's stream"
    n, _ = m.normals_curls()
    torch.cuda.synchronize()
    assert np.abs(n.cpu().numpy() - _normals_curls(v, t)[0]).max() < 1.2e-7
