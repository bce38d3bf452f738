"""What tgmm_batch_time_kernel reports as a launch's bytes: of the search, those
of the queries that the iterations searched for and looked at; of the others,
what their kernels read and write, in both modes."""
import pytest

from tgmm_amd import em
from test_gpu_knn_look import _resting

pytestmark = pytest.mark.gpu

K, ITERS = 5, 24


@pytest.fixture(scope="module")
def frame():
    return _resting()


def _batch(frame, lanes, voxel=False):
    b = em.Batch([frame], em.make_opts(K=K, max_iter=ITERS, scale=(1.0, 1.0, 5.0), voxel=voxel))
    b.set_tiles(dict(b.get_tiles(), knn_lanes=lanes))
    return b


@pytest.mark.parametrize("lanes", [0, 1, 2, 4, 64])
def test_search(frame, lanes):
    S, G = frame.S, frame.G
    whole, look = S * (16 + 8 * K) + 32 * G, 8 * S
    with _batch(frame, lanes) as b:
        ms, first = b.time_kernel("knn", 1)  # the first iteration searches whole
        assert ms > 0 and first == whole
        ms, avg = b.time_kernel("knn", ITERS)
    print("lanes %d: %.0f of %d bytes a launch" % (lanes, avg, whole), flush=True)
    # most means rest after a few iterations: those only look, and search little
    assert (whole + (ITERS - 1) * look) / ITERS <= avg < 0.6 * whole


def test_others(frame):
    S, G, N = frame.S, frame.G, frame.N
    with _batch(frame, 2) as b:
        got = {k: b.time_kernel(k, 3)[1] for k in ("loglik", "estep", "mstep")}
    assert got == dict(loglik=8 * N + S * (44 + 4 * K) + 64 * G, estep=S * (84 + 8 * K) + 96 * G,
                       mstep=125 * G + 88 * S)
    with _batch(frame, 2, voxel=True) as b:
        got = {k: b.time_kernel(k, 3)[1] for k in ("loglik", "estep", "mstep")}
    assert got == dict(loglik=N * (20 + 4 * K) + 64 * G, estep=N * (20 + 8 * K) + 96 * G,
                       mstep=125 * G + 20 * N)
