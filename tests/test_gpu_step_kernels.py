"""The batch tests once more on the step kernels and their graphs: runs of small
slabs are resident by default, and graphs of steps are then never replayed."""
import pytest

from cardioid_amd import hip
import test_gpu_batch as TB
import test_gpu_checkpoint as TC
import test_gpu_serve as TS

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module", autouse=True)
def gpu():
    if not torch.cuda.is_available():
        pytest.skip("no HIP device")
    hip.lib()
    yield


@pytest.fixture
def closed(monkeypatch):
    """hip.Batch with the resident form off; the batches closed so far, each of
    which is asserted to have run no resident step."""
    done = []

    class StepBatch(hip.Batch):
        def __init__(self, *args, **kw):
            super().__init__(*args, **kw)
            self.set_resident(False)

        def close(self):
            if self.h:
                done.append(self.resident())
                assert done[-1] == {"on": False, "steps": 0, "tiles": 0}
            super().close()

    monkeypatch.setattr(hip, "Batch", StepBatch)
    return done


def test_fp64_batch_matches_oracle_per_slab(closed):
    TB.test_fp64_batch_matches_oracle_per_slab()
    assert len(closed) == 1


@pytest.mark.parametrize("mode", ["fp64_fused", "mixed_fused"])
def test_arrivals_and_departures_with_graphs(closed, mode):
    TB.test_alone_equals_in_batch_with_arrivals_and_departures(mode)
    assert len(closed) == 5


def test_graph_replay_equals_direct_launches(closed):
    TB.test_graph_replay_equals_direct_launches()
    assert len(closed) == 3


@pytest.mark.parametrize("mode", ["fp64_fma", "mixed_fused"])
def test_graph_follows_the_live_tiles(closed, mode):
    TB.test_graph_follows_the_live_tiles(mode)
    assert closed


def test_configuration_A(closed):
    TB.test_configuration_A_batch_alone_equals_in_batch_and_other_modes_refuse()
    assert closed


@pytest.mark.parametrize("mode,tol", [("fp64_fused", 0.0), ("mixed_fused", 0.01)])
def test_evicted_and_resumed(closed, tmp_path, mode, tol):
    TC.test_batch_slab_evicted_and_resumed(tmp_path, mode, tol)
    assert closed


def test_requests_alone_equal_requests_in_the_mix(closed):
    TS.test_results_alone_equal_results_in_the_mix()
    assert closed
