"""A batch step that fails after some of its iterations are queued: the next poll reports the states the device has."""
import numpy as np
import pytest

from eggpu_amd import native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [9, 14])  # one reduce launch, and two
@pytest.mark.parametrize("graphs", ["0", "1"])
def test_poll_after_a_failed_step(gpu_ready, monkeypatch, scale, graphs):
    print(f"failed step scale={scale} graphs={graphs}", flush=True)
    monkeypatch.setenv("EGGPU_AMD_BATCH_GRAPHS", graphs)
    with native.DeviceGraph.rmat(scale, 8, seed=3) as g:
        monkeypatch.setenv("EGGPU_AMD_TEST_FAIL_STEP", "3")
        failing = g.batch()
        monkeypatch.delenv("EGGPU_AMD_TEST_FAIL_STEP")
        plain = g.batch()
        try:
            for b in (failing, plain):
                b.assign(0, [1, 2], max_iter=100, tol=0.0)
                b.step(2)
                assert b.poll()["iterations"][0] == 2
                b.step(2)
            with pytest.raises(native.EgxError):
                failing.step(5)
            # launched one by one, three iterations were queued; a captured step never runs
            done = 4 + (3 if graphs == "0" else 0)
            if done > 4:
                plain.step(done - 4)
            got, want = failing.poll(), plain.poll()
            assert got["iterations"][0] == done
            assert all(np.array_equal(got[k], want[k]) for k in got)
            failing.step(1)
            plain.step(1)
            assert failing.poll()["iterations"][0] == done + 1
            assert np.array_equal(failing.result(0), plain.result(0))
        finally:
            failing.close()
            plain.close()
