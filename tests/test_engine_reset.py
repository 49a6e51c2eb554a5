"""QeRun reset: a run's own buffers hold the states of a fresh run again."""
import numpy as np
import pytest

from conftest import GOLDEN, ROOT
from qwen_mi355x import engine as E
from qwen_mi355x import model as M

OPS_BRIDGE = ROOT / "oracle" / "lib" / "libqwen_ops_bridge.so"


@pytest.mark.parametrize("device", [False, pytest.param(True, marks=pytest.mark.gpu)])
def test_reset_equals_a_fresh_run(device):
    """Every state part is zero after a reset whatever wrote it (a prefill, a
    step, a write of states), the snapshots included, and the outputs are a
    fresh run's; a call that is refused before it runs changes nothing of that."""
    fixture = M.load_fixture(GOLDEN / "hybrid.json")
    c, w = M.fixture_config_and_weights(fixture)
    m = E.Model(w) if device else E.Model(w, bridge=OPS_BRIDGE, kind=E.KIND_CPU_TEST)
    ids = fixture["ids"]
    capacity = len(ids) + 4
    want = m.new_run(capacity, chunk=3).prefill(ids)
    run = m.new_run(capacity, chunk=3, snapshots=2)
    layer = c.layer_types.index("full_attention")
    for _ in range(2):
        run.prefill(ids)
        run.step(ids[0])
        run.verify_rollback(ids[:2])
        run.set_position(capacity)
        run.write_state(layer, 2, np.ones(run.state_size(layer, 2), np.float32))
        run.reset()
        assert run.position == 0
        run.set_position(capacity)
        for part, v in run.inspect_state().items():
            assert not v.any(), part
        run.reset()
        assert np.array_equal(run.prefill(ids), want)
        run.reset()
    with pytest.raises(E.EngineError):
        run.step(10**6)
    run.reset()
    assert np.array_equal(run.prefill(ids), want)


@pytest.mark.parametrize("device", [False, pytest.param(True, marks=pytest.mark.gpu)])
@pytest.mark.parametrize("how", ["step", "prefill", "verify"])
def test_failed_run_starts_over(device, how):
    """A forward that fails on the way (keys so large that the scores and then the
    logits are not finite) leaves the run refused until a reset, which builds it anew: its
    states are zero, its outputs and its one-launch plan a fresh run's."""
    fixture = M.load_fixture(GOLDEN / "hybrid.json")
    c, w = M.fixture_config_and_weights(fixture)
    m = E.Model(w) if device else E.Model(w, bridge=OPS_BRIDGE, kind=E.KIND_CPU_TEST)
    ids = fixture["ids"]
    capacity = len(ids) + 4
    fresh = m.new_run(capacity, chunk=3, snapshots=2)
    want = fresh.prefill(ids)
    want_step = fresh.step(ids[0])
    run = m.new_run(capacity, chunk=3, snapshots=2)
    layer = c.layer_types.index("full_attention")
    call = {"step": lambda: run.step(ids[0]), "prefill": lambda: run.prefill(ids),
            "verify": lambda: run.verify_rollback(ids[:2])}[how]
    for _ in range(2):
        run.prefill(ids[:3])
        run.write_state(layer, 2, np.full(run.state_size(layer, 2), 3e38, np.float32))  # scores overflow
        with pytest.raises(E.EngineError, match="NaN/Inf|non-finite"):
            call()
        with pytest.raises(E.EngineError, match="failed"):
            call()
        with pytest.raises(E.EngineError, match="poisoned"):
            run.state(layer, 2)
        run.reset()
        assert run.position == 0 and run.decode_plan == fresh.decode_plan
        run.set_position(capacity)
        for part, v in run.inspect_state().items():
            assert not v.any(), part
        run.reset()
        assert np.array_equal(run.prefill(ids), want)
        assert np.array_equal(run.step(ids[0]), want_step)
        run.reset()
