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
    fresh run's; a failed run starts over as well."""
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
