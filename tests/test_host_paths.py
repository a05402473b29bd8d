"""What the library's host code allocates, launches and waits for, on the
stand-in HIP runtime (tests/fake_hip): no GPU."""
from __future__ import annotations

import fakehip
import pytest

pytestmark = fakehip.needed


@pytest.mark.parametrize("copies", [1, 8])
def test_tallies_wait_for_every_stream(copies):
    """A run may have been given a stream that does not wait for the plan's:
    the device is waited for before the packets are counted and before the
    fluence is copied into linear order."""
    r = fakehip.run(f"""
        import models
        m = models.base(n=10)
        plan = api.MCPlan(m)
        plan.set_fluence_copies({copies})
        plan.simulate(100, stream=C.c_void_p(0x20))
        log()
        plan.tallies()
        result(log=log())
    """)
    events = [ln.split()[0] + " " + ln.split()[1] for ln in r["log"]]
    device = events.index("sync device")
    assert not any(e.startswith(("launch", "memcpy")) for e in events[:device])
    assert any("mc_linear_nfr" in e for e in events[device:])
