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


HEAT = """
from test_gpu_heat_lines import line_case
T0, Om0, P = line_case((35, 21, 18), 0.3, steps=6)
"""


def modes(log):
    """The modes (0 row by row, 1 from factors, 2 building them) of the FP32 line sweeps launched."""
    names = [ln.split()[1] for ln in log if "heat_sweep_lines32" in ln]
    return {int(n.split("heat_sweep_lines32")[1].split("ELi")[2].split("EL")[0]) for n in names}


@pytest.mark.parametrize("room", [0, 1, 2, 3])  # of the three line factors
def test_fp32_runs_without_memory_for_line_factors(room):
    r = fakehip.run(HEAT + f"""
plan = api.HeatPlan(T0, Om0, P, precision="fp32", graph_steps=2)
voxels = 35 * 21 * 18
fake.fake_peak(1)
before = fake.fake_peak(0)
fake.fake_set_limit(before + {room} * voxels * 4)
log()
plan.advance(6, 0.3, 1)
first = log()
fake.fake_peak(1)
held = fake.fake_peak(0) - before
fake.fake_set_limit(1 << 40)
plan.advance(6, 0.3, 1)
result(first=first, held=held, second=log(), voxels=voxels)
""")
    # with too little room: none kept, rows computed on the way; used when there is room again
    assert modes(r["first"]) == ({1, 2} if room == 3 else {0})
    assert r["held"] == (12 * r["voxels"] if room == 3 else 0)
    assert modes(r["second"]) == (set() if room == 3 else {1, 2})  # (a replay of the first run's graph launches no kernel)


ADJOINT = """
from test_gpu_heat_lines import line_case
T0, Om0, P = line_case((16, 16, 16), 0.05, steps=200)
state = 16 ** 3 * 8
def peak(**kw):
    fake.fake_peak(1)
    r = api.heat_adjoint(T0, Om0, P, **kw)
    return fake.fake_peak(1)
"""


def test_adjoint_falls_back_to_checkpoints_when_the_kept_states_leave_no_room():
    """The states that are kept where they fit never take the room of what the
    reverse sweep cannot do without."""
    r = fakehip.run(ADJOINT + """
base = peak(grads=False, checkpointEvery=200) - state  # less its one checkpoint
peaks = []
# from room for the checkpointed run (10 checkpoints and 21 states of a segment beside the sweep's 6 fields) to more
# than the kept one needs
for states in (40, 100, 200, 203, 206, 207, 208, 300):
    fake.fake_set_limit(base + states * state)
    peaks.append((peak(checkpointEvery=20) - base) / state)
result(peaks=peaks)
""")
    assert all(p < 40 for p in r["peaks"][:5]) and all(p > 200 for p in r["peaks"][5:])


def test_adjoint_memory_is_bounded_by_the_caller():
    """Kept states take at most 1 GiB beside an explicit checkpoint period (4 GiB
    without one), what the caller allows, or what the checkpoints would take;
    calls that run together share the limit."""
    r = fakehip.run(ADJOINT + """
base = peak(grads=False, checkpointEvery=200) - state
sweep = 6 * state
def states(**kw):
    return (peak(**kw) - base - sweep) / state
out = dict(
    default=states(),
    period=states(checkpointEvery=20),
    none=states(checkpointEvery=20, maxStateBytes=0),          # 10 checkpoints, 21 states of a segment
    short=states(checkpointEvery=20, maxStateBytes=200 * state),
    enough=states(checkpointEvery=20, maxStateBytes=201 * state),
    asked=states(checkpointEvery=200, maxStateBytes=0),        # as many as one segment
    unset=states(maxStateBytes=0),                             # every 100 steps
)
limits = []
def note(*a, **kw):
    limits.append(kw["maxStateBytes"])
api.heat_adjoint = note
one = (T0, Om0, P, None)
api.heat_adjoints([one] * 8, workers=4, checkpointEvery=20)
api.heat_adjoints([one] * 2, workers=4)
api.heat_adjoints(iter([one] * 8), workers=8, maxStateBytes=800)
result(out=out, limits=sorted(set(limits)))
""")
    assert r["out"] == {"default": 201, "period": 201, "none": 31, "short": 31, "enough": 201, "asked": 201, "unset": 103}
    assert r["limits"] == [100, 1 << 28, 2 << 30]


def test_adjoint_refuses_a_negative_memory_limit():
    r = fakehip.run(ADJOINT + """
try:
    peak(maxStateBytes=-1)
    result(code=0)
except _lib.MCMError as e:
    result(code=e.code)
""")
    assert r["code"] == -1


@pytest.mark.parametrize("kind", ["batch", "multi"])
def test_fluence_copies_of_a_batch_follow_its_packets(kind):
    """Copies pay by the packet and cost by the voxel: n copies from n packets in
    256 voxels."""
    r = fakehip.run(f"""
import models
plan = api.MCPlan(models.base(n=40))
out = {{}}
for packets in (1, 499, 501, 999, 1001, 1999, 2001, 20000):
    items = [(0, packets, 1, 0)] * 16
    log()
    plan.batch(items) if {kind == "batch"} else api.multi_run([plan], [(0, *it) for it in items])
    slices = [int(l.split()[1]) / (16 * 40 ** 3 * 8) for l in log() if l.startswith("malloc ")]
    out[packets] = max(slices)
result(**{{str(k): v for k, v in out.items()}})
""")
    assert r == {"1": 1, "499": 1, "501": 2, "999": 2, "1001": 4, "1999": 4, "2001": 8, "20000": 8}


def test_a_multi_grid_launch_downloads_through_one_pinned_block():
    r = fakehip.run("""
import models
m = models.base(n=130)
plans = [api.MCPlan(m) for _ in range(3)]
log()
api.multi_run(plans, [(k, 0, 100, 1, 0) for k in range(3)])
result(pinned=[l for l in log() if l.startswith("pinned")])
""")
    assert len(r["pinned"]) == 1


def covered(log, kernel):
    """Workgroups of each launch of a kernel."""
    return [int(ln.split()[2]) for ln in log if ln.startswith("launch ") and kernel in ln]


@pytest.mark.parametrize("kind", ["criteria", "plain", "batch", "multi", "grad"])
def test_runs_take_smaller_launches_where_packet_records_do_not_fit(kind):
    """A launch's records (64 bytes a packet, 112 with escapes) are the only
    memory a run needs by the packet: with room for an eighth of them the run is
    cut into eight launches, with no room for 4096 packets it is refused."""
    r = fakehip.run(f"""
import models
kind = {kind!r}
m = models.cases()["criteria_scatter" if kind == "criteria" else "pencil_bt1"]()
plan = api.MCPlan(m)
N = 1 << 20
size = 64 if kind in ("criteria", "grad") else 112
def go():
    if kind == "batch":
        plan.batch([(0, N, 1, 0)])
    elif kind == "multi":
        api.multi_run([plan], [(0, 0, N, 1, 0)])
    elif kind == "grad":
        plan.absorbed_power(((0, 1), (0, 1), (0, 1)), N)
    else:
        plan.simulate(N)
# what the call needs beside the records
other = api.MCPlan(m)
plan, kept = other, plan
fake.fake_peak(1)
before = fake.fake_peak(0)
go()
rest = fake.fake_peak(1) - before - size * N
other.close()
plan = kept
fake.fake_peak(1)
before = fake.fake_peak(1)
log()
fake.fake_set_limit(before + rest + size * N // 8)
go()
cut = log()
used = fake.fake_peak(1) - before - rest
plan.close()
plan = api.MCPlan(m)
fake.fake_peak(1)
fake.fake_set_limit(fake.fake_peak(1) + rest + size * 4000)
try:
    go()
    code = 0
except _lib.MCMError as e:
    code = e.code
result(cut=cut, used=used, whole=size * N // 8, code=code)
""")
    kernel = "mc_gradI" if kind == "grad" else "mc_transport"
    assert len(covered(r["cut"], kernel)) == 8
    assert r["used"] == r["whole"]
    assert r["code"] == -2


BIG = """
from test_gpu_heat_lines import line_case
T0, Om0, P = line_case((128, 128, 129), 0.05, steps=0)
plan = api.HeatPlan(T0, Om0, P)
log()
"""


def test_large_downloads_do_without_threads():
    """A thread that cannot be started, for whatever reason, leaves its stripe to the caller's."""
    r = fakehip.run(BIG + """
fake.fake_fail_threads(1)
plan.download(f64=False)
result(bytes=sum(int(l.split()[1]) for l in log() if l.startswith("download ")), L=int(T0.size))
""")
    assert r["bytes"] >= 8 * r["L"]  # T and Omega


@pytest.mark.parametrize("nth", [1, 3, 5])
def test_a_failed_download_leaves_nothing_under_way(nth):
    """The other stripes' copies into the pinned block have ended before the error
    is returned: the block is used again, or freed, by what comes next."""
    r = fakehip.run(BIG + f"""
fake.fake_fail_downloads({nth})
try:
    plan.download(f64=False)
    code = 0
except _lib.MCMError as e:
    code = e.code
result(code=code, log=log())
""")
    assert r["code"] == -3
    assert r["log"][-1] == "sync stream"
