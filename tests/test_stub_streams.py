"""Host-side order of the engine's work, with the device left out
(stub_lib): what is still running when a call returns."""
from __future__ import annotations

import stub_lib


def test_adjoint_that_fails_leaves_nothing_running():
    """Each device allocation of a first adjoint fails in turn: when the call
    returns, no stream holds work that reads the caller's cotangent."""
    out = stub_lib.run("""
        st = state()
        for k in range(20):
            with ag.Context(0) as ctx, ag.Analytic(ctx, st) as e:
                maps, dmaps = device(4 * st.n_maps * st.points), device(4 * st.n_maps * st.points)
                e.forward(maps)
                before = stub.stub_launches()
                stub.stub_fail_from(k)
                try:
                    e.adjoint(dmaps)
                except ag.AgError as err:
                    print("failed", k, stub.stub_pending(), err.status)
                else:
                    print("done", k, stub.stub_pending(), len({s for _, s in launched(before)}))
                    break
                finally:
                    stub.stub_fail_from(-1)
        """).splitlines()
    assert out[-1].startswith("done") and len(out) > 6       # several allocations, then none failed
    assert out[-1].split()[2:] == ["0", "2"]                 # both compute streams worked
    for line in out[:-1]:
        assert line.split()[2] == "0", line


def test_destroy_waits_for_every_stream():
    """An engine goes when its work on each of the context's streams is done."""
    out = stub_lib.run("""
        st = state()
        with ag.Context(0) as ctx:
            e = ag.Analytic(ctx, st)
            for s in (1, 2, 3):     # as a call cut short would leave them
                stub.hipMemsetAsync(C.c_void_p(device(16)), 0, C.c_size_t(16), C.c_void_p(s))
            print(stub.stub_pending())
            e.close()
            print(stub.stub_pending())
        """).split()
    assert out == ["14", "0"]


# A constant dielectric on a grid of 884,736 points: its far field may run beside the
# near one, into 8 bytes a point (blocks are rounded up by an eighth at most).
FLAT = """
st = dataclasses.replace(state(), dddiel=0, inv_diel_cal=83.0, n1=(96, 96, 96), ne=(48, 48, 48), _keep=[])
wide = 8 * st.points


def blocks(first):
    return [s for s in map(stub.stub_malloc_size, range(first, stub.stub_mallocs())) if wide <= s <= wide * 9 // 8]
"""


def test_host_calls_take_no_wide_far_field():
    """Map sets to host memory never run the two fields beside each other, so they
    take no block for it; plans of one context share theirs."""
    out = stub_lib.run(FLAT + """
with ag.Context(0) as ctx:
    first = stub.stub_mallocs()
    ctx.maps_plain(st)
    print(len(blocks(first)))
    first = stub.stub_mallocs()
    maps = device(4 * st.n_maps * st.points)
    with ctx.plan(st) as a, ctx.plan(st) as b:
        after = stub.stub_launches()
        a.execute(maps)
        b.execute(maps)
        print(len(blocks(first)), len({s for name, s in launched(after) if "k_far" in name and "k_far_add" not in name}),
              sum("k_far_add" in name for name, _ in launched(after)))
""").split("\n")
    assert out[0] == "0"
    assert out[1] == "1 1 2"


def test_no_room_for_a_wide_far_field():
    """A plan whose far field finds no room for running beside the near one runs one
    after the other instead of failing."""
    out = stub_lib.run(FLAT + """
with ag.Context(0) as ctx:
    maps = device(4 * st.n_maps * st.points)
    stub.stub_fail_above(wide - 1)
    with ctx.plan(st) as p:
        after = stub.stub_launches()
        p.execute(maps)
        names = [n for n, _ in launched(after)]
        print(sum("k_far_add" in n for n in names), len({s for n, s in launched(after)}),
              sum("5k_far" in n for n in names))
""").split()
    assert out == ["0", "1", "1"]
