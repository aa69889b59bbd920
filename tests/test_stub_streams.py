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
