"""Element flags of a call that fails between the kernel that raised them and
their read-back: the next call must not see them.  The failure is forced from
the host (PH_HIP_FAIL_AFTER=n+k refuses the launches after the first k of
operation n+1, before they are issued), in a fresh child process each."""
import os
import subprocess
import sys
import textwrap

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _child(code, fail_after):
    env = dict(os.environ, PH_HIP_FAIL_AFTER=fail_after)
    env["PYTHONPATH"] = os.pathsep.join([os.path.join(ROOT, "ph-core_amd"), os.path.join(ROOT, "tests"),
                                         env.get("PYTHONPATH", "")])
    print(f"child with PH_HIP_FAIL_AFTER={fail_after}", flush=True)
    r = subprocess.run([sys.executable, "-c", textwrap.dedent(code)], env=env, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


# the finish of a small reduction; the pre-fold of rows of over 64 column tiles
@pytest.mark.parametrize("shape,what", [([7, 50], "reduction finish"), ([2, 70000], "reduction pre-fold")])
def test_flags_of_a_failed_reduction_are_dropped(shape, what):
    out = _child(f"""
        import numpy as np
        import phase
        phase.init(0)
        x = phase.NArray.from_numpy(np.full({shape}, 1 << 20, np.int32))
        one = phase.NArray.from_numpy(np.ones({shape}, np.int32))
        try:
            x.process(lambda v: v * v).slices_sum(0)   # the tile kernel raises, the next launch is refused
            raise SystemExit("not refused")
        except phase.DeviceError as e:
            assert "{what}" in str(e), str(e)
        assert np.array_equal((one + one).to_numpy(), np.full({shape}, 2, np.int32))
        assert one.slices_sum(0) == [{shape[1]}.0] * {shape[0]}
        for k in range(2):                             # and flags are reported as ever
            try:
                x.process(lambda v: v * v).slices_sum(0)
                raise SystemExit("no overflow")
            except phase.OverflowError:
                pass
            assert one.sum() == one.size
        print("clean")
    """, "0+1")
    assert "clean" in out


def test_second_run_of_a_bounded_sum_refused():
    """Int32 values whose bounds leave Int32 and whose totals do not: the exact
    run that would decide is refused, and the flags hold none of the first's."""
    out = _child("""
        import ctypes as C
        import os
        import numpy as np
        import phase
        from test_gpu_alias_deep import _desc

        class Prog(C.Structure):  # r0 = input 0
            _fields_ = [(n, C.c_int32) for n in ("n_insn", "n_in", "out_reg", "out_dtype")] + [("insn", C.c_int64 * 96)]

        phase.init(0)
        lib = C.CDLL(os.path.join(phase.LIB_DIR, "libphhip.so"))
        top = 2**31 - 1
        x = phase.NArray.from_numpy(np.array([top, -top] * 50, np.int32))
        s = phase.NArray.from_numpy(np.zeros(1))
        d, p = _desc(0, 100, [100]), Prog(1, 1, 0, 0)
        ins, fl = (C.c_void_p * 1)(x.device_ptr), C.c_int32(77)
        rc = lib.ph_reduce(C.byref(p), 1, ins, C.byref(d), -1, 1, 0, C.c_void_p(s.device_ptr), None, C.byref(fl))
        assert rc == -10 and fl.value == 0, (rc, fl.value)
        print("refused")
    """, "1")
    assert "refused" in out
