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
