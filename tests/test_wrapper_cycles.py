"""A context and its objects in one garbage cycle (an application object that a
callback refers back to, the frames of a failed call): the collector clears the
weak references within the cycle and calls the finalizers in any order, and
still ppm_destroy comes after every object's destroy call, each once.  CPU only:
the library is replaced by a recorder, as in the teardown tests."""
import subprocess
import sys

import pytest

from test_wrapper_teardown import ROOT, SCRIPT

NAMES = ["ppm_batch_destroy", "ppm_session_destroy", "ppm_map_destroy", "ppm_photons_destroy", "ppm_scene_destroy"]


@pytest.mark.parametrize("order", ["c, ds, ph, m, s, b", "b, s, m, ph, ds, c", "ph, c, b, ds, s, m"])
def test_cycle_destroys_the_context_last(order):
    code = SCRIPT + f'''
import gc
gc.disable()
class App:
    pass
app = App()
app.all = [{order}]
app.back = app
del app, c, ds, ph, m, s, b
gc.collect()
os.write(1, b"collected\\n")
'''
    out = subprocess.run([sys.executable, "-c", code, ROOT], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stderr
    calls = out.stdout.split()
    assert calls[-1] == "collected" and sorted(calls[:-1]) == sorted(NAMES + ["ppm_destroy"]), calls
    assert calls[-2] == "ppm_destroy", calls


def test_objects_closed_one_by_one():
    code = SCRIPT + "\ns.close(); s.close(); ds.close(); c.close(); m.close(); del b\nos.write(1, b'closed\\n')\n"
    out = subprocess.run([sys.executable, "-c", code, ROOT], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stderr
    calls = out.stdout.split()
    assert calls[:2] == ["ppm_session_destroy", "ppm_scene_destroy"] and calls[-2:] == ["ppm_destroy", "closed"], calls
    assert sorted(calls[:-1]) == sorted(NAMES + ["ppm_destroy"]), calls
