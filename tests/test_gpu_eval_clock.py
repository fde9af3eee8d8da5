"""Reading vd_eval's kernel time touches no stream: the words lie in page-locked memory the kernel has
written.  So it may be read in the middle of a graph capture (where a copy would be refused and end the
capture), waits for nobody, and costs the front end's device-pointer call, which reads it each time,
nothing."""
import ctypes as C
import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CAPTURE_GLOBAL = 0   # hipStreamCaptureModeGlobal


def hip_runtime():
    """The HIP runtime that libvdock has loaded."""
    with open("/proc/self/maps") as f:
        path, = {m.group(0) for m in re.finditer(r"/\S*libamdhip64\.so\S*", f.read())}
    return C.CDLL(path)


@pytest.mark.parametrize("n", [1, 70000])   # one workgroup, and as many as a launch takes
def test_time_read_during_a_capture(module_ctx, n):
    import vdock
    from vdock import workloads
    ctx = module_ctx
    workloads.small_scene(vdock, ctx)
    lid = ctx.add_ligand(vdock.synth_ligand(12, 3, 2))
    conf = np.zeros((n, 7 + ctx.ligand_info(lid).n_torsions), dtype=np.float32)
    conf[:, 3] = 1
    ctx.eval(lid, conf)
    before = ctx.eval_last_ms()
    assert before > 0
    hip = hip_runtime()
    stream, graph = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreate(C.byref(stream)) == 0
    print("capture begins", flush=True)
    assert hip.hipStreamBeginCapture(stream, CAPTURE_GLOBAL) == 0
    during = ctx.eval_last_ms()
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0 and graph.value
    assert hip.hipGraphDestroy(graph) == 0 and hip.hipStreamDestroy(stream) == 0
    assert during == before
