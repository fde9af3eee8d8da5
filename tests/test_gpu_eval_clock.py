"""Reading vd_eval's kernel time waits for nobody else and may happen in the middle of a graph capture
(where a copy on the null stream would be refused and end the capture): the words lie in page-locked
memory the kernel has written, or, after many workgroups on small host arrays, come over on the
context's own stream.  For the front end's device-pointer call, which reads them each time, it is no
call of the runtime at all."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CAPTURE_GLOBAL = 0   # hipStreamCaptureModeGlobal


# one workgroup, more than write to the host's memory, and arrays that are copied
@pytest.mark.parametrize("n", [1, 3000, 70000])
def test_time_read_during_a_capture(module_ctx, n):
    import vdock
    from vdock import workloads
    ctx = module_ctx
    workloads.small_scene(vdock, ctx)
    lid = ctx.add_ligand(vdock.synth_ligand(12, 3, 2))
    conf = np.zeros((n, 7 + ctx.ligand_info(lid).n_torsions), dtype=np.float32)
    conf[:, 3] = 1
    ctx.eval(lid, conf)
    first = ctx.eval_last_ms()
    assert first > 0
    ctx.eval(lid, conf)   # its time is read for the first time during the capture
    hip = C.CDLL(vdock.LIB_PATH)   # looks names up in the library's own HIP runtime
    stream, graph = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreate(C.byref(stream)) == 0
    print("capture begins", flush=True)
    assert hip.hipStreamBeginCapture(stream, CAPTURE_GLOBAL) == 0
    during = ctx.eval_last_ms()
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0 and graph.value
    assert hip.hipGraphDestroy(graph) == 0 and hip.hipStreamDestroy(stream) == 0
    assert 0.1 * first < during < 10 * first
    assert ctx.eval_last_ms() == during
