"""A context on a stream that the caller made: the stream is the caller's again
once the context's objects are closed."""
import ctypes as C
import weakref

import numpy as np
import pytest

from gpu_common import ctx, say, small_scene

import ppmpa_amd as P
from ppmpa_amd import _abi as A

pytestmark = pytest.mark.gpu

NON_BLOCKING, RELAXED = 1, 2  # hipStreamNonBlocking, hipStreamCaptureModeRelaxed


def _context_on(stream):
    c = P.Context.__new__(P.Context)
    c.lib, c.h, c._objs, c._live = A.load(), C.c_void_p(), weakref.WeakSet(), {}
    assert c.lib.ppm_create(C.byref(c.h), 0, stream) == 0
    return c


def test_destroy_leaves_the_stream_alone():
    """The caller captures a graph on its stream while the context, which has
    staged results and keeps a block, is destroyed: waiting for the stream
    would end the capture with an error."""
    say("caller stream: destroy during a capture")
    hip = A.load()  # its symbols include those of the HIP runtime that it is linked to
    stream, graph = C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreateWithFlags(C.byref(stream), NON_BLOCKING) == 0
    want = P.trace_classic(ctx(), P.DeviceScene(ctx(), small_scene("caustic", 64, 48)), 3, 1)
    c = _context_on(stream)
    ds = P.DeviceScene(c, small_scene("caustic", 64, 48))
    got = P.trace_classic(c, ds, 3, 1)
    ds.close()
    assert hip.hipStreamBeginCapture(stream, RELAXED) == 0
    c.close()
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert hip.hipGraphDestroy(graph) == 0
    assert hip.hipStreamSynchronize(stream) == 0
    assert hip.hipStreamDestroy(stream) == 0
    assert np.array_equal(got, want)
