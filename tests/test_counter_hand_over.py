"""ResetIDBuffer returns when its kernel has handed the counter over, not when the stream is idle, so
the kernel has to order its clear before the hand-over: work on another stream, enqueued after the
call, must find the counter 0 and keep what it writes there."""
from __future__ import annotations

import ctypes as C
import re
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT


def test_clear_is_ordered_before_the_hand_over(tmp_path):
    """In the kernel's own assembly: the clear is waited for, and written back to where other queues
    see it, before the word the host watches is stored."""
    sys.path.insert(0, str(ROOT / "svo-tracer_amd"))
    import build as recipe

    out = tmp_path / "wavefront.s"
    subprocess.run([recipe.HIPCC, "-x", "hip", *recipe.COMMON, *recipe.DEVICE_ONLY, "--cuda-device-only", "-S",
                    str(recipe.CSRC / "wavefront.hip"), "-o", str(out)], check=True, capture_output=True)
    body = re.search(r"^\S*take_counter_kernel\S*:.*?s_endpgm", out.read_text(), re.M | re.S).group(0)
    ops = [line.split()[0:2] for line in body.splitlines() if line.startswith("\t")]
    stores = [i for i, op in enumerate(ops) if op[0].startswith("global_store")]
    assert [ops[i][0] for i in stores] == ["global_store_dword", "global_store_dwordx2"], body
    between = ops[stores[0] + 1:stores[1]]
    assert ["s_waitcnt", "vmcnt(0)"] in between and any(op[0] == "buffer_wbl2" for op in between), body


@pytest.mark.gpu
def test_other_streams_find_it_cleared(svo, gpu):
    hip = C.CDLL("libamdhip64.so.7")
    B = svo.BufferName
    gpu.InitBuffer(B.ChildRequestID, np.zeros(1, np.uint32))
    p = C.c_void_p(gpu.DevicePointer(B.ChildRequestID))
    stream, word = C.c_void_p(), (C.c_uint32 * 1)()
    assert hip.hipStreamCreateWithFlags(C.byref(stream), 1) == 0
    for k in range(1, 201):
        gpu.WriteBuffer(B.ChildRequestID, np.full(1, k, np.uint32))
        assert gpu.ResetIDBuffer(B.ChildRequestID) == k
        assert hip.hipMemcpyAsync(word, p, C.c_size_t(4), 2, stream) == 0  # device to host
        assert hip.hipStreamSynchronize(stream) == 0
        assert word[0] == 0
        word[0] = 1000 + k
        assert hip.hipMemcpyAsync(p, word, C.c_size_t(4), 1, stream) == 0  # host to device
        assert hip.hipStreamSynchronize(stream) == 0
        assert gpu.ResetIDBuffer(B.ChildRequestID) == 1000 + k
    assert hip.hipStreamDestroy(stream) == 0
