"""The matvec on device buffers (q4hip_mv_run_noalloc), whose kernels quantize x themselves, against
q4hip_mv_run: rows of each kernel's block counts and around its limits, ragged row counts, and y written
over x (which takes a quantize launch of its own).  28672 rows of 64 blocks are the most whose workgroups
quantize x, 28673 take two launches.  Bit for bit.
"""
import ctypes

import numpy as np
import pytest

import synth
from test_zz_no_alloc import DevBuf, _hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,nb", [(896, 28), (17, 28), (40000, 28), (1536, 48), (100, 48), (64, 1), (65, 27), (130, 63),
                                  (129, 64), (896, 152), (48, 480), (48, 481), (28672, 64), (28673, 64)])
def test_device_call_equals_run(N, nb):
    import q4hip
    hip = _hip()
    assert hip.hipSetDevice(0) == 0
    K = 32 * nb
    rng = np.random.default_rng(N + nb)
    if N < 20000 or nb < 64:
        w = synth.quantize_q4_0(rng.standard_normal(N * K, dtype=np.float32) * np.float32(0.02))
    else:                                       # the same format without quantizing 58 million values
        w = rng.integers(0, 256, (N * nb, 18), dtype=np.uint8)
        w[:, :2] = np.frombuffer(np.float16(0.005).tobytes(), np.uint8)
        w = w.reshape(-1)
    x = rng.standard_normal(K, dtype=np.float32)
    x[:32] = 0                                  # a zero block
    print(f"{N} x {K}", flush=True)
    mv = q4hip.Matvec(w, N, K)
    want = mv.run(x)
    stream = ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(stream)) == 0
    buf, y = DevBuf(hip, 4 * (K + N + 1)), DevBuf(hip, 4 * N)
    try:
        host = np.zeros(K + N + 1, np.float32)
        host[1:1 + K] = x                       # x at 4-byte alignment only
        buf.put(host)
        xp = buf.p.value + 4
        for _ in range(2):
            mv.run_device(xp, y.p.value, stream.value)
        assert hip.hipStreamSynchronize(stream) == 0
        assert np.array_equal(y.get(N).view(np.uint32), want.view(np.uint32))
        mv.run_device(xp, xp + 4 * (K // 2), stream.value)      # y over x's second half
        assert hip.hipStreamSynchronize(stream) == 0
        got = buf.get(K + N + 1)[1 + K // 2:1 + K // 2 + N]
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    finally:
        buf.free()
        y.free()
        hip.hipStreamDestroy(stream)
