"""The matvec on device buffers (q4hip_mv_run_noalloc), whose kernels quantize x themselves, against
q4hip_mv_run: rows of each kernel's block counts and around its limits, ragged row counts, and y written
over x (which takes a quantize launch of its own).  Bit for bit.
"""
import numpy as np
import pytest

import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,nb", [(896, 28), (17, 28), (40000, 28), (1536, 48), (100, 48), (64, 1), (65, 27), (130, 63),
                                  (129, 64), (896, 152), (48, 480), (48, 481)])
def test_device_call_equals_run(N, nb):
    import q4hip
    import torch
    K = 32 * nb
    rng = np.random.default_rng(N + nb)
    w = synth.quantize_q4_0(rng.standard_normal(N * K, dtype=np.float32) * np.float32(0.02))
    x = rng.standard_normal(K, dtype=np.float32)
    x[:32] = 0                                  # a zero block
    print(f"{N} x {K}", flush=True)
    mv = q4hip.Matvec(w, N, K)
    want = mv.run(x)
    s = torch.cuda.Stream()
    buf = torch.zeros(K + N + 1, device="cuda")
    off = 1                                     # x at 4-byte alignment only
    buf[off:off + K] = torch.from_numpy(x).cuda()
    y = torch.zeros(N, device="cuda")
    torch.cuda.synchronize()
    for _ in range(2):
        mv.run_device(buf.data_ptr() + 4 * off, y.data_ptr(), s.cuda_stream)
    torch.cuda.synchronize()
    assert np.array_equal(y.cpu().numpy().view(np.uint32), want.view(np.uint32))
    mv.run_device(buf.data_ptr() + 4 * off, buf.data_ptr() + 4 * (off + K // 2), s.cuda_stream)   # over x's second half
    torch.cuda.synchronize()
    assert np.array_equal(buf[off + K // 2:off + K // 2 + N].cpu().numpy().view(np.uint32), want.view(np.uint32))
