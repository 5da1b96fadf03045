"""GPU: drop-in products of growing and shrinking sizes (the pinned buffers
grow and are reused), from several threads, equal the device call's bits."""
import threading

import numpy as np
import pytest

from inferno_hip import formats as F
from inferno_hip import synth

pytestmark = pytest.mark.gpu

CALLS = [(F.Q4_K, 16, 256), (F.Q8_0, 1, 32), (F.Q6_K, 4100, 512), (F.Q5_K, 33, 12288), (F.Q4_K, 70000, 256),
         (F.Q8_0, 17, 2080)]


@pytest.fixture(scope="module")
def ih():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import inferno_hip
    assert inferno_hip.quant_kernels_available(), inferno_hip._lib.last_error()
    return inferno_hip


def test_sizes_and_threads(ih):
    import torch
    gemv = ih.quantized_kernels.GEMV_BY_QTYPE
    rng = np.random.default_rng(0)
    cases = []
    for qt, n, k in CALLS + CALLS[::-1]:
        w = synth.matrix(qt, n, k, synth.stream_for(n + k, f"d{qt}"))
        x = rng.standard_normal(k).astype(np.float32)
        wp = ih.pack_weights(qt, torch.from_numpy(w).cuda(), n, k)
        want = ih.gemm_q(qt, wp, torch.from_numpy(x).cuda(), n, k, flags=ih.GEMM_F32 | ih.GEMM_PACKED).cpu().numpy()[0]
        cases.append((qt, n, k, w, x, want))
    bad = []

    def work():
        for qt, n, k, w, x, want in cases:
            out = np.full(n + 8, 7.0, np.float32)
            gemv[qt](out, w, x, k, n)
            if not np.array_equal(out[:n], want) or (out[n:] != 7.0).any():
                bad.append((qt, n, k))

    threads = [threading.Thread(target=work) for _ in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
