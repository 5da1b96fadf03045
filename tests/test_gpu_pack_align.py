"""GPU: the packers take a GGUF matrix at any byte address, every row count
and unit count around a tile and a workgroup's four units, and write exactly
ihip_packed_bytes bytes of the layout's numpy statement (the gated layout:
that of the rows in its order)."""
import numpy as np
import pytest

from _packref import pack_ref

from inferno_hip import formats as F
from inferno_hip import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ih():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import inferno_hip
    assert inferno_hip.quant_kernels_available(), inferno_hip._lib.last_error()
    return inferno_hip


@pytest.mark.parametrize("qt", F.QTYPES)
@pytest.mark.parametrize("offset", [0, 1, 2, 7])
@pytest.mark.parametrize("N,units", [(1, 1), (15, 3), (17, 5), (48, 4)])
def test_pack_any_address(ih, qt, offset, N, units):
    import torch
    K = units * 256 - (96 if qt == F.Q8_0 and units % 2 else 0)
    w = synth.matrix(qt, N, K, synth.stream_for(N + K, f"pa{qt}"))
    buf = torch.zeros(w.size + offset, dtype=torch.uint8, device="cuda")
    buf[offset:] = torch.from_numpy(w).cuda()
    nb = ih.packed_bytes(qt, N, K)
    out = torch.full((nb + 64,), 0xA5, dtype=torch.uint8, device="cuda")
    ih.pack_weights(qt, buf[offset:], N, K, out=out)
    got = out.cpu().numpy()
    assert np.array_equal(got[:nb], pack_ref(qt, w, N, K)) and (got[nb:] == 0xA5).all()


@pytest.mark.parametrize("qt", F.QTYPES)
@pytest.mark.parametrize("Fh,units", [(8, 1), (24, 3), (40, 5)])
def test_pack_gated(ih, qt, Fh, units):
    import torch
    K = units * 256
    w = synth.matrix(qt, 2 * Fh, K, synth.stream_for(Fh + K, f"pg{qt}"))
    rows = w.reshape(2 * Fh, -1)
    order = [r for t in range(Fh // 8) for r in (*range(8 * t, 8 * t + 8), *range(Fh + 8 * t, Fh + 8 * t + 8))]
    got = ih.pack_weights_gated(qt, torch.from_numpy(w).cuda(), Fh, K).cpu().numpy()
    assert np.array_equal(got, pack_ref(qt, np.ascontiguousarray(rows[order]).reshape(-1), 2 * Fh, K))
