"""GPU: the MLP with a K-sliced [gate; up] (its partials summed by down's
input stage) equals, bit for bit, the two matmul calls with the product
materialised, and the same call on a workspace of the undeferred size; at one
and several slices and token tiles, both layouts and precisions."""
import pytest

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


def _w(ih, qt, n, k, name, packed):
    import torch
    w = torch.from_numpy(synth.matrix(qt, n, k, synth.stream_for(n + k, name))).cuda()
    return ih.pack_weights(qt, w, n, k) if packed else w


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("M,H,Fh,flags", [(5, 512, 256, 1), (9, 2304, 512, 1), (32, 4096, 256, 1), (33, 4096, 256, 1),
                                          (16, 4096, 512, 0), (64, 2304, 768, 2), (64, 4096, 256, 0)])
def test_mlp_sliced_gate_up(ih, packed, M, H, Fh, flags):
    import torch
    fl = flags | (ih.GEMM_PACKED if packed else 0)
    gu, dn = _w(ih, F.Q4_K, 2 * Fh, H, "gu", packed), _w(ih, F.Q6_K, H, Fh, "dn", packed)
    x0 = torch.randn(M, H, device="cuda", generator=torch.Generator("cuda").manual_seed(M + H))
    nw = 1 + 0.1 * torch.randn(H, device="cuda", generator=torch.Generator("cuda").manual_seed(3))
    ref = x0.clone()
    g = ih.gemm_q_ex(F.Q4_K, gu, ref, 2 * Fh, H, act=ih.ACT_RMSNORM, norm_w=nw, flags=fl)
    ih.gemm_q_ex(F.Q6_K, dn, g, H, Fh, act=ih.ACT_SILU_MUL, flags=fl | ih.GEMM_ACCUM, out=ref)
    need = ih.mlp_ws_bytes(F.Q4_K, F.Q6_K, M, H, Fh, fl)
    gws = ih.quantized_kernels.gemm_ws_bytes
    plain = ((M * 2 * Fh * 4 + 255) // 256 * 256) + max(gws(F.Q4_K, M, 2 * Fh, H, fl), gws(F.Q6_K, M, H, Fh, fl | ih.GEMM_ACCUM))
    assert need >= plain
    for size in (need, plain):
        ws = torch.full((size + 64,), 0x7F, dtype=torch.uint8, device="cuda")
        x = x0.clone()
        ih.mlp_forward_(F.Q4_K, gu, F.Q6_K, dn, x, H, Fh, norm_w=nw, flags=fl, ws=ws[:size])
        assert torch.equal(x, ref), size
        assert bool((ws[size:] == 0x7F).all())
