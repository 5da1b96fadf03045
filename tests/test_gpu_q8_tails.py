"""GPU: Q8_0 in GGUF layout with every length of the last unit: the bits of the
packed layout, and the fp64 product."""
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


@pytest.mark.parametrize("M", [3, 11, 20, 64])
@pytest.mark.parametrize("blocks", [1, 3, 9, 15, 65, 71])
def test_q8_0_gguf_tails(ih, M, blocks):
    import torch
    N, K = 50, 32 * blocks
    w = torch.from_numpy(synth.matrix(F.Q8_0, N, K, synth.stream_for(K, "t"))).cuda()
    x = torch.randn(M, K, device="cuda", generator=torch.Generator("cuda").manual_seed(K))
    for fl in (ih.GEMM_F32, ih.GEMM_HALF):
        a = ih.gemm_q(F.Q8_0, w, x, N, K, flags=fl)
        b = ih.gemm_q(F.Q8_0, ih.pack_weights(F.Q8_0, w, N, K), x, N, K, flags=fl | ih.GEMM_PACKED)
        assert torch.equal(a, b)
        d = ih.dequant(F.Q8_0, w, N * K).view(N, K).double()
        ref = x.double() @ d.t()
        # two fp16 limbs: 2^-21 an activation; one limb: 2^-11 (rms sums: the norms' ratio)
        assert float((a.double() - ref).norm() / ref.norm()) < (2.0 ** -20 if fl == ih.GEMM_F32 else 2.0 ** -10)
