"""Q4Dispatch.run_gemm_npu on bf16 rows: the bf16 kernels in place of the float32
ones between two conversions."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 2, 16, 17, 32, 33, 200])
@pytest.mark.parametrize("offset", [0, 1])
def test_run_gemm_bf16_rows(orc, dev, B, offset):
    """bf16 rows give the float64 product within its float32 bound and half a
    bf16 ulp (2^-8 of the value), as the same rows widened to float32 do (the
    route before), on either side of both kernels' token thresholds; rows that
    are not 16-byte aligned (offset 1) keep the float32 route."""
    import alveare_amd as aa
    from alveare_amd.runtime import Q4Dispatch, ResidentWeight

    N, K = 700, 1056
    print(f"\n[dispatch] B={B} offset={offset}", flush=True)
    W = torch.from_numpy(orc.synth_q4(N, K, 3)).to(dev)
    d = Q4Dispatch(K, 4 * K, device=dev)
    rw = ResidentWeight(W.reshape(-1), tuple(W.shape))
    flat = torch.from_numpy(orc.synth_normal(B * K + 1, 4)).to(dev).to(torch.bfloat16)
    X = flat[offset:offset + B * K].view(B, K)
    ref = X.double() @ aa.dequant_q4(W, N, K).double().T
    bound = (3 * K + 8) * 2.0 ** -24 * (X.double().abs() @ aa.dequant_q4(W, N, K).double().abs().T)
    bound = 1.01 * bound + ref.abs() * 2.0 ** -8 + 1e-30
    for x in (X, X.float()):
        y = d.run_gemm_npu(rw, x)
        assert y.dtype == torch.bfloat16 and tuple(y.shape) == (B, N)
        assert ((y.double() - ref).abs() <= bound).all()
