"""The two ways of forming dQ (recomputing S and dP, or from the dS that the dK/dV pass stores): dK and dV have the same bits
in both, and so has dQ where a workgroup is one group (more 128-row blocks per pass than half the CUs); two groups add two
partial sums in the recomputing kernel where the other adds the tiles in order."""

import math

import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

SCALE = 1.0 / math.sqrt(128.0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("B,T,H,groups", [(1, 65, 2, 2), (1, 300, 4, 2), (1, 1000, 16, 2), (2, 777, 16, 1), (3, 400, 16, 1),
                                          (1, 2047, 16, 1), (1, 2500, 16, 1)])
def test_paths_agree_bit_for_bit(B, T, H, groups, causal, dtype):
    from dirktensor_amd import Context, flash_attention_backward, flash_attention_forward

    if groups == 1:
        cus = torch.cuda.get_device_properties(0).multi_processor_count
        assert 2 * B * H * ((T + 127) // 128) > cus
    g = torch.Generator(device="cuda").manual_seed(T)
    q, k, v, do = (torch.randn((B, T, H, 128), generator=g, device="cuda").to(dtype) for _ in range(4))
    r = flash_attention_forward(q, k, v, SCALE, causal)
    out = []
    for path in ("recompute", "from_ds"):
        ctx = Context(0)
        ctx.set_bwd_dq_path(path)
        x = flash_attention_backward(do, r.output, r.softmax_m, r.softmax_l, q, k, v, SCALE, causal, ctx=ctx)
        torch.cuda.synchronize()
        out.append((x.d_Q, x.d_K, x.d_V))
    (q0, k0, v0), (q1, k1, v1) = out
    assert torch.equal(k0, k1) and torch.equal(v0, v1)
    if groups == 1:
        assert torch.equal(q0, q1)
    else:  # the same terms, rounded in another order: fp32 sums, and bf16 results that fall to the other side of a tie
        assert float((q0.double() - q1.double()).norm() / q1.double().norm()) < (1e-6 if dtype == torch.float32 else 1e-3)
