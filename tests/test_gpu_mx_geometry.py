"""The MX row kernel's two lane geometries: on both sides of the grid size where the nibble layout
goes from two to four rows per lane (d_state 128; the other widths stay at two), the compact update equals the reference layout's bit for bit."""
import pytest
import torch

from hybrid_quant import mamba_state_8b_kernel as ms

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bsz", [23, 24])  # 5888 and 6144 workgroups of 256 heads
@pytest.mark.parametrize("n", [64, 128, 256])
@pytest.mark.parametrize("stochastic", [True, False])
def test_compact_equals_reference_layout(gpu, diag, bsz, n, stochastic):
    diag.set("LQ_MX_REQUIRE_ROWS")
    nh, p_, ng = 256, 17, 8  # 17 rows: most of a workgroup's row slots are past the end
    gen = torch.Generator(device=gpu).manual_seed(n + bsz)
    h0 = torch.randn(bsz, nh, p_, n, device=gpu, generator=gen)
    caches = [ms.allocate_state_kernel_cache(h0, format_bits=4, layout=layout)
              for layout in ("reference", "compact")]
    x = torch.randn(bsz, nh, p_, device=gpu, generator=gen).to(torch.bfloat16)
    dt = torch.randn(bsz, nh, 1, device=gpu, generator=gen).to(torch.bfloat16).expand(bsz, nh, p_)
    A = (-torch.rand(nh, 1, 1, device=gpu, generator=gen)).expand(nh, p_, n)
    B, C = (torch.randn(bsz, ng, n, device=gpu, generator=gen).to(torch.bfloat16) for _ in range(2))
    for _ in range(2):
        ys = [ms.mx_state_selective_update(c, x, dt, A, B, C, dt_softplus=True, stochastic=stochastic)
              for c in caches]
        assert torch.equal(*ys)
    back = ms.convert_state_cache_layout(caches[1], "reference")
    for name in ("q_state", "shared_exp", "micro_exp"):
        assert torch.equal(getattr(back, name), getattr(caches[0], name)), name
