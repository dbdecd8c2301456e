"""silu(gate) * up at the edges of its vector kernel: below one vector, last
elements past the vectors, work-groups that are not full, buffers off a 16-byte
boundary, and the result in gate's place."""
import numpy as np
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("n,shift", [(1, 0), (3, 0), (4, 0), (7, 0), (1023, 0), (1024, 0),
                                     (2048, 0), (2052, 0), (4097, 0), (4097, 1),
                                     (4 * 256 * 1024 + 4099, 0)])
def test_silu_mul_rows(orc, n, shift):
    import torch

    import hypno_amd as hk
    rng = np.random.default_rng(n)
    g = (rng.standard_normal(n) * 4).astype(np.float32)
    g[: 3] = [-100.0, 100.0, 0.0][: n]  # exp overflows: -0
    u = rng.standard_normal(n).astype(np.float32)
    ref = orc.silu_mul(g, u)

    def put(a):
        d = torch.empty(n + shift, dtype=torch.float32, device="cuda")[shift:]
        d.copy_(torch.from_numpy(a))
        return d

    dg, du = put(g), put(u)
    got = hk.silu_mul(dg, du, out=torch.full((n + 4,), float("nan"), device="cuda"))
    hk.silu_mul(dg, du, out=dg)
    torch.cuda.synchronize()
    assert torch.isnan(got[n:]).all()  # nothing past the end
    got = got[:n].cpu().numpy()
    assert np.array_equal(got, dg.cpu().numpy())
    # two exponentials within an ulp or two, a sum, a quotient and a product
    assert np.all(np.abs(got - ref) <= 8 * 2.0 ** -23 * np.abs(ref) + 1e-37)
