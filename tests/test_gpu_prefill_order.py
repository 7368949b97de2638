"""GPU: a prompt's attention at the numbers of workgroups where their order changes (256 CUs, two workgroups each), against float64."""
import pytest
import torch

from qtip_amd import ops

pytestmark = pytest.mark.gpu


# workgroups of 64 queries by a head: 256 and 257 to 512 (the second ones shortest first), more (longest first), heads that do
# not come out even on eight XCDs, one head
@pytest.mark.parametrize("n,heads,kv,D", ((512, 32, 32, 128), (513, 32, 8, 64), (1000, 32, 32, 128), (1025, 32, 4, 64), (900, 35, 7, 64),
                                          (2100, 9, 3, 128), (1300, 1, 1, 128)))
def test_attention_in_any_order_of_workgroups(n, heads, kv, D):
    g = torch.Generator(device="cuda").manual_seed(n)
    q, k, v = (torch.randn(n, h * D, generator=g, device="cuda").half() for h in (heads, kv, kv))
    ang = torch.rand(n, D // 2, generator=g, device="cuda") * 6
    cos, sin = (torch.cat((t, t), -1).half() for t in (ang.cos(), ang.sin()))
    caches = [torch.zeros(1, kv, n + 9, D, dtype=torch.float16, device="cuda") for _ in range(2)]
    got = ops.prefill_attention(q, k, v, cos, sin, *caches, torch.arange(n, device="cuda"), heads, kv, D).view(n, heads, D)

    def rotated(x, h):
        x = x.view(n, h, D)
        turned = torch.cat((-x[..., D // 2:], x[..., :D // 2]), -1)
        return (x * cos[:, None] + turned * sin[:, None]).double()

    qq, kk, vv = rotated(q, heads), rotated(k, kv), v.view(n, kv, D).double()
    mask = torch.ones(n, n, dtype=torch.bool, device="cuda").tril()
    for h in range(heads):
        s = (qq[:, h] @ kk[:, h * kv // heads].T * D**-0.5).masked_fill(~mask, float("-inf"))
        want = s.softmax(-1) @ vv[:, h * kv // heads]
        # correctly rounded but for few: 2**-11 of a value at most, 2.0e-4 in 2-norm
        assert (got[:, h].double() - want).norm() <= 2.5e-4 * want.norm()
