"""GPU parity of the expert products on the persistent 128 x 256 tiles, and on
the 128 x 128 tiles that take their place where a k loop is under 256: a
token's outputs do not depend on how many tokens a call has, so they agree bit
for bit with the streaming kernel's, which the same tokens take in chunks."""
import pytest
import torch

import moe_cases

pytestmark = pytest.mark.gpu


# (tokens, experts, dim, hidden, shared, router bias): the smallest k loops and
# rows per expert, columns that end within a tile, an expert without rows, rows
# past the grouping's capacity, more tiles than workgroups, partial row tiles, and
# too few tiles for one product or both (128 x 128 tiles there)
@pytest.mark.parametrize("tokens,experts,dim,hidden,shared,bias", [
    (1025, 4, 256, 256, 256, None), (2048, 16, 768, 512, 256, None),
    (1100, 3, 320, 448, 320, (9.0, 9.0, -90.0)), (4099, 5, 768, 512, 256, (4.0, 2.0, 0.0, 0.0, 0.0)),
    (513, 2, 512, 320, 704, None), (8200, 32, 256, 320, 256, None), (20001, 16, 768, 512, 256, None),
    (3000, 3, 768, 448, 320, (9.0, 9.0, -90.0)), (1200, 8, 768, 512, 256, None),
    # k loops under 256 in both products, in the second only (its shared, its
    # routed rows): even and skewed segments with partial last tiles
    (4099, 5, 192, 128, 64, (4.0, 2.0, 0.0, 0.0, 0.0)), (1100, 3, 64, 192, 192, (9.0, 9.0, -90.0)),
    (2051, 4, 768, 512, 192, (4.0, 2.0, 0.0, 0.0)), (4097, 8, 320, 64, 448, None)])
def test_persistent_tiles(tokens, experts, dim, hidden, shared, bias):
    from parrot import hip_moe
    print(f"persistent experts T={tokens} E={experts} {dim}/{hidden}/{shared}", flush=True)
    module = moe_cases.moe_module(experts, seed=tokens, dim=dim, hidden=hidden, shared=shared)
    x = moe_cases.inputs(tokens, seed=tokens, dim=dim)
    bias = None if bias is None else torch.tensor(bias)

    def layer(rows):
        r = hip_moe.route(module, rows, False, logit_bias=bias)
        return hip_moe.grouped_hip_experts(module, rows, r.indices, r.weights, grouping=r.grouping)

    with torch.no_grad():
        got = layer(x)
        again = layer(x)
        # 64 tokens: under 96 rows per expert on average for any E >= 2
        ref = torch.cat([layer(x[i:i + 64]) for i in range(0, tokens, 64)])
    assert torch.equal(got, again)
    assert torch.equal(got, ref)
