"""The fused q_activation decode (core.py:131-139, :142-183) off its common
path, against the separate launches: infinite activations, whose weights are NaN."""
import pytest
import torch

pytestmark = pytest.mark.gpu

F = 3000


def operator(H, T, seed):
    """Random bucket lists: every token in 8 random buckets, shared by all groups."""
    from prismkv_amd import Native8B
    gen = torch.Generator(device="cuda").manual_seed(seed)
    k, v = (torch.randn(8, H + T, 128, generator=gen, device="cuda").to(torch.bfloat16) for _ in range(2))
    q = torch.randn(8, 4, 128, generator=gen, device="cuda").to(torch.bfloat16)
    W = torch.randn(8, F, 128, generator=gen, device="cuda") / 128 ** 0.5
    b = 0.05 * torch.randn(8, F, generator=gen, device="cuda")
    tok = torch.arange(H, device="cuda").repeat_interleave(8)
    order = (torch.randint(0, F, (8 * H,), generator=gen, device="cuda") * H + tok).unique()
    feat, tok = order // H, order % H
    n = torch.bincount(feat, minlength=F)
    csr = tok.int().expand(8, -1).contiguous()
    offsets = torch.cat((torch.zeros(1, dtype=torch.int64, device="cuda"), n.cumsum(0))).int().expand(8, -1).contiguous()
    zeros = torch.zeros(8, F, 128, device="cuda")
    return Native8B.from_tables(H, n.expand(8, -1), zeros, zeros, csr, offsets), q, k, v, W, b


@pytest.mark.parametrize("H", [3000, 150000])
@pytest.mark.parametrize("heads", [1, 3])
def test_infinite_activations(H, heads):
    # the first heads overflow in buckets 7 and 40, which every other head ranks high:
    # their scores are NaN and neither is selected
    op, q, k, v, W, b = operator(H, 5, H + heads)
    W[:, :, :2] = 0
    W[:, 7, 0] = W[:, 40, 0] = 3e38
    W[:, 7, 1] = W[:, 40, 1] = 9.0
    q[:, :, :2] = 0
    q[:, :heads, 0] = 5.0
    q[:, heads:, 1] = 5.0
    op.set_query_encoders(W, b, torch.ones(8))
    op.router = "q_activation"
    op.route(q)
    want_out = op.attention(q, k, v).clone()
    names = ("features", "valid", "raw", "count")
    want = {x: getattr(op, x).clone() for x in names}
    ids = [op.ids[g, :op.count[g]].clone() for g in range(8)]
    assert not bool(((op.features == 7) | (op.features == 40)).logical_and(op.valid > 0).any())
    assert bool((op.count > 0).all())
    got = op(q, k, v)
    for x in names:
        assert torch.equal(getattr(op, x), want[x]), x
    for g in range(8):
        assert torch.equal(op.ids[g, :op.count[g]], ids[g]), g
    # bf16 outputs of two exact softmaxes: at most a rounding of 2^-9 apart
    assert float((got.float() - want_out.float()).norm()) <= 4e-3 * float(want_out.float().norm())
    assert op.decode_errors() == 0
