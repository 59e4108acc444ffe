"""The index update (append_index, core.py:186-201) on keys and tables off the
ordinary range: infinite keys and squares past fp32 in the moments' quotients."""
import pytest
import torch

from tests.test_gpu_encode import D, F, G, H, inputs
from tests.test_gpu_selection import membership

pytestmark = pytest.mark.gpu


def merged(a, b, ma, mb, va, vb):
    """core.py:194-199 in fp32, divisions as torch makes them."""
    den = (a + b).clamp_min(1)
    return (a * ma + b * mb) / den, (a * va + b * vb) / den + (a * b) / (den * den) * (ma - mb).square()


@pytest.mark.parametrize("kind", ["infinite key", "squares past fp32", "infinite table", "large table"])
def test_append_moments_where_fp32_ends(kind):
    from prismkv_amd import Native8B
    from prismkv_amd.native8b import untile_moments
    block = 200
    k, W, b, center, scale = inputs(block, 11)
    gen = torch.Generator(device="cuda").manual_seed(12)
    counts = torch.full((G, F), 3, dtype=torch.int64, device="cuda")
    mean = torch.randn(G, F, D, generator=gen, device="cuda")
    var = torch.rand(G, F, D, generator=gen, device="cuda")
    # dim 9 does not reach the activations, so the block's memberships stay ordinary
    W[:, :, 9] = 0
    if kind == "infinite key":
        # each infinite key is in the buckets that see it (elsewhere 0 times infinity is NaN)
        W.zero_()
        W[:, :8, 3] = 1e-3
        W[:, 8:16, 4] = -1e-3
        b.zero_()
        b[:, :16] = 1.0
        k[:, H + 5, 3] = float("inf")
        k[:, H + 6, 4] = float("-inf")
        center.zero_()
    if kind == "squares past fp32":
        k[:, H::2, 9] = 3e19
        k[:, H + 1::2, 9] = -3e19
    if kind == "infinite table":
        mean[:, ::3, 9] = float("inf")
        mean[:, 1::3, 9] = float("-inf")
        var[:, :, 10] = float("inf")
    if kind == "large table":  # a * var overflows
        var[:, :, 10] = 3e38
        mean[:, :, 9] = -3e38
    csr = torch.arange(9000, dtype=torch.int32, device="cuda").remainder(H).expand(G, -1).contiguous()
    offsets = (3 * torch.arange(F + 1, dtype=torch.int32, device="cuda")).expand(G, -1).contiguous()
    op = Native8B.from_tables(H, counts, mean, var, csr, offsets, center=center, capacity=H + block)
    op.set_encoder_tables(W, b, scale, 8)
    op.append(k, block)
    torch.cuda.synchronize()
    got_mean, got_var = untile_moments(op.moments)
    flat = membership(op, H, block)
    for g in range(G):
        feat, tok = flat[g] % F, flat[g] // F
        assert kind != "infinite key" or bool((feat[tok == 5] < 8).all() and (tok == 5).sum() == (tok == 6).sum() == 8)
        n = torch.bincount(feat, minlength=F).float()[:, None]
        x = k[g, H:].float()[tok]
        den = n.clamp_min(1)
        mb = torch.zeros(F, D, device="cuda").index_add_(0, feat, x) / den
        vb = torch.zeros(F, D, device="cuda").index_add_(0, feat, (x - mb[feat]).square()) / den
        want = merged(counts[g].float()[:, None], n, mean[g], mb, var[g], vb)
        for what, got, w in (("mean", got_mean[g], want[0]), ("variance", got_var[g], want[1])):
            odd = ~w.isfinite()
            # at the last finite octave an order of additions may reach infinity and another not
            clear = odd | (w.abs() < 1e38)
            assert bool(odd.any()) or what == "mean"
            same = (got == w) | (got.isnan() & w.isnan()) | ~odd
            assert bool(same[clear].all()), (kind, g, what, got[~same][:4], w[~same][:4])
            assert torch.allclose(got[clear & ~odd], w[clear & ~odd], rtol=1e-4, atol=2e-5), (kind, g, what)
