"""The encode of the index update and build (relu((k - center) / scale W^T + b),
src/prismkv/core.py:47-48,98) where its f16 split or its tiles can go wrong:
blocks around its 16-token steps, its 64-token stages and a workgroup's range of
tokens, rows and buckets of extreme magnitudes (scaled per row and per bucket),
and rows and buckets that are not split (beyond 2^60, infinite or NaN, or of few
significant dims)."""
import numpy as np
import pytest
import torch

from oracle import expect

pytestmark = pytest.mark.gpu

F, G, D, H = 3000, 8, 128, 40


def run_append(k, W, b, center, scale, block, key_mean=8):
    from prismkv_amd import Native8B
    zeros = torch.zeros(G, F, dtype=torch.int64, device="cuda")
    op = Native8B.from_tables(H, zeros, torch.zeros(G, F, D, device="cuda"), torch.zeros(G, F, D, device="cuda"),
                              torch.zeros(G, 1, dtype=torch.int32, device="cuda"),
                              torch.zeros(G, F + 1, dtype=torch.int32, device="cuda"), center=center,
                              capacity=H + block)
    op.set_encoder_tables(W, b, scale, key_mean)
    op.append(k, block)
    torch.cuda.synchronize()
    return op, op.update_activations(block)


def inputs(block, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    k = torch.randn(G, H + block, D, generator=gen, device="cuda").to(torch.bfloat16)
    W = torch.randn(G, F, D, generator=gen, device="cuda") / D ** 0.5
    b = 0.05 * torch.randn(G, F, generator=gen, device="cuda")
    center = 0.1 * torch.randn(G, D, generator=gen, device="cuda")
    scale = torch.linspace(0.7, 2.0, G, device="cuda")
    return k, W, b, center, scale


def check(k, W, b, center, scale, act, rows=slice(None), buckets=slice(None)):
    for g in range(G):
        # x in fp32 with the device's operations, the sums in 64 bits
        x = ((k[g, H:].float() - center[g]) / scale[g])[rows].cpu().numpy()
        w, bg = W[g][buckets].cpu().numpy(), b[g][buckets].cpu().numpy()
        want = np.maximum(x.astype(np.float64) @ w.astype(np.float64).T + bg, 0.0)
        # the bound of any fp32 summation order of the 128 products (expect.encode_error_bound)
        bound = (D + 2) * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(w).astype(np.float64).T) + \
            2.0 ** -24 * np.abs(bg)
        got = act[g][rows][:, buckets].cpu().numpy().astype(np.float64)
        assert (np.abs(got - want) <= bound + 1e-45).all(), (g, float(np.abs(got - want).max()))


@pytest.mark.parametrize("block", [1, 15, 31, 33, 255, 256, 257, 513, 4096])
def test_encode_tile_edges(block):
    k, W, b, center, scale = inputs(block, 400 + block)
    op, act = run_append(k, W, b, center, scale, block)
    check(k, W, b, center, scale, act)
    assert int(op.n.sum()) == G * 8 * block  # the budget, exactly


def test_encode_is_closer_to_64_bits_than_an_fp32_chain():
    # the split's products and sums are off by less than 128 fp32 roundings: 1.4e-7
    # measured, 2.1e-7 for fp32 MFMA chains; the bound lies between the two
    k, W, b, center, scale = inputs(1024, 5)
    _, act = run_append(k, W, b, center, scale, 1024)
    x = (k[:, H:].float() - center[:, None]) / scale[:, None, None]
    want = torch.stack([torch.relu(x[g].double() @ W[g].double().T + b[g].double()) for g in range(G)])
    assert float((act.double() - want).norm() / want.norm()) < 1.8e-7


@pytest.mark.parametrize("exponent", [-100, -59, -30, 30, 55])
def test_encode_row_and_bucket_scales(exponent):
    # keys and buckets spread over 2^exponent: per-row and per-bucket powers of two (and,
    # beyond 2^60, the plain fp32 chains) keep the relative precision of each
    k, W, b, center, scale = inputs(300, 71)
    center.zero_()
    k[:, H::3] = (k[:, H::3].float() * 2.0 ** exponent).to(torch.bfloat16)
    W[:, ::5] *= 2.0 ** (-exponent)
    b[:, ::5] = 0.0
    b[:, 1::5] = 0.0
    _, act = run_append(k, W, b, center, scale, 300)
    check(k, W, b, center, scale, act)


def test_encode_rows_and_buckets_that_are_not_split():
    k, W, b, center, scale = inputs(290, 72)
    center.zero_()
    k[:, H + 7] = 0                      # a zero row: relu(b)
    k[2, H + 40, 5] = float("inf")       # its activations: +inf or 0 with the sign of W's column
    k[3, H + 41] = float("nan")          # all NaN sums: relu keeps none
    W[4, 17] = 0                         # a dead bucket
    W[5, 2999, 3] = float("inf")
    W[6, 64] = W[6, 64] * 2.0 ** 80      # beyond the split's range
    b[6, 64] = 0
    _, act = run_append(k, W, b, center, scale, 290)
    assert torch.equal(act[:5, 7], torch.relu(b[:5]))
    want = torch.where(W[2, :, 5] > 0, float("inf"), 0.0)
    assert torch.equal(act[2, 40], want)
    assert not bool(act[3, 41].any())
    assert torch.equal(act[4, :, 17], torch.relu(b[4, 17]).expand(290))
    x = (k[5, H:].float() / scale[5])[:, 3]
    rows = torch.arange(290, device="cuda") != 7
    assert torch.equal(act[5, rows, 2999], torch.where(x[rows] > 0, float("inf"), 0.0))
    rest = [r for r in range(290) if r not in (7, 40, 41)]
    check(k, W, b, center, scale, act, rows=rest, buckets=[f for f in range(F) if f != 2999])


@pytest.mark.parametrize("block", [16, 17, 63, 65, 80, 81, 129, 1023, 1041, 2000])
def test_encode_steps_and_stages(block):
    # token ranges of whole 16-token steps, rows split 64 at a time: blocks that end inside either
    k, W, b, center, scale = inputs(block, 900 + block)
    op, act = run_append(k, W, b, center, scale, block)
    check(k, W, b, center, scale, act)
    assert int(op.n.sum()) == G * 8 * block


@pytest.mark.parametrize("exponent", [-59, -40, 40, 59])
def test_encode_key_scales(exponent):
    # the row's power of two is folded into the division by the key scale; where the
    # divisor would leave the normal range the plain fp32 chains take over
    k, W, b, center, scale = inputs(100, 33)
    center.zero_()
    k[:, H:] = (k[:, H:].float() * 2.0 ** exponent).to(torch.bfloat16)
    k[:, H + 1::4] = (k[:, H + 1::4].float() * 2.0 ** (exponent // 2)).to(torch.bfloat16)
    scale = scale * 2.0 ** exponent
    _, act = run_append(k, W, b, center, scale, 100)
    check(k, W, b, center, scale, act)


@pytest.mark.parametrize("where", ["buckets", "keys"])
@pytest.mark.parametrize("dims,norm", [(1, 3.2e-8), (4, 4.9e-8), (16, 8.5e-8), (79, 1.8e-7)])
def test_encode_of_few_dims(where, dims, norm):
    # a sum of few products has few roundings in fp32, fewer than the split's operands
    # cost it: fp32 chains measure 2.5e-8, 3.9e-8, 7.5e-8 and 1.6e-7 (2-norm), the split
    # 0.8 to 1.0e-7.  Every third row or bucket is such a one, the others are dense
    k, W, b, center, scale = inputs(200, 81)
    center.zero_()
    b.zero_()
    if where == "buckets":
        W[:, ::3, dims:] = 0
        pick = (slice(None), slice(0, F, 3))
    else:
        k[:, H::3, dims:] = 0
        pick = (slice(0, None, 3), slice(None))
    _, act = run_append(k, W, b, center, scale, 200)
    x = (k[:, H:].float() / scale[:, None, None])[:, pick[0]]
    want = torch.stack([torch.relu(x[g].double() @ W[g, pick[1]].double().T) for g in range(G)])
    got = act[:, pick[0], pick[1]].double()
    assert float((got - want).norm() / want.norm()) < norm
    if dims == 1:  # one product, one rounding
        assert bool(((got - want).abs() <= 2.0 ** -24 * want).all())


def test_encode_of_a_key_with_one_large_dim():
    # the other dims fall toward f16's subnormals once the largest one is at 2^15: 2.0e-7 by
    # fp32 chains, 2.4e-7 split
    k, W, b, center, scale = inputs(200, 82)
    b.zero_()
    k[:, :, 7] = (k[:, :, 7].float() * 2.0 ** 18).to(torch.bfloat16)
    W[:, :, 7] = 0
    _, act = run_append(k, W, b, center, scale, 200)
    x = (k[:, H:].float() - center[:, None]) / scale[:, None, None]
    want = torch.stack([torch.relu(x[g].double() @ W[g].double().T) for g in range(G)])
    assert float((act.double() - want).norm() / want.norm()) < 2.15e-7
