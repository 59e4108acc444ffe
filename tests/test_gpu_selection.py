"""The batch-wide positive Top-k of the index update and build (core.py:13-26)
over the routes its kernels take: the candidate list of the sampled floor, a
list that the sample misjudged (too short, too long), calls that collect none
(a large budget), ties by the thousand in one workgroup's buffer and beyond it,
and buckets of more members than the moments' lists hold."""
import numpy as np
import pytest
import torch

import oracle
from tests.test_gpu_encode import D, F, G, H, inputs, run_append

pytestmark = pytest.mark.gpu


def membership(op, lo, n):
    """Flat indices token * F + bucket, ascending, of each group's bits [lo, lo + n)."""
    t = torch.arange(lo, lo + n, device="cuda")
    out = []
    for g in range(G):
        on = (op.bits[g][:, t // 32] >> (t % 32)) & 1  # [F, n]
        out.append(on.T.contiguous().reshape(-1).nonzero().flatten())
    return out


def check_moments(op, k, flat):
    """Counts exactly, means and variances of the members' keys in 64 bits."""
    from prismkv_amd.native8b import untile_moments
    mean, var = untile_moments(op.moments)
    for g in range(G):
        feat, tok = flat[g] % F, flat[g] // F
        n = torch.bincount(feat, minlength=F)
        assert torch.equal(op.n[g, :F].long(), n)
        x = k[g].double()
        m = torch.zeros(F, D, dtype=torch.float64, device="cuda").index_add_(0, feat, x[tok]) / n.clamp_min(1)[:, None]
        # two-pass fp32: n roundings of the sum and of the squares, each of 2^-24 of the running magnitude
        assert torch.allclose(mean[g].double(), m, rtol=1e-5, atol=2e-5)
        v = torch.zeros(F, D, dtype=torch.float64, device="cuda").index_add_(0, feat, (x[tok] - m[feat]) ** 2)
        assert torch.allclose(var[g].double(), v / n.clamp_min(1)[:, None], rtol=1e-4, atol=2e-5)


@pytest.mark.parametrize("block,buckets,key_mean", [
    (64, 9, 8),         # ties inside one workgroup's buffer
    (600, 3000, 8),     # every value ties: more candidates than the list holds
    (4096, 9, 8),       # 36864 ties listed; buckets of 3640 members
    (4096, 3000, 8),    # list overflow at the largest block
    (100, 5, 8),        # fewer positive values than the budget
    (300, 3000, 2000),  # a budget beyond the list: no candidates collected
    (300, 700, 3000),   # a budget of every value
])
def test_append_ties(block, buckets, key_mean):
    k, W, b, center, scale = inputs(block, 900 + block)
    W.zero_()
    b.zero_()
    b[:, :buckets] = 1.0
    op, _ = run_append(k, W, b, center, scale, block, key_mean)
    # the first block * key_mean ties in flat order
    flat = (torch.arange(block, device="cuda")[:, None] * F + torch.arange(buckets, device="cuda")).flatten()
    flat = flat[:block * key_mean]
    for got in membership(op, H, block):
        assert torch.equal(got, flat)
    check_moments(op, k[:, H:], [flat] * G)


@pytest.mark.parametrize("history,buckets,key_mean", [(5000, 9, 8), (5000, 3000, 8), (5000, 5, 8), (4500, 3000, 2500),
                                                      (70000, 9, 8)])
def test_build_ties(history, buckets, key_mean):
    # beyond 4096 keys the levels of the search are launches of their own
    from prismkv_amd import Native8B
    gen = torch.Generator(device="cuda").manual_seed(history)
    k = torch.randn(G, history, D, generator=gen, device="cuda").to(torch.bfloat16)
    W = torch.zeros(G, F, D, device="cuda")
    b = torch.zeros(G, F, device="cuda")
    b[:, :buckets] = 1.0
    op = Native8B.from_keys(k, history, W, b, torch.ones(G), key_mean)
    torch.cuda.synchronize()
    flat = (torch.arange(history, device="cuda")[:, None] * F + torch.arange(buckets, device="cuda")).flatten()
    flat = flat[:history * key_mean]
    for got in membership(op, 0, history):
        assert torch.equal(got, flat)
    check_moments(op, k, [flat] * G)


@pytest.mark.parametrize("block,loud", [(1024, 5), (4096, 1), (4096, 700), (130, 3)])
def test_append_uneven_tokens(block, loud):
    # a few tokens hold most of the memberships, so the sample's floor is far off
    k, W, b, center, scale = inputs(block, 40 + loud)
    k[:, H + 1:H + 1 + loud] *= 30
    op, act = run_append(k, W, b, center, scale, block)
    got = membership(op, H, block)
    for g in (0, 5):
        want = oracle.positive_global_topk(act[g].cpu().numpy(), 8 * block)
        assert np.array_equal(np.sort(want), got[g].cpu().numpy())
    check_moments(op, k[:, H:], got)


@pytest.mark.parametrize("history", [6000, 40000])
def test_build_without_activations_is_the_build_with_them(history):
    from prismkv_amd import Native8B
    k, W, b, _, scale = inputs(history - H, 7)
    k[:, ::97] *= 20
    ops = [Native8B.from_keys(k, history, W, b, scale, 8, keep_activations=keep) for keep in (False, True)]
    torch.cuda.synchronize()
    for name in ("bits", "n", "moments", "center"):
        assert torch.equal(getattr(ops[0], name), getattr(ops[1], name)), name
    assert int(ops[0].n.sum()) == G * 8 * history


def test_summarize_reads_rows_of_any_alignment():
    # bitmap rows of an odd number of words (the kernel's 16-byte reads do not apply)
    from prismkv_amd import _lib
    from prismkv_amd.native8b import tile_moments
    n, rw = 9000, (9000 + 31) // 32  # 282 words
    lib = _lib.load()
    gen = torch.Generator(device="cuda").manual_seed(3)
    k = torch.randn(1, n, D, generator=gen, device="cuda").to(torch.bfloat16)
    bits = torch.randint(-2 ** 31, 2 ** 31 - 1, (1, F, rw), generator=gen, device="cuda", dtype=torch.int32)
    bits &= torch.randint(-2 ** 31, 2 ** 31 - 1, (1, F, rw), generator=gen, device="cuda", dtype=torch.int32)
    bits[:, 1::2] = 0
    bits[:, ::64] = -1  # every token: 9000 members
    center = torch.zeros(1, D, device="cuda")
    counts = torch.zeros(1, 3008, dtype=torch.int32, device="cuda")
    moments = torch.zeros(1, 94, 256, 32, device="cuda")
    work = torch.zeros(lib.query("prismkv_summarize_work_bytes", 1), dtype=torch.uint8, device="cuda")
    lib.call("prismkv_summarize", k.data_ptr(), bits.data_ptr(), center.data_ptr(), counts.data_ptr(), moments.data_ptr(),
             work.data_ptr(), 1, n, 0, n * D, rw, _lib.nbytes(work), stream=torch.cuda.current_stream().cuda_stream)
    on = ((bits[0][:, :, None] >> torch.arange(32, device="cuda", dtype=torch.int32)) & 1).reshape(F, -1)[:, :n].double()
    c = on.sum(1)
    assert torch.equal(counts[0, :F].double(), c)
    x = k[0].double()
    m = (on @ x) / c.clamp_min(1)[:, None]
    v = (on @ (x * x)) / c.clamp_min(1)[:, None] - m * m
    tiles = tile_moments(m[None].float(), v[None].float())
    assert torch.allclose(moments, tiles, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("first,second", [("ties", "plain"), ("wide", "plain"), ("plain", "wide")])
def test_append_after_append(first, second):
    # each call leaves the counts of its candidates' digits cleared for the next, whichever
    # way it took: thousands of ties in one digit, or values beyond the digits' octave
    from prismkv_amd import Native8B
    block = 1100
    k, W, b, center, scale = inputs(2 * block, 3)
    for i, kind in enumerate((first, second)):
        rows = slice(H + i * block, H + (i + 1) * block)
        if kind == "ties":
            k[:, rows] = k[:, H:H + 1]
        if kind == "wide":  # half the tokens scaled by 2^0 .. 2^12
            k[:, H + i * block:H + (i + 1) * block:2] *= 2.0 ** torch.randint(0, 13, (block // 2, 1), device="cuda")
    zeros = torch.zeros(G, F, dtype=torch.int64, device="cuda")
    op = Native8B.from_tables(H, zeros, torch.zeros(G, F, D, device="cuda"), torch.zeros(G, F, D, device="cuda"),
                              torch.zeros(G, 1, dtype=torch.int32, device="cuda"),
                              torch.zeros(G, F + 1, dtype=torch.int32, device="cuda"), center=center,
                              capacity=H + 2 * block)
    op.set_encoder_tables(W, b, scale, 8)
    for i in range(2):
        op.append(k[:, :H + (i + 1) * block], block)
        act = op.update_activations(block)
        got = membership(op, H + i * block, block)
        for g in range(G):
            want = oracle.positive_global_topk(act[g].cpu().numpy(), 8 * block)
            assert np.array_equal(np.sort(want), got[g].cpu().numpy()), (i, g)


@pytest.mark.parametrize("history,heavy", [(6000, 511), (6000, 513), (32768, 2100), (32769, 2100), (40000, 16385)])
def test_build_heavy_buckets(history, heavy):
    # buckets around the lengths of the token lists, beside ordinary ones: a wave's list
    # of 512 (up to 32768 keys), a workgroup's of 2048, and none
    from prismkv_amd import Native8B
    gen = torch.Generator(device="cuda").manual_seed(heavy)
    k = torch.randn(G, history, D, generator=gen, device="cuda").to(torch.bfloat16)
    k[:, :, 0] = 0
    k[:, :heavy, 0] = 64.0
    W = torch.randn(G, F, D, generator=gen, device="cuda") / D ** 0.5
    W[:, 5::1000] = 0
    W[:, 5::1000, 0] = 8.0  # far above the others for the first `heavy` keys, 0 for the rest
    op = Native8B.from_keys(k, history, W, torch.zeros(G, F, device="cuda"), torch.ones(G), 8)
    torch.cuda.synchronize()
    assert (op.n[:, 5:F:1000] >= heavy).all()
    check_moments(op, k, membership(op, 0, history))


@pytest.mark.parametrize("block,key_mean", [(1024, 60), (1024, 74), (1024, 76), (1024, 100), (4096, 42), (300, 300)])
def test_append_of_many_per_key(block, key_mean):
    # memberships per key around those that the sample can count
    k, W, b, center, scale = inputs(block, key_mean)
    op, act = run_append(k, W, b, center, scale, block, key_mean)
    got = membership(op, H, block)
    for g in (0, 5):
        want = oracle.positive_global_topk(act[g].cpu().numpy(), key_mean * block)
        assert np.array_equal(np.sort(want), got[g].cpu().numpy())
    check_moments(op, k[:, H:], got)


def sampled(block):
    """The tokens whose activations place the floor (sample_token)."""
    S = min(block, 128)
    r = torch.arange(S)
    return r if S == block else r * block // S + ((r * 0x9E3779B9 & 0xFFFFFFFF) >> 8) % (block // S)


@pytest.mark.parametrize("block", [200, 600, 1024, 4096])
@pytest.mark.parametrize("kind", ["low floor", "high floor", "few values", "two values"])
def test_append_with_a_list_of_no_use(kind, block):
    # the sample misjudges: the members are found from the dense activations, by many
    # workgroups and the last of them
    k, W, b, center, scale = inputs(block, 60 + block)
    tok = (H + sampled(block)).cuda()
    loud = torch.ones(H + block, device="cuda")
    if kind == "low floor":  # the others are the loud ones: more candidates than the list holds
        loud[H:] = 30.0
        loud[tok] = 1.0
    else:  # the sampled ones are: fewer candidates than the budget
        loud[tok] = 30.0
    k = (k.float() * loud[:, None]).to(torch.bfloat16)
    if kind == "few values":  # and all the positive ones together are fewer
        center.zero_()
        k[:, H:][:, loud[H:] == 1.0] = 0
        b.fill_(-60.0)
    if kind == "two values":  # the larger one four times a token, the other more often than the list holds
        W.zero_()
        b.fill_(1.0)
        b[:, ::750] = 1.0 + 2.0 ** -22
    op, act = run_append(k, W, b, center, scale, block)
    got = membership(op, H, block)
    for g in (0, 3):
        want = oracle.positive_global_topk(act[g].cpu().numpy(), 8 * block)
        assert np.array_equal(np.sort(want), got[g].cpu().numpy())
    check_moments(op, k[:, H:], got)
