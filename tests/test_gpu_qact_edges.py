"""The fused q_activation decode (core.py:131-139, :142-183) off its common
path, against the separate launches: infinite activations, whose weights are
NaN, group counts whose launches have 64 to 256 workgroups per group, and a
captured call."""
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


@pytest.mark.parametrize("H,T", [(1, 2), (777, 5), (9000, 0), (65537, 33), (300001, 7)])
@pytest.mark.parametrize("groups", [1, 2, 4])
def test_other_group_counts_equal_the_separate_launches(groups, H, T):
    # 256, 128 and 64 workgroups per group (Native8B's 8 groups have 32)
    from prismkv_amd import _lib
    op, q, k, v, W, b = operator(H, T, groups + H)
    lib = op.lib
    q, k, v, W, b = (x[:groups].contiguous() for x in (q, k, v, W, b))
    scale = torch.linspace(0.5, 1.5, groups, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream
    cap = op.capacity

    def work(name, *args):
        return torch.zeros(max(lib.query(name, *args), 16), dtype=torch.uint8, device="cuda")

    def outputs():
        return dict(features=torch.full((groups, 64), 3, dtype=torch.int64, device="cuda"),
                    valid=torch.full((groups, 64), 3.0, device="cuda"),
                    raw=torch.full((groups,), 3, dtype=torch.int32, device="cuda"),
                    ids=torch.full((groups, cap), 3, dtype=torch.int32, device="cuda"),
                    count=torch.full((groups,), 3, dtype=torch.int32, device="cuda"),
                    out=torch.full((groups, 4, 128), 3.0, dtype=torch.bfloat16, device="cuda"))

    want, got = outputs(), outputs()
    at = {x: t.data_ptr() for x, t in want.items()}
    qact, union, state = (work("prismkv_route_qact_work_bytes", groups), work("prismkv_union_work_bytes", groups, H),
                          work("prismkv_attend_work_bytes", groups, 64))
    lib.call("prismkv_route_qact", q.data_ptr(), W.data_ptr(), b.data_ptr(), scale.data_ptr(), op.n.data_ptr(),
             qact.data_ptr(), at["features"], at["valid"], at["raw"], 0, groups, _lib.nbytes(qact), stream=stream)
    lib.call("prismkv_union_n", op.bits.data_ptr(), at["features"], at["valid"], union.data_ptr(), at["ids"], at["count"],
             groups, H, op.row_words, cap, 64, _lib.nbytes(union), stream=stream)
    lib.call("prismkv_attend", q.data_ptr(), k.data_ptr(), v.data_ptr(), at["ids"], at["count"], state.data_ptr(),
             at["out"], groups, H, T, k.stride(0), v.stride(0), cap, 64, _lib.nbytes(state), stream=stream)
    at = {x: t.data_ptr() for x, t in got.items()}
    qact, decode = work("prismkv_route_qact_work_bytes", groups), work("prismkv_decode_work_bytes", groups, cap)
    for _ in range(2):
        lib.call("prismkv_decode_qact", q.data_ptr(), W.data_ptr(), b.data_ptr(), scale.data_ptr(), op.n.data_ptr(),
                 op.bits.data_ptr(), k.data_ptr(), v.data_ptr(), qact.data_ptr(), decode.data_ptr(), at["features"],
                 at["valid"], at["raw"], at["ids"], at["count"], at["out"], groups, H, T, cap, op.row_words, k.stride(0),
                 v.stride(0), cap, _lib.nbytes(qact), _lib.nbytes(decode), stream=stream)
        assert int(decode[:4].view(torch.int32)) == 0  # no wait gave up
        for x in ("features", "valid", "raw", "count"):
            assert torch.equal(got[x], want[x]), x
        for g in range(groups):
            assert torch.equal(got["ids"][g, :want["count"][g]], want["ids"][g, :want["count"][g]])
        a, e = got["out"].float(), want["out"].float()
        assert bool(e.isfinite().all()) and float((a - e).norm()) <= 4e-3 * float(e.norm()) + 1e-6


def test_accepted_beside_the_refused():
    # the argument set of test_fused_q_activation_refuses_what_the_decode_refuses, on real memory
    op, q, k, v, W, b = operator(100, 4, 1)
    op.set_query_encoders(W, b, torch.ones(8))
    op.router = "q_activation"
    call = getattr(op.lib.cdll, "prismkv_decode_qact")
    need = op.lib.query("prismkv_decode_work_bytes", 8, 100), op.lib.query("prismkv_route_qact_work_bytes", 8)
    good = [x.data_ptr() for x in (q, W, op.b_query, op.query_scale, op.n, op.bits, k, v, op.qact_work, op.decode_work,
                                   op.features, op.valid, op.raw, op.ids, op.count, op.out)]
    good += [8, 100, 4, 100, op.row_words, k.stride(0), v.stride(0), op.capacity, need[1], need[0],
             torch.cuda.current_stream().cuda_stream]
    assert op.capacity >= 100 and call(*good) == 0
    torch.cuda.synchronize()
    assert op.decode_errors() == 0
    for at, value in ((24, need[1] - 1), (25, need[0] - 1), (17, 0), (18, -1), (1, 0)):
        args = list(good)
        args[at] = value
        assert call(*args) == -1, (at, value)


@pytest.mark.parametrize("H", [700, 40000])
def test_captured_launches(H):
    # the two launches replayed from a HIP graph on new queries, with eager calls between
    op, q, k, v, W, b = operator(H, 9, H)
    op.set_query_encoders(W, b, torch.ones(8))
    op.router = "q_activation"
    names = ("features", "valid", "raw", "count", "out")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        op(q, k, v)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        op(q, k, v)
    for i in range(4):
        q.copy_(torch.randn(q.shape, generator=torch.Generator().manual_seed(i)))
        op(q, k, v)
        want = {x: getattr(op, x).clone() for x in names}
        ids = [op.ids[g, :op.count[g]].clone() for g in range(8)]
        for x in names + ("ids",):
            getattr(op, x).fill_(3)
        graph.replay()
        torch.cuda.synchronize()
        for x in names:
            assert torch.equal(getattr(op, x), want[x]), (i, x)
        for g in range(8):
            assert torch.equal(op.ids[g, :op.count[g]], ids[g]), (i, g)
    assert op.decode_errors() == 0


@pytest.mark.parametrize("H,T", [(700, 0), (700, 3), (70000, 0), (70000, 5)])
def test_no_bucket_of_positive_weight(H, T):
    # two groups whose activations are all 0, one of NaN queries: the tail alone, or nothing
    op, q, k, v, W, b = operator(H, T, H + T)
    W[2:4] = 0
    b[2:4] = -1.0
    q[5] = float("nan")
    op.set_query_encoders(W, b, torch.ones(8))
    op.router = "q_activation"
    op.route(q)
    want_out = op.attention(q, k, v).clone()
    count, valid, raw = op.count.clone(), op.valid.clone(), op.raw.clone()
    got = op(q, k, v)
    assert count[[2, 3, 5]].tolist() == [0, 0, 0] and torch.equal(op.count, count)
    assert torch.equal(op.valid, valid) and torch.equal(op.raw, raw)
    assert torch.equal(got.isnan(), want_out.isnan())
    a, e = got.float().nan_to_num(), want_out.float().nan_to_num()
    assert float((a - e).norm()) <= 4e-3 * float(e.norm())
    assert op.decode_errors() == 0
