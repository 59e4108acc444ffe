"""prismkv_check_ids (the id checks of attend, core.py:176-179) at the ends of
its argument range."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_the_largest_count_of_ids():
    # indices near 2^31: 17 GB of ids, of which the last three are checked for
    from prismkv_amd import _lib
    n, H = 2 ** 31 - 1, 1 << 20
    ids = torch.arange(n, device="cuda").remainder_(H)
    ids[-1] = H
    out = torch.full((n + 8192,), -7, dtype=torch.int32, device="cuda")
    meta = torch.zeros(2, dtype=torch.int32, device="cuda")
    _lib.load().call("prismkv_check_ids", ids.data_ptr(), out.data_ptr(), meta.data_ptr(), n, H,
                     stream=torch.cuda.current_stream().cuda_stream)
    assert meta.tolist() == [n, 3]  # one out of range, the others many times
    ids[-1] = 0  # clamped
    assert torch.equal(out[:n:4097], ids[::4097].int()) and torch.equal(out[n - 9000:n], ids[-9000:].int())
    assert bool((out[n:] == -7).all())


def check(ids, H):
    from prismkv_amd import _lib
    out = torch.full((len(ids),), -7, dtype=torch.int32, device="cuda")
    meta = torch.zeros(2, dtype=torch.int32, device="cuda")
    _lib.load().call("prismkv_check_ids", ids.data_ptr(), out.data_ptr(), meta.data_ptr(), len(ids), H,
                     stream=torch.cuda.current_stream().cuda_stream)
    return out, meta


@pytest.mark.parametrize("H", [1, 32, 33, 64, 65, 1000, 2049, 1 << 19, (1 << 19) + 1, 1 << 20])
def test_every_id_and_one_twice(H):
    # the bits' places around the powers of two
    ids = torch.randperm(H, generator=torch.Generator().manual_seed(H)).cuda()
    out, meta = check(ids, H)
    assert meta.tolist() == [H, 0] and torch.equal(out.long(), ids)
    assert check(torch.cat((ids, ids[H // 2:H // 2 + 1])), H)[1].tolist() == [H + 1, 2]
    ids[H // 3] = H
    assert check(ids, H)[1].tolist() == [H, 1]


def test_consecutive_ids_cost_what_others_do():
    # 151 us of either (503 of consecutive ones where 32 of them share an LDS word)
    from tests.test_gpu_index_cost import shortest
    H = 600000
    ordered = torch.arange(H, device="cuda")
    mixed = ordered[torch.randperm(H, generator=torch.Generator().manual_seed(1)).cuda()]
    assert shortest(lambda: check(ordered, H)) < 2 * shortest(lambda: check(mixed, H))


def test_refusals():
    from prismkv_amd import _lib
    lib = _lib.load()
    ids = torch.arange(4, device="cuda")
    out = torch.zeros(4, dtype=torch.int32, device="cuda")
    meta = torch.zeros(2, dtype=torch.int32, device="cuda")
    call = getattr(lib.cdll, "prismkv_check_ids")
    good = [ids.data_ptr(), out.data_ptr(), meta.data_ptr(), 4, 1 << 20, torch.cuda.current_stream().cuda_stream]
    for at, value in ((0, 0), (1, 0), (2, 0), (3, -1), (3, 2 ** 31), (4, 0), (4, -1), (4, (1 << 20) + 1)):
        args = list(good)
        args[at] = value
        assert call(*args) == -1, (at, value)
    assert call(*good) == 0 and meta.tolist() == [4, 0] and out.tolist() == [0, 1, 2, 3]
    assert call(0, *good[1:3], 0, *good[4:]) == 0 and meta.tolist() == [0, 0]
