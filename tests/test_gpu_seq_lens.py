"""get_seq_lens as one launch, against the same tensor arithmetic in 64 bits
and against its other forms (other types, strides, broadcasting, CPU)."""
import pytest
import torch

from paceserve_amd.kv_transfer import append as ap

pytestmark = pytest.mark.gpu


def expect(indptr, last, page_size):
    pages = indptr.long()[1:] - indptr.long()[:-1]
    return (torch.clamp(pages - 1, min=0) * page_size + last.long()).to(torch.int32)


@pytest.mark.parametrize("page_size", [1, 16, 48])
@pytest.mark.parametrize("batch", [1, 2, 255, 256, 257, 1000])
def test_every_form_gives_the_same(gpu, batch, page_size):
    gen = torch.Generator().manual_seed(batch)
    counts = torch.randint(0, 9, (batch,), generator=gen)      # requests without pages among them
    indptr = torch.cat([torch.zeros(1, dtype=torch.long), counts.cumsum(0)]).to(torch.int32)
    last = torch.randint(0, page_size + 1, (batch,), generator=gen).to(torch.int32)
    want = expect(indptr, last, page_size)
    g_ip, g_last = indptr.to(gpu), last.to(gpu)
    assert ap._one_launch(g_ip, g_last, page_size)
    got = ap.get_seq_lens(g_ip, g_last, page_size)
    assert got.dtype == torch.int32 and got.device == g_ip.device and torch.equal(got.cpu(), want)
    spread = torch.zeros(2 * batch, dtype=torch.int32, device=gpu)
    spread[::2] = g_last
    for a, b in ((indptr, last), (g_ip.long(), g_last), (g_ip, spread[::2])):
        assert batch == 1 or not ap._one_launch(a, b, page_size)    # one element has no stride
        assert torch.equal(ap.get_seq_lens(a, b, page_size).cpu(), want)
    one = ap.get_seq_lens(g_ip, g_last[:1], page_size)         # one length for all requests
    assert torch.equal(one.cpu(), expect(indptr, last[:1], page_size))
    assert ap.get_seq_lens(g_ip[:1], g_last[:0], page_size).numel() == 0
    both = torch.vmap(lambda x: ap.get_seq_lens(g_ip, x, page_size))(torch.stack([g_last, g_last + 1]))
    assert torch.equal(both.cpu(), torch.stack([want, want + 1]))


def test_wraps_as_tensor_arithmetic_does(gpu):
    ip = torch.tensor([0, 2 ** 31 - 1, -2 ** 31, 5], dtype=torch.int32)
    last = torch.tensor([2 ** 31 - 1, 3, -7], dtype=torch.int32)
    assert torch.equal(ap.get_seq_lens(ip.to(gpu), last.to(gpu), 4097).cpu(), ap.get_seq_lens(ip, last, 4097))


def test_a_function_mode_sees_the_arithmetic(gpu):
    seen = []

    class Mode(torch.overrides.TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            seen.append(func)
            return func(*args, **(kwargs or {}))

    ip, last = (torch.tensor(x, dtype=torch.int32, device=gpu) for x in ([0, 3, 7], [2, 4]))
    assert ap._one_launch(ip, last, 4)
    with Mode():
        got = ap.get_seq_lens(ip, last, 4)
    assert torch.clamp in seen and got.tolist() == [10, 16]
