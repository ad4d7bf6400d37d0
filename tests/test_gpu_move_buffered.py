"""Movement through a transfer buffer (pace_kv_move_buffered): the buffer and
the destination hold what a pack and an unpack leave there, for pages that
fill, miss or straddle a wave's 1 KiB row, fewer buffer layers than layers,
ids outside their pools, and pools that share memory."""
import pytest
import torch

from paceserve_amd.kv_transfer import ops

pytestmark = pytest.mark.gpu


def pool(layers, pages, page_bytes, gen, dev):
    # float8 elements: one byte each, so any multiple of 16 bytes is a page
    shape = (pages, 2, 1, 1, page_bytes // 2)
    return [torch.randint(0, 120, shape, dtype=torch.uint8, generator=gen).to(dev).view(torch.float8_e4m3fn)
            for _ in range(layers)]


def u8(t):
    return t.view(torch.uint8)


def expect(src, s_ids, dst, d_ids, k):
    """(buffer, destination) of a gather into k layers and a scatter out of
    them, chunk after chunk, on the CPU."""
    src, dst = [u8(t).cpu() for t in src], [u8(t).cpu().clone() for t in dst]
    buf = torch.zeros((k, len(s_ids)) + tuple(src[0].shape[1:]), dtype=torch.uint8)
    for lb in range(0, len(src), k):
        for l in range(lb, min(lb + k, len(src))):
            for j, s in enumerate(s_ids):
                if 0 <= s < src[l].shape[0]:
                    buf[l - lb, j] = src[l][s]
        for l in range(lb, min(lb + k, len(src))):
            for j, d in enumerate(d_ids):
                if 0 <= d < dst[l].shape[0]:
                    dst[l][d] = buf[l - lb, j]
    return buf, dst


@pytest.mark.parametrize("bad", [False, True])
@pytest.mark.parametrize("k", [2, 5, 70])
@pytest.mark.parametrize("page_bytes", [32, 352, 992, 1024, 1056, 2048, 3072, 5120])
def test_buffer_and_destination_match_pack_then_unpack(gpu, page_bytes, k, bad):
    L, N = (70, 11) if k == 70 else (5, 40)     # 70 layers: more than one launch
    gen = torch.Generator().manual_seed(page_bytes + k)
    src, dst = pool(L, N, page_bytes, gen, gpu), pool(L, N, page_bytes, gen, gpu)
    n = N - 4
    s_ids = torch.randperm(N, generator=gen)[:n].tolist()
    d_ids = torch.randperm(N, generator=gen)[:n].tolist()
    if bad:
        s_ids[1], s_ids[n - 1], d_ids[2], d_ids[n - 1] = -1, N, N + 7, -2 ** 31
    want_buf, want_dst = expect(src, s_ids, dst, d_ids, k)
    buf = torch.zeros((k, n) + tuple(src[0].shape[1:]), dtype=torch.uint8, device=gpu).view(torch.float8_e4m3fn)
    err = torch.zeros(1, dtype=torch.int32, device=gpu)
    ids = [torch.tensor(t, dtype=torch.int32, device=gpu) for t in (s_ids, d_ids)]
    ops.move_buffered(src, ids[0], dst, ids[1], buf, err=err)
    assert torch.equal(u8(buf).cpu(), want_buf)
    for l in range(L):
        assert torch.equal(u8(dst[l]).cpu(), want_dst[l]), f"layer {l}"
    assert int(err.item()) == (4 * L if bad else 0)


@pytest.mark.parametrize("how", ["same", "shifted", "one layer", "interleaved"])
def test_pools_that_share_memory_are_packed_before_they_are_unpacked(gpu, how):
    """A page may be source and destination at once: every source page is
    read before the first destination page is written.  The interleaved
    layers share none, though each pool's span covers the other's."""
    L, N, page_bytes = 4, 24, 3072
    gen = torch.Generator().manual_seed(3)
    whole = torch.stack([u8(t) for t in pool(2 * L, 2 * N, page_bytes, gen, gpu)]).view(torch.float8_e4m3fn)
    src = [whole[l, :N] for l in range(L)]
    dst = {"same": src, "shifted": [whole[l, N // 2:N // 2 + N] for l in range(L)],
           "one layer": [src[2]] + [whole[L + l, :N] for l in range(1, L)],
           "interleaved": [whole[l, N:] for l in range(L)]}[how]
    s_ids = torch.randperm(N, generator=gen).tolist()
    d_ids = torch.randperm(N, generator=gen).tolist()
    k = 4
    want_buf, want_dst = expect(src, s_ids, dst, d_ids, k)
    buf = torch.empty((k, N) + tuple(src[0].shape[1:]), dtype=torch.float8_e4m3fn, device=gpu)
    ids = [torch.tensor(t, dtype=torch.int32, device=gpu) for t in (s_ids, d_ids)]
    ops.move_buffered(src, ids[0], dst, ids[1], buf)
    assert torch.equal(u8(buf).cpu(), want_buf)
    for l in range(L):
        assert torch.equal(u8(dst[l]).cpu(), want_dst[l]), f"layer {l}"
