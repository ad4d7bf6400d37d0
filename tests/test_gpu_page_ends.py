"""Pages that are no whole number of 1 KiB rows are copied end to end: pack,
unpack, move and promotion of pages around the sizes where the split changes
(21 vectors: 336 bytes) and where a wave holds one, two or many pages, with
page counts that leave a last wave of one vector, part of it or all of it."""
import pytest
import torch

from paceserve_amd.core.block_manager import NativeBlockAllocator
from paceserve_amd.kv_transfer import ops
from paceserve_amd.kv_transfer.migrate import KVMigrator

pytestmark = pytest.mark.gpu
PAGE_BYTES = [32, 64, 320, 352, 480, 496, 512, 544, 1008, 1056, 1536, 3104]


def pool(layers, pages, page_bytes, gen, dev):
    shape = (layers, pages, 2, 1, 1, page_bytes // 2)
    whole = torch.randint(0, 120, shape, dtype=torch.uint8, generator=gen).to(dev)
    return whole, list(whole.view(torch.float8_e4m3fn))


def ids_of(n, pages, gen, bad):
    t = torch.randperm(pages, generator=gen)[:n]
    if bad:
        t[0], t[n // 2], t[n - 1] = -1, pages, -2 ** 31
    return t.tolist()


def in_pool(ids, pages):
    return [j for j, p in enumerate(ids) if 0 <= p < pages]


@pytest.mark.parametrize("bad", [False, True])
@pytest.mark.parametrize("n", [1, 2, 33, 1025])
@pytest.mark.parametrize("page_bytes", PAGE_BYTES)
def test_pack_unpack_move(gpu, page_bytes, n, bad):
    L, N = 3, n + 5
    gen = torch.Generator().manual_seed(page_bytes * 2048 + n)
    (src, src_l), (dst, dst_l) = pool(L, N, page_bytes, gen, gpu), pool(L, N, page_bytes, gen, gpu)
    s_ids, d_ids = ids_of(n, N, gen, bad), ids_of(n, N, gen, bad)
    dev = [torch.tensor(t, dtype=torch.int32, device=gpu) for t in (s_ids, d_ids)]
    err = torch.zeros(1, dtype=torch.int32, device=gpu)
    before = dst.cpu()

    buf = torch.zeros((L, n) + tuple(src.shape[2:]), dtype=torch.uint8, device=gpu).view(torch.float8_e4m3fn)
    ops.pack(src_l, dev[0], buf, err=err)
    want = torch.zeros((L, n) + tuple(src.shape[2:]), dtype=torch.uint8)
    ok = in_pool(s_ids, N)
    want[:, ok] = src.cpu()[:, [s_ids[j] for j in ok]]
    assert torch.equal(buf.view(torch.uint8).cpu(), want)
    skipped = n - len(ok)
    assert int(err.item()) == L * skipped

    ops.unpack(buf, dst_l, dev[1], err=err)
    ok = in_pool(d_ids, N)
    want_dst = before.clone()
    want_dst[:, [d_ids[j] for j in ok]] = want[:, ok]
    assert torch.equal(dst.cpu(), want_dst)
    assert int(err.item()) == L * (skipped + n - len(ok))

    dst.copy_(before)
    err.zero_()
    ops.move(src_l, dev[0], dst_l, dev[1], err=err)
    ok = [j for j in in_pool(s_ids, N) if 0 <= d_ids[j] < N]
    want_dst = before.clone()
    want_dst[:, [d_ids[j] for j in ok]] = src.cpu()[:, [s_ids[j] for j in ok]]
    assert torch.equal(dst.cpu(), want_dst)
    assert int(err.item()) == L * (n - len(ok))


@pytest.mark.parametrize("n", [31775, 31776])        # the last pack by scalar ids, and the first by lanes' own
def test_packs_around_64_mib(gpu, n):
    L, page_bytes = 2, 1056
    gen = torch.Generator().manual_seed(n)
    src, src_l = pool(L, n + 5, page_bytes, gen, gpu)
    ids = torch.randperm(n + 5, generator=gen)[:n]
    ids[0], ids[n - 1] = -1, n + 5
    buf = torch.zeros((L, n) + tuple(src.shape[2:]), dtype=torch.uint8, device=gpu).view(torch.float8_e4m3fn)
    err = torch.zeros(1, dtype=torch.int32, device=gpu)
    ops.pack(src_l, ids.to(torch.int32).to(gpu), buf, err=err)
    want = torch.zeros((L, n) + tuple(src.shape[2:]), dtype=torch.uint8, device=gpu)
    want[:, 1:-1] = src[:, ids[1:-1].to(gpu)]
    assert torch.equal(buf.view(torch.uint8), want)
    assert int(err.item()) == 2 * L


@pytest.mark.parametrize("mode", ["fused", "buffer"])
@pytest.mark.parametrize("n", [1, 33, 512, 513])     # up to 512 ids travel in the kernel arguments
@pytest.mark.parametrize("page_bytes", PAGE_BYTES)
def test_promotion(gpu, page_bytes, n, mode):
    L, N = 3, n + 5
    gen = torch.Generator().manual_seed(page_bytes * 2048 + n)
    (src, src_l), (dst, dst_l) = pool(L, N, page_bytes, gen, gpu), pool(L, N, page_bytes, gen, gpu)
    before = dst.cpu()
    s_ids, free = ids_of(n, N, gen, False), torch.randperm(N, generator=gen).tolist()
    plan = KVMigrator(src_l, dst_l, NativeBlockAllocator(1, N, free)).promote([s_ids], mode=mode)
    want = before.clone()
    want[:, plan.dst_ids] = src.cpu()[:, s_ids]
    assert torch.equal(dst.cpu(), want)


@pytest.mark.parametrize("n", [1, 33, 512, 513])     # up to 512 ids travel in the kernel arguments
@pytest.mark.parametrize("page_bytes", [32, 480, 1056, 2048, 3072])
def test_host_ids(gpu, page_bytes, n):
    """Lists and CPU tensors of page ids, through the device and the host
    legs, in one chunk and in several."""
    L, N = 5, n + 5
    gen = torch.Generator().manual_seed(page_bytes * 2048 + n)
    (src, src_l), (dst, dst_l) = pool(L, N, page_bytes, gen, gpu), pool(L, N, page_bytes, gen, gpu)
    s_ids, d_ids = ids_of(n, N, gen, False), ids_of(n, N, gen, False)
    picked = src.cpu()[:, s_ids]
    want = dst.cpu()
    want[:, d_ids] = picked
    buf = ops.pack(src_l, s_ids)
    assert torch.equal(buf.view(torch.uint8).cpu(), picked)
    ops.unpack(buf, dst_l, torch.tensor(d_ids))
    assert torch.equal(dst.cpu(), want)
    for k in (L, 2):
        host = torch.empty(buf.shape, dtype=buf.dtype, pin_memory=True)
        dst[:, d_ids] = 0
        with ops.Stager(-(-k * n * page_bytes // 256) * 256, 2) as st:
            st.pack_to_host(src_l, s_ids, host, k)
            torch.cuda.synchronize()
            assert torch.equal(host.view(torch.uint8), picked)
            st.unpack_from_host(host, dst_l, d_ids, k)
            assert torch.equal(dst.cpu(), want)


def test_pinned_ids_are_read_in_stream_order(gpu):
    """Pinned ids that earlier work on the stream writes, in a pack and a pack
    to host, and in a graph whose replays follow the ids' new values."""
    L, N, n, page_bytes = 3, 40, 7, 1024
    gen = torch.Generator().manual_seed(11)
    src, src_l = pool(L, N, page_bytes, gen, gpu)
    ids = torch.zeros(n, dtype=torch.int32, pin_memory=True)
    host = torch.empty((L, n) + tuple(src.shape[2:]), dtype=torch.uint8, pin_memory=True)
    buf = torch.empty(host.shape, dtype=torch.uint8, device=gpu).view(torch.float8_e4m3fn)

    def new_ids():
        return torch.randperm(N, generator=gen)[:n].to(torch.int32)

    with ops.Stager(L * n * page_bytes, 2) as st:
        want = new_ids()
        late = want.to(gpu)
        torch.cuda.synchronize()
        torch.cuda._sleep(20_000_000)
        ids.copy_(late, non_blocking=True)
        ops.pack(src_l, ids, buf)
        st.pack_to_host(src_l, ids, host.view(torch.float8_e4m3fn), L)
        torch.cuda.synchronize()
    assert torch.equal(buf.view(torch.uint8).cpu(), src.cpu()[:, want.long()])
    assert torch.equal(host, src.cpu()[:, want.long()])

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.pack(src_l, ids, buf)
    for _ in range(4):
        ids.copy_(new_ids())
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(buf.view(torch.uint8).cpu(), src.cpu()[:, ids.long()])
        assert torch.equal(ops.pack(src_l, ids.tolist()).view(torch.uint8).cpu(), src.cpu()[:, ids.long()])
