"""One-chunk copies between pages and pinned host memory go in one kernel per
direction: payloads of less than a round of its lanes, exactly one round, one
vector more and many, pages that fill, miss or straddle a KiB, more layers than
a launch takes, and page ids outside the pool."""
import pytest
import torch

from paceserve_amd import _native
from paceserve_amd.kv_transfer import ops

pytestmark = pytest.mark.gpu
# A round is 4 workgroups x 256 lanes x 16 vectors out (256 KiB) and 16 x 256 x
# 8 in (512 KiB).  (layers, pages, page bytes)
SHAPES = [(1, 1, 32), (3, 5, 160), (1, 16, 16384), (1, 32, 16384), (2, 8193, 32), (4, 33, 1056), (70, 3, 2048),
          (5, 40, 65536)]


def pool(layers, pages, page_bytes, gen, dev):
    shape = (layers, pages, 2, 1, 1, page_bytes // 2)
    whole = torch.randint(0, 120, shape, dtype=torch.uint8, generator=gen).to(dev)
    return whole, list(whole.view(torch.float8_e4m3fn))


@pytest.mark.parametrize("bad", [False, True])
@pytest.mark.parametrize("layers,n,page_bytes", SHAPES)
def test_out_in_and_round_trip(gpu, layers, n, page_bytes, bad):
    N = n + 5
    gen = torch.Generator().manual_seed(n * page_bytes)
    (src, src_l), (dst, dst_l) = pool(layers, N, page_bytes, gen, gpu), pool(layers, N, page_bytes, gen, gpu)
    s_ids, d_ids = torch.randperm(N, generator=gen)[:n], torch.randperm(N, generator=gen)[:n]
    if bad:
        s_ids[0], s_ids[n - 1], d_ids[n // 2] = -1, N, -2 ** 31
    s_ok, d_ok = (s_ids >= 0) & (s_ids < N), (d_ids >= 0) & (d_ids < N)
    ids = [t.to(torch.int32).to(gpu) for t in (s_ids, d_ids)]
    err = torch.zeros(1, dtype=torch.int32, device=gpu)
    before = dst.cpu()
    host = torch.full((layers, n) + tuple(src.shape[2:]), 121, dtype=torch.uint8, pin_memory=True)
    want = host.clone()
    want[:, s_ok] = src.cpu()[:, s_ids[s_ok]]
    want_dst = before.clone()
    want_dst[:, d_ids[d_ok]] = want[:, d_ok]
    content = host.view(torch.float8_e4m3fn)
    with ops.Stager(-(-layers * n * page_bytes // 256) * 256, 2) as st:
        st.pack_to_host(src_l, ids[0], content, layers, err=err)
        torch.cuda.synchronize()
        assert torch.equal(host, want)
        assert int(err.item()) == layers * int((~s_ok).sum())
        st.unpack_from_host(content, dst_l, ids[1], layers, err=err)
        assert torch.equal(dst.cpu(), want_dst)
        assert int(err.item()) == layers * int((~s_ok).sum() + (~d_ok).sum())

        dst.copy_(before)
        host.fill_(121)
        st.roundtrip(src_l, ids[0], dst_l, ids[1], content, layers)
        torch.cuda.synchronize()
        assert torch.equal(host, want)
        assert torch.equal(dst.cpu(), want_dst)


def test_host_memory_that_no_kernel_copies(gpu):
    """Pageable memory, and pinned memory off a 16-byte boundary, still go
    through the device slots."""
    layers, n, page_bytes = 3, 7, 1056
    gen = torch.Generator().manual_seed(1)
    (src, src_l), (dst, dst_l) = pool(layers, n, page_bytes, gen, gpu), pool(layers, n, page_bytes, gen, gpu)
    ids = torch.randperm(n, generator=gen)
    size = layers * n * page_bytes
    for raw in (torch.empty(size, dtype=torch.uint8), torch.empty(size + 8, dtype=torch.uint8, pin_memory=True)[8:]):
        host = raw.view(torch.float8_e4m3fn)
        with ops.Stager(-(-size // 256) * 256, 2) as st:
            st.pack_to_host(src_l, ids, host, layers)
            torch.cuda.synchronize()
            assert torch.equal(raw.view(layers, n, -1), src.cpu()[:, ids].reshape(layers, n, -1))
            st.unpack_from_host(host, dst_l, ids, layers)
            assert torch.equal(dst.cpu()[:, ids], src.cpu()[:, ids])
            dst.zero_()
            st.roundtrip(src_l, ids, dst_l, ids, host, layers)
            assert torch.equal(dst.cpu()[:, ids], src.cpu()[:, ids])


@pytest.mark.parametrize("bad", [False, True])
@pytest.mark.parametrize("layers,n,page_bytes", [(1, 1, 1024), (3, 33, 1056), (70, 5, 2048), (2, 900, 1024), (5, 40, 65536),
                                                 (3, 50, 1008), (3, 40, 32), (5, 700, 496), (70, 9, 512),
                                                 (2, 5000, 528), (70, 20, 2048), (1, 8, 65536), (4, 8, 65536)])
def test_swaps(gpu, layers, n, page_bytes, bad):
    """Pages with ids on both sides; a page whose id is out of range on either
    is skipped and counted once.  Pages of up to 512 bytes, small swaps (512
    KiB in, 2 MiB out) and the rest go by three kernels."""
    N, M = n + 5, n + 3
    gen = torch.Generator().manual_seed(n * page_bytes)
    src, src_l = pool(layers, N, page_bytes, gen, gpu)
    host = ops.HostPagePool(layers, M, tuple(src.shape[2:]), torch.float8_e4m3fn)
    d_ids, h_ids = torch.randperm(N, generator=gen)[:n], torch.randperm(M, generator=gen)[:n]
    if bad:
        d_ids[0], h_ids[n - 1], h_ids[n // 2], d_ids[n // 2] = -1, M, -2 ** 31, N
    ok = (d_ids >= 0) & (d_ids < N) & (h_ids >= 0) & (h_ids < M)
    ids = [t.to(torch.int32).to(gpu) for t in (d_ids, h_ids)]
    err = torch.zeros(1, dtype=torch.int32, device=gpu)
    for l, t in enumerate(host.layers):
        t.view(torch.uint8).fill_(121 + l % 2)
    want = torch.stack([t.view(torch.uint8) for t in host.layers]).clone()
    want[:, h_ids[ok]] = src.cpu()[:, d_ids[ok]]
    ops.swap_out(src_l, ids[0], host, ids[1], err=err)
    torch.cuda.synchronize()
    assert torch.equal(torch.stack([t.view(torch.uint8) for t in host.layers]), want)
    before = torch.randint(0, 120, tuple(src.shape), dtype=torch.uint8, generator=gen)
    src.copy_(before)
    ops.swap_in(host, ids[1], src_l, ids[0], err=err)
    before[:, d_ids[ok]] = want[:, h_ids[ok]]
    assert torch.equal(src.cpu(), before)
    assert int(err.item()) == 2 * layers * int((~ok).sum())


@pytest.mark.parametrize("second", ["one chunk", "chunks"])
def test_a_round_trip_reads_what_the_one_before_it_wrote(gpu, second):
    """A migration chain on two streams, its first call held up: the second
    call's source pages are the first one's destination."""
    layers, n, page_bytes = 6, 12, 4096
    gen = torch.Generator().manual_seed(4)
    (a, a_l), (b, b_l), (c, c_l) = (pool(layers, n, page_bytes, gen, gpu) for _ in range(3))
    ids = torch.randperm(n, generator=gen).to(torch.int32).to(gpu)
    size = layers * n * page_bytes
    hosts = [torch.empty(size, dtype=torch.uint8, pin_memory=True) for _ in range(2)]
    x, y = torch.cuda.Stream(gpu), torch.cuda.Stream(gpu)
    torch.cuda.synchronize()
    with ops.Stager(size, 3) as st:
        with torch.cuda.stream(x):
            torch.cuda._sleep(20_000_000)
            st.roundtrip(a_l, ids, b_l, ids, hosts[0], layers)
        with torch.cuda.stream(y):
            st.roundtrip(b_l, ids, c_l, ids, hosts[1], layers if second == "one chunk" else 2)
        torch.cuda.synchronize()
    assert torch.equal(b.cpu(), a.cpu()) and torch.equal(c.cpu(), a.cpu())


@pytest.mark.parametrize("first", ["unpack", "roundtrip", "roundtrip in chunks"])
@pytest.mark.parametrize("second", ["unpack", "roundtrip"])
def test_calls_into_the_same_pages_land_in_call_order(gpu, first, second):
    """Two calls on two streams, the first held up: the second's pages stay.
    The same for two packs into one host buffer."""
    layers, n, page_bytes = 4, 12, 4096
    gen = torch.Generator().manual_seed(5)
    (src, src_l), (dst, dst_l) = pool(layers, n, page_bytes, gen, gpu), pool(layers, n, page_bytes, gen, gpu)
    other, other_l = pool(layers, n, page_bytes, gen, gpu)
    ids = torch.arange(n, dtype=torch.int32, device=gpu)
    size = layers * n * page_bytes
    hosts = [torch.empty((layers, n) + tuple(src.shape[2:]), dtype=torch.uint8, pin_memory=True) for _ in range(3)]
    contents = [h.view(torch.float8_e4m3fn) for h in hosts]
    for host, pages in zip(hosts, (src, other)):
        host.copy_(pages.cpu())
    a, b = torch.cuda.Stream(gpu), torch.cuda.Stream(gpu)
    torch.cuda.synchronize()

    def call(st, kind, i):
        if kind == "unpack":
            st.unpack_from_host(contents[i], dst_l, ids, layers)
        else:
            st.roundtrip((src_l, other_l)[i], ids, dst_l, ids, contents[i], 1 if "chunks" in kind else layers)

    with ops.Stager(size, 3) as st:
        with torch.cuda.stream(a):
            torch.cuda._sleep(20_000_000)
            call(st, first, 0)
        with torch.cuda.stream(b):
            call(st, second, 1)
        torch.cuda.synchronize()
        assert torch.equal(dst.cpu(), other.cpu())

        with torch.cuda.stream(a):
            torch.cuda._sleep(20_000_000)
            st.pack_to_host(src_l, ids, contents[2], layers)
        with torch.cuda.stream(b):
            st.pack_to_host(other_l, ids, contents[2], layers)
        torch.cuda.synchronize()
        assert torch.equal(hosts[2], other.cpu())


def test_one_chunk_legs_in_a_graph(gpu):
    """Captured with the library's own calls, replayed among eager calls on
    the same stager: each replay copies what the pages hold then."""
    layers, n, page_bytes = 4, 12, 4096
    gen = torch.Generator().manual_seed(6)
    (src, src_l), (dst, dst_l) = pool(layers, n, page_bytes, gen, gpu), pool(layers, n, page_bytes, gen, gpu)
    ids = torch.randperm(n, generator=gen).to(torch.int32).to(gpu)
    host = torch.empty((layers, n) + tuple(src.shape[2:]), dtype=torch.uint8, pin_memory=True)
    spare = torch.empty_like(host).pin_memory()
    sp, dp, lib = ops.as_pool(src_l), ops.as_pool(dst_l), _native.load()
    with ops.Stager(layers * n * page_bytes, 2) as st:
        st.pack_to_host(src_l, ids, spare.view(torch.float8_e4m3fn), layers)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            stream = torch.cuda.current_stream().cuda_stream
            _native.check(lib.pace_kv_pack_to_host(st._handle, sp.table(), layers, n, ids.data_ptr(), n, page_bytes,
                                                   layers, host.data_ptr(), None, stream))
            _native.check(lib.pace_kv_unpack_from_host(st._handle, host.data_ptr(), dp.table(), layers, n,
                                                       ids.data_ptr(), n, page_bytes, layers, None, stream))
        for i in range(4):
            src.copy_(torch.randint(0, 120, tuple(src.shape), dtype=torch.uint8, generator=gen))
            dst.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(dst.cpu(), src.cpu())
            assert torch.equal(host, src.cpu()[:, ids.cpu().long()])
            st.pack_to_host(src_l, ids, spare.view(torch.float8_e4m3fn), layers)
            st.roundtrip(src_l, ids, dst_l, ids, spare, layers)
            torch.cuda.synchronize()
            assert torch.equal(spare.reshape(host.shape), host)


@pytest.mark.parametrize("kind", ["pack", "unpack", "roundtrip"])
def test_close_waits_for_one_chunk_calls(gpu, kind):
    """A closed stager's calls have finished, on a stream that was held up."""
    layers, n, page_bytes = 4, 12, 4096
    gen = torch.Generator().manual_seed(7)
    (src, src_l), (dst, dst_l) = pool(layers, n, page_bytes, gen, gpu), pool(layers, n, page_bytes, gen, gpu)
    ids = torch.arange(n, dtype=torch.int32, device=gpu)
    host = torch.empty((layers, n) + tuple(src.shape[2:]), dtype=torch.uint8, pin_memory=True)
    host.copy_(src.cpu()) if kind == "unpack" else host.fill_(121)
    content, stream = host.view(torch.float8_e4m3fn), torch.cuda.Stream(gpu)
    torch.cuda.synchronize()
    with ops.Stager(layers * n * page_bytes, 2) as st, torch.cuda.stream(stream):
        torch.cuda._sleep(20_000_000)
        if kind == "pack":
            st.pack_to_host(src_l, ids, content, layers)
        elif kind == "unpack":
            st.unpack_from_host(content, dst_l, ids, layers)
        else:
            st.roundtrip(src_l, ids, dst_l, ids, content, layers)
        st.close()
    assert torch.equal(host, src.cpu())
    assert kind == "pack" or torch.equal(dst.cpu(), src.cpu())


@pytest.mark.parametrize("call", ["pack_to_host", "unpack_from_host", "pack_to_host_inline", "unpack_from_host_inline"])
def test_missing_page_ids_leave_everything_as_it_was(gpu, call):
    layers, n, page_bytes = 3, 5, 1024
    gen = torch.Generator().manual_seed(8)
    src, src_l = pool(layers, n, page_bytes, gen, gpu)
    before, p, lib = src.cpu(), ops.as_pool(src_l), _native.load()
    host = torch.full((layers, n, page_bytes), 121, dtype=torch.uint8, pin_memory=True)
    stream = torch.cuda.current_stream().cuda_stream
    with ops.Stager(-(-layers * n * page_bytes // 256) * 256, 2) as st:
        pages = (p.table(), layers, n, None, n, page_bytes, layers)
        args = (*pages, host.data_ptr()) if call.startswith("pack") else (host.data_ptr(), *pages)
        assert getattr(lib, "pace_kv_" + call)(st._handle, *args, None, stream) == _native.PACE_KV_EINVAL
        torch.cuda.synchronize()
    assert torch.equal(src.cpu(), before) and bool((host == 121).all())


def test_more_vectors_than_one_launch_takes(gpu):
    """A launch takes 2^31 vectors: three layers of 2^30 go in two.  Two pages
    of each layer are copied, the rest of the 16384 are out of range."""
    layers, n, page_bytes = 3, 1 << 14, 1 << 20
    gen = torch.Generator().manual_seed(9)
    src, src_l = pool(layers, 2, page_bytes, gen, gpu)
    host = ops.HostPagePool(layers, 2, tuple(src.shape[2:]), torch.float8_e4m3fn)
    d_ids, h_ids = (torch.full((n,), -1, dtype=torch.int32) for _ in range(2))
    d_ids[0], d_ids[-1], h_ids[0], h_ids[-1] = 1, 0, 0, 1
    d_ids, h_ids = d_ids.to(gpu), h_ids.to(gpu)
    err = torch.zeros(1, dtype=torch.int32, device=gpu)
    ops.swap_out(src_l, d_ids, host, h_ids, err=err)
    torch.cuda.synchronize()
    assert torch.equal(torch.stack([t.view(torch.uint8) for t in host.layers]), src.cpu().flip(1))
    assert int(err.item()) == layers * (n - 2)
    before = src.cpu()
    src.zero_()
    ops.swap_in(host, h_ids, src_l, d_ids, err=err)
    assert torch.equal(src.cpu(), before)
    assert int(err.item()) == 2 * layers * (n - 2)
