"""Paged append where a wave holds whole KiB of one row, parts of two or many
short rows: both forms against the oracle, at row sizes around the wave's 64
vectors, page sizes that are and are not powers of two, batches of more
requests than the search loads in one round, and runs of empty requests."""
import numpy as np
import pytest
import torch

from oracle import kv_oracle as orc
from paceserve_amd import _native
from paceserve_amd.kv_transfer import append as ap


def i32(x, dev):
    return torch.tensor(np.asarray(x), dtype=torch.int32, device=dev)


@pytest.mark.gpu
@pytest.mark.parametrize("P,R", [(1, 5), (3, 70), (16, 700)])
@pytest.mark.parametrize("row_bytes", [16, 48, 256, 1008, 1024, 1040, 1536, 3072, 16400])
def test_rows_around_a_wave_match_the_oracle(gpu, row_bytes, P, R):
    print(f"append rows of {row_bytes} bytes, P={P} R={R}", flush=True)
    rng = np.random.default_rng(row_bytes + R)
    prior, app = rng.integers(0, 20, R), rng.integers(0, 4, R)
    app[R // 3: R // 3 + R // 2] = 0            # a run of requests that append nothing
    app[0], app[-1] = 5, 2
    total = prior + app
    pages = -(-total // P)
    NP = int(pages.sum()) + 3
    kv_indptr = np.concatenate([[0], np.cumsum(pages)])
    kv_indices = rng.permutation(NP)[: kv_indptr[-1]]
    last = np.where(total == 0, 0, (total - 1) % P + 1)
    append_indptr = np.concatenate([[0], np.cumsum(app)])
    nnz = int(append_indptr[-1])
    rand = lambda *shape: rng.integers(0, 120, shape).astype(np.uint8)  # noqa: E731
    k, v, cache = rand(nnz, 1, row_bytes), rand(nnz, 1, row_bytes), rand(NP, 2, P, 1, row_bytes)
    bi, pos = orc.get_batch_indices_positions(append_indptr, orc.get_seq_lens(kv_indptr, last, P), nnz)
    bad = int(nnz // 2)                          # its page does not exist
    kv_indices = np.where(np.arange(len(kv_indices)) == kv_indptr[bi[bad]] + pos[bad] // P, NP, kv_indices)
    ok = kv_indices[kv_indptr[bi] + pos // P] < NP
    want = cache.copy()
    for i in np.nonzero(ok)[0]:
        page = kv_indices[kv_indptr[bi[i]] + pos[i] // P]
        want[page, 0, pos[i] % P], want[page, 1, pos[i] % P] = k[i], v[i]
    f8 = lambda x: torch.from_numpy(x).to(gpu).view(torch.float8_e4m3fn)  # noqa: E731
    args = (i32(kv_indices, gpu), i32(kv_indptr, gpu), i32(last, gpu))
    for form in ("two calls", "fused"):
        got, err = f8(cache), torch.zeros(1, dtype=torch.int32, device=gpu)
        if form == "fused":
            ap.append_paged_kv_cache_indptr(f8(k), f8(v), i32(append_indptr, gpu), got, *args, err=err)
        else:
            ap.append_paged_kv_cache(f8(k), f8(v), i32(bi, gpu), i32(pos, gpu), got, *args, err=err)
        np.testing.assert_array_equal(got.view(torch.uint8).cpu().numpy(), want, err_msg=form)
        assert int(err.item()) == int((~ok).sum()), form


@pytest.mark.parametrize("nnz,row_bytes", [(1 << 24, 256), (1 << 24, 16384), (1 << 23, 16400)])
def test_batches_past_the_limit_are_refused_on_the_host(nnz, row_bytes):
    lib = _native.load()
    rc = lib.pace_kv_append(0x1000, 0x1000, row_bytes, nnz, 0x1000, 0x1000, 4, 0x1000, 8, 0x1000, 8, 0x1000, 16,
                            row_bytes, None, None)
    assert rc == _native.PACE_KV_ERANGE and b"too many tokens" in lib.pace_kv_last_error()


@pytest.mark.gpu
@pytest.mark.parametrize("row_bytes", [8192, 8208])    # whole KiB, and rows end to end
def test_more_rows_than_one_launch_takes(gpu, row_bytes):
    """A launch takes 2^25 waves; the tokens around the split land in their
    pages, and all others, of a request without pages, are counted."""
    first_launch = 2 ** 25 // -(-row_bytes // 1024)
    nnz, n, P = first_launch + 70, 170, 16
    print(f"append {nnz} rows of {row_bytes} bytes", flush=True)
    whole = torch.empty((nnz + 1, 1, row_bytes), dtype=torch.uint8, device=gpu)    # values: one row on from the keys
    tail = torch.randint(0, 120, (n + 1, 1, row_bytes), dtype=torch.uint8)
    whole[-n - 1:] = tail.to(gpu)
    f8 = whole.view(torch.float8_e4m3fn)
    pages = -(-n // P)
    NP = pages + 2
    table = np.random.default_rng(1).permutation(NP)[:pages]
    args = (i32(table, gpu), i32([0, 0, pages], gpu), i32([0, n - (pages - 1) * P], gpu))
    want = torch.full((NP, 2, P, 1, row_bytes), 121, dtype=torch.uint8)
    at, slot = torch.from_numpy(table)[torch.arange(n) // P], torch.arange(n) % P
    want[at, 0, slot], want[at, 1, slot] = tail[:-1], tail[1:]
    for form in ("two calls", "fused"):
        cache = torch.full(want.shape, 121, dtype=torch.uint8, device=gpu)
        err = torch.zeros(1, dtype=torch.int32, device=gpu)
        got = cache.view(torch.float8_e4m3fn)
        if form == "fused":
            ap.append_paged_kv_cache_indptr(f8[:-1], f8[1:], i32([0, nnz - n, nnz], gpu), got, *args, err=err)
        else:
            bi = torch.full((nnz,), -1, dtype=torch.int32, device=gpu)
            bi[-n:] = 1
            pos = torch.zeros(nnz, dtype=torch.int32, device=gpu)
            pos[-n:] = torch.arange(n, dtype=torch.int32, device=gpu)
            ap.append_paged_kv_cache(f8[:-1], f8[1:], bi, pos, got, *args, err=err)
        assert torch.equal(cache.cpu(), want), form
        assert int(err.item()) == nnz - n, form
