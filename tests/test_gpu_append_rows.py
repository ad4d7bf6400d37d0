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
