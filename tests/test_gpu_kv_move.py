"""Prefix moves between compact rows and the blocked cache, a workgroup per 16-token block: partial last blocks, many
blocks through a permuted table with spare blocks, ids outside the planes.  Bits are moved as they are (NaN payloads
among them): the cache equals the layout written out element by element, tokens past the prefix keep the cache's old
contents, and the way back gives the rows (zeros for a block outside the planes)."""

import numpy as np
import pytest

from pvlc_testlib import W, from_dev, log, pvlc, scatter_rows, to_dev, to_dev_i32

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("table", ["contiguous", "permuted", "bad ids"])
@pytest.mark.parametrize("tokens", [1, 15, 16, 17, 31, 257, 1000])
def test_pack_and_unpack_move_every_bit(tokens, table):
    import torch
    log(f"case: kv move tokens={tokens} {table}")
    rng = np.random.default_rng(tokens)
    k, v = (rng.integers(0, 1 << 16, tokens * W, dtype=np.uint16) for _ in range(2))
    used = (tokens + 15) // 16
    nb = used + (0 if table == "contiguous" else 4)
    ids = np.arange(used) if table == "contiguous" else rng.permutation(nb)[:used]
    want_k, want_v = (rng.integers(0, 1 << 16, nb * 16 * W, dtype=np.uint16) for _ in range(2))
    d_k, d_v = to_dev(want_k), to_dev(want_v)
    rows_k, rows_v = k.copy(), v.copy()
    given = ids.astype(np.int32)
    live = np.arange(used)
    if table == "bad ids":
        bad = rng.permutation(used)[:(used + 2) // 3]
        given[bad] = np.where(np.arange(len(bad)) % 2 == 0, -1, nb)
        live = np.setdiff1d(live, bad)
        for b in bad:
            rows_k[b * 16 * W:(b + 1) * 16 * W] = 0
            rows_v[b * 16 * W:(b + 1) * 16 * W] = 0
    for b in live:
        n = min(16, tokens - b * 16)
        part = slice(b * 16 * W, (b * 16 + n) * W)
        scatter_rows(want_k, want_v, k[part], v[part], n, [ids[b]])
    d_table = None if table == "contiguous" else to_dev_i32(given)
    pvlc.kv_pack_f16(to_dev(k), to_dev(v), tokens, d_k, d_v, nb, block_table=d_table)
    back_k, back_v = (torch.full((tokens * W + 64,), 7, dtype=torch.int16, device="cuda") for _ in range(2))
    pvlc.kv_unpack_f16(d_k, d_v, tokens, back_k, back_v, nb, block_table=d_table)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(from_dev(d_k), want_k)
    np.testing.assert_array_equal(from_dev(d_v), want_v)
    for back, rows in ((back_k, rows_k), (back_v, rows_v)):
        got = from_dev(back)
        np.testing.assert_array_equal(got[:tokens * W], rows)
        assert np.all(got[tokens * W:] == 7), "unpack wrote past the rows"


@pytest.mark.parametrize("tokens", [16, 31, 300])
@pytest.mark.parametrize("shift", [1, 4])
def test_operands_need_their_elements_alignment_only(tokens, shift):
    """Rows and planes that begin 2 or 8 bytes after a 16-byte boundary."""
    import torch
    log(f"case: kv move tokens={tokens} shifted by {2 * shift} bytes")
    rng = np.random.default_rng(tokens)
    used = (tokens + 15) // 16
    k, v = (rng.integers(0, 1 << 16, tokens * W, dtype=np.uint16) for _ in range(2))
    planes = [rng.integers(0, 1 << 16, used * 16 * W, dtype=np.uint16) for _ in range(2)]
    shifted = lambda a: to_dev(np.concatenate([np.zeros(shift, np.uint16), a, np.full(64, 7, np.uint16)]))[shift:]  # noqa: E731
    d_rows, d_planes = [shifted(k), shifted(v)], [shifted(p) for p in planes]
    backs = [shifted(np.zeros(tokens * W, np.uint16)) for _ in range(2)]
    assert all(x.data_ptr() % 16 == 2 * shift for x in d_rows + d_planes + backs)
    pvlc.kv_pack_f16(*d_rows, tokens, *d_planes, used)
    pvlc.kv_unpack_f16(*d_planes, tokens, *backs, used)
    torch.cuda.synchronize()
    for b in range(used):
        n = min(16, tokens - b * 16)
        part = slice(b * 16 * W, (b * 16 + n) * W)
        scatter_rows(*planes, k[part], v[part], n, [b])
    for d, want in zip(d_planes + backs, planes + [k, v]):
        got = from_dev(d)
        np.testing.assert_array_equal(got[:-64], want)
        assert np.all(got[-64:] == 7), "wrote past the end"
