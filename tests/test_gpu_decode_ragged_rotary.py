"""Ragged batches with rotary tables, rotated queries and explicit positions, in both regimes: one launch of up to 512
workgroups (which adds a generation to its arrival counters) and the streaming kernel with 4 and with 2 waves (which
leaves the counters alone), on both sides of 512 workgroups and of 64 sequences.  Positions anywhere in the tables, not
at the row's place, and outside them (error bit 4: that sequence is not rotated); refused lengths beside them.

The appended keys equal the oracle's apply_rope_neox of the key at that position rounded to fp16, bit for bit; outputs
against a 64-bit softmax over the fp16 rows and the query rotated and rounded the same way, within the bounds of
test_gpu_decode_ragged_single.py."""

import math

import numpy as np
import pytest

import oracle as O
from pvlc_testlib import W, log, pvlc, scatter_rows, to_dev, to_dev_f32, to_dev_i32
from test_gpu_decode_ragged_single import Batch, workspace

pytestmark = pytest.mark.gpu
BASE, TABLE_ROWS = 500000.0, 5000


def rotated(x, heads, pos, f32):
    """fp16 of `heads` rows at table position pos (None: not rotated), from their f32 or fp16 values."""
    x = np.ascontiguousarray(x, np.float32).ravel()
    if pos is not None:
        x = O.rope_neox_f32(x, heads, 128, 128, [pos] * heads, BASE)
    return O.f32_to_f16(x).view(np.float16).reshape(heads, 128)


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n,max_context,partition,streams", [
    (13, 2010, 0, False),    # automatic, one launch
    (32, 512, 64, False),    # 512 workgroups
    (33, 512, 64, True),     # 528 workgroups, 2 waves
    (64, 900, 400, True),    # 4 waves, one sequence per lane
    (65, 900, 400, True),    # through LDS
    (130, 600, 512, True),
    (20, 6200, 0, True),     # automatic partition
])
def test_positions_and_rotated_queries(n, max_context, partition, streams, f32):
    import torch
    log(f"case: ragged rotary {n} seqs max_context={max_context} partition={partition} f32={f32}")
    r = np.random.default_rng(n + partition)
    lens = [int(t) for t in r.integers(0, max_context, n)]
    lens[0], lens[1], lens[-1] = max_context - 1, 0, max_context - 2
    lens[n // 2] = -5  # refused
    batch = Batch(lens, max_context, n)
    positions = r.integers(0, TABLE_ROWS, n).astype(np.int32)
    positions[2], positions[n - 2], positions[5] = -1, TABLE_ROWS, TABLE_ROWS - 1
    if f32:  # operands that fp16 does not hold: rotated as f32, rounded once
        batch.q, batch.nk, batch.nv = (r.standard_normal(x.shape, dtype=np.float32) for x in (batch.q, batch.nk, batch.nv))
    dt = torch.float32 if f32 else torch.float16
    cos, sin = pvlc.rope_table(BASE, TABLE_ROWS)
    tables = to_dev_f32(cos), to_dev_f32(sin), to_dev_i32(batch.tables), to_dev_i32(np.array(lens, np.int32))
    ws = workspace(n, max_context, partition)
    for rotate_query, given in [(True, True), (False, True), (True, False)]:
        label = f"{n} seqs rotate_query={rotate_query} positions {'given' if given else 'from lengths'}"
        d_k, d_v, d_p = to_dev(batch.k), to_dev(batch.v), to_dev_i32(positions)
        q, nk, nv = (torch.from_numpy(x).cuda().to(dt) for x in (batch.q, batch.nk, batch.nv))
        out = torch.full((n, 16, 128), float("nan"), dtype=dt, device="cuda")
        operands = dict(query=None, new_key=None, new_value=None, out=None) if f32 else dict(query=q, new_key=nk, new_value=nv, out=out)
        args = pvlc.paged_decode_args(num_seqs=n, num_blocks=batch.nb, max_blocks_per_seq=batch.tables.shape[1], key_cache=d_k,
                                      value_cache=d_v, workspace=ws, workspace_bytes=ws.numel(), max_context=max_context,
                                      block_tables=tables[2], cache_lens=tables[3], rope_cos=tables[0], rope_sin=tables[1],
                                      rope_rows=TABLE_ROWS, positions=d_p if given else None, rotate_query=rotate_query,
                                      partition_tokens=partition, **operands)
        pvlc.workspace_init(ws, 256)  # the error word
        before = ws[256:256 + 8 * n].clone()
        if f32:
            pvlc.paged_decode_f32io(args, q, nk, nv, out)
        else:
            pvlc.paged_decode_f16(args)
        torch.cuda.synchronize()
        assert torch.equal(before, ws[256:256 + 8 * n]) == streams, f"{label}: not the regime it is meant for"
        # the refused length; positions outside the tables where they are given or taken from a length beyond them
        outside = [i for i in range(n) if batch.valid[i] and not 0 <= (positions[i] if given else lens[i]) < TABLE_ROWS]
        assert pvlc.workspace_error(ws, ws.numel()) == 1 | (4 if outside else 0)
        got, want_k, want_v = out.cpu().numpy(), batch.k.copy(), batch.v.copy()
        for s, t in enumerate(lens):
            if not batch.valid[s]:
                assert np.all(np.isnan(got[s])), f"{label}: refused sequence {s} was written"
                continue
            pos = None if s in outside else int(positions[s] if given else t)
            key, value = rotated(batch.nk[s], 2, pos, f32), rotated(batch.nv[s], 2, None, f32)
            rk, rv = (np.concatenate([batch.rows[s][i], (key, value)[i].ravel().view(np.uint16)]) for i in (0, 1))
            scatter_rows(want_k, want_v, rk, rv, t + 1, batch.tables[s])
            query = rotated(batch.q[s], 16, pos if rotate_query else None, f32).astype(np.float64)
            keys, values = (x.view(np.float16).astype(np.float64).reshape(t + 1, 2, 128) for x in (rk, rv))
            want = np.empty((16, 128))
            for h in range(16):
                sc = keys[:, h // 8] @ query[h] / math.sqrt(128)
                p = np.exp(sc - sc.max())
                want[h] = (p / p.sum()) @ values[:, h // 8]
            rel = np.linalg.norm(got[s] - want) / np.linalg.norm(want)
            assert rel <= (4e-6 if f32 else 1e-3), f"{label}: sequence {s} T={t + 1}: rel {rel}"
        np.testing.assert_array_equal(d_k.cpu().numpy().view(np.uint16), want_k)
        np.testing.assert_array_equal(d_v.cpu().numpy().view(np.uint16), want_v)
