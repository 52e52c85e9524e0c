"""Ragged batches small enough for one workgroup per (partition, kv head, sequence) in one launch: lengths at the edges
of tiles and partitions, sequences without cached rows, lengths that are refused (error bit 1, sequence left alone),
block ids outside the planes (error bit 2), and both regimes in turn over one workspace.  Outputs against a 64-bit
softmax over the fp16 rows: relative L2 per sequence at most 1e-3 for the fp16 output (weights and output rounded to
2^-11), 4e-6 for the f32 one (weights as hi + lo fp16 pairs, f32 sums); caches bit for bit."""

import math

import numpy as np
import pytest

from pvlc_testlib import W, gather_rows, log, pvlc, scatter_rows, to_dev, to_dev_i32

pytestmark = pytest.mark.gpu


class Batch:
    """Cached rows of ragged sequences in a paged pool; cache_len -5 and beyond the table stand for refused lengths."""

    def __init__(self, cache_lens, max_context, seed):
        r = np.random.default_rng(seed)
        self.lens, self.max_context, n = cache_lens, max_context, len(cache_lens)
        per = (max_context + 15) // 16
        self.nb = n * per + 3
        self.tables = r.permutation(self.nb)[:n * per].reshape(n, per).astype(np.int32)
        self.valid = [0 <= t < per * 16 for t in cache_lens]
        half = lambda m: r.standard_normal(m).astype(np.float16)  # noqa: E731
        self.k, self.v = half(self.nb * 16 * W).view(np.uint16), half(self.nb * 16 * W).view(np.uint16)
        self.rows = [(half(max(t, 0) * W).view(np.uint16), half(max(t, 0) * W).view(np.uint16)) if ok else None
                     for t, ok in zip(cache_lens, self.valid)]
        for s in range(n):
            if self.valid[s]:
                scatter_rows(self.k, self.v, *self.rows[s], cache_lens[s], self.tables[s])
        self.q, self.nk, self.nv = half(n * 2048).reshape(n, 16, 128), half(n * W).reshape(n, 2, 128), half(n * W).reshape(n, 2, 128)

    def run(self, f32, ws, partition=0, tables=None):
        import torch
        n, dt = len(self.lens), torch.float32 if f32 else torch.float16
        d_k, d_v = to_dev(self.k), to_dev(self.v)
        q, nk, nv = (torch.from_numpy(x).cuda().to(dt) for x in (self.q, self.nk, self.nv))
        out = torch.full((n, 16, 128), float("nan"), dtype=dt, device="cuda")
        d_t, d_l = to_dev_i32(self.tables if tables is None else tables), to_dev_i32(np.array(self.lens, np.int32))
        operands = dict(query=None, new_key=None, new_value=None, out=None) if f32 else dict(query=q, new_key=nk, new_value=nv, out=out)
        args = pvlc.paged_decode_args(num_seqs=n, num_blocks=self.nb, max_blocks_per_seq=self.tables.shape[1], key_cache=d_k,
                                      value_cache=d_v, workspace=ws, workspace_bytes=ws.numel(), max_context=self.max_context,
                                      block_tables=d_t, cache_lens=d_l, partition_tokens=partition, **operands)
        if f32:
            pvlc.paged_decode_f32io(args, q, nk, nv, out)
        else:
            pvlc.paged_decode_f16(args)
        torch.cuda.synchronize()
        err = pvlc.workspace_error(ws, ws.numel())
        return out.cpu().numpy(), d_k.cpu().numpy().view(np.uint16), d_v.cpu().numpy().view(np.uint16), err

    def check(self, f32, ws, label, partition=0):
        out, k, v, err = self.run(f32, ws, partition)
        assert err == (0 if all(self.valid) else 1)
        want_k, want_v = self.k.copy(), self.v.copy()
        for s, t in enumerate(self.lens):
            if not self.valid[s]:
                assert np.all(np.isnan(out[s])), f"{label}: refused sequence {s} was written"
                continue
            rk, rv = (np.concatenate([self.rows[s][i], (self.nk, self.nv)[i][s].ravel().view(np.uint16)]) for i in (0, 1))
            scatter_rows(want_k, want_v, rk, rv, t + 1, self.tables[s])
            keys, values = (x.view(np.float16).astype(np.float64).reshape(t + 1, 2, 128) for x in (rk, rv))
            want = np.empty((16, 128))
            for h in range(16):
                sc = keys[:, h // 8] @ self.q[s, h].astype(np.float64) / math.sqrt(128)
                p = np.exp(sc - sc.max())
                want[h] = (p / p.sum()) @ values[:, h // 8]
            rel = np.linalg.norm(out[s] - want) / np.linalg.norm(want)
            assert rel <= (4e-6 if f32 else 1e-3), f"{label}: sequence {s} T={t + 1}: rel {rel}"
        np.testing.assert_array_equal(k, want_k)
        np.testing.assert_array_equal(v, want_v)


def workspace(num_seqs, max_context, partition=0):
    import torch
    nbytes = pvlc.decode_workspace_bytes(num_seqs, max_context, partition)
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    pvlc.workspace_init(ws, nbytes)
    return ws


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("lens,max_context", [
    ([0, 0], 16),                                                    # nothing cached, one partition
    ([0, 1, 14, 15, 16, 17, 62, 63, 64, 65, 127, 128], 200),         # tile and partition edges, ends inside and at a tile
    ([2000, 0, 1999, 300, 255, 256, 257, 511, 512, 1, 90, 1023, 1024], 2010),  # 1 to 8 partitions a sequence
    ([383, 384, 5] * 42 + [20, 0], 385),                             # 256 units: every sequence in one or two partitions
])
def test_ragged_lengths(lens, max_context, f32):
    log(f"case: ragged single launch {len(lens)} seqs max_context={max_context} f32={f32}")
    batch = Batch(lens, max_context, len(lens))
    ws = workspace(len(lens), max_context)
    for rep in range(2):
        batch.check(f32, ws, f"{len(lens)} seqs, call {rep}")


def test_refused_lengths_leave_their_sequences_alone():
    log("case: ragged single launch with refused lengths")
    batch = Batch([-5, 40, 704, 699, 0, 1 << 20], 700, 3)
    batch.check(False, workspace(6, 700), "refused lengths")


def test_block_ids_outside_the_planes_are_reported():
    log("case: ragged single launch with a bad block id")
    batch = Batch([100, 40, 250], 300, 4)
    tables = batch.tables.copy()
    tables[1, 2] = batch.nb  # the block that sequence 1 appends to
    out, k, v, err = batch.run(False, workspace(3, 300), tables=tables)
    assert err == 2
    for s in (0, 2):
        gk, _ = gather_rows(k, v, batch.lens[s] + 1, batch.tables[s])
        np.testing.assert_array_equal(gk[:batch.lens[s] * W], batch.rows[s][0])
        assert np.all(np.isfinite(out[s]))


def test_both_regimes_share_a_workspace():
    """Explicit 16-token partitions of 24 sequences make 24 x 2 x 32 workgroups (streaming), 256-token ones 96."""
    lens = [511, 3, 100, 256, 17, 480] * 4
    batch = Batch(lens, 512, 9)
    ws = workspace(24, 512, 16)
    for rep, partition in enumerate([16, 256, 0, 16, 64, 256]):
        log(f"case: shared workspace, partition {partition}")
        batch.check(False, ws, f"partition {partition}, call {rep}", partition)


def test_automatic_launches_record_their_partition():
    """Ragged automatic launches of either regime over one workspace leave the partition they ran with in the word after
    the error word (so never an earlier launch's), the first sequence refused or not; an explicit partition leaves it."""
    words = lambda: ws[4:12].cpu().numpy().view(np.uint32)  # noqa: E731
    ws = workspace(64, 1300)  # the largest of the launches below
    for lens, max_context, streams in [([2, 0, 13], 16, False), ([1299] * 64, 1300, True), ([1999, 5, 300], 2010, False),
                                       ([-5, 700], 701, False), ([1299] * 64, 1300, True), ([40] * 5, 300, False)]:
        log(f"case: recorded partition {len(lens)} seqs max_context={max_context}")
        assert pvlc.decode_workspace_bytes(len(lens), max_context) <= ws.numel()
        pvlc.workspace_init(ws, 256)  # the error word of the refused sequence
        batch = Batch(lens, max_context, len(lens))
        batch.check(False, ws, f"{len(lens)} seqs")
        plan, (chosen, units) = pvlc.decode_partition(len(lens), max_context), (int(w) for w in words())
        assert units > 0 and chosen == pvlc.decode_streaming_partition(np.array(lens, np.int32), max_context, units)
        assert streams or chosen == plan
        batch.check(False, ws, "explicit", 32 if max_context < 500 else 512)
        assert int(words()[0]) == chosen


@pytest.mark.parametrize("f32", [False, True])
def test_batches_of_changing_size_share_a_workspace(f32):
    """A serving loop keeps one workspace, zeroed once, while its batch grows and shrinks: the partials of a small batch
    must not lie where a larger one counts arrivals.  Single launches of 3 to 256 sequences, streaming ones between."""
    batches = [Batch([2000 - 37 * i for i in range(3)], 2010, 31), Batch([383 - 5 * i for i in range(40)], 400, 32),
               Batch([900 - 11 * i for i in range(64)], 1000, 33), Batch([96 - i % 17 for i in range(256)], 97, 34),
               Batch([383, 384, 5] * 42 + [20, 0], 385, 35)]
    import torch
    ws = torch.empty(max(pvlc.decode_workspace_bytes(len(b.lens), b.max_context) for b in batches), dtype=torch.uint8, device="cuda")
    pvlc.workspace_init(ws, ws.numel())
    for rep, i in enumerate([0, 1, 0, 3, 2, 4, 1, 3, 0, 4]):
        log(f"case: one workspace, batch of {len(batches[i].lens)}, call {rep} f32={f32}")
        batches[i].check(f32, ws, f"batch of {len(batches[i].lens)}, call {rep}")
