"""How the streaming decode kernel numbers its items: up to 64 sequences one per lane of every wave, more through LDS,
with quotients taken by a reciprocal.  The quotient over its whole range on the CPU (edges of every divisor, the
reciprocal one unit in the last place off either way); on the GPU both sides of 64 sequences with empty, refused and
edge lengths, the partition that the kernel settles on against its host replay, outputs and caches as the ragged
single launch's tests hold them."""

import numpy as np
import pytest

from pvlc_testlib import log, pvlc


def test_quotients_by_reciprocal_are_exact():
    for d in range(1, 4097):
        x = np.arange(0, (1 << 19) - d, d, dtype=np.int64)
        x = np.concatenate([x, x + d - 1, x + d // 2])
        x = x[x + d < 1 << 19]
        r = np.float32(1) / np.float32(d)
        for rcp in (r, np.nextafter(r, np.float32(0)), np.nextafter(r, np.float32(2))):
            got = ((x.astype(np.float32) + np.float32(0.5)) * rcp).astype(np.int64)
            np.testing.assert_array_equal(got, x // d, err_msg=f"divisor {d}")


def lengths(n, max_context):
    r = np.random.default_rng(n)
    lens = [int(t) for t in r.integers(max_context - 40, max_context, n)]
    for i, t in enumerate([0, 511, 512, 1023, 1024, -5, 767, 768, 1 << 20, 0, -5]):
        if 5 * i + 1 < n and t < max_context or t == 1 << 20 and n > 50:
            lens[5 * i + 1] = t
    lens[-1] = max_context - 1
    return lens


@pytest.mark.gpu
@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n,max_context", [(1, 6200), (2, 6200), (63, 1300), (64, 1300), (65, 1300), (64, 800), (130, 800)])
def test_both_sides_of_one_sequence_per_lane(n, max_context, f32):
    from test_gpu_decode_ragged_single import Batch, workspace
    log(f"case: streaming numbering {n} seqs max_context={max_context} f32={f32}")
    lens = lengths(n, max_context)
    batch = Batch(lens, max_context, n)
    ws = workspace(n, max_context)
    assert pvlc.decode_partition(n, max_context) == 512
    for rep in range(2):
        batch.check(f32, ws, f"{n} seqs, call {rep}")
        chosen, units = (int(w) for w in ws[4:12].cpu().numpy().view(np.uint32))
        assert chosen == pvlc.decode_streaming_partition(np.array(lens, np.int32), max_context, units)
    explicit = workspace(n, max_context, 400)
    batch.check(f32, explicit, f"{n} seqs, explicit partition", 400)
