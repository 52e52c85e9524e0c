"""Sessions of one runtime take over the buffers of finished ones: capacities that grow and shrink, two sessions alive at
once, and a session dropped without finishing in between.  Every session's rows come back bit for bit and its attention
equals a 64-bit softmax over its own fp16-rounded rows (relative L2 at most 4e-6: weights as hi + lo fp16 pairs, f32
sums), so nothing of an earlier session is left in the planes, the workspace or the staging."""

import math

import numpy as np
import pytest

from pvlc_testlib import log, pvlc

pytestmark = pytest.mark.gpu


class Live:
    def __init__(self, runtime, prefix, capacity, seed):
        r = np.random.default_rng(seed)
        self.r, self.t = r, prefix
        self.k, self.v = (r.standard_normal((capacity, 2, 128), dtype=np.float32) for _ in range(2))
        self.session = runtime.begin_decoder_kv_session(
            pvlc.DecoderKvSessionDescriptor(prefix, capacity, self.k.ravel(), self.v.ravel()))

    def step(self):
        q, k, v = (self.r.standard_normal((h, 128), dtype=np.float32) for h in (16, 2, 2))
        got = self.session.step(pvlc.DecoderKvSessionStep(q.ravel(), k.ravel(), v.ravel())).attention.reshape(16, 128)
        self.k[self.t], self.v[self.t] = k, v
        self.t += 1
        keys, values = (x[:self.t].astype(np.float16).astype(np.float64) for x in (self.k, self.v))
        for h in range(16):
            s = keys[:, h // 8] @ q[h].astype(np.float16).astype(np.float64) / math.sqrt(128)
            p = np.exp(s - s.max())
            want = (p / p.sum()) @ values[:, h // 8]
            assert np.linalg.norm(got[h] - want) <= 4e-6 * np.linalg.norm(want)

    def finish(self):
        snap = self.session.finish()
        assert snap.cache_tokens == self.t
        np.testing.assert_array_equal(snap.key_cache.view(np.uint32), self.k.ravel().view(np.uint32))
        np.testing.assert_array_equal(snap.value_cache.view(np.uint32), self.v.ravel().view(np.uint32))


def test_sessions_over_reused_buffers():
    runtime = pvlc.NativeRuntime(0)
    for seed, (a, b) in enumerate([((300, 320), (17, 33)), ((16, 17), (900, 1000)), ((1, 2), (300, 301)),
                                   ((513, 700), (40, 64))]):
        log(f"case: sessions {a} and {b} on one runtime")
        first, second = Live(runtime, *a, seed=seed), Live(runtime, *b, seed=100 + seed)
        first.step()
        second.step()
        first.finish()
        third = Live(runtime, 5, 9, seed=200 + seed)  # takes the first's buffers while the second lives
        third.step()
        second.finish()
        third.step()
        if seed % 2:
            third.finish()
        else:
            del third  # dropped without finishing
    runtime.close()


def test_the_larger_set_is_kept():
    """Two sessions that lived side by side end in either order: the larger one's buffers serve the next large session
    (no device memory is allocated for it), and the runtime gives everything back."""
    import torch
    used = lambda: base - torch.cuda.mem_get_info()[0]  # noqa: E731
    torch.cuda.synchronize()
    small, large, large_bytes = (5, 40), (9, 32768), 2 * 32768 * 512
    for order in ("small first", "large first"):
        log(f"case: session buffers kept, {order}")
        base = torch.cuda.mem_get_info()[0]
        runtime = pvlc.NativeRuntime(0)
        a, b = Live(runtime, *large, seed=1), Live(runtime, *small, seed=2)
        both = used()
        assert both >= large_bytes
        for x in (b, a) if order == "small first" else (a, b):
            x.step()
            x.finish()
        assert large_bytes <= used() <= both
        kept = used()
        c = Live(runtime, *large, seed=3)
        assert used() == kept, "a large session allocated beside the kept buffers"
        c.step()
        c.finish()
        runtime.close()
        assert used() < large_bytes
