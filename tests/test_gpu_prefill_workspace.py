"""One prefill workspace, zeroed once, for prompts of different lengths in turn: the partials of a shorter prompt's split
blocks lie where a longer one counts arrivals, which begin at zero all the same.  Odd and even numbers of query blocks;
every output row against a 64-bit softmax, within the bounds of test_gpu_prefill_wave.py."""

import pytest

from pvlc_testlib import W, log, pvlc
from test_gpu_prefill_wave import check, exact, operands

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f32", [False, True])
def test_prompts_of_different_lengths_share_a_workspace(f32):
    import torch
    lengths = [3500, 6000, 3100, 5210, 5200, 6000]
    nbytes = max(pvlc.prefill_workspace_bytes(n) for n in lengths)
    ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
    pvlc.workspace_init(ws, nbytes)
    dt = torch.float32 if f32 else torch.float16
    for rep, n in enumerate(lengths):
        log(f"case: shared prefill workspace N={n} f32={f32}")
        q, k, v = operands(n, n + rep)
        nb = (n + 15) // 16
        kc, vc = (torch.zeros(nb * 16 * W, dtype=torch.float16, device="cuda") for _ in range(2))
        out = torch.full((n, 16, 128), float("nan"), dtype=dt, device="cuda")
        call = pvlc.paged_prefill_f32io if f32 else pvlc.paged_prefill_f16
        call(tokens=n, num_blocks=nb, key_cache=kc, value_cache=vc, query=q.to(dt), key=k.to(dt), value=v.to(dt), out=out,
             workspace=ws, workspace_bytes=nbytes)
        torch.cuda.synchronize()
        check(out, exact(q, k, v), f32, f"N={n} f32={f32} call {rep}")
