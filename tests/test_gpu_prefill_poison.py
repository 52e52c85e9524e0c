"""Prefill into planes that hold NaN or infinity, as recycled or uninitialised memory may: a partly filled last block
keeps its other tokens, which must not reach any output (their weights are 0, and 0 times NaN is NaN).  Lengths of every
form, with one and with 15 tokens in the last block, and the last block at every place of a 64-key step; every output
row against a 64-bit softmax within the bounds of test_gpu_prefill_wave.py, and the other tokens' bits untouched."""

import pytest

from pvlc_testlib import W, log, pvlc
from test_gpu_prefill_wave import check, exact, operands

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n,workspace", [(95, False), (97, False), (111, False), (211, False), (769, False), (1157, False),
                                         (3073, True), (3103, True), (3109, True), (3130, True), (3500, True), (3151, False)])
def test_stale_tokens_of_the_last_block_reach_no_output(n, workspace, f32):
    import torch
    q, k, v = operands(n, n + 1)
    want = exact(q, k, v)
    dt = torch.float32 if f32 else torch.float16
    nb = (n + 15) // 16
    nbytes = pvlc.prefill_workspace_bytes(n) if workspace else 0
    ws = torch.empty(max(nbytes, 256), dtype=torch.uint8, device="cuda")
    pvlc.workspace_init(ws, ws.numel())
    call = pvlc.paged_prefill_f32io if f32 else pvlc.paged_prefill_f16
    for poison in (0x7e00, 0x7c00, 0xfc00):  # NaN, +inf, -inf
        log(f"case: prefill over poison {poison:#x} N={n} workspace={workspace} f32={f32}")
        bits = poison - (1 << 16) if poison >= 1 << 15 else poison
        kc, vc = (torch.full((nb * 16 * W,), bits, dtype=torch.int16, device="cuda") for _ in range(2))
        out = torch.zeros(n, 16, 128, dtype=dt, device="cuda")
        call(tokens=n, num_blocks=nb, key_cache=kc, value_cache=vc, query=q.to(dt), key=k.to(dt), value=v.to(dt), out=out,
             workspace=ws if workspace else None, workspace_bytes=nbytes)
        torch.cuda.synchronize()
        check(out, want, f32, f"N={n} f32={f32} over {poison:#x}")
        values = vc.view(nb, 2, 128, 16)
        assert bool((values[-1, :, :, (n - 1) % 16 + 1:] == bits).all()), "tokens past the prompt were written"
