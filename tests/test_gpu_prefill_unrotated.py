"""Prefill without rotary in both operand widths: no tables, and tables that do not hold any position (error bit 4, no
rotation).  The f32 entry point gets no fp16 query, so nothing may be read through that pointer.  Every output row
against a 64-bit softmax over the same fp16-exact operands; relative L2 at most 1e-3 for the fp16 output (weights and
output rounded to 2^-11), 4e-6 for the f32 one (weights as hi + lo fp16 pairs, f32 sums)."""

import math

import pytest

from pvlc_testlib import W, log, pvlc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tables", [False, True])
@pytest.mark.parametrize("n,workspace", [(40, False), (3500, True)])
def test_prefill_without_rotary(n, workspace, tables):
    import torch
    log(f"case: unrotated prefill N={n} workspace={workspace} tables={tables}")
    g = torch.Generator(device="cuda").manual_seed(n)
    q, k, v = (torch.randn(n, h, 128, generator=g, device="cuda").half() for h in (16, 2, 2))
    want = torch.empty(n, 16, 128, dtype=torch.float64, device="cuda")
    mask = torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1)
    for h in range(16):
        s = (q[:, h].double() @ k[:, h // 8].double().t().contiguous() / math.sqrt(128)).masked_fill(mask, -math.inf)
        want[:, h] = torch.softmax(s, -1) @ v[:, h // 8].double().contiguous()
    nb = (n + 15) // 16
    nbytes = pvlc.prefill_workspace_bytes(n) if workspace else 0
    ws = torch.zeros(nbytes, dtype=torch.uint8, device="cuda") if nbytes else None
    rope = {}
    if tables:
        rope = dict(rope_cos=torch.full((4, 64), 0.5, device="cuda"), rope_sin=torch.full((4, 64), 0.5, device="cuda"),
                    rope_rows=4, positions=torch.arange(n, dtype=torch.int32, device="cuda") + 4)
    for dt, call, bound in ((torch.float16, pvlc.paged_prefill_f16, 1e-3), (torch.float32, pvlc.paged_prefill_f32io, 4e-6)):
        kc, vc = (torch.zeros(nb * 16 * W, dtype=torch.float16, device="cuda") for _ in range(2))
        out = torch.full((n, 16, 128), float("nan"), dtype=dt, device="cuda")
        err = torch.zeros(1, dtype=torch.int32, device="cuda")
        call(tokens=n, num_blocks=nb, key_cache=kc, value_cache=vc, query=q.to(dt), key=k.to(dt), value=v.to(dt),
             out=out, error_word=err, workspace=ws, workspace_bytes=nbytes, **rope)
        torch.cuda.synchronize()
        assert int(err.item()) == (4 if tables else 0)
        rel = float((out.double() - want).norm() / want.norm())
        log(f"[parity] unrotated prefill N={n} {dt}: rel_l2={rel:.3e}")
        assert rel <= bound
