"""The prefill attention that spreads a query block's heads and keys over workgroups and waves (prompts of 97 to 3072
tokens, any greater length without a workspace, and the one-launch form of up to 96 tokens), around the edges it can go wrong at: query blocks and 32-key steps partly
filled, waves without a step, the switch of its one- and two-head forms, block ids reloaded after 32 steps a wave, and
the first lengths of the pair schedule.  Every output row against a 64-bit softmax over the same fp16 operands, in both
operand widths, through a permuted block table with spare blocks.

Bounds, relative L2 over all rows: f32 output 4e-6 (weights as hi + lo fp16 pairs, 2^-22, and f32 sums of at most 2 x 128
products and N weighted values); fp16 output 1e-3 (weights and output rounded to 2^-11 each)."""

import math

import pytest

from pvlc_testlib import W, log, pvlc

pytestmark = pytest.mark.gpu


def run(n, f32, q, k, v, workspace=False):
    """Causal prefill without rotary; operands fp16 tensors, given as f32 to the f32 entry point."""
    import torch
    nb = (n + 15) // 16 + 5
    table = torch.randperm(nb, generator=torch.Generator().manual_seed(n))[:(n + 15) // 16].int().cuda()
    kc, vc = (torch.zeros(nb * 16 * W, dtype=torch.float16, device="cuda") for _ in range(2))
    dt = torch.float32 if f32 else torch.float16
    out = torch.full((n * 2048 + 64,), float("nan"), dtype=dt, device="cuda")
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    nbytes = pvlc.prefill_workspace_bytes(n) if workspace else 0
    ws = None
    if nbytes:
        ws = torch.empty(nbytes, dtype=torch.uint8, device="cuda")
        pvlc.workspace_init(ws, nbytes)
    call = pvlc.paged_prefill_f32io if f32 else pvlc.paged_prefill_f16
    call(tokens=n, num_blocks=nb, key_cache=kc, value_cache=vc, query=q.to(dt), key=k.to(dt), value=v.to(dt), out=out,
         block_table=table, error_word=err, workspace=ws, workspace_bytes=nbytes)
    torch.cuda.synchronize()
    assert int(err.item()) == 0
    assert bool(torch.isnan(out[n * 2048:]).all()), "prefill wrote past the output"
    return out[:n * 2048].view(n, 16, 128)


def exact(q, k, v):
    import torch
    n = q.shape[0]
    out = torch.empty(n, 16, 128, dtype=torch.float64, device="cuda")
    mask = torch.ones(n, n, dtype=torch.bool, device="cuda").triu(1)
    for h in range(16):
        s = (q[:, h].double() @ k[:, h // 8].double().t().contiguous() / math.sqrt(128)).masked_fill(mask, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, h // 8].double().contiguous()
    return out


def operands(n, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(n, h, 128, generator=g, device="cuda").half() for h in (16, 2, 2)]


def check(got, want, f32, label):
    rel = float((got.double() - want).norm() / want.norm())
    log(f"[parity] {label}: rel_l2={rel:.3e}")
    assert rel <= (4e-6 if f32 else 1e-3)


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 32, 33, 65, 129, 255, 768, 769, 1100, 3072, 4200])
def test_every_row_at_the_edges(n, f32):
    log(f"case: wave prefill N={n} f32={f32}")
    q, k, v = operands(n, n)
    check(run(n, f32, q, k, v), exact(q, k, v), f32, f"N={n} f32={f32}")


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n", [3072, 3073, 3500])
def test_both_sides_of_the_pair_schedule(n, f32):
    """With a workspace: 3072 tokens run the wave form, 3073 (a last block of one token) and 3500 the pair schedule."""
    log(f"case: prefill with a workspace N={n} f32={f32}")
    q, k, v = operands(n, n + 7)
    check(run(n, f32, q, k, v, workspace=True), exact(q, k, v), f32, f"N={n} f32={f32} workspace")


@pytest.mark.parametrize("n", [200, 1000])
def test_a_step_of_minus_infinite_scores_has_weight_zero(n):
    """Keys 32..63 (one wave's whole first step) score -infinity for every query: their weights are 0, wherever the
    wave that holds them stands in the merge."""
    log(f"case: -inf scores N={n}")
    q, k, v = operands(n, 3 * n)
    q[:, :, 0] = q[:, :, 0].abs() + 1
    k[32:64, :, 0] = -math.inf
    for f32 in (False, True):
        check(run(n, f32, q, k, v), exact(q, k, v), f32, f"-inf step N={n} f32={f32}")


@pytest.mark.parametrize("n,workspace", [(1500, False), (3500, True), (4096, True)])
def test_scores_rising_over_the_waves_steps(n, workspace):
    """Scores that grow along the keys move every wave's softmax reference again and again, and in the pair schedule
    (3500 and 4096 tokens) leave the two parts of a block with references far apart."""
    log(f"case: rising scores N={n} workspace={workspace}")
    q, k, v = operands(n, 99)
    import torch
    ramp = torch.linspace(0, 6, n, device="cuda").half()
    q[:, :, 1] = 12
    k[:, :, 1] = ramp[:, None] * 8
    for f32 in (False, True):
        check(run(n, f32, q, k, v, workspace), exact(q, k, v), f32, f"rising N={n} f32={f32}")
