"""Prompts of up to 96 tokens run as one launch that appends and attends together; with a query scratch, and beyond 96
tokens, they run as two.  Both are compared over every form that the one launch accepts: partly filled blocks and 32-key
steps, both operand widths, with and without rotary, positions inside and outside the tables, permuted and identity
tables, a block id outside the planes, and key rows that lie in the output (which stay with the two launches).

The caches and the error word are the same bit for bit.  The outputs differ by the order of the f32 sums only: relative
L2 2e-6 for f32 outputs (sums of N weighted values at 2^-24, weights as hi + lo pairs of 2^-22), 1e-3 for fp16 ones
(output and weights rounded to 2^-11, the weights against another reference of the exponent)."""

import pytest

from pvlc_testlib import W, log, pvlc

pytestmark = pytest.mark.gpu


def rows(n, f32, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    dt = torch.float32 if f32 else torch.float16
    return [torch.randn(n, h, 128, generator=g, device="cuda").to(dt) for h in (16, 2, 2)]


def call(n, f32, operands, table, nb, cos=None, sin=None, positions=None, scratch=False, out=None):
    import torch
    q, k, v = operands
    g = torch.Generator(device="cuda").manual_seed(5)
    kc, vc = (torch.randn(nb * 16 * W, generator=g, device="cuda").half() for _ in range(2))
    if out is None:
        out = torch.full((n + 1, 16, 128), float("nan"), dtype=q.dtype, device="cuda")
    err = torch.zeros(1, dtype=torch.int32, device="cuda")
    qs = torch.empty(n, 16, 128, dtype=torch.float16, device="cuda") if scratch else None
    (pvlc.paged_prefill_f32io if f32 else pvlc.paged_prefill_f16)(
        tokens=n, num_blocks=nb, key_cache=kc, value_cache=vc, query=q, key=k, value=v, out=out, block_table=table,
        rope_cos=cos, rope_sin=sin, rope_rows=0 if cos is None else cos.shape[0], positions=positions, query_scratch=qs,
        error_word=err)
    torch.cuda.synchronize()
    return out, kc, vc, int(err.item())


def compare(one, two, f32, n, attention=True):
    import torch
    assert one[3] == two[3], "error words"
    for a, b in zip(one[1:3], two[1:3]):
        assert torch.equal(a.view(torch.int16), b.view(torch.int16)), "caches"
    if attention:
        a, b = one[0][:n].double(), two[0][:n].double()
        rel = float((a - b).norm() / b.norm())
        log(f"[parity] short prefill N={n} f32={f32}: rel_l2={rel:.3e}")
        assert rel <= (2e-6 if f32 else 1e-3)
    assert bool(torch.isnan(one[0][n:]).all()), "wrote past the output"


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n", [1, 8, 15, 16, 17, 31, 32, 33, 63, 64, 65, 80, 81, 95, 96, 97])
def test_one_launch_against_two(n, f32):
    import torch
    blocks = (n + 15) // 16
    operands = rows(n, f32, n)
    angle = torch.arange(n + 9, device="cuda")[:, None] * 0.7 ** torch.arange(64, device="cuda")[None, :]
    cos, sin = angle.cos().float().contiguous(), angle.sin().float().contiguous()
    table = torch.randperm(blocks + 3, generator=torch.Generator().manual_seed(n))[:blocks].int().cuda()
    inside = (torch.arange(n, device="cuda") + 5).int()
    outside = inside.clone()
    outside[n // 2] = n + 9
    outside[n - 1] = -1
    for label, kw in (("identity, no rotary", dict(table=None)), ("paged, rotary", dict(table=table, cos=cos, sin=sin)),
                      ("paged, positions", dict(table=table, cos=cos, sin=sin, positions=inside)),
                      ("positions outside the tables", dict(table=None, cos=cos, sin=sin, positions=outside))):
        log(f"case: short prefill N={n} f32={f32} {label}")
        one = call(n, f32, operands, nb=blocks + 3, **kw)
        two = call(n, f32, operands, nb=blocks + 3, scratch=True, **kw)
        assert one[3] == (4 if label.startswith("positions out") else 0)
        compare(one, two, f32, n)


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("n", [17, 90])
def test_a_block_id_outside_the_planes_is_reported_and_not_stored(n, f32):
    import torch
    blocks = (n + 15) // 16
    operands = rows(n, f32, n)
    for bad in (-1, blocks):
        table = torch.arange(blocks, device="cuda", dtype=torch.int32)
        table[-1] = bad
        log(f"case: short prefill N={n} f32={f32} block id {bad}")
        one, two = (call(n, f32, operands, table, blocks, scratch=s) for s in (False, True))
        assert one[3] == 2
        compare(one, two, f32, n, attention=False)


def test_key_rows_inside_the_output():
    """The keys lie where the output goes: read before it is written, as with two launches."""
    import torch
    n = 90
    log("case: short prefill, keys in the output")
    q, k, v = rows(n, True, 3)
    out = torch.full((n + 1, 16, 128), float("nan"), device="cuda")
    kin = out.view(-1)[2048 * 30:2048 * 30 + n * W].view(n, 2, 128)
    kin.copy_(k)
    one = call(n, True, (q, kin, v), None, 6, out=out)
    two = call(n, True, (q, k, v), None, 6, scratch=True)
    compare(one, two, True, n)
