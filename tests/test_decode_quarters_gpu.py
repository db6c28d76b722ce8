"""Decode items by one wave and by four: the same bits, and the oracle's result (GPU).

A split's tokens are kept in quarters; small launches give every quarter a
wave, larger ones walk them with one.  Lengths sit at the edges of tiles (32),
quarters (64) and splits (256).  Launches of few rows of two to four splits fold a
row in one workgroup: the same bits again.
"""

import pytest
import torch

from oracle.paged_attention import paged_attention_cpu
from paged_cases import random_decode_case
from test_decode_gpu import TOL

pytestmark = pytest.mark.gpu

ONE_SPLIT = [0, 1, 16, 31, 32, 33, 63, 64, 65, 96, 127, 128, 129, 161, 191, 192, 193, 224, 255, 256]
LONGER = ONE_SPLIT + [257, 288, 320, 321, 447, 511, 512, 513, 705, 1000]
# Past 64 splits of 256 tokens a split doubles.  Rows of more than four splits have
# no quarters: one wave an item in every launch.
LONG = [16384, 16385, 16640, 17000]


def by_row(run, case, append):
    """Each row of the case in a launch of its own."""
    outs = []
    for r in range(len(case.lengths)):
        outs.append(run(case, slice(r, r + 1), append))
    return torch.cat(outs)


def launch(case, rows, append):
    from vllm_rlt_amd import ops

    q, tables, lengths = case.q[rows], case.tables[rows], case.lengths[rows]
    if not append:
        return ops.paged_decode(q, case.key_slice, case.value_slice, tables, lengths)
    k, v, blocks, offsets = (t[rows] for t in append)
    return ops.paged_decode_append(
        q, case.key_slice, case.value_slice, tables, lengths, k.contiguous(), v.contiguous(), blocks.contiguous(),
        offsets.contiguous(),
    )


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("lengths", [ONE_SPLIT, LONGER, LONG], ids=["one_split", "longer", "long"])
def test_one_wave_and_four_give_the_same_bits(lengths, dtype, fused):
    heads = 4 if lengths is LONG else 16
    # Rows alone are small launches; the batch repeats them until it is a large one.
    case = random_decode_case(lengths, hq=heads, hkv=heads, d=128, dtype=dtype, seed=len(lengths))
    dev = case.to("cuda")
    append = None
    if fused:
        last = (dev.lengths.long() - 1).clamp(min=0)
        blocks = dev.tables[torch.arange(len(lengths), device="cuda"), last // 16].long()
        blocks[dev.lengths == 0] = -1  # nowhere
        # The new token is what the page already holds: every launch appends the same bytes.
        safe = blocks.clamp(min=0)
        append = (dev.key_slice[safe, last % 16], dev.value_slice[safe, last % 16], blocks, last % 16)
    alone = by_row(launch, dev, append)
    copies = max(1, 4200 // (heads * len(lengths)))
    many = random_case_copies(dev, copies)
    batch = launch(many, slice(None), tuple(t.repeat((copies,) + (1,) * (t.ndim - 1)) for t in append) if append else None)
    torch.cuda.synchronize()
    print(f"[decode quarters] {dtype} fused={fused} rows={len(lengths) * copies}", flush=True)
    assert torch.equal(batch, alone.repeat(copies, 1, 1))
    atol, rtol = TOL[dtype]
    expect = paged_attention_cpu(case.q, case.key_slice, case.value_slice, case.tables, case.lengths)
    torch.testing.assert_close(alone.cpu(), expect, atol=atol, rtol=rtol)


@pytest.mark.parametrize("fused", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("splits,rows", [(2, 1), (2, 32), (3, 7), (3, 32), (4, 9), (4, 16)])
def test_rows_in_one_workgroup_give_the_same_bits(splits, rows, dtype, fused):
    edges = [n for n in LONGER if n <= 256 * splits] + [256 * splits - d for d in (1, 0, 64, 65, 33)]
    lengths = [edges[(5 * i + splits) % len(edges)] for i in range(rows - 1)] + [256 * splits]
    case = random_decode_case(lengths, hq=16, hkv=16, d=128, dtype=dtype, seed=rows + splits)
    dev = case.to("cuda")
    append = None
    if fused:
        last = (dev.lengths.long() - 1).clamp(min=0)
        blocks = dev.tables[torch.arange(rows, device="cuda"), last // 16].long()
        blocks[dev.lengths == 0] = -1
        safe = blocks.clamp(min=0)
        append = (dev.key_slice[safe, last % 16], dev.value_slice[safe, last % 16], blocks, last % 16)
    few = launch(dev, slice(None), append)
    copies = 1100 // rows  # past every limit of the small launches
    many = random_case_copies(dev, copies)
    batch = launch(many, slice(None), tuple(t.repeat((copies,) + (1,) * (t.ndim - 1)) for t in append) if append else None)
    torch.cuda.synchronize()
    assert torch.equal(batch, few.repeat(copies, 1, 1))
    atol, rtol = TOL[dtype]
    expect = paged_attention_cpu(case.q, case.key_slice, case.value_slice, case.tables, case.lengths)
    torch.testing.assert_close(few.cpu(), expect, atol=atol, rtol=rtol)


@pytest.mark.parametrize("tokens", [16, 200, 256, 700, 1300])
@pytest.mark.parametrize("heads", [(4, 4), (16, 16), (32, 8), (16, 4), (12, 12)])
def test_every_row_and_head_is_served_once(heads, tokens):
    """Left-over groups dealt out by rows: 1 to 7 of them (kv heads / 4 x splits, modulo 8), odd row counts."""
    hq, hkv = heads
    lengths = [1 + (37 * i) % tokens for i in range(66)] + [tokens]
    case = random_decode_case(lengths, hq=hq, hkv=hkv, d=128, dtype=torch.bfloat16, seed=tokens)
    dev = case.to("cuda")
    out = launch(random_case_copies(dev, 5), slice(None), None).view(5, len(lengths), hq, 128)
    assert all(torch.equal(out[0], o) for o in out[1:])
    atol, rtol = TOL[torch.bfloat16]
    expect = paged_attention_cpu(case.q, case.key_slice, case.value_slice, case.tables, case.lengths)
    torch.testing.assert_close(out[0].cpu(), expect, atol=atol, rtol=rtol)


@pytest.mark.parametrize("lengths", [[160, 200], [160, 420], [160, 1000], [160, 3000]], ids=str)
def test_a_tile_of_minus_infinity_scores(lengths):
    # The first tiles of a split, of a quarter and of a later split's quarter hold
    # only scores of -inf: weights of 0, as the oracle has them.
    case = random_decode_case(lengths, hq=16, hkv=16, d=128, dtype=torch.bfloat16, seed=lengths[1])
    case.q[:, 3, 7] = 1.5
    for r, n in enumerate(lengths):
        for first in (0, 64, 320):
            if first + 32 < n:
                case.key_slice[case.tables[r, first // 16 : first // 16 + 2].long(), :, 3, 7] = float("-inf")
    expect = paged_attention_cpu(case.q, case.key_slice, case.value_slice, case.tables, case.lengths)
    assert expect.isfinite().all()
    dev = case.to("cuda")
    atol, rtol = TOL[torch.bfloat16]
    for copies in (1, 12, 200):  # four waves an item, whole rows, one wave an item
        out = launch(random_case_copies(dev, copies), slice(None), None).view(copies, len(lengths), 16, 128)
        assert all(torch.equal(out[0], o) for o in out[1:])
        torch.testing.assert_close(out[0].cpu(), expect, atol=atol, rtol=rtol)


@pytest.mark.parametrize("lengths", [[32, 96, 224], [96, 288, 480], [96, 544, 992]], ids=str)
def test_an_infinite_value_in_the_last_token(lengths):
    # Rows that end with a full first tile of a quarter: its second tile is loaded
    # beyond the row, from the last token, and 0 x Inf would be a NaN.
    case = random_decode_case(lengths, hq=16, hkv=16, d=128, dtype=torch.bfloat16, seed=lengths[1])
    for r, n in enumerate(lengths):
        case.value_slice[int(case.tables[r, (n - 1) // 16]), (n - 1) % 16, 3, 7] = float("inf")
    expect = paged_attention_cpu(case.q, case.key_slice, case.value_slice, case.tables, case.lengths)
    assert (expect == float("inf")).sum() == len(lengths) and not expect.isnan().any()
    dev = case.to("cuda")
    atol, rtol = TOL[torch.bfloat16]
    for copies in (1, 8, 200):  # four waves an item, whole rows, one wave an item
        out = launch(random_case_copies(dev, copies), slice(None), None).view(copies, len(lengths), 16, 128)
        assert all(torch.equal(out[0], o) for o in out[1:])
        torch.testing.assert_close(out[0].cpu(), expect, atol=atol, rtol=rtol)


def random_case_copies(case, copies):
    """The case with its rows repeated; the copies read the same pages."""
    from dataclasses import replace

    return replace(
        case, q=case.q.repeat(copies, 1, 1), tables=case.tables.repeat(copies, 1), lengths=case.lengths.repeat(copies)
    )
