"""Packed prefill at the edges of its kernels' ranges, against the CPU oracle (GPU).

Tolerances are those of the other prefill tests: the storage type's rounding
of the output and of the probabilities (bf16 2^-9, fp16 2^-12 relative, at
outputs of order 1), fp32 1e-5.
"""

import pytest
import torch

from oracle.paged_attention import paged_attention_cpu
from test_decode_gpu import TOL, ragged_prefill_case

pytestmark = pytest.mark.gpu


def run_prefill(q, kp, vp, tables, lens, cu, chunks, **kw):
    from vllm_rlt_amd import ops

    out = ops.paged_prefill(
        q if q.is_cuda else q.cuda(), kp.cuda(), vp.cuda(), tables.cuda(), lens.cuda(), cu.cuda(), max(chunks), **kw
    )
    torch.cuda.synchronize()
    return out.cpu()


@pytest.mark.parametrize("num_seqs", [1, 15, 16, 17, 64, 65, 511])
def test_ranking_at_its_size_limits(num_seqs):
    # Sequences are ranked in registers up to 16 and through LDS up to 512: every
    # sequence's query tiles must be found exactly once, equal lengths among them.
    g = torch.Generator().manual_seed(num_seqs)
    prefixes = [int(x) for x in torch.randint(0, 3, (num_seqs,), generator=g) * 64]
    chunks = [int(x) for x in torch.randint(0, 4, (num_seqs,), generator=g)]
    chunks[0] = 130
    q, kp, vp, tables, lens, cu, row_tables, row_lengths = ragged_prefill_case(
        torch.bfloat16, 8, 8, 128, prefixes, chunks, num_seqs
    )
    print(f"[prefill ranking] num_seqs={num_seqs}", flush=True)
    out = run_prefill(q, kp, vp, tables, lens, cu, chunks)
    atol, rtol = TOL[torch.bfloat16]
    torch.testing.assert_close(out, paged_attention_cpu(q, kp, vp, row_tables, row_lengths), atol=atol, rtol=rtol)


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
def test_a_query_that_is_not_finite_leaves_the_other_rows_alone(bad):
    # q is staged in the LDS rows of the second V buffer, which the first MFMA
    # phase multiplies by P = 0: nothing of it may reach another row.
    prefixes, chunks = [70, 0], [140, 33]
    q, kp, vp, tables, lens, cu, row_tables, row_lengths = ragged_prefill_case(
        torch.bfloat16, 8, 8, 128, prefixes, chunks, 3
    )
    plain = run_prefill(q, kp, vp, tables, lens, cu, chunks)
    rows = [5, 131, 150]
    poisoned = q.clone()
    poisoned[rows, 3, 17] = bad
    out = run_prefill(poisoned, kp, vp, tables, lens, cu, chunks)
    keep = torch.ones(out.shape[:2], dtype=torch.bool)
    keep[rows, 3] = False
    assert torch.equal(out[keep], plain[keep])


def test_query_rows_far_apart():
    # A row stride past the direct staging's 32-bit offsets takes the kernel that
    # loads q through registers.
    prefixes, chunks = [40], [5]
    q, kp, vp, tables, lens, cu, row_tables, row_lengths = ragged_prefill_case(
        torch.bfloat16, 8, 8, 128, prefixes, chunks, 11
    )
    wide = torch.empty_strided(q.shape, (1 << 23, 128, 1), dtype=q.dtype, device="cuda")
    wide.copy_(q)
    out = torch.empty(q.shape, dtype=q.dtype, device="cuda")
    run_prefill(wide, kp, vp, tables, lens, cu, chunks, out=out)
    atol, rtol = TOL[torch.bfloat16]
    torch.testing.assert_close(out.cpu(), paged_attention_cpu(q, kp, vp, row_tables, row_lengths), atol=atol, rtol=rtol)
