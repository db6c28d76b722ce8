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


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(
    "hq,hkv,prefixes,chunks",
    [
        (8, 8, [2047], [1]),  # one row, every segment full
        (8, 2, [959, 1022, 1025], [1, 2, 3]),  # 15, 16 and 17 key tiles: two segments from 16 on
        (16, 16, [3000], [130]),  # two query tiles; the last segment is cut short
        (16, 4, [5000, 0, 40], [64, 33, 7]),  # a long sequence beside ones too short to cut
        (8, 8, [0], [1500]),  # no prefix: the first query tiles end before the later segments
        (32, 8, [2600, 130], [129, 128]),
    ],
)
def test_cut_key_ranges(dtype, hq, hkv, prefixes, chunks):
    # Few query tiles over long contexts: keys in segments and a merge.  The
    # workspace starts as NaN, so a partial that is read is one that was written.
    from vllm_rlt_amd import ops

    q, kp, vp, tables, lens, cu, row_tables, row_lengths = ragged_prefill_case(dtype, hq, hkv, 128, prefixes, chunks, 21)
    need = ops.prefill_split_workspace_bytes(len(q), len(chunks), tables.shape[1], hq, hkv, 128, 16, dtype)
    assert 0 < need <= 17 << 20
    print(f"[prefill cut] {hq}/{hkv} prefixes={prefixes} chunks={chunks} {dtype}", flush=True)
    args = [t.cuda() for t in (q, kp, vp, tables, lens, cu)]
    workspace = torch.full((need,), 0xFF, dtype=torch.uint8, device="cuda")
    out = ops._paged_prefill(*args, max(chunks), None, None, workspace, True)
    plain = ops.paged_prefill(*args, max(chunks), workspace=workspace)  # a given workspace: never cut
    torch.cuda.synchronize()
    atol, rtol = TOL[dtype]
    expect = paged_attention_cpu(q, kp, vp, row_tables, row_lengths)
    torch.testing.assert_close(out.cpu(), expect, atol=atol, rtol=rtol)
    torch.testing.assert_close(plain.cpu(), expect, atol=atol, rtol=rtol)
    assert torch.equal(ops.paged_prefill(*args, max(chunks)), out)


def test_cut_key_ranges_beside_a_context_shorter_than_its_chunk():
    # Rows that see no key are zeros whether or not another sequence is cut.
    from vllm_rlt_amd import ops

    chunks, contexts = [300, 16, 5], [3, 1500, 1]
    q, kp, vp, tables, _, cu, row_tables, _ = ragged_prefill_case(torch.bfloat16, 8, 8, 128, [0, 1484, 0], chunks, 5)
    row_lengths = torch.tensor(
        [max(0, n - (c - 1 - i)) for n, c in zip(contexts, chunks) for i in range(c)], dtype=torch.int32
    )
    out = torch.full(q.shape, 7.0, dtype=q.dtype, device="cuda")
    ops.paged_prefill(
        q.cuda(), kp.cuda(), vp.cuda(), tables.cuda(), torch.tensor(contexts, dtype=torch.int32).cuda(), cu.cuda(),
        max(chunks), out=out,
    )
    torch.cuda.synchronize()
    atol, rtol = TOL[torch.bfloat16]
    torch.testing.assert_close(out.cpu(), paged_attention_cpu(q, kp, vp, row_tables, row_lengths), atol=atol, rtol=rtol)
    assert torch.count_nonzero(out.cpu()[row_lengths == 0]) == 0


@pytest.mark.parametrize(
    "hq,hkv,prefixes,chunks",
    [
        (16, 16, [0], [1]),
        (16, 16, [31, 32, 33], [1, 31, 33]),  # rows and keys around a 32-row, 32-key tile
        (8, 2, [255, 700], [65, 32]),  # every wave a tile; grouped heads
        (3, 3, [9000], [40]),  # a wave's tiles past one batch of page ids
        (4, 1, [0, 5] * 40, [0, 3] * 40),  # more sequences than lanes, empty ones among them
    ],
)
def test_fp32_matrix_kernel(hq, hkv, prefixes, chunks):
    q, kp, vp, tables, lens, cu, row_tables, row_lengths = ragged_prefill_case(
        torch.float32, hq, hkv, 128, prefixes, chunks, 17
    )
    print(f"[prefill fp32] {hq}/{hkv} prefixes={prefixes[:3]} chunks={chunks[:3]}", flush=True)
    atol, rtol = TOL[torch.float32]
    for scale, sign in ((None, 1), (-(128**-0.5), -1)):
        out = run_prefill(q, kp, vp, tables, lens, cu, chunks, scale=scale)
        torch.testing.assert_close(out, paged_attention_cpu(sign * q, kp, vp, row_tables, row_lengths), atol=atol, rtol=rtol)
    # Rows off 16 bytes take the per-token path: the same attention.
    shifted = torch.cat([q.new_zeros(1), q.flatten()]).cuda()[1:].view(q.shape)
    apart = run_prefill(shifted, kp, vp, tables, lens, cu, chunks)
    torch.testing.assert_close(apart, run_prefill(q, kp, vp, tables, lens, cu, chunks), atol=atol, rtol=rtol)


def test_fp32_context_shorter_than_its_chunk():
    chunks, contexts = [70, 3], [20, 1]
    q, kp, vp, tables, _, cu, row_tables, _ = ragged_prefill_case(torch.float32, 4, 4, 128, [0, 0], chunks, 2)
    row_lengths = torch.tensor([max(0, n - (c - 1 - i)) for n, c in zip(contexts, chunks) for i in range(c)], dtype=torch.int32)
    out = run_prefill(q, kp, vp, tables, torch.tensor(contexts, dtype=torch.int32), cu, chunks)
    atol, rtol = TOL[torch.float32]
    torch.testing.assert_close(out, paged_attention_cpu(q, kp, vp, row_tables, row_lengths), atol=atol, rtol=rtol)
    assert torch.count_nonzero(out[row_lengths == 0]) == 0


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_fp32_value_that_is_not_finite_reaches_only_the_rows_that_see_it(bad):
    # A masked key has P = 0, and 0 times its V is a NaN: rows before the token
    # must be what they are without it, the rows that see it as the oracle has them.
    prefixes, chunks = [70, 0, 300], [100, 40, 33]
    q, kp, vp, tables, lens, cu, row_tables, row_lengths = ragged_prefill_case(
        torch.float32, 8, 4, 128, prefixes, chunks, 23
    )
    clean = run_prefill(q, kp, vp, tables, lens, cu, chunks)
    first = {}  # sequence -> its first poisoned token
    for s, token, head, dims in ((0, 120, 1, slice(17, 18)), (0, 137, 3, slice(0, 128)), (1, 39, 2, slice(64, 70)),
                                 (2, 317, 0, slice(127, 128))):
        vp[int(tables[s, token // 16]), token % 16, head, dims] = bad
        first.setdefault(s, token)
    print(f"[prefill fp32] V {bad}", flush=True)
    out = run_prefill(q, kp, vp, tables, lens, cu, chunks)
    seq = torch.repeat_interleave(torch.arange(len(chunks)), torch.tensor(chunks))
    before = row_lengths <= torch.tensor([first[int(s)] for s in seq])
    assert before.any() and torch.equal(out[before], clean[before])
    expect = paged_attention_cpu(q, kp, vp, row_tables, row_lengths)
    atol, rtol = TOL[torch.float32]
    torch.testing.assert_close(out, expect, atol=atol, rtol=rtol, equal_nan=True)


@pytest.mark.parametrize(
    "hq,hkv,prefixes,chunks",
    [(16, 16, [4000], [1]), (16, 16, [2000, 700], [8, 3]), (32, 8, [2500], [7]), (8, 8, [0, 40, 900], [1, 1, 16])],
)
def test_few_fp32_rows_stay_on_the_per_token_path(hq, hkv, prefixes, chunks):
    # A row tile of the matrix-core kernel costs 1 row as much as 32, and one
    # workgroup walks all its keys: few rows are decoded one by one, as by paged_decode.
    from vllm_rlt_amd import ops

    q, kp, vp, tables, lens, cu, row_tables, row_lengths = ragged_prefill_case(
        torch.float32, hq, hkv, 128, prefixes, chunks, 31
    )
    out = run_prefill(q, kp, vp, tables, lens, cu, chunks)
    rows = ops.paged_decode(q.cuda(), kp.cuda(), vp.cuda(), row_tables.cuda(), row_lengths.int().cuda())
    assert torch.equal(out, rows.cpu())
    given = torch.empty(
        ops.prefill_workspace_bytes(len(q), len(chunks), tables.shape[1], hq, hkv, 128, 16, torch.float32),
        dtype=torch.uint8, device="cuda",
    )
    assert torch.equal(run_prefill(q, kp, vp, tables, lens, cu, chunks, workspace=given), out)
    atol, rtol = TOL[torch.float32]
    torch.testing.assert_close(out, paged_attention_cpu(q, kp, vp, row_tables, row_lengths), atol=atol, rtol=rtol)


@pytest.mark.parametrize(
    "hq,hkv,prefixes,chunks",
    [
        (32, 1, [0], [1]),
        (32, 1, [9000], [40]),  # a wave's tiles past one batch of page ids
        (4, 1, [0, 205] * 40, [0, 40] * 40),  # more sequences than lanes, empty ones among them
        (3, 3, [31, 32, 33], [255, 256, 257]),
    ],
)
def test_fp32_matrix_kernel_where_it_is_taken(hq, hkv, prefixes, chunks):
    from vllm_rlt_amd import ops

    q, kp, vp, tables, lens, cu, row_tables, row_lengths = ragged_prefill_case(
        torch.float32, hq, hkv, 128, prefixes, chunks, 37
    )
    print(f"[prefill fp32] {hq}/{hkv} prefixes={prefixes[:3]} chunks={chunks[:3]}", flush=True)
    out = run_prefill(q, kp, vp, tables, lens, cu, chunks)
    rows = ops.paged_decode(q.cuda(), kp.cuda(), vp.cuda(), row_tables.cuda(), row_lengths.int().cuda())
    if len(q) > 1:
        assert not torch.equal(out, rows.cpu())  # not the per-token path, whose bits are these
    atol, rtol = TOL[torch.float32]
    torch.testing.assert_close(out, paged_attention_cpu(q, kp, vp, row_tables, row_lengths), atol=atol, rtol=rtol)
    short = [max(1, n // 3) for n in lens.tolist()]  # a context shorter than its chunk: rows that see no key
    seen = torch.tensor([max(0, n - (c - 1 - i)) for n, c in zip(short, chunks) for i in range(c)], dtype=torch.int32)
    out = run_prefill(q, kp, vp, tables, torch.tensor(short, dtype=torch.int32), cu, chunks)
    torch.testing.assert_close(out, paged_attention_cpu(q, kp, vp, row_tables, seen), atol=atol, rtol=rtol)


@pytest.mark.parametrize(
    "hq,prefixes,chunks,cut",
    [
        (8, [1217], [16], True),  # 20 key tiles, room for 3 segments and more
        (8, [1200], [16], False),  # 19
        (8, [1217, 1000], [16, 40], True),  # the longest sequence decides for the others
        (16, [1700, 10], [129, 300], True),  # 29 tiles; five query tiles, room for 3
        (16, [1292], [700], True),  # 32 tiles, halves: six query tiles of 16 heads
        (16, [1284], [700], False),  # 31
        (32, [0, 700, 1300], [300, 300, 300], False),  # nine query tiles of 32 heads: 256 items without a cut
        (16, [1600, 1600, 1600], [300, 300, 300], False),  # nine of 16 heads: halves would be 288 items
        (16, [170, 512, 853, 1194, 1536, 1877], [143, 304, 89, 196, 35, 250], True),  # 11, of which 5 are cut: 256
    ],
)
def test_keys_are_cut_where_the_merge_pays(hq, prefixes, chunks, cut):
    from vllm_rlt_amd import ops

    q, kp, vp, tables, lens, cu, row_tables, row_lengths = ragged_prefill_case(
        torch.bfloat16, hq, 8, 128, prefixes, chunks, 41
    )
    args = [t.cuda() for t in (q, kp, vp, tables, lens, cu)]
    out = ops.paged_prefill(*args, max(chunks))
    spare = torch.empty(1, dtype=torch.uint8, device="cuda")
    plain = ops.paged_prefill(*args, max(chunks), workspace=spare)  # a given workspace: never cut
    # A cut rounds P against a segment's own maximum, so the two differ in last bits.
    assert torch.equal(out, plain) != cut
    some = torch.randperm(len(q), generator=torch.Generator().manual_seed(1))[:60]
    atol, rtol = TOL[torch.bfloat16]
    expect = paged_attention_cpu(q[some], kp, vp, row_tables[some], row_lengths[some])
    torch.testing.assert_close(out.cpu()[some], expect, atol=atol, rtol=rtol)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_batch_invariant_rows_keep_their_bits_in_any_launch(dtype):
    from vllm_rlt_amd import ops
    from vllm_rlt_amd.paged_attention import HipPagedAttention

    prefixes, chunks = [3000, 100, 900, 0], [40, 300, 200, 500]
    q, kp, vp, tables, lens, cu, _, _ = ragged_prefill_case(dtype, 16, 16, 128, prefixes, chunks, 43)
    q, kp, vp, tables, lens, cu = (t.cuda() for t in (q, kp, vp, tables, lens, cu))
    one = torch.tensor([0, chunks[0]], dtype=torch.int32, device="cuda")
    alone = (q[: chunks[0]], kp, vp, tables[:1], lens[:1], one, chunks[0])
    together = (q, kp, vp, tables, lens, cu, max(chunks))
    attention = HipPagedAttention("cuda", dtype, 128, 16, batch_invariant=True)
    for call in (lambda *a: ops.paged_prefill(*a, batch_invariant=True), attention.prefill):
        assert torch.equal(call(*alone), call(*together)[: chunks[0]])
    attention.batch_invariant = False
    for call in (ops.paged_prefill, attention.prefill):  # what it is an option for
        assert not torch.equal(call(*alone), call(*together)[: chunks[0]])
        atol, rtol = TOL[dtype]
        torch.testing.assert_close(call(*alone), call(*together)[: chunks[0]], atol=atol, rtol=rtol)
