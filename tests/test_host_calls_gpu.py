"""The direct host calls take exactly the calls they should, to the same results (GPU).

Forcing the Python path (no host module) and taking the direct one must agree
bit for bit; calls the direct path leaves alone must end as they do without it.
"""

import pytest
import torch

from paged_cases import random_decode_case
from test_decode_gpu import ragged_prefill_case

pytestmark = pytest.mark.gpu


@pytest.fixture
def python_path(monkeypatch):
    """Runs a call through the Python path."""
    from vllm_rlt_amd import ops

    def run(f):
        with monkeypatch.context() as m:
            m.setattr(ops, "_host_calls", lambda t: (None, 0))
            return f()

    return run


def direct(f, module_call):
    """f(), asserting that the direct call took it."""
    from vllm_rlt_amd import _native

    taken = []
    host = _native.host

    class Spy:
        def __getattr__(self, name):
            def call(*args):
                out = getattr(host, name)(*args)
                taken.append((name, out is not None))
                return out

            return call

    _native.host = Spy()
    try:
        out = f()
    finally:
        _native.host = host
    assert (module_call, True) in taken, taken
    return out


def bits(t):
    return t.contiguous().view(torch.uint8)


def decode_args(case):
    last = case.lengths.long() - 1
    rows = torch.arange(len(case.lengths), device="cuda")
    blocks = case.tables[rows, last // 16].long()
    k, v = torch.randn_like(case.key_slice[: len(rows), 0]), torch.randn_like(case.key_slice[: len(rows), 0])
    return k, v, blocks, last % 16


@pytest.mark.parametrize("dtype,hq,hkv,d", [(torch.bfloat16, 16, 16, 128), (torch.float16, 8, 2, 64), (torch.float32, 4, 4, 40)])
@pytest.mark.parametrize("n_write", [None, 2])
def test_decode_append(python_path, dtype, hq, hkv, d, n_write):
    from vllm_rlt_amd import ops
    from vllm_rlt_amd.paged_attention import HipPagedAttention

    case = random_decode_case([1, 33, 300, 700], hq=hq, hkv=hkv, d=d, dtype=dtype, seed=d).to("cuda")
    k, v, blocks, offsets = decode_args(case)
    pools = (case.key_slice.clone(), case.value_slice.clone())

    def run(out=None, workspace=None, scale=None):
        case.key_slice.copy_(pools[0])
        case.value_slice.copy_(pools[1])
        got = ops.paged_decode_append(
            case.q, case.key_slice, case.value_slice, case.tables, case.lengths, k, v, blocks, offsets, n_write=n_write,
            out=out, workspace=workspace, scale=scale,
        )
        return got, case.key_slice.clone(), case.value_slice.clone()

    expect = python_path(run)
    for a, b in zip(direct(run, "decode"), expect):
        assert torch.equal(bits(a), bits(b))  # unused slots hold NaN
    out = torch.empty_like(case.q)
    space = torch.empty(ops.decode_workspace_bytes(4, hq, hkv, d), dtype=torch.uint8, device="cuda")
    assert direct(lambda: run(out, space), "decode")[0] is out
    assert torch.equal(out, expect[0])
    assert torch.equal(direct(lambda: run(scale=0.25), "decode")[0], python_path(lambda: run(scale=0.25))[0])
    plain = lambda: ops.paged_decode(case.q, case.key_slice, case.value_slice, case.tables, case.lengths)  # noqa: E731
    assert torch.equal(direct(plain, "decode"), python_path(plain))
    attention = HipPagedAttention("cuda", dtype, d, 16)
    first = attention(case.q, case.key_slice, case.value_slice, case.tables, case.lengths)  # grows the workspace
    again = lambda: attention(case.q, case.key_slice, case.value_slice, case.tables, case.lengths)  # noqa: E731
    assert torch.equal(direct(again, "decode"), first)


def test_prefill_and_rope(python_path):
    from vllm_rlt_amd import ops

    for dtype, shift in ((torch.bfloat16, 0), (torch.float32, 0), (torch.bfloat16, 1)):
        chunks = [40, 3]
        q, kp, vp, tables, lens, cu, _, _ = ragged_prefill_case(dtype, 8, 8, 128, [100, 0], chunks, 5)
        q = torch.cat([q.flatten(), q.new_zeros(8)]).cuda()[shift:][: q.numel()].view(q.shape)  # off 16 bytes when shifted
        rest = [t.cuda() for t in (kp, vp, tables, lens, cu)]
        run = lambda: ops.paged_prefill(q, *rest, max(chunks))  # noqa: E731
        assert torch.equal(direct(run, "prefill"), python_path(run))
    q, k, v = (torch.randn(5, 4, 64, device="cuda", dtype=torch.bfloat16) for _ in range(3))
    angle = torch.randn(5, 64, device="cuda")
    cos, sin = angle.cos().bfloat16(), angle.sin().bfloat16()
    blocks, offsets = torch.arange(5, device="cuda"), torch.arange(5, device="cuda") * 3
    results = []
    for how in (lambda f: direct(f, "rope"), python_path):
        pools = [torch.zeros(6, 2, 16, 4, 64, device="cuda", dtype=torch.bfloat16) for _ in range(2)]
        out = how(lambda: ops.rope_kv_append(*pools, 1, blocks, offsets, q, k, v, cos, sin, n_rows=4))
        results.append((out, *pools))
    for a, b in zip(*results):
        assert torch.equal(a, b)


def test_calls_left_to_python():
    from vllm_rlt_amd import ops

    case = random_decode_case([20, 40], hq=4, hkv=4, d=128, dtype=torch.bfloat16, seed=1).to("cuda")
    expect = ops.paged_decode(case.q, case.key_slice, case.value_slice, case.tables, case.lengths)

    class Sub(torch.Tensor):
        pass

    sub = case.q.as_subclass(Sub)
    out = ops.paged_decode(sub, case.key_slice, case.value_slice, case.tables, case.lengths)
    assert type(out) is Sub and torch.equal(out.as_subclass(torch.Tensor), expect)
    with pytest.raises(ValueError, match="one entry per row"):
        ops.paged_decode(case.q, case.key_slice, case.value_slice, case.tables[:1], case.lengths)
    with pytest.raises(ValueError, match="int32"):
        ops.paged_decode(case.q, case.key_slice, case.value_slice, case.tables, case.lengths.long())
    with pytest.raises(ValueError, match="ROCm device"):
        ops.paged_decode(case.q, case.key_slice, case.value_slice, case.tables.cpu(), case.lengths)
    with pytest.raises(ValueError, match="out must match"):
        ops.paged_decode(case.q, case.key_slice, case.value_slice, case.tables, case.lengths, out=case.q.float())
    with pytest.raises(ValueError, match="workspace must hold"):
        ops.paged_decode(
            case.q, case.key_slice, case.value_slice, case.tables, case.lengths, workspace=case.q.new_empty(8)
        )
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda q: ops.paged_decode(q, case.key_slice, case.value_slice, case.tables, case.lengths))(
            case.q[None]
        )
    empty = ops.paged_decode(case.q[:0], case.key_slice, case.value_slice, case.tables[:0], case.lengths[:0])
    assert empty.shape == (0, 4, 128)
    # An argument the library refuses: its status becomes its ValueError.
    with pytest.raises(ValueError, match="scale"):
        ops.paged_prefill(
            case.q, case.key_slice, case.value_slice, case.tables[:1], case.lengths[:1],
            torch.tensor([0, 2], dtype=torch.int32, device="cuda"), 2, scale=0.0,
        )


@pytest.mark.parametrize("n_write", [3, 1 << 40, 1 << 63, 1 << 70])
def test_an_append_of_more_rows_than_there_are_is_refused(n_write):
    from vllm_rlt_amd import ops
    from vllm_rlt_amd.paged_attention import HipPagedAttention

    case = random_decode_case([20, 40], hq=4, hkv=4, d=128, dtype=torch.bfloat16, seed=1).to("cuda")
    args = (case.q, case.key_slice, case.value_slice, case.tables, case.lengths, *decode_args(case))
    with pytest.raises(ValueError, match="n_write"):
        ops.paged_decode_append(*args, n_write=n_write)
    attention = HipPagedAttention("cuda", torch.bfloat16, 128, 16)
    attention.reserve_decode(2, 4, 4)
    with pytest.raises(ValueError, match="n_write"):
        attention.decode_append(*args, n_write=n_write)


def test_prefill_on_the_attention_objects_workspace():
    from vllm_rlt_amd.paged_attention import HipPagedAttention

    for dtype, d in ((torch.bfloat16, 128), (torch.float32, 128), (torch.bfloat16, 256)):
        chunks = [40, 3]
        q, kp, vp, tables, lens, cu, _, _ = ragged_prefill_case(dtype, 8, 8, d, [100, 0], chunks, 5)
        args = [t.cuda() for t in (q, kp, vp, tables, lens, cu)]
        attention = HipPagedAttention("cuda", dtype, d, 16)
        first = attention.prefill(*args, max(chunks))  # reserves the workspace, if the path needs one
        if attention.workspace_bytes == 0:
            attention.reserve(1)
        assert torch.equal(direct(lambda: attention.prefill(*args, max(chunks)), "prefill"), first)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_the_attention_object_without_host_calls(python_path, dtype):
    from vllm_rlt_amd.paged_attention import HipPagedAttention

    case = random_decode_case([1, 33, 300, 700], hq=8, hkv=8, d=128, dtype=dtype, seed=3).to("cuda")
    decode = (case.q, case.key_slice, case.value_slice, case.tables, case.lengths)
    append = (*decode, *decode_args(case))
    q, kp, vp, tables, lens, cu, _, _ = ragged_prefill_case(dtype, 8, 8, 128, [100, 0], [40, 3], 5)
    prefill = [t.cuda() for t in (q, kp, vp, tables, lens, cu)]
    attention = HipPagedAttention("cuda", dtype, 128, 16)
    attention.reserve_decode(4, 8, 8)
    for run in (lambda: attention(*decode), lambda: attention.decode_append(*append), lambda: attention.prefill(*prefill, 40)):
        assert torch.equal(python_path(run), run())


def test_side_stream_and_capture():
    from vllm_rlt_amd.paged_attention import HipPagedAttention

    case = random_decode_case([200, 90], hq=16, hkv=16, d=128, dtype=torch.bfloat16, seed=9).to("cuda")
    attention = HipPagedAttention("cuda", torch.bfloat16, 128, 16)
    call = lambda: attention(case.q, case.key_slice, case.value_slice, case.tables, case.lengths)  # noqa: E731
    expect = call()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        out = direct(call, "decode")
    side.synchronize()
    assert torch.equal(out, expect)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = direct(call, "decode")
    for i in range(3):
        case.q.normal_()
        graph.replay()
        assert torch.equal(captured, call())
    # A captured workspace outlives its growth.
    held = attention.workspace_bytes
    attention.reserve(held + 1)
    assert attention.held_bytes == held
