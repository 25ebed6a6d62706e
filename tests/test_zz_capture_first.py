"""Operators as the first call of their stream, recorded into a graph: the scratch arena cannot grow then. Scratch that only
makes a call faster (padded copies of ragged operands, partial sums along K, shared key blocks of the attention
gradient) is done without; what a call cannot do without is reported. Every accepted call is replayed three times, with eager
work and a synchronisation in between, and compared with the eager call, which has all the scratch it asks for and so
may add in another order: the one-normalisation bounds of tests/util.py."""
import pytest
import torch

from cgpt_amd import capi, ops
from tests.util import DTYPE_IDS, DTYPES, STOL, assert_scaled_close, randint, randn

pytestmark = pytest.mark.gpu

MIB = 1 << 20


def check_recorded(device, call, outputs, arena=0):
    """`call(stream)` eagerly, then with an arena of `arena` bytes under capture, then replays."""
    stream = torch.cuda.Stream(device=device)
    torch.cuda.synchronize()
    call(stream)
    stream.synchronize()
    want = [t.clone() for t in outputs]
    torch.cuda.synchronize()
    capi.call("cgptx_release_scratch")
    if arena:  # the loss of rows of one logit takes 4 bytes of scratch per row
        rows = arena // 4
        logits, targets = torch.zeros(rows, 1, device=device), torch.zeros(rows, dtype=torch.int32, device=device)
        loss = torch.empty(1, device=device)
        torch.cuda.synchronize()
        ops.cross_entropy_forward(loss, logits, targets, rows, stream)
        stream.synchronize()
    assert capi.lib().cgptx_scratch_bytes(stream.cuda_stream) == arena
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
        call(stream)
    for replay in range(3):
        for t in outputs:
            t.fill_(7.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        for i, (t, w) in enumerate(zip(outputs, want)):
            assert_scaled_close(t, w, STOL[t.dtype], f"output {i} of replay {replay}")


LINEAR_SHAPES = [  # [rows, in, out]
    (1, 5, 3),           # nothing is a whole 16-byte chunk
    (33, 50, 70),
    (130, 1000, 72),     # K no multiple of a K tile
    (2000, 1025, 300),   # long ragged K
    (300, 768, 3000),    # whole chunks, the input gradient split along K
    (64, 8192, 64),      # whole chunks, K of one tile split
]


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("shape", LINEAR_SHAPES, ids=str)
@pytest.mark.parametrize("arena", [0, MIB], ids=["none", "1MiB"])
def test_linear(device, dtype, shape, arena):
    rows, k, n = shape
    x, w, dy = (t.to(device) for t in (randn((rows, k), dtype, 1), randn((n, k), dtype, 2, 0.05), randn((rows, n), dtype, 3)))
    y, dx, dw = torch.empty_like(dy), torch.empty_like(x), torch.empty_like(w)
    if shape != (64, 8192, 64) or dtype == torch.float32:
        check_recorded(device, lambda s: ops.linear_forward(y, x, w, stream=s), [y], arena)
    if shape != (300, 768, 3000) or dtype == torch.float32 or arena:
        check_recorded(device, lambda s: ops.linear_backward(dx, None, None, dy, x, w, stream=s), [dx], arena)
    check_recorded(device, lambda s: ops.linear_backward(None, dw, None, dy, x, w, stream=s), [dw], arena)
    if dtype == torch.float32 or n % 8 != 0:
        check_recorded(device, lambda s: ops.linear_backward(dx, dw, None, dy, x, w, stream=s), [dx, dw], arena)


@pytest.mark.parametrize("dtype", DTYPES[1:], ids=DTYPE_IDS[1:])
def test_weight_gradient_of_a_long_batch_insists_on_its_scratch(device, dtype):
    """One 128 x 128 tile and 8192 rows: unsplit it would run on one compute unit, at every replay."""
    dy, x = (torch.ones(8192, 128, dtype=dtype, device=device) for _ in range(2))
    w, dw = torch.ones(128, 128, dtype=dtype, device=device), torch.empty(128, 128, dtype=dtype, device=device)
    stream = torch.cuda.Stream(device=device)
    torch.cuda.synchronize()
    capi.call("cgptx_release_scratch")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
        with pytest.raises(capi.CgptxCaptureError):
            ops.linear_backward(None, dw, None, dy, x, w, stream=stream)


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("with_lse", [True, False])
@pytest.mark.parametrize("arena", [4, 8, 12])
def test_attention_gradient(device, dtype, with_lse, arena):
    """One sequence of 512: the key blocks are shared between workgroups, whose partial sums the smaller arenas have no or
    not all the room for."""
    c = dict(num_query_heads=8, num_kv_heads=2, head_dim=128)
    q, do = randn((1, 512, 8, 128), dtype, 1).to(device), randn((1, 512, 8, 128), dtype, 2).to(device)
    k, v = randn((1, 512, 2, 128), dtype, 3).to(device), randn((1, 512, 2, 128), dtype, 4).to(device)
    out, lse = torch.empty_like(q), torch.empty((1, 512, 8), device=device)
    options = ops.FlashAttentionOptions(**c)
    ops.flash_gqa_attention_forward_with_lse(out, lse, q, k, v, None, options)
    torch.cuda.synchronize()
    grads = [torch.empty_like(t) for t in (q, k, v)]
    if with_lse:
        check_recorded(device, lambda s: ops.flash_gqa_attention_backward_with_lse(*grads, do, out, lse, q, k, v, s, options), grads, arena * MIB)
    else:
        check_recorded(device, lambda s: ops.flash_gqa_attention_backward(*grads, do, q, k, v, s, options), grads, arena * MIB)


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
def test_cut_cross_entropy(device, dtype):
    """[2000, 256] x [521, 256]: the logits fit the arena, the room to split the gradients' contractions does not."""
    x, w = randn((2000, 256), dtype, 1).to(device), randn((521, 256), dtype, 2, 0.05).to(device)
    targets = randint(521, (2000,), 3).to(device)
    loss, dx, dw = torch.empty(1, device=device), torch.empty_like(x), torch.empty_like(w)
    arena = 4 if dtype == torch.float32 else 2  # 2000 rows of 521 logits take 4.0 or 2.0 MiB, padded 4.15 or 2.08
    for room in (arena, arena + 1):
        check_recorded(device, lambda s: ops.cut_cross_entropy_forward_backward(loss, dx, dw, x, w, targets, 2000, s), [loss, dx, dw], room * MIB)


def test_a_recorded_call_keeps_its_scratch(device):
    """A caller's graph, whose kernels work in the arena as it was: a later call that makes the arena grow leaves that block where it
    is, replays give what they gave, and cgptx_release_scratch gives all of it back."""
    stream = torch.cuda.Stream(device=device)
    rows = 2 << 20  # 4 bytes of scratch per row
    logits, targets = torch.randn(2 * rows, 2, device=device), torch.zeros(2 * rows, dtype=torch.int32, device=device)
    loss = torch.empty(1, device=device)

    def call(count):
        ops.cross_entropy_forward(loss, logits[:count], targets[:count], count, stream)

    free = []
    for _ in range(20):
        torch.cuda.synchronize()
        capi.call("cgptx_release_scratch")
        free.append(torch.cuda.mem_get_info()[0])
        call(rows)
        stream.synchronize()
        want = loss.clone()
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
            call(rows)
        for _ in range(3):
            call(2 * rows)
            stream.synchronize()
            assert capi.lib().cgptx_scratch_bytes(stream.cuda_stream) == 8 * rows
            loss.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(loss, want)
        del graph
    assert free[1] - free[-1] <= 18 * 4 * rows // 2  # the smaller blocks, kept in every round, would be twice that
