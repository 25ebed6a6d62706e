"""GPU parity tests: embedding gather/scatter (bit-exact), dense cross-entropy, AdamW."""
import math

import numpy as np
import pytest
import torch

from cgpt_amd import ops
from oracle import cpu_ops, oracle64
from tests.util import DTYPES, DTYPE_IDS, TOL, assert_close, launches, randint, randn, to_np

pytestmark = pytest.mark.gpu


def dev(t, device):
    return t.to(device).contiguous()


# ---------------------------------------------------------------------- Embedding
@pytest.mark.parametrize("dtype,tol", [(torch.float16, 1e-2), (torch.bfloat16, 5e-2), (torch.float32, 1e-6)])
def test_embedding_backward_repeated_tokens_known_answer(device, dtype, tol):
    """tests/embedding_test.cu:183-203."""
    dy = torch.tensor([1, 2, 3, 4, 0.5, 1.5, -1, 2, 7, 8, 9, 10.0]).reshape(3, 4).to(dtype)
    ids = torch.tensor([1, 1, 2], dtype=torch.int32)
    gw = torch.full((3, 4), 5.0, dtype=dtype, device=device)
    ops.embedding_backward(gw, dev(dy, device), dev(ids, device), 3)
    assert np.abs(to_np(gw).reshape(-1) - [0, 0, 0, 0, 1.5, 3.5, 2, 6, 7, 8, 9, 10]).max() <= tol


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("tokens,vocab,hidden,accumulate", [
    (64, 7, 16, False), (64, 7, 16, True), (1000, 50, 24, True), (4096, 1000, 128, False), (300, 5, 7, True),
    (1, 3, 8, False), (4097, 900, 40, True), (6000, 50, 24, False),
])
def test_embedding_backward_bit_exact(device, tokens, vocab, hidden, accumulate, dtype):
    """Heavy id collisions, out-of-range ids, odd widths: which rows receive which tokens is integer work
    and the per-add rounding follows the CPU operator, so the whole table is compared bit for bit."""
    ids = randint(vocab + 2, (tokens,), 3)  # ids vocab and vocab+1 are out of range and must be skipped
    dy = randn((tokens, hidden), dtype, 4)
    gw = randn((vocab, hidden), dtype, 5)
    dgw = dev(gw, device).clone()
    cpu_ops.embedding_backward(gw, dy, ids, True, accumulate)
    ops.embedding_backward(dgw, dev(dy, device), dev(ids, device), tokens, None,
                           ops.EmbeddingBackwardOptions(accumulate_weight=accumulate))
    assert torch.equal(dgw.cpu(), gw)


def test_embedding_backward_all_tokens_same_id(device):
    dtype = torch.bfloat16
    ids = torch.full((5000,), 3, dtype=torch.int32)
    dy = randn((5000, 64), dtype, 6)
    gw = torch.zeros(8, 64, dtype=dtype)
    dgw = torch.ones(8, 64, dtype=dtype, device=device)
    cpu_ops.embedding_backward(gw, dy, ids)
    ops.embedding_backward(dgw, dev(dy, device), dev(ids, device), 5000)
    assert torch.equal(dgw.cpu(), gw)


def test_embedding_backward_training_shape_bit_exact_and_deterministic(device):
    """32768 tokens into a [32000, 1024] bf16 table that already holds the lm_head gradient (tied weights)."""
    dtype = torch.bfloat16
    ids = randint(32000, (32768,), 7)
    dy = randn((32768, 1024), dtype, 8)
    base = randn((32000, 1024), dtype, 9)
    want = base.clone()
    cpu_ops.embedding_backward(want, dy, ids, True, True)
    d_ids, d_dy = dev(ids, device), dev(dy, device)
    results = []
    for _ in range(2):
        got = dev(base, device).clone()
        ops.embedding_backward(got, d_dy, d_ids, 32768, None, ops.EmbeddingBackwardOptions(accumulate_weight=True))
        results.append(got.cpu())
    assert torch.equal(results[0], results[1])
    assert torch.equal(results[0], want)
    # integer side: exactly the rows named by the ids changed
    changed = (results[0] != base).any(dim=1).nonzero().flatten().tolist()
    assert set(changed) <= set(ids.tolist())


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
def test_embedding_forward_bit_exact(device, dtype):
    for vocab, hidden, tokens in ((11, 24, 40), (100, 1024, 256), (7, 5, 9)):
        w = randn((vocab, hidden), dtype, 10)
        ids = randint(vocab + 1, (tokens,), 11)
        out = torch.empty(tokens, hidden, dtype=dtype)
        cpu_ops.embedding_forward(out, ids, w)
        dout = torch.full((tokens, hidden), 9.0, dtype=dtype, device=device)
        ops.embedding_forward(dout, dev(ids, device), tokens, dev(w, device))
        assert torch.equal(dout.cpu(), out)


def test_embedding_argument_errors(device):
    gw = torch.zeros(3, 4, device=device)
    dy = torch.zeros(2, 4, device=device)
    ids = torch.zeros(2, dtype=torch.int32, device=device)
    with pytest.raises(ValueError):
        ops.embedding_backward(gw, dy, ids, 3)
    with pytest.raises(ValueError):
        ops.embedding_backward(gw, dy.half(), ids, 2)
    with pytest.raises(ValueError):
        ops.embedding_backward(gw, dy, ids, 0)


# ------------------------------------------------------------------ Cross entropy
def test_cross_entropy_known_answers(device):
    """tests/cross_entropy_test.cu:33-56."""
    logits = torch.tensor([1, 2, 3, 1, 1, 1.0]).reshape(2, 3).to(device)
    targets = torch.tensor([2, 0], dtype=torch.int32, device=device)
    loss, grad = torch.zeros(1, device=device), torch.zeros(2, 3, device=device)
    ops.cross_entropy_forward_backward(loss, grad, logits, targets, 2)
    want = (math.log(math.exp(1) + math.exp(2) + math.exp(3)) - 3 + math.log(3)) / 2
    assert abs(loss.item() - want) <= 1e-5
    assert np.abs(to_np(grad).reshape(-1) -
                  [0.0450153, 0.1223642, -0.1673795, -0.3333333, 0.1666667, 0.1666667]).max() <= 1e-5
    only = torch.zeros(1, device=device)
    ops.cross_entropy_forward(only, logits, targets, 2)
    assert abs(only.item() - want) <= 1e-5
    loss, grad = torch.zeros(1, device=device), torch.zeros(1, 2, device=device)
    ops.cross_entropy_forward_backward(loss, grad, torch.zeros(1, 2, device=device),
                                       torch.tensor([0], dtype=torch.int32, device=device), 1, None, 1024.0)
    assert abs(loss.item() - math.log(2)) <= 1e-6
    assert grad.reshape(-1).tolist() == [-512.0, 512.0]
    with pytest.raises(ValueError):  # target count does not match the rows (tests/cross_entropy_test.cu:58-63)
        ops.cross_entropy_forward_backward(loss, torch.zeros(2, 3, device=device), torch.zeros(2, 3, device=device),
                                           targets, 1)


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("rows,vocab", [(5, 11), (64, 1000), (7, 32000), (3, 50257), (16, 8), (2, 50264), (2, 65544)])
def test_cross_entropy_parity(device, rows, vocab, dtype):
    # Rows of up to 16384 vectors stay in registers, wherever they start: 2, 8 or 16 vectors per thread of 512, 16 of 1024 (fp32
    # 50257 .. 65536). Longer ones stream (fp32 65544). The edges of each: test_gpu_kernel_boundaries.py.
    logits = randn((rows, vocab), dtype, 12, 3.0)
    targets = randint(vocab, (rows,), 13)
    targets[0] = vocab + 5  # out of range: no loss, gradient stays the softmax
    loss, grad = torch.empty(1), torch.empty_like(logits)
    cpu_ops.cross_entropy_forward_backward(loss, grad, logits, targets, 1024.0)
    dloss, dgrad = torch.zeros(1, device=device), torch.empty_like(logits, device=device)
    ops.cross_entropy_forward_backward(dloss, dgrad, dev(logits, device), dev(targets, device), rows, None, 1024.0)
    l64, g64 = oracle64.cross_entropy(to_np(logits), targets.numpy(), 1024.0)
    assert abs(dloss.item() - l64) <= 1e-4 * max(1.0, abs(l64))
    assert abs(dloss.item() - loss.item()) <= 1e-4 * max(1.0, abs(l64))
    assert_close(dgrad, grad, TOL[dtype], "grad vs float32 checker")
    assert_close(dgrad, g64, TOL[dtype], "grad vs float64")
    only = torch.zeros(1, device=device)
    ops.cross_entropy_forward(only, dev(logits, device), dev(targets, device), rows)
    assert abs(only.item() - l64) <= 1e-4 * max(1.0, abs(l64))


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
def test_cross_entropy_rows_that_start_off_a_16_byte_boundary(device, dtype):
    """A vocabulary that is not a multiple of the vector width: every row starts at another offset from a 16-byte
    boundary. In place (gradient = logits), and with a gradient whose rows have a different offset than the logits'."""
    rows, vocab = 9, 50257
    logits = randn((rows, vocab), dtype, 21, 3.0)
    targets = randint(vocab, (rows,), 22)
    l64, g64 = oracle64.cross_entropy(to_np(logits), targets.numpy(), 8.0)
    d_targets = dev(targets, device)
    in_place, loss = dev(logits, device).clone(), torch.zeros(1, device=device)
    ops.cross_entropy_forward_backward(loss, in_place, in_place, d_targets, rows, None, 8.0)
    assert abs(loss.item() - l64) <= 1e-4 * max(1.0, abs(l64))
    assert_close(in_place, g64, TOL[dtype], "in place")
    storage = torch.empty(rows * vocab + 1, dtype=dtype, device=device)
    shifted = storage[1:].view(rows, vocab)  # one element off the logits' alignment
    ops.cross_entropy_forward_backward(loss, shifted, dev(logits, device), d_targets, rows, None, 8.0)
    assert_close(shifted, g64, TOL[dtype], "gradient rows at another offset")


def test_cross_entropy_training_shape_rows_sum_to_zero(device):
    """[8192, 32000] bf16 (a quarter of the training rows; 524 MB): every gradient row sums to ~0, the target
    entry is the only negative one, the loss equals the float64 value on a row sample, twice identical."""
    dtype = torch.bfloat16
    rows, vocab = 8192, 32000
    logits = randn((rows, vocab), dtype, 14, 2.0)
    targets = randint(vocab, (rows,), 15)
    dl, dt = dev(logits, device), dev(targets, device)
    runs = []
    for _ in range(2):
        loss, grad = torch.zeros(1, device=device), torch.empty_like(dl)
        ops.cross_entropy_forward_backward(loss, grad, dl, dt, rows, None, 1024.0)
        runs.append((loss.item(), grad))
    assert runs[0][0] == runs[1][0] and torch.equal(runs[0][1], runs[1][1])
    grad = runs[0][1].float()
    assert grad.sum(dim=1).abs().max().item() <= 2e-2 * 1024.0 / rows * 40
    negatives = (grad < 0).sum(dim=1)
    assert torch.all(negatives == 1)
    assert torch.equal((grad < 0).float().argmax(dim=1).int().cpu(), targets)
    sample = slice(0, 64)
    l64, g64 = oracle64.cross_entropy(to_np(logits[sample]), targets[sample].numpy(), 1024.0 * 64 / rows)
    assert_close(runs[0][1][sample], g64, TOL[dtype], "grad rows vs float64")
    full = torch.empty(1)
    cpu_ops.cross_entropy_forward(full, logits, targets)
    assert abs(runs[0][0] - full.item()) <= 1e-4 * full.item()


# -------------------------------------------------------------------------- AdamW
@pytest.mark.parametrize("dtype,tol", [(torch.float32, 2e-6), (torch.float16, 2e-3), (torch.bfloat16, 1e-2)])
def test_adamw_step_known_answers(device, dtype, tol):
    """tests/adamw_test.cu:21-57."""
    p = torch.tensor([1.0, -2.0]).to(dtype).to(device)
    g = torch.tensor([0.1, -0.2]).to(dtype).to(device)
    state = ops.AdamWState.for_parameter(p)
    options = ops.AdamWOptions(learning_rate=0.1, beta1=0.9, beta2=0.999, epsilon=1e-8, weight_decay=0.01)
    assert ops.adamw_step(p, g, state, options)
    assert np.abs(to_np(p) - [0.899, -1.898]).max() <= tol
    assert np.abs(to_np(state.first_moment) - [0.01, -0.02]).max() <= tol
    assert np.abs(to_np(state.second_moment) - [0.00001, 0.00004]).max() <= tol
    assert state.step == 1
    assert ops.adamw_step(p, g, state, options)
    assert np.abs(to_np(p) - [0.798101, -1.796102]).max() <= tol
    assert state.step == 2

    p = torch.tensor([1.0, -1.0]).to(dtype).to(device)
    g = torch.tensor([8.0, 0.0]).to(dtype).to(device)
    state = ops.AdamWState.for_parameter(p)
    options = ops.AdamWOptions(learning_rate=0.1, weight_decay=0.0, loss_scale=4.0, max_grad_norm=1.0)
    assert ops.adamw_step(p, g, state, options)
    assert np.abs(to_np(p) - [0.9, -1.0]).max() <= tol
    assert np.abs(to_np(state.master_parameter) - [0.9, -1.0]).max() <= 2e-6
    before = p.clone()
    g = torch.tensor([float("inf"), 0.0]).to(dtype).to(device)
    assert not ops.adamw_step(p, g, state, options)
    assert torch.equal(p, before) and state.step == 1


def test_adamw_validation(device):
    p = torch.zeros(1, device=device)
    state = ops.AdamWState.for_parameter(p)
    with pytest.raises(ValueError):
        ops.adamw_step(p, torch.zeros(2, device=device), state)
    with pytest.raises(ValueError):
        ops.adamw_step(p, torch.zeros(1, device=device), state, ops.AdamWOptions(beta2=1.0))


def test_adamw_batched_non_finite_gradient(device):
    """tests/adamw_test.cu:70-91."""
    p = torch.tensor([1.0, -1.0], device=device)
    g = torch.tensor([1.0, 0.0], device=device)
    state = ops.AdamWState.for_parameter(p)
    ws = ops.AdamWWorkspace()
    entry = [ops.AdamWBatchEntry(p, g, state)]
    ops.adamw_step_many_async(entry, ops.AdamWOptions(learning_rate=0.1, weight_decay=0.0), ws)
    assert ops.adamw_check(ws)
    assert np.abs(to_np(p) - [0.9, -1.0]).max() <= 1e-6 and state.step == 1
    g.copy_(torch.tensor([float("inf"), 0.0]))
    ops.adamw_step_many_async(entry, ops.AdamWOptions(), ws)
    assert not ops.adamw_check(ws)
    assert np.abs(to_np(p) - [0.9, -1.0]).max() <= 1e-6 and state.step == 1
    # the sticky flag was cleared by the check; a finite step goes through again
    g.copy_(torch.tensor([1.0, 0.0]))
    ops.adamw_step_many_async(entry, ops.AdamWOptions(learning_rate=0.1, weight_decay=0.0), ws)
    assert ops.adamw_check(ws) and state.step == 2
    with pytest.raises(ValueError):  # the workspace is bound to its first entry list
        ops.adamw_step_many_async(entry + entry, ops.AdamWOptions(), ws)


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
def test_adamw_many_parity_three_steps(device, dtype):
    """Ragged tensor sizes (1 .. 70001 elements, crossing the 4096-element chunking), global-norm clipping,
    loss scale 1024, three steps, against the float64 statement of src/optim/adamw.cu:148-187."""
    sizes = [1, 7, 4096, 4097, 70001, 513, 8192]
    params = [randn((n,), dtype, 100 + i, 0.5) for i, n in enumerate(sizes)]
    d_params = [dev(p, device).clone() for p in params]
    states = [ops.AdamWState.for_parameter(p) for p in d_params]
    d_grads = [torch.empty_like(p) for p in d_params]
    entries = [ops.AdamWBatchEntry(p, g, s) for p, g, s in zip(d_params, d_grads, states)]
    ws = ops.AdamWWorkspace()
    options = ops.AdamWOptions(learning_rate=3e-4, beta1=0.9, beta2=0.95, epsilon=1e-8, weight_decay=0.1,
                               loss_scale=1024.0, max_grad_norm=1.0)
    masters = [to_np(p) for p in params]
    ms = [np.zeros(n) for n in sizes]
    vs = [np.zeros(n) for n in sizes]
    step = 0
    for it in range(3):
        grads = [randn((n,), dtype, 200 + 10 * it + i, 1024.0 * 0.01) for i, n in enumerate(sizes)]
        for dg, g in zip(d_grads, grads):
            dg.copy_(g)
        ops.adamw_step_many_async(entries, options, ws)
        ok, masters, ms, vs, step = oracle64.adamw(None, [to_np(g) for g in grads], masters, ms, vs, step, 3e-4, 0.9,
                                                   0.95, 1e-8, 0.1, 1024.0, 1.0)
        assert ok
    assert ops.adamw_check(ws) and states[0].step == 3 == step
    for p, s, m64, mm, vv in zip(d_params, states, masters, ms, vs):
        assert_close(s.master_parameter, m64, 1e-5, "master")
        assert_close(s.first_moment, mm, 1e-5, "m")
        assert np.abs(to_np(s.second_moment) - vv).max() <= 1e-5 * max(1e-12, np.abs(vv).max()) + 1e-12
        assert_close(p, m64, TOL[dtype], "param")
        assert torch.equal(p, s.master_parameter.to(dtype))


@pytest.mark.parametrize("sizes", [
    [4096 * (i % 3) + i for i in range(1, 65)], [4096 * (i % 2) + 7 * i for i in range(1, 66)],  # one and two starts a lane
    [1 + 37 * i % 5000 for i in range(256)], [1 + 37 * i % 5000 for i in range(257)],            # the most that are read at once, and one more
    [3, 2045 * 4096, 4096], [3, 2046 * 4096, 4097, 5],                                           # 2047 chunks, one a block, and 2050, four
], ids=["64", "65", "256", "257", "one-chunk", "four-chunks"])
def test_adamw_finds_every_chunk(device, sizes):
    """One clipped step over many tensors, and over as many chunks as the statistics pass changes its blocks at, against float64:
    a chunk that is taken for another tensor's or left out moves the norm and its elements."""
    params = [randn((n,), torch.float32, 500 + i, 0.5) for i, n in enumerate(sizes)]
    grads = [randn((n,), torch.float32, 900 + i, 1.0 + i % 7) for i, n in enumerate(sizes)]
    d_params = [dev(p, device).clone() for p in params]
    states = [ops.AdamWState.for_parameter(p) for p in d_params]
    entries = [ops.AdamWBatchEntry(p, dev(g, device), s) for p, g, s in zip(d_params, grads, states)]
    ws = ops.AdamWWorkspace()
    ops.adamw_step_many_async(entries, ops.AdamWOptions(learning_rate=3e-4, beta1=0.9, beta2=0.95, epsilon=1e-8, weight_decay=0.1,
                                                        loss_scale=2.0, max_grad_norm=1.0), ws)
    ok, masters, ms, vs, step = oracle64.adamw(None, [to_np(g) for g in grads], [to_np(p) for p in params], [np.zeros(n) for n in sizes],
                                               [np.zeros(n) for n in sizes], 0, 3e-4, 0.9, 0.95, 1e-8, 0.1, 2.0, 1.0)
    assert ok and ops.adamw_check(ws)
    for s, m64, mm in zip(states, masters, ms):
        assert_close(s.master_parameter, m64, 1e-5, "master")
        assert np.abs(to_np(s.first_moment) - mm).max() <= 1e-5 * max(1e-12, np.abs(mm).max())


def test_adamw_matches_cpu_restatement_single_tensor(device):
    n = 10007
    p, g = randn((n,), torch.float32, 300), randn((n,), torch.float32, 301, 5.0)
    dp, dg = dev(p, device).clone(), dev(g, device)
    state = ops.AdamWState.for_parameter(dp)
    master, m, v = p.clone(), torch.zeros(n), torch.zeros(n)
    options = ops.AdamWOptions(learning_rate=1e-2, beta2=0.95, weight_decay=0.1, loss_scale=2.0, max_grad_norm=1.0)
    for step in (1, 2):
        assert cpu_ops.adamw(p, g, master, m, v, step, 1e-2, 0.9, 0.95, 1e-8, 0.1, 2.0, 1.0)
        assert ops.adamw_step(dp, dg, state, options)
    assert_close(dp, p, 1e-6, "param")
    assert_close(state.first_moment, m, 1e-6, "m")
    assert_close(state.second_moment, v, 1e-6, "v")


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("tokens,hidden,frequent", [
    (64, 64, 64), (65, 64, 65),            # the longest segment of one wavefront, the shortest of a workgroup
    (300, 72, 129), (300, 33, 130),        # one row past a batch of 128; a partial and an unaligned slice of columns
    (200, 64, 97), (200, 40, 159), (200, 31, 71),  # past the batches of 96 and 64 rows, and up to one row short of 160
    (4200, 128, 4097), (9000, 96, 8000),     # more tokens than are ordered at a time
])
def test_embedding_backward_frequent_ids_bit_exact(device, tokens, hidden, frequent, dtype):
    """Ids that take a large share of the batch, between other ids and ids past the vocabulary."""
    vocab = 50
    g = torch.Generator().manual_seed(tokens + hidden)
    ids = torch.randint(0, vocab + 3, (tokens,), generator=g)
    where = torch.randperm(tokens, generator=g)[:frequent]
    ids[where] = torch.where(torch.arange(frequent) % 3 == 0, 7, 8) if frequent > 1000 else 7
    dy = randn((tokens, hidden), dtype, 3)
    for accumulate in (False, True):
        want = randn((vocab, hidden), dtype, 4)
        got = want.to(device)
        # Additions in token order, each rounded to the storage type; ids past the vocabulary are skipped.
        base = want.clone() if accumulate else torch.zeros_like(want)
        for i in range(tokens):
            if ids[i] < vocab:
                base[ids[i]] = (base[ids[i]].float() + dy[i].float()).to(dtype)
        ops.embedding_backward(got, dy.to(device), ids.to(torch.int32).to(device), tokens,
                               options=ops.EmbeddingBackwardOptions(accumulate_weight=accumulate))
        assert torch.equal(got.cpu(), base)


def test_adamw_entry_list_longer_than_it_says(device):
    """The entries are written into an array of len(entries): a list with more in it than that (here one that lies, in earnest
    one that another thread extends) is refused and nothing is written behind the array."""
    class Short(list):
        def __len__(self):
            return 1

    p, g = torch.ones(4, device=device), torch.ones(4, device=device)
    entry = ops.AdamWBatchEntry(p, g, ops.AdamWState.for_parameter(p))
    with pytest.raises(IndexError):
        ops.adamw_step_many_async(Short([entry, entry]), ops.AdamWOptions(), ops.AdamWWorkspace())


def _added_in_token_order(ids, dy, table, accumulate):
    """Row by row what the scatter promises: additions in token order, each rounded to the storage type."""
    out = table.clone() if accumulate else torch.zeros_like(table)
    order = torch.sort(ids, stable=True).indices
    ids_sorted, rows = ids[order], dy[order].float()
    starts = torch.cat([torch.zeros(1, dtype=torch.long), (ids_sorted[1:] != ids_sorted[:-1]).nonzero().flatten() + 1, torch.tensor([len(ids)])])
    lengths, first = starts[1:] - starts[:-1], starts[:-1]
    segment_ids = ids_sorted[first]
    keep = segment_ids < len(table)
    lengths, first, segment_ids = lengths[keep], first[keep], segment_ids[keep]
    acc = out[segment_ids].float()
    for k in range(int(lengths.max())):  # the k-th token of every segment that has one
        live = lengths > k
        acc[live] = (acc[live] + rows[first[live] + k]).to(dy.dtype).float()
    out[segment_ids] = acc.to(dy.dtype)
    return out


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("tokens,vocab,hidden,frequent", [
    (5000, 4096, 8, {}), (5000, 4097, 8, {}), (5000, 4098, 7, {}),  # one id per wavefront, two, and an odd number of them
    (5000, 4099, 8, {4098: 70, 2048: 66, 2049: 65, 0: 80}),          # long and short ids in one wavefront
    (16384, 3000, 8, {2999: 100}), (16448, 3000, 8, {2999: 100}),    # 256 positions to look at for long ids, and one more
    (20000, 3000, 9, {5: 90, 1024: 65, 2999: 300}),                   # some in every workgroup of the grouping
    (20000, 3000, 8, {1500: 300}),                                    # in the middle one only
    (70000, 9, 8, {4: 20000, 7: 9000}),                               # two windows of positions, several lists in each
    (66000, 5000, 7, {17: 8192, 18: 4096}),                           # whole lists
])
def test_embedding_backward_splits_bit_exact(device, tokens, vocab, hidden, frequent, dtype):
    """Where the grouping's marks, the row kernel's wavefronts and the ordering of long segments change over."""
    g = torch.Generator().manual_seed(tokens + vocab)
    ids = torch.randint(0, vocab + 2, (tokens,), generator=g)
    where = torch.randperm(tokens, generator=g)
    for id, count in frequent.items():
        ids[where[:count]] = id
        where = where[count:]
    dy, table = randn((tokens, hidden), dtype, 3), randn((vocab, hidden), dtype, 4)
    d_ids, d_dy = ids.to(torch.int32).to(device), dy.to(device)
    for accumulate in (False, True):
        got = table.to(device)
        ops.embedding_backward(got, d_dy, d_ids, tokens, options=ops.EmbeddingBackwardOptions(accumulate_weight=accumulate))
        assert torch.equal(got.cpu(), _added_in_token_order(ids, dy, table, accumulate))


@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("tokens,vocab", [
    (4097, 300),       # ranges of 128 ids, the last one partly filled; one id more than a round of loads
    (40707, 120),      # one range: wavefronts whose list holds all of their tokens, and one token more
    (45000, 120),      # no wavefront's list holds its tokens
    (33000, 33000),    # ranges of 256 ids
    (140000, 4300000), # ranges of 32768 ids: more tokens than an entry of a list can name
])
def test_embedding_backward_grouping_bit_exact(device, tokens, vocab, offset):
    """The grouping with and without its lists, from an id list that does and does not begin on 16 bytes."""
    g = torch.Generator().manual_seed(tokens + offset)
    ids = torch.randint(0, vocab, (tokens,), generator=g)
    dy, table = randn((tokens, 1), torch.float32, 3), randn((vocab, 1), torch.float32, 4)
    d_ids = torch.zeros(tokens + offset, dtype=torch.int32, device=device)[offset:]
    d_ids.copy_(ids)
    got = table.to(device)
    ops.embedding_backward(got, dy.to(device), d_ids, tokens, options=ops.EmbeddingBackwardOptions(accumulate_weight=False))
    assert torch.equal(got.cpu(), _added_in_token_order(ids, dy, table, False))


def test_embedding_backward_keeps_non_finite_rows_to_their_ids(device):
    """Long segments read past their last token's row into the same row again: nothing of it is added."""
    ids = torch.arange(1000) % 3
    for hidden in (64, 33):
        dy = randn((1000, hidden), torch.float32, 3)
        dy[999] = float("inf")  # id 0
        got = torch.empty(3, hidden, device=device)
        ops.embedding_backward(got, dy.to(device), ids.to(torch.int32).to(device), 1000)
        want = _added_in_token_order(ids, dy, torch.zeros(3, hidden), False)
        assert torch.equal(got.cpu(), want) and torch.isfinite(got[1:]).all() and torch.isinf(got[0]).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32], ids=["bf16", "f32"])
def test_adamw_of_more_state_than_the_memory_cache_gives_the_bits_of_less(device, dtype):
    """22.4 million elements are 256 MiB of fp32 state: beyond them the update accesses it as what is used once. Without clipping
    every element is updated by itself, so one call over all gives what calls over parts give."""
    count = (256 << 20) // 12 + 4096 * 3 + 17
    generator = torch.Generator(device=device).manual_seed(3)
    start = torch.randn(count, device=device, generator=generator).to(dtype)
    grads = [torch.randn(count, device=device, generator=generator).mul_(0.01).to(dtype) for _ in range(2)]
    options = ops.AdamWOptions(learning_rate=3e-4, weight_decay=0.1, max_grad_norm=float("inf"))
    results = []
    for parts in (1, 3):
        edges = [count * i // parts // 64 * 64 for i in range(parts)] + [count]
        parameter, gradient, master = start.clone(), torch.empty_like(start), start.to(torch.float32, copy=True)
        first, second = torch.zeros_like(master), torch.zeros_like(master)
        calls = []
        for a, b in zip(edges, edges[1:]):
            state = ops.AdamWState(master[a:b], first[a:b], second[a:b])
            calls.append(([ops.AdamWBatchEntry(parameter[a:b], gradient[a:b], state)], ops.AdamWWorkspace()))
        for g in grads:
            gradient.copy_(g)
            for entries, workspace in calls:
                ops.adamw_step_many_async(entries, options, workspace)
        results.append((parameter, master, first, second))
    for name, one, three in zip(("parameter", "master", "first", "second"), *results):
        assert torch.equal(one, three), name


@pytest.mark.parametrize("dtype,rows,vocab", [(torch.bfloat16, 1511, 50257), (torch.float32, 2311, 16381), (torch.float16, 19, 8 * 1024 * 1024 // 64 - 3)],
                         ids=["bf16", "f32", "f16"])
def test_cross_entropy_of_more_logits_than_the_memory_cache_gives_the_rows_of_few(device, dtype, rows, vocab):
    """Beyond 288 MiB logits and gradients are accessed as what is used once; a row's gradient is what a call over few rows gives for it
    (the same scale / rows). The last shape is a small one of long rows at odd addresses."""
    generator = torch.Generator(device=device).manual_seed(5)
    logits = torch.randn(rows, vocab, device=device, generator=generator).to(dtype)
    targets = torch.randint(0, vocab, (rows,), device=device, generator=generator, dtype=torch.int32)
    loss, gradient = torch.empty(1, device=device), torch.empty_like(logits)
    ops.cross_entropy_forward_backward(loss, gradient, logits, targets, rows, gradient_scale=float(rows))
    total = 0.0
    for first in range(0, rows, 300):
        part = slice(first, min(first + 300, rows))
        few = part.stop - part.start
        part_loss, part_gradient = torch.empty(1, device=device), torch.empty_like(logits[part])
        ops.cross_entropy_forward_backward(part_loss, part_gradient, logits[part], targets[part].contiguous(), few, gradient_scale=float(few))
        assert torch.equal(gradient[part], part_gradient)
        total += part_loss.item() * few
    assert abs(loss.item() - total / rows) <= 1e-6 * abs(loss.item())
    only = torch.empty(1, device=device)
    ops.cross_entropy_forward(only, logits, targets, rows)
    assert only.item() == loss.item()


@pytest.mark.parametrize("rows", [1, 63, 64, 65, 128, 129, 1023, 1024, 1025, 2049, 4096, 4097, 9001])
def test_mean_loss_counts_every_row_once(device, rows):
    """Rows of equal logits all have the loss that one of them has alone, and rows whose target lies outside the vocabulary have none: their
    sum in 64 bits is exact in any order, so the mean is known to the last bit, at the edges of the tree of 1024 sums that takes it."""
    vocab = 40
    z = torch.full((rows, vocab), 0.5, device=device)
    for seed in range(3):
        keep = randint(2, (rows,), rows + seed) == 1
        y = torch.where(keep, 7, vocab).to(torch.int32).to(device)
        one, loss = torch.empty(1, device=device), torch.empty(1, device=device)
        ops.cross_entropy_forward(one, z[:1], torch.full((1,), 7, dtype=torch.int32, device=device), 1)
        ops.cross_entropy_forward(loss, z, y, rows)
        total = np.float32(float(one.item()) * int(keep.sum()))
        assert loss.item() == total * (np.float32(1.0) / np.float32(rows))


@pytest.mark.parametrize("dtype,vocab", [(torch.bfloat16, 1003), (torch.float32, 9000), (torch.float16, 140000)], ids=["bf16", "f32", "f16"])
@pytest.mark.parametrize("rows", [1, 2, 127, 128, 129])
def test_mean_loss_of_few_rows_comes_from_the_rows_launch(device, dtype, vocab, rows):
    """Up to 128 rows the last workgroup takes the mean (longer rows than the registers hold: a launch of its own). Three calls in a row
    and three replays: the workgroups' counter is left as it was found. The bound is the rounding of a row's loss, 2^-24 of values around
    log V and of the largest logit, in rows and in their mean, and that of the fast exponential and logarithm, a few units each."""
    logits = randn((rows, vocab), dtype, rows + vocab)
    targets = randint(vocab, (rows,), rows)
    wide = logits.double()
    want = (torch.logsumexp(wide, 1) - wide.gather(1, targets.long()[:, None])[:, 0]).mean().item()
    z, y = dev(logits, device), dev(targets, device)
    loss, gradient = torch.empty(1, device=device), torch.empty_like(z)
    for with_gradient in (True, False):
        def call():
            if with_gradient:
                ops.cross_entropy_forward_backward(loss, gradient, z, y, rows)
            else:
                ops.cross_entropy_forward(loss, z, y, rows)
        seen = set()
        for _ in range(3):
            loss.fill_(float("nan"))
            call()
            seen.add(loss.item())
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            call()
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=stream):
                call()
            for _ in range(3):
                loss.fill_(float("nan"))
                graph.replay()
                call()
                seen.add(loss.item())
        assert len(seen) == 1
        assert abs(seen.pop() - want) <= 2e-6 * max(1.0, abs(want))
    long_rows = vocab > 131072 and dtype != torch.float32
    assert launches(lambda: ops.cross_entropy_forward(loss, z, y, rows)) == (1 if rows <= 128 and not long_rows else 2)


@pytest.mark.parametrize("dtype,rows,vocab", [(torch.bfloat16, 3011, 50257), (torch.float16, 1201, 131071), (torch.float32, 4721, 16381)],
                         ids=["bf16", "f16", "f32"])
def test_cross_entropy_without_a_gradient_or_in_place_over_the_memory_cache(device, dtype, rows, vocab):
    """More than 288 MiB of logits alone: the loss without a gradient, and with the gradient in the logits' own place, are those of calls over
    few rows, which access them otherwise."""
    assert rows * vocab * dtype.itemsize > 288 << 20
    generator = torch.Generator(device=device).manual_seed(6)
    logits = torch.randn(rows, vocab, device=device, generator=generator).to(dtype)
    targets = torch.randint(0, vocab, (rows,), device=device, generator=generator, dtype=torch.int32)
    loss, total = torch.empty(1, device=device), 0.0
    want = torch.empty_like(logits)
    for first in range(0, rows, 300):
        part = slice(first, min(first + 300, rows))
        few = part.stop - part.start
        ops.cross_entropy_forward_backward(loss, want[part], logits[part], targets[part].contiguous(), few, gradient_scale=float(few))
        only = torch.empty(1, device=device)
        ops.cross_entropy_forward(only, logits[part], targets[part].contiguous(), few)
        assert only.item() == loss.item()
        total += loss.item() * few
    ops.cross_entropy_forward(loss, logits, targets, rows)
    assert abs(loss.item() - total / rows) <= 1e-6 * abs(loss.item())
    in_place = torch.empty(1, device=device)
    ops.cross_entropy_forward_backward(in_place, logits, logits, targets, rows, gradient_scale=float(rows))
    assert in_place.item() == loss.item()
    assert torch.equal(logits, want)
