"""GPU tests at the sizes where one kernel, tile, split or unrolling gives way to the next: the first and last sizes of each
range, with the oracle of the operator's own tests."""
import numpy as np
import pytest
import torch

from cgpt_amd import ops
from oracle import cpu_ops, oracle64
from tests.test_gpu_attention import make_inputs, oracle_args, run_backward, run_forward
from tests.util import DTYPE_IDS, DTYPES, STOL, TOL, assert_close, assert_scaled_close, launches, randint, randn, to_np

pytestmark = pytest.mark.gpu

ATTENTION = [
    dict(b=1, qs=64, ks=64, hq=2, hkv=1, d=128),                        # one key tile: blocks of 128 rows
    dict(b=1, qs=65, ks=65, hq=4, hkv=2, d=128),                        # two key tiles of 64 rows, one row in the second block
    dict(b=1, qs=1, ks=129, hq=2, hkv=1, d=64, off=128),                # one query, three key tiles: parts of two and one
    dict(b=2, qs=63, ks=192, hq=2, hkv=2, d=96, causal=False),          # odd number of key tiles, padded columns
    dict(b=1, qs=130, ks=300, hq=2, hkv=1, d=40, off=20, scale=0.2),    # keys that no query sees, 64-wide heads
    dict(b=32, qs=64, ks=65, hq=8, hkv=8, d=128, causal=False),         # 256 blocks of 64 rows: the last call in two parts
    dict(b=33, qs=64, ks=65, hq=8, hkv=8, d=128, causal=False),         # 264: the first one in blocks of 128
    dict(b=64, qs=40, ks=65, hq=8, hkv=2, d=64, causal=False),          # 512 with 64-wide heads
    dict(b=65, qs=40, ks=65, hq=8, hkv=2, d=64, causal=False),
    dict(b=1, qs=390, ks=390, hq=6, hkv=2, d=128),                      # few key blocks: shared between workgroups, ragged end
    dict(b=3, qs=330, ks=330, hq=4, hkv=2, d=64),                       # 6 (batch, kv-head) pairs: shared key blocks, no even share of the XCDs
    dict(b=8, qs=260, ks=300, hq=8, hkv=2, d=128, off=40),              # 16 pairs: two for each XCD
    dict(b=30, qs=130, ks=150, hq=4, hkv=2, d=128, off=20),             # 360 blocks of 64 rows: causal blocks of 128, ragged end
]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("case", range(len(ATTENTION)))
def test_attention_around_the_choice_of_blocks(device, case, dtype):
    """Bounds as in the operator's parity tests; every result twice with the same bits, gradients added to what is there."""
    c = ATTENTION[case]
    q, k, v, do = make_inputs(c, dtype, 700 + 10 * case)
    out, lse = run_forward(device, q, k, v, c)
    want_out, want_lse = oracle64.attention_forward(to_np(q), to_np(k), to_np(v), *oracle_args(c))
    assert_close(out, want_out, TOL[dtype], "O")
    assert_close(lse, want_lse, 1e-3, "LSE")
    want = oracle64.attention_backward(to_np(do), to_np(q), to_np(k), to_np(v), *oracle_args(c))
    got = run_backward(device, do, q, k, v, c)
    base = (randn(q.shape, dtype, 91), randn(k.shape, dtype, 92), randn(v.shape, dtype, 93))
    added = run_backward(device, do, q, k, v, c, accumulate=True, base=base)
    for g, a, w, start, name in zip(got, added, want, base, ("dQ", "dK", "dV")):
        assert_scaled_close(g, w, STOL[dtype], name)
        assert_scaled_close(a, w + to_np(start), STOL[dtype], f"{name} accumulate")
    for g, again in zip(got, run_backward(device, do, q, k, v, c)):
        assert torch.equal(g, again)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("case", range(len(ATTENTION)))
def test_attention_gradients_without_saved_statistics_around_the_choice_of_blocks(device, case, dtype):
    """The launch that makes the statistics itself, in one and in two parts: the bits of the one that is given them."""
    c = ATTENTION[case]
    q, k, v, do = make_inputs(c, dtype, 900 + 10 * case)
    for got, want in zip(run_backward(device, do, q, k, v, c, with_lse=False), run_backward(device, do, q, k, v, c)):
        assert torch.equal(got, want)


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("rows,fin,fout", [
    (1, 4096, 64), (33, 4096, 40), (64, 5024, 96),        # few tiles, long K: 32- and 64-wide tiles in K slices
    (3000, 64, 40), (4999, 136, 72),                      # the same for the weight gradient, K ends inside a K tile
    (257, 2048, 264), (512, 1536, 1536),                  # tiles of 64 and 128 in slices, ragged edges
])
def test_contractions_in_k_slices_are_exact_on_integers(device, rows, fin, fout, dtype):
    """Small integers: every product and partial sum is exact in fp32 (at most 4 x 5024 < 2^24), so the result is the rounded
    exact value whatever the tile and the slices."""
    g = torch.Generator().manual_seed(rows + fin + fout)
    x, w, dy = (torch.randint(-2, 3, shape, generator=g).double() for shape in ((rows, fin), (fout, fin), (rows, fout)))
    on = lambda t: t.to(dtype).to(device)
    y, gi, gw = (torch.full(shape, float("nan"), dtype=dtype, device=device) for shape in ((rows, fout), (rows, fin), (fout, fin)))
    ops.linear_forward(y, on(x), on(w))
    ops.linear_backward(gi, gw, None, on(dy), on(x), on(w))
    for name, got, exact in zip(("Y", "dX", "dW"), (y, gi, gw), (x @ w.T, dy @ w, dy.T @ x)):
        assert torch.equal(got.cpu(), exact.to(dtype)), name


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("rows,fin,fout", [
    (16300, 2048, 760), (16300, 760, 2048),  # Y and dX on 256 x 192 tiles, ragged rows and columns
    (2048, 760, 16304), (2040, 768, 16384),  # dW: both operands as they lie, a K tile half empty
])
def test_contractions_whose_columns_leave_square_tiles_idle_are_exact_on_integers(device, rows, fin, fout, dtype):
    """Some 750 columns are three tiles of 256, which is 192 of them for 256 compute units, or four of 192. Every sum is exact in
    fp32 (at most 4 x 16304 < 2^24), so each result is the rounded exact value, alone and added to what is there."""
    g = torch.Generator(device=device).manual_seed(rows + fin)
    x, w, dy = (torch.randint(-2, 3, shape, generator=g, device=device).float() for shape in ((rows, fin), (fout, fin), (rows, fout)))
    on = lambda t: t.to(dtype)
    y, gi, gw = (torch.full(shape, float("nan"), dtype=dtype, device=device) for shape in ((rows, fout), (rows, fin), (fout, fin)))
    ops.linear_forward(y, on(x), on(w))
    ops.linear_backward(gi, None, None, on(dy), on(x), on(w))
    ops.linear_backward(None, gw, None, on(dy), on(x), on(w))
    exact = (x @ w.T.contiguous(), dy @ w, dy.T.contiguous() @ x)
    for name, got, want in zip(("Y", "dX", "dW"), (y, gi, gw), exact):
        assert torch.equal(got, on(want)), name
    added = ops.LinearBackwardOptions(accumulate_input=True, accumulate_weight=True)
    ops.linear_backward(gi, None, None, on(dy), on(x), on(w), options=added)
    ops.linear_backward(None, gw, None, on(dy), on(x), on(w), options=added)
    for name, got, want in zip(("dX", "dW"), (gi, gw), exact[1:]):
        assert torch.equal(got, on(want + on(want).float())), name


@pytest.mark.parametrize("rows,fin,fout", [(33, 480, 576), (121, 192, 896), (690, 352, 512), (2837, 256, 128), (5399, 608, 640)])
def test_fp32_gradients_of_one_call_are_as_near_to_64_bits_as_one_by_one(device, rows, fin, fout):
    """Whatever shares a launch adds no longer chains in fp32 than the calls by themselves. The error of a sum of random terms,
    taken over a whole gradient, varies by a few per cent from one order of additions to another of the same length (the
    smallest gradient here has 128 elements: 1 / sqrt(2 x 128)); a chain twice as long has 1.4 times the error."""
    g = torch.Generator(device=device).manual_seed(rows)
    x, w, dy = (torch.randn(shape, device=device, generator=g) for shape in ((rows, fin), (fout, fin), (rows, fout)))
    together, alone = ({name: torch.empty(shape, device=device) for name, shape in (("dX", (rows, fin)), ("dW", (fout, fin)), ("db", (fout,)))}
                       for _ in range(2))
    ops.linear_backward(*together.values(), dy, x, w)
    for name in alone:
        ops.linear_backward(*(alone[n] if n == name else None for n in alone), dy, x, w)
    exact = {"dX": dy.double() @ w.double(), "dW": dy.double().T.contiguous() @ x.double(), "db": dy.double().sum(0)}
    for name in ("db",):
        off, before = ((t[name].double() - exact[name]).norm() / exact[name].norm() for t in (together, alone))
        assert off <= 1.25 * before, (name, float(off), float(before))


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("rows,fin,fout", [
    *((12288, k, 4096) for k in (32, 64, 96, 160, 352)),   # 256 x 256 tiles: one K step, whole K tiles, a step more
    *((3500, k, 3496) for k in (32, 96, 128, 320, 352)),   # 128 x 128 tiles, two and more workgroups on a CU, ragged edges
    (2000, 992, 2048), (2000, 1024, 2048), (1990, 1056, 2040),  # one workgroup per CU, more operand tiles in flight
    (2048, 4096 + 32, 4096),                                # both gradients' K an odd number of K steps long as well
])
def test_contractions_whose_last_k_tile_is_half_filled_are_exact_on_integers(device, rows, fin, fout, dtype):
    """As above (products of -1 .. 1, at most 12288 of them): K tiles are two K steps long, and what a load brings in past the
    last step of a row is the next row, which no sum may see."""
    g = torch.Generator(device=device).manual_seed(rows + fin + fout)
    x, w, dy = (torch.randint(-1, 2, shape, generator=g, device=device).float() for shape in ((rows, fin), (fout, fin), (rows, fout)))
    on = lambda t: t.to(dtype)
    y, gi, gw = (torch.full(shape, float("nan"), dtype=dtype, device=device) for shape in ((rows, fout), (rows, fin), (fout, fin)))
    ops.linear_forward(y, on(x), on(w))
    ops.linear_backward(gi, gw, None, on(dy), on(x), on(w))
    for name, got, exact in zip(("Y", "dX", "dW"), (y, gi, gw), (x @ w.T, dy @ w, dy.T.contiguous() @ x)):
        assert torch.equal(got, exact.to(dtype)), name


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("steps", [1026, 1028, 1033])
def test_weight_gradients_are_cut_into_equal_k_slices(device, steps, dtype):
    """A long weight gradient's K steps (32 rows, 16 in fp32) are dealt out to its slices evenly, an odd number each where that
    is what they come to. The cuts are read off the sums: column j of dY holds 2^24 in step 0, 1 in step j and -2^24 in step
    j + 1 (as products). A 1 behind the 2^24 of its own slice is lost, 2^24 + 1 being no float; so is one that is the last of
    a later slice, where it meets the 2^24 alone."""
    rows = steps * (16 if dtype == torch.float32 else 32)
    width = 1024
    dy = torch.zeros(steps, rows // steps, width, dtype=dtype, device=device)
    column = torch.arange(width, device=device)
    dy[0, 0] = 4096
    dy[column + 1, 0, column] = 2.0 ** -12
    dy[column + 2, 0, column] = -4096
    x = torch.full((rows, width), 4096, dtype=dtype, device=device)
    gw = torch.full((width, width), float("nan"), dtype=dtype, device=device)
    ops.linear_backward(None, gw, None, dy.view(rows, width), x, x[:width])
    assert torch.equal(gw, gw[:, :1].expand_as(gw))
    kept = gw[:, 0].cpu()
    assert ((kept == 0) | (kept == 1)).all()
    length = int(kept.nonzero()[0]) + 1  # the first step that is not slice 0's
    slices = -(-steps // length)
    assert slices > 1 and length == -(-steps // slices), (length, slices)
    lost = {j for j in range(1, width + 1) if j < length or (j + 1) % length == 0}
    assert set((kept == 0).nonzero().flatten().add(1).tolist()) == lost


def column_sums_in_order(parts, hidden, units):
    """parts [P, H] in float32, added over P in the order that the column reductions promise."""
    count = len(parts)
    slices = max(1, min(2 * units // -(-hidden // 64), count // 16, 4096 // (16 if hidden <= 256 else 32)))
    if slices > 1:
        chunk = -(-count // slices)
        folded = np.zeros((slices, hidden), np.float32)
        for i in range(slices):
            own = parts[i * chunk:(i + 1) * chunk]
            eighths = np.zeros((8, hidden), np.float32)
            for p, row in enumerate(own):
                eighths[p % 8] += row
            for w in range(4):
                folded[i] += eighths[w] + eighths[w + 4]
        parts, count = folded, slices
    total = np.zeros(hidden, np.float32)
    for w in range(4):
        running = np.zeros((4, hidden), np.float32)
        p = w
        while p + 12 < count:
            for u in range(4):
                running[u] += parts[p + 4 * u]
            p += 16
        for q in range(p, count, 4):
            running[0] += parts[q]
        total += (running[0] + running[1]) + (running[2] + running[3])
    return total


@pytest.mark.parametrize("rows,width", [
    *((rows, width) for rows in (300, 4096, 65536) for width in (1, 16, 20, 256, 300, 1024)),  # 60, 64, 256 parts; 16 or 32 columns
    (4096, 9000), (4096, 16448),                                                               # few slices, one slice
])
def test_column_sums_add_in_their_order(device, rows, width):
    """A bias's gradient in fp32 whose parts are one row each, so that the order of additions is all there is to it: that order
    is part of what the norms' weight gradients promise a training step."""
    parts = 64 if rows < 65536 else 256
    per_part = -(-rows // parts)
    values = (torch.randn(parts, width, generator=torch.Generator().manual_seed(width)) * 3).float()
    values[-(-rows // per_part):] = 0
    dy = torch.zeros(rows, width, device=device)
    dy[torch.arange(0, rows, per_part, device=device)] = values[:-(-rows // per_part)].to(device)
    x = torch.zeros(rows, 4, device=device)
    db = torch.full((width,), float("nan"), device=device)
    ops.linear_backward(None, None, db, dy, x, torch.zeros(width, 4, device=device))
    units = torch.cuda.get_device_properties(device).multi_processor_count
    want = column_sums_in_order(values.numpy(), width, units)
    assert np.array_equal(db.cpu().numpy(), want)


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("accumulate", [False, True])
@pytest.mark.parametrize("rows,fin,fout", [
    (1, 64, 64), (31, 64, 32), (33, 40, 72), (300, 256, 100),   # tiles of 32 and 64, one and more per gradient, ragged edges
    (128, 768, 2048), (2000, 1024, 2048), (1999, 1000, 2040),   # more workgroups than compute units
    (70, 256, 5003),                                            # output gradient in padded rows
    (33, 40, 96), (131, 72, 160), (1999, 1000, 2048),           # ragged edges in the shared launch
])
def test_linear_gradients_in_one_launch_are_exact_on_integers(device, rows, fin, fout, accumulate, dtype):
    """dX, dW and db of a small call share a launch, behind a copy of 16-bit output gradients whose rows are no whole K steps (the
    other ragged calls go their own way, several launches). Products and sums of small integers are exact in fp32 (at most 4 x 5003 + 2),
    so every result is the rounded exact value; all three overwritten and all three added to what is there."""
    g = torch.Generator().manual_seed(rows + fin + fout)
    ints = lambda *shape: torch.randint(-2, 3, shape, generator=g).double()
    x, w, dy = ints(rows, fin), ints(fout, fin), ints(rows, fout)
    blank = [torch.zeros(shape, dtype=dtype, device=device) for shape in ((rows, fin), (fout, fin), fout, (rows, fout), (rows, fin), (fout, fin))]
    enqueued = launches(lambda: ops.linear_backward(*blank))
    if fout % 32 == 0:
        assert enqueued == 1
    elif fin % 32 == 0 and dtype != torch.float32:
        assert enqueued == 2
    else:
        assert enqueued > 2
    start = {"dX": ints(rows, fin), "dW": ints(fout, fin), "db": ints(fout)}
    got = {name: t.to(dtype).to(device) if accumulate else torch.full(t.shape, float("nan"), dtype=dtype, device=device)
           for name, t in start.items()}
    ops.linear_backward(got["dX"], got["dW"], got["db"], dy.to(dtype).to(device), x.to(dtype).to(device), w.to(dtype).to(device),
                        options=ops.LinearBackwardOptions(accumulate_input=accumulate, accumulate_weight=accumulate,
                                                          accumulate_bias=accumulate))
    for name, exact in (("dX", dy @ w), ("dW", dy.T @ x), ("db", dy.sum(0))):
        assert torch.equal(got[name].cpu(), (exact + (start[name] if accumulate else 0)).to(dtype)), name


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("vectors", [1024, 1025, 4096, 4097, 8192, 8193, 16384, 16385])
@pytest.mark.parametrize("tail", [0, 1])
def test_cross_entropy_around_the_held_row_lengths(device, vectors, tail, dtype):
    """Rows of exactly as many 16-byte vectors as a kernel holds and of one more, with and without a tail element."""
    rows, vocab = 3, vectors * (16 // torch.empty(0, dtype=dtype).element_size()) + tail
    logits, targets = randn((rows, vocab), dtype, vectors, 3.0), randint(vocab, (rows,), vectors + 1)
    targets[0] = vocab - 1
    loss, grad = torch.zeros(1, device=device), torch.empty((rows, vocab), dtype=dtype, device=device)
    # A scale of the order of the vocabulary, so that the bound sees the softmax and not only the target's column.
    ops.cross_entropy_forward_backward(loss, grad, logits.to(device), targets.to(device), rows, None, 4096.0)
    want_loss, want = oracle64.cross_entropy(to_np(logits), targets.numpy(), 4096.0)
    assert abs(loss.item() - want_loss) <= 1e-4 * max(1.0, abs(want_loss))
    assert_close(grad, want, TOL[dtype], "gradient")


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("more", [-1, 0, 1])
def test_swiglu_backward_around_the_choice_of_unrolling(device, more, dtype):
    """One vector per thread below two tiles of 1024 vectors per compute unit, four from there on."""
    units = torch.cuda.get_device_properties(device).multi_processor_count
    count = (units * 2 * 1024 + more) * (16 // torch.empty(0, dtype=dtype).element_size())
    g, u, dy = randn((count,), dtype, 8, 2.0), randn((count,), dtype, 9), randn((count,), dtype, 10)
    want_g, want_u = torch.empty_like(g), torch.empty_like(u)
    cpu_ops.swiglu_backward(want_g, want_u, dy, g, u)
    got_g, got_u = torch.empty_like(g, device=device), torch.empty_like(u, device=device)
    ops.swiglu_backward(got_g, got_u, dy.to(device), g.to(device), u.to(device))
    assert_close(got_g, want_g, TOL[dtype], "dgate")
    assert_close(got_u, want_u, TOL[dtype], "dup")


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("value", [float("inf"), float("nan")], ids=["inf", "nan"])
@pytest.mark.parametrize("rows,fin,fout", [
    (1, 5, 3), (33, 50, 70), (7, 131, 257),              # operands in padded copies
    (100, 64, 96), (33, 4096, 40),                       # 32- and 64-wide tiles, K slices
    (257, 2048, 264), (1100, 320, 520),                  # tiles of 64 and 128, ragged edges
])
def test_contractions_keep_non_finite_values_to_their_row_and_column(device, rows, fin, fout, value, dtype):
    """An Inf or a NaN in an operand reaches the row or column of the product that it belongs to and nothing beside it, whatever
    the kernel reads past the operands' ends; the rest is exact (small integers)."""
    g = torch.Generator().manual_seed(rows + fin)
    x, w, dy = (torch.randint(-2, 3, shape, generator=g).double() for shape in ((rows, fin), (fout, fin), (rows, fout)))
    for tensor, (i, j) in [("x", (rows - 1, fin - 1)), ("w", (fout - 1, fin - 1)), ("dy", (rows - 1, fout - 1)), ("x", (rows // 2, 0)),
                           ("w", (0, fin // 2)), ("dy", (0, fout // 2))]:
        planted = {"x": x.clone(), "w": w.clone(), "dy": dy.clone()}
        planted[tensor][i, j] = value
        on = lambda name: planted[name].to(dtype).to(device)
        y, gi, gw = (torch.empty(shape, dtype=dtype, device=device) for shape in ((rows, fout), (rows, fin), (fout, fin)))
        ops.linear_forward(y, on("x"), on("w"))
        ops.linear_backward(gi, gw, None, on("dy"), on("x"), on("w"))
        whole = slice(None)
        touched = {"x": {"Y": (i, whole), "dW": (whole, j)}, "w": {"Y": (whole, i), "dX": (whole, j)},
                   "dy": {"dX": (i, whole), "dW": (j, whole)}}[tensor]
        for name, got, exact in zip(("Y", "dX", "dW"), (y, gi, gw), (x @ w.T, dy @ w, dy.T @ x)):
            got, exact = got.cpu(), exact.to(dtype)
            if name in touched:
                assert not torch.isfinite(got[touched[name]]).any(), f"{tensor}[{i}, {j}] {name}"
                got[touched[name]] = exact[touched[name]] = 0
            assert torch.equal(got, exact), f"{tensor}[{i}, {j}] {name}"


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("vocab", [7, 1003, 8192, 50257, 131073])
def test_cross_entropy_with_non_finite_logits(device, vocab, dtype):
    """-Inf logits (masked classes) have probability 0, single ones and whole vectors of them; an Inf or a NaN spoils its own
    row's gradient, the Inf the loss, and no other row."""
    rows = 6
    logits = randn((rows, vocab), dtype, vocab, 2.0)
    targets = torch.tensor([0, 1, 2, 3, 4, 5], dtype=torch.int32)
    logits[1, vocab - 1] = logits[1, 6] = -float("inf")
    logits[2, vocab // 2:] = -float("inf")
    logits[3, :3] = -float("inf")

    def run(z):
        loss, grad = torch.zeros(1, device=device), torch.empty((rows, vocab), dtype=dtype, device=device)
        ops.cross_entropy_forward_backward(loss, grad, z.to(device), targets.to(device), rows, None, 4096.0)
        return loss.item(), grad.cpu()

    loss, grad = run(logits)
    want_loss, want = oracle64.cross_entropy(to_np(logits), targets.numpy(), 4096.0)
    assert abs(loss - want_loss) <= 1e-4 * max(1.0, abs(want_loss))
    assert_close(grad, want, TOL[dtype], "gradient")
    for value in (float("inf"), float("nan")):
        for row, col in ((0, 0), (4, vocab - 1), (5, vocab // 2)):
            spoiled = logits.clone()
            spoiled[row, col] = value
            bad_loss, bad = run(spoiled)
            others = torch.arange(rows) != row
            assert not torch.isfinite(bad[row]).all() and (np.isnan(value) or not np.isfinite(bad_loss))
            assert torch.equal(bad[others], grad[others])
