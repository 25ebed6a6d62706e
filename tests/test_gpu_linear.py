"""GPU parity tests of linear_forward / linear_backward (MFMA contraction kernels, padded copies of ragged operands) against
the CPU checker and float64 matmuls, through the C-ABI. The general kernel of operands that cannot be copied:
test_zz_capture_first.py."""
import numpy as np
import pytest
import torch

from cgpt_amd import capi, ops
from oracle import cpu_ops, oracle64
from tests.util import DTYPES, DTYPE_IDS, TOL, assert_close, launches, randn, to_np

pytestmark = pytest.mark.gpu


def dev(t, device):
    return t.to(device).contiguous()


def test_linear_backward_known_answer_and_accumulation(device):
    """tests/linear_backward_test.cu:20-45 (F32, 2x3)."""
    x = torch.tensor([1, 2, 3, 4, 5, 6.0]).reshape(2, 3).to(device)
    w = torch.tensor([1, 0, 2, -1, 3, 1.0]).reshape(2, 3).to(device)
    dy = torch.tensor([2, -1, 3, 4.0]).reshape(2, 2).to(device)
    gi, gw, gb = torch.zeros(2, 3, device=device), torch.zeros(2, 3, device=device), torch.zeros(2, device=device)
    ops.linear_backward(gi, gw, gb, dy, x, w)
    assert gi.reshape(-1).tolist() == [3, -3, 3, -1, 12, 10]
    assert gw.reshape(-1).tolist() == [14, 19, 24, 15, 18, 21]
    assert gb.tolist() == [5, 3]
    options = ops.LinearBackwardOptions(accumulate_input=True, accumulate_weight=True, accumulate_bias=True)
    ops.linear_backward(gi, gw, gb, dy, x, w, None, None, options)
    assert gi.reshape(-1).tolist() == [6, -6, 6, -2, 24, 20]
    assert gw.reshape(-1).tolist() == [28, 38, 48, 30, 36, 42]
    assert gb.tolist() == [10, 6]


def test_linear_backward_batched_f16_known_answer(device):
    """tests/linear_backward_test.cu:47-58."""
    f16 = torch.float16
    x = torch.tensor([1, 2, 3, 4, 5, 6, 7, 8.0]).reshape(2, 2, 2).to(f16).to(device)
    w = torch.tensor([1, 2, 3, 4, 5, 6.0]).reshape(3, 2).to(f16).to(device)
    dy = torch.arange(1, 13, dtype=torch.float32).reshape(2, 2, 3).to(f16).to(device)
    gi, gw, gb = torch.empty_like(x), torch.empty_like(w), torch.empty(3, dtype=f16, device=device)
    ops.linear_backward(gi, gw, gb, dy, x, w)
    assert np.abs(to_np(gi).reshape(-1) - [22, 28, 49, 64, 76, 100, 103, 136]).max() <= 0.1
    assert np.abs(to_np(gw).reshape(-1) - [118, 140, 134, 160, 150, 180]).max() <= 0.2
    assert np.abs(to_np(gb) - [22, 26, 30]).max() <= 0.1


def check_against_float64(got, want64, dtype, what, terms):
    """A dot product of `terms` rounded inputs: compare relative to the result's scale."""
    scale = max(1.0, float(np.abs(want64).max()))
    err = np.abs(to_np(got) - want64).max()
    assert np.isfinite(to_np(got)).all()
    assert err <= TOL[dtype] * scale, f"{what}: abs err {err:.3e} vs scale {scale:.3e}"


SHAPES = [  # rows, in, out
    (5, 7, 3), (33, 20, 17), (64, 64, 64), (128, 128, 256), (256, 192, 128), (136, 64, 72), (200, 256, 264),
    (384, 1024, 256), (1024, 320, 1024),
    # every reduction length (in for Y, out for dX, rows for dW) is an odd multiple of 32
    (288, 96, 160), (1056, 160, 352),
    # a single K tile; partial tiles in both directions with more work items than persistent blocks
    (64, 32, 64), (1000, 96, 520), (4104, 64, 2056),
]


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("rows,fin,fout", SHAPES)
def test_linear_forward_backward_parity(device, rows, fin, fout, dtype):
    x, w = randn((rows, fin), dtype, 1), randn((fout, fin), dtype, 2, 0.1)
    dy, b = randn((rows, fout), dtype, 3), randn((fout,), dtype, 4)
    dx_, dw_, ddy_, db_ = dev(x, device), dev(w, device), dev(dy, device), dev(b, device)

    y = torch.empty(rows, fout, dtype=dtype, device=device)
    ops.linear_forward(y, dx_, dw_, None, None, db_)
    check_against_float64(y, oracle64.linear_forward(to_np(x), to_np(w), to_np(b)), dtype, "y", fin)

    gi = torch.full((rows, fin), 5.0, dtype=dtype, device=device)
    gw = torch.full((fout, fin), 5.0, dtype=dtype, device=device)
    gb = torch.full((fout,), 5.0, dtype=dtype, device=device)
    ops.linear_backward(gi, gw, gb, ddy_, dx_, dw_)
    dx64, dw64, db64 = oracle64.linear_backward(to_np(dy), to_np(x), to_np(w))
    check_against_float64(gi, dx64, dtype, "dX", fout)
    check_against_float64(gw, dw64, dtype, "dW", rows)
    check_against_float64(gb, db64, dtype, "db", rows)

    if rows * fin * fout <= 256 * 192 * 128:  # the scalar CPU checker is O(rows*in*out)
        ci, cw, cb = torch.empty_like(x), torch.empty_like(w), torch.empty_like(b)
        cpu_ops.linear_backward(ci, cw, cb, dy, x, w)
        check_against_float64(gi, to_np(ci), dtype, "dX vs checker", fout)
        check_against_float64(gw, to_np(cw), dtype, "dW vs checker", rows)
        check_against_float64(gb, to_np(cb), dtype, "db vs checker", rows)

    # accumulate adds the same product onto what is there
    before = (gi.clone(), gw.clone(), gb.clone())
    options = ops.LinearBackwardOptions(accumulate_input=True, accumulate_weight=True, accumulate_bias=True)
    ops.linear_backward(gi, gw, gb, ddy_, dx_, dw_, None, None, options)
    check_against_float64(gi, to_np(before[0]) + dx64, dtype, "dX accumulate", fout)
    check_against_float64(gw, to_np(before[1]) + dw64, dtype, "dW accumulate", rows)
    check_against_float64(gb, to_np(before[2]) + db64, dtype, "db accumulate", rows)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_linear_backward_integer_valued_inputs_are_exact(device, dtype):
    """Small integers make every product and partial sum exactly representable: the MFMA path (incl. split-K
    for dW) must return the exact integers whatever the summation order."""
    rows, fin, fout = 2048, 256, 128
    g = torch.Generator().manual_seed(5)
    x = torch.randint(-2, 3, (rows, fin), generator=g).to(dtype)
    w = torch.randint(-2, 3, (fout, fin), generator=g).to(dtype)
    dy = torch.randint(-1, 2, (rows, fout), generator=g).to(dtype)
    dx64, dw64, db64 = oracle64.linear_backward(to_np(dy), to_np(x), to_np(w))
    gi = torch.empty(rows, fin, dtype=dtype, device=device)
    gw = torch.empty(fout, fin, dtype=dtype, device=device)
    ops.linear_backward(gi, gw, None, dev(dy, device), dev(x, device), dev(w, device))
    assert np.array_equal(to_np(gi), to_np(torch.tensor(dx64).to(dtype)))
    assert np.array_equal(to_np(gw), to_np(torch.tensor(dw64).to(dtype)))
    y = torch.empty(rows, fout, dtype=dtype, device=device)
    ops.linear_forward(y, dev(x, device), dev(w, device))
    assert np.array_equal(to_np(y), to_np(torch.tensor(to_np(x) @ to_np(w).T).to(dtype)))


def test_linear_backward_layer_shapes_of_the_104m_model(device):
    """One layer's projection shapes at 4096 of the 32768 training rows (k/v 256x1024, q/o 1024x1024,
    gate/up 2048x1024, down 1024x2048), bf16, against float64 matmuls, run twice bit-identically."""
    dtype = torch.bfloat16
    rows = 4096
    for fout, fin in ((256, 1024), (1024, 1024), (2048, 1024), (1024, 2048)):
        x, w, dy = randn((rows, fin), dtype, 6), randn((fout, fin), dtype, 7, 0.02), randn((rows, fout), dtype, 8)
        dx64, dw64, _ = oracle64.linear_backward(to_np(dy), to_np(x), to_np(w))
        outs = []
        for _ in range(2):
            gi = torch.empty(rows, fin, dtype=dtype, device=device)
            gw = torch.empty(fout, fin, dtype=dtype, device=device)
            ops.linear_backward(gi, gw, None, dev(dy, device), dev(x, device), dev(w, device))
            outs.append((gi.cpu(), gw.cpu()))
        assert torch.equal(outs[0][0], outs[1][0]) and torch.equal(outs[0][1], outs[1][1])
        check_against_float64(outs[0][0], dx64, dtype, f"dX {fout}x{fin}", fout)
        check_against_float64(outs[0][1], dw64, dtype, f"dW {fout}x{fin}", rows)


@pytest.mark.parametrize("fout,fin", [(256, 1024), (1024, 1024), (4096, 1024), (1024, 2048), (32000, 1024)],
                         ids=["kv-256x1024", "q-o-1024x1024", "gate_up-4096x1024", "down-1024x2048", "lm_head-32000x1024"])
def test_linear_backward_at_the_32768_training_rows_sampled_against_float64(device, fout, fin):
    """linear_backward at the real row count of a B=32, T=1024 step (the weight gradient's split-K depth is the 32768
    rows; the classifier shape is the one the cut cross-entropy contracts), bf16. Checked against float64 dot products
    on samples that touch every output tile: 256 rows of dX (two per 256-row tile, all columns), 64 rows and 64 columns
    of dW (all of the other index, i.e. sums over all 32768 rows), with the tolerance of the 16-bit parity bar relative
    to each result's scale. Inputs are made on the device; only the sampled slices travel to the host."""
    dtype = torch.bfloat16
    rows = 32768
    gen = torch.Generator(device=device).manual_seed(fout + fin)
    x = torch.randn(rows, fin, device=device, generator=gen).to(dtype)
    w = (torch.randn(fout, fin, device=device, generator=gen) * 0.02).to(dtype)
    dy = torch.randn(rows, fout, device=device, generator=gen).to(dtype)
    gi = torch.empty(rows, fin, dtype=dtype, device=device)
    gw = torch.empty(fout, fin, dtype=dtype, device=device)
    ops.linear_backward(gi, gw, None, dy, x, w)
    torch.cuda.synchronize()
    rng = np.random.default_rng(fout * 7 + fin)
    # dX rows: two per 256-row tile.
    picked = np.sort(np.concatenate([tile * 256 + rng.choice(256, 2, replace=False) for tile in range(rows // 256)]))
    index = torch.as_tensor(picked, device=device)
    want = to_np(dy[index]) @ to_np(w)
    check_against_float64(gi[index], want, dtype, f"dX rows {fout}x{fin}", fout)
    # dW rows (outputs o) and columns (inputs i), each a sum over all rows: accumulated over row chunks on the host.
    some_out = np.sort(rng.choice(fout, 64, replace=False))
    some_in = np.sort(rng.choice(fin, 64, replace=False))
    out_index, in_index = torch.as_tensor(some_out, device=device), torch.as_tensor(some_in, device=device)
    want_rows = np.zeros((64, fin))
    want_cols = np.zeros((fout, 64))
    for r0 in range(0, rows, 2048):
        dy_chunk, x_chunk = dy[r0:r0 + 2048], x[r0:r0 + 2048]
        want_rows += to_np(dy_chunk[:, out_index]).T @ to_np(x_chunk)
        want_cols += to_np(dy_chunk).T @ to_np(x_chunk[:, in_index])
    check_against_float64(gw[out_index], want_rows, dtype, f"dW rows {fout}x{fin}", rows)
    check_against_float64(gw[:, in_index], want_cols, dtype, f"dW columns {fout}x{fin}", rows)
    # dX columns over all rows for the layer shapes (the classifier's dY is too large to widen on the host).
    if fout <= 4096:
        want_dx_cols = np.concatenate([to_np(dy[r0:r0 + 4096]) @ to_np(w[:, in_index]) for r0 in range(0, rows, 4096)])
        check_against_float64(gi[:, in_index], want_dx_cols, dtype, f"dX columns {fout}x{fin}", fout)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("count,rows,fout,fin", [
    (8, 2048, 256, 512),    # 16 tiles: the launch splits the row sum
    (3, 1056, 512, 264),    # ragged columns, three slices' worth of K tiles
    (5, 4096, 768, 1024),   # 60 tiles
    (40, 1024, 2048, 256),  # 320 tiles: more than one round of the persistent blocks
    (2, 520, 96, 200),      # out_features not a multiple of 256: separate weight gradients
    (1, 2048, 256, 512),    # a stack of one
], ids=["8x256x512", "3x512x264", "5x768x1024", "40x2048x256", "fallback", "single"])
def test_linear_backward_weights_stacked_matches_float64_and_integers(device, count, rows, fout, fin, dtype):
    """The weight gradients of several layers in one launch against float64 products (the bound of the single
    weight gradient), and exact on small integers whatever the number of slices the launch picks."""
    g = torch.Generator().manual_seed(11)
    dy = (torch.randn((count, rows, fout), generator=g) * 1.0).to(dtype)
    x = (torch.randn((count, rows, fin), generator=g) * 1.0).to(dtype)
    gw = torch.full((count, fout, fin), 7.0, dtype=dtype, device=device)
    ops.linear_backward_weights_stacked(gw, dev(dy, device), dev(x, device))
    for j in range(count):
        want = to_np(dy[j]).T @ to_np(x[j])
        check_against_float64(gw[j].cpu(), want, dtype, f"dW of layer {j}", rows)
    # twice, bit-identical
    again = torch.empty_like(gw)
    ops.linear_backward_weights_stacked(again, dev(dy, device), dev(x, device))
    assert torch.equal(gw, again)
    if dtype != torch.float32:
        dy = torch.randint(-1, 2, (count, rows, fout), generator=g).to(dtype)
        x = torch.randint(-2, 3, (count, rows, fin), generator=g).to(dtype)
        ops.linear_backward_weights_stacked(gw, dev(dy, device), dev(x, device))
        for j in range(count):
            want = torch.tensor(to_np(dy[j]).T @ to_np(x[j])).to(dtype)
            assert np.array_equal(to_np(gw[j]), to_np(want)), f"layer {j}"


def test_linear_backward_weights_stacked_with_strided_layers_and_errors(device):
    """Layers taken out of larger blocks (strides beyond rows x features), and the argument checks."""
    dtype = torch.bfloat16
    count, rows, fout, fin = 4, 1024, 256, 256
    g = torch.Generator().manual_seed(12)
    dy_block = torch.randn((count, rows + 64, fout), generator=g).to(dtype).to(device)
    x_block = torch.randn((count, rows + 32, fin), generator=g).to(dtype).to(device)
    dy, x = dy_block[:, :rows], x_block[:, :rows]
    gw = torch.empty((count, fout, fin), dtype=dtype, device=device)
    ops.linear_backward_weights_stacked(gw, dy, x)
    for j in range(count):
        check_against_float64(gw[j].cpu(), to_np(dy[j]).T @ to_np(x[j]), dtype, f"dW of layer {j}", rows)
    with pytest.raises(ValueError):
        ops.linear_backward_weights_stacked(gw, dy[:3], x)
    with pytest.raises(ValueError):
        ops.linear_backward_weights_stacked(gw, dy, x[:, :, :128])
    with pytest.raises(ValueError):
        ops.linear_backward_weights_stacked(gw.cpu(), dy, x)


def test_linear_argument_errors(device):
    x, w, dy = torch.zeros(4, 8, device=device), torch.zeros(3, 8, device=device), torch.zeros(4, 3, device=device)
    gi, gw, gb = torch.zeros_like(x), torch.zeros_like(w), torch.zeros(3, device=device)
    with pytest.raises(ValueError):
        ops.linear_backward(gi, gw, gb, torch.zeros(4, 4, device=device), x, w)
    with pytest.raises(ValueError):
        ops.linear_backward(gi, gw, gb, dy, x.half(), w)
    with pytest.raises(ValueError):
        ops.linear_backward(gi, torch.zeros(3, 7, device=device), gb, dy, x, w)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("rows,fin,hidden", [(4096, 256, 1664), (4104, 64, 1664), (2056, 96, 3328), (64, 32, 64), (520, 96, 200)],
                         ids=["fused", "fused-ragged-rows", "fused-wide", "small", "unaligned-columns"])
def test_linear_swiglu_forward_equals_the_two_operators(device, rows, fin, hidden, dtype):
    """Gate/up projection with the SwiGLU product from its epilogue (one contraction over interleaved
    gate and up columns when the shape fills the chip) against linear_forward into the concatenated
    layout followed by swiglu_forward: the same bits, and the float64 product within the 16-bit tolerance."""
    g = torch.Generator().manual_seed(rows + hidden)
    x = torch.randn(rows, fin, generator=g).to(dtype).to(device)
    w = (torch.randn(2 * hidden, fin, generator=g) * 0.3).to(dtype).to(device)
    want_gate_up = torch.empty(rows, 2 * hidden, dtype=dtype, device=device)
    want_act = torch.empty(rows, hidden, dtype=dtype, device=device)
    ops.linear_forward(want_gate_up, x, w)
    ops.swiglu_forward(want_act, want_gate_up)
    got_gate_up = torch.full_like(want_gate_up, float("nan"))
    got_act = torch.full_like(want_act, float("nan"))
    ops.linear_swiglu_forward(got_gate_up, got_act, x, w)
    torch.cuda.synchronize()
    assert torch.equal(got_gate_up, want_gate_up)
    assert torch.equal(got_act, want_act)
    exact = x.double().cpu() @ w.double().cpu().t()
    gate, up = exact[:, :hidden], exact[:, hidden:]
    reference = gate / (1 + torch.exp(-gate)) * up
    err = (got_act.double().cpu() - reference).abs().max() / reference.abs().max()
    assert err <= 2e-2


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("rows,out,hidden", [(4096, 256, 3328), (4104, 64, 3328), (4096, 96, 3336), (64, 32, 64), (520, 96, 200)],
                         ids=["fused", "fused-ragged-rows", "fused-ragged-columns", "small", "unaligned-columns"])
def test_linear_swiglu_backward_equals_the_two_operators(device, rows, out, hidden, dtype):
    """Input gradient of the down projection with the SwiGLU gradient from its epilogue (when the shape
    fills the chip) against linear_backward followed by the packed swiglu_backward: the same bits, rows and
    columns past the matrix untouched, and the float64 gradient within the 16-bit tolerance."""
    g = torch.Generator().manual_seed(rows + hidden + 1)
    dy = torch.randn(rows, out, generator=g).to(dtype).to(device)
    w = (torch.randn(out, hidden, generator=g) * 0.3).to(dtype).to(device)
    gate_up = torch.randn(rows, 2 * hidden, generator=g).to(dtype).to(device)
    act = torch.empty(rows, hidden, dtype=dtype, device=device)  # the projection's input: unused by its input gradient
    d_act = torch.empty(rows, hidden, dtype=dtype, device=device)
    want = torch.empty(rows, 2 * hidden, dtype=dtype, device=device)
    ops.linear_backward(d_act, None, None, dy, act, w)
    ops.swiglu_backward_packed(want, d_act, gate_up)
    guarded = torch.full((rows + 8, 2 * hidden), 7.0, dtype=dtype, device=device)  # rows after the output
    got = guarded[:rows]
    work = torch.empty_like(d_act)
    ops.linear_swiglu_backward(got, work, dy, w, gate_up)
    torch.cuda.synchronize()
    assert torch.equal(got, want)
    assert bool((guarded[rows:] == 7.0).all())
    exact = dy.double().cpu() @ w.double().cpu()
    gate, up = gate_up.double().cpu()[:, :hidden], gate_up.double().cpu()[:, hidden:]
    sig = 1 / (1 + torch.exp(-gate))
    reference = torch.cat([exact * up * sig * (1 + gate * (1 - sig)), exact * gate * sig], dim=1)
    err = (got.double().cpu() - reference).abs().max() / reference.abs().max()
    assert err <= 2e-2


def test_linear_swiglu_backward_argument_errors(device):
    bf = torch.bfloat16
    dy = torch.zeros(8, 16, dtype=bf, device=device)
    w = torch.zeros(16, 32, dtype=bf, device=device)
    gate_up = torch.zeros(8, 64, dtype=bf, device=device)
    grad = torch.zeros(8, 64, dtype=bf, device=device)
    work = torch.zeros(8, 32, dtype=bf, device=device)
    ops.linear_swiglu_backward(grad, work, dy, w, gate_up)  # valid
    with pytest.raises(ValueError):
        ops.linear_swiglu_backward(grad, torch.zeros(8, 16, dtype=bf, device=device), dy, w, gate_up)
    with pytest.raises(ValueError):
        ops.linear_swiglu_backward(grad, work, dy, torch.zeros(15, 32, dtype=bf, device=device), gate_up)
    with pytest.raises(ValueError):
        ops.linear_swiglu_backward(grad.float(), work, dy, w, gate_up)
    from cgpt_amd import capi
    with pytest.raises(ValueError):  # the C entry point rejects null tensors itself
        capi.call("cgptx_linear_swiglu_backward", grad.data_ptr(), None, dy.data_ptr(), w.data_ptr(), gate_up.data_ptr(),
                  8, 32, 16, 1, None)


def test_linear_swiglu_forward_argument_errors(device):
    x = torch.zeros(8, 32, dtype=torch.bfloat16, device=device)
    w = torch.zeros(64, 32, dtype=torch.bfloat16, device=device)
    gate_up = torch.zeros(8, 64, dtype=torch.bfloat16, device=device)
    act = torch.zeros(8, 32, dtype=torch.bfloat16, device=device)
    ops.linear_swiglu_forward(gate_up, act, x, w)  # valid
    with pytest.raises(ValueError):
        ops.linear_swiglu_forward(gate_up, torch.zeros(8, 16, dtype=torch.bfloat16, device=device), x, w)
    with pytest.raises(ValueError):
        ops.linear_swiglu_forward(gate_up, act, x, torch.zeros(63, 32, dtype=torch.bfloat16, device=device))
    with pytest.raises(ValueError):
        ops.linear_swiglu_forward(gate_up, act.float(), x, w)
    from cgpt_amd import capi
    with pytest.raises(ValueError):  # the C entry point rejects null tensors itself
        capi.call("cgptx_linear_swiglu_forward", None, act.data_ptr(), x.data_ptr(), w.data_ptr(), 8, 32, 32, 1, None)


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("rows,fin,fout", [
    (1, 64, 64), (63, 64, 96), (65, 96, 64), (129, 160, 136),      # 64-wide tiles with a ragged last row; short K tiles in dW
    (3001, 512, 1024), (2049, 1024, 2048),                         # 128-wide tiles
    (8197, 1024, 2048),                                            # 256-wide tiles
    (77, 100, 31), (130, 33, 129), (258, 130, 66), (4099, 257, 515),  # widths that are not whole chunks: padded copies, C by elements
    (40, 72, 24), (40, 24, 72),                                    # whole chunks, but K ends inside a K tile
])
@pytest.mark.parametrize("accumulate", [False, True], ids=["overwrite", "accumulate"])
def test_linear_ragged_shapes_integer_valued_inputs_are_exact(device, rows, fin, fout, accumulate, dtype):
    """Small integers: every product and partial sum is exact in fp32, so the result is the rounded exact value whatever
    the order of additions."""
    g = torch.Generator().manual_seed(rows + fin + fout)
    integers = lambda *shape: torch.randint(-2, 3, shape, generator=g).double()
    x, w, dy, b = integers(rows, fin), integers(fout, fin), integers(rows, fout), integers(fout)
    base = [integers(rows, fin), integers(fout, fin), integers(fout)] if accumulate else [0, 0, 0]
    want = [x @ w.T + b, dy @ w + base[0], dy.T @ x + base[1], dy.sum(0) + base[2]]
    on = lambda t: t.to(dtype).to(device)
    y = torch.full((rows, fout), float("nan"), dtype=dtype, device=device)
    gi, gw, gb = (on(v) if accumulate else torch.full(shape, float("nan"), dtype=dtype, device=device)
                  for v, shape in zip(base, ((rows, fin), (fout, fin), (fout,))))
    ops.linear_forward(y, on(x), on(w), bias=on(b))
    options = ops.LinearBackwardOptions(accumulate_input=accumulate, accumulate_weight=accumulate, accumulate_bias=accumulate)
    ops.linear_backward(gi, gw, gb, on(dy), on(x), on(w), options=options)
    for name, got, exact in zip(("Y", "dX", "dW", "db"), (y, gi, gw, gb), want):
        assert torch.equal(got.cpu(), exact.to(dtype)), name


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("behind,before", [("db", "dW"), ("dW", "dX"), ("db", "dX")])
def test_overlapping_gradients_are_written_one_after_the_other(device, behind, before, dtype):
    """Gradients that share memory hold what the last of dX, dW, db leaves. Small calls run all three in one launch, whose
    workgroups are in no order: not these."""
    rows, fin, fout = 128, 256, 192
    g = torch.Generator().manual_seed(rows)
    x, w, dy = (torch.randint(-2, 3, shape, generator=g).to(dtype).to(device) for shape in ((rows, fin), (fout, fin), (rows, fout)))
    shapes = {"dX": (rows, fin), "dW": (fout, fin), "db": (fout,)}
    # `behind` begins within the last sixteen elements of `before`.
    size = {name: int(np.prod(shape)) for name, shape in shapes.items()}
    shared = torch.zeros(size[before] + size[behind], dtype=dtype, device=device)
    place = {name: torch.zeros(shape, dtype=dtype, device=device) for name, shape in shapes.items()}
    place[before] = shared[:size[before]].view(shapes[before])
    place[behind] = shared[size[before] - 16:][:size[behind]].view(shapes[behind])

    def at_once(to):
        ops.linear_backward(to["dX"], to["dW"], to["db"], dy, x, w)

    assert launches(lambda: at_once(place)) > 1
    shared.zero_()
    at_once(place)
    got = shared.clone()
    shared.zero_()
    for name in ("dX", "dW", "db"):
        ops.linear_backward(*(place[n] if n == name else None for n in ("dX", "dW", "db")), dy, x, w)
    assert torch.equal(got, shared)
    apart = {name: torch.zeros(shape, dtype=dtype, device=device) for name, shape in shapes.items()}
    assert launches(lambda: at_once(apart)) == 1


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("rows,fin,fout", [
    (2000, 1024, 2048),                      # a workgroup per CU, one sum over K; dW's K ends inside a K tile
    (4100, 768, 768), (5005, 1032, 288),     # dW in K slices, rows and columns that end inside a tile, an odd last slice
    (8193, 1024, 1024),                      # more workgroups than the chip holds at once
])
@pytest.mark.parametrize("accumulate", [False, True], ids=["overwrite", "accumulate"])
def test_both_gradients_on_large_tiles_share_a_launch(device, rows, fin, fout, accumulate, dtype):
    """Small integers: exact in any order of additions. Three passes into poisoned memory: the counters by which the last
    workgroup of a tile knows itself start each from zero."""
    g = torch.Generator().manual_seed(rows + fin)
    integers = lambda *shape: torch.randint(-1, 2, shape, generator=g).float()
    x, w, dy = integers(rows, fin), integers(fout, fin), integers(rows, fout)
    base = [integers(rows, fin), integers(fout, fin), integers(fout)]
    want = [dy @ w, dy.T @ x, dy.sum(0)]  # whole numbers far below 2^24: exact in fp32
    x, w, dy = (t.to(dtype).to(device) for t in (x, w, dy))
    outputs = [torch.empty(shape, dtype=dtype, device=device) for shape in ((rows, fin), (fout, fin), (fout,))]
    options = ops.LinearBackwardOptions(accumulate_input=accumulate, accumulate_weight=accumulate, accumulate_bias=accumulate)
    for _ in range(3):
        for out, old in zip(outputs, base):
            out.copy_(old) if accumulate else out.fill_(float("nan"))
        ops.linear_backward(*outputs, dy, x, w, options=options)
        for name, got, exact, old in zip(("dX", "dW", "db"), outputs, want, base):
            assert torch.equal(got.cpu(), (exact + old if accumulate else exact).to(dtype)), name
    assert launches(lambda: ops.linear_backward(*outputs, dy, x, w, options=options)) == 1


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("rows,fin,fout", [
    (2000, 1024, 2048),   # a workgroup per CU and all of its LDS
    (4100, 768, 768),     # two per CU, dW in K slices
])
@pytest.mark.parametrize("shifted", ["dX", "dW", "both"])
@pytest.mark.parametrize("accumulate", [False, True], ids=["overwrite", "accumulate"])
def test_large_gradients_wherever_they_start(device, rows, fin, fout, accumulate, shifted, dtype):
    """Gradients that start on no multiple of 16 bytes are stored element by element, by one launch all the same, and nothing
    beside them is written."""
    g = torch.Generator().manual_seed(rows + fin)
    integers = lambda *shape: torch.randint(-1, 2, shape, generator=g).float()
    x, w, dy = integers(rows, fin), integers(fout, fin), integers(rows, fout)
    base = [integers(rows, fin), integers(fout, fin), integers(fout)]
    want = [dy @ w, dy.T @ x, dy.sum(0)]  # whole numbers far below 2^24: exact in fp32
    x, w, dy = (t.to(dtype).to(device) for t in (x, w, dy))
    buffers, outputs = [], []
    for name, old in zip(("dX", "dW", "db"), base):
        first = 16 + (3 if shifted in (name, "both") else 0)
        buffer = torch.full((old.numel() + 48,), 7.0, dtype=dtype, device=device)
        outputs.append(buffer[first:first + old.numel()].view(old.shape))
        outputs[-1].copy_(old) if accumulate else outputs[-1].fill_(float("nan"))
        buffers.append((buffer, first))
    options = ops.LinearBackwardOptions(accumulate_input=accumulate, accumulate_weight=accumulate, accumulate_bias=accumulate)
    ops.linear_backward(*outputs, dy, x, w, options=options)
    for name, got, exact, old, (buffer, first) in zip(("dX", "dW", "db"), outputs, want, base, buffers):
        assert torch.equal(got.cpu(), (exact + old if accumulate else exact).to(dtype)), name
        assert (buffer[:first] == 7.0).all() and (buffer[first + old.numel():] == 7.0).all(), name
    assert launches(lambda: ops.linear_backward(*outputs, dy, x, w, options=options)) == 1


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_gradients_in_k_slices_replay_from_a_graph(device, dtype):
    """dW in K slices, recorded: replays between eager calls with another number of slices on the same counters, which all start
    from zero, and with partial tiles that make the arena grow, under which the recorded ones stay where they were. Then replays on
    another stream beside eager work of the first: they share the counters and their results are undefined, but what comes after
    them is not."""
    shapes = [(4100, 768, 768), (5005, 1024, 1024)]  # five slices, three
    g = torch.Generator().manual_seed(5)
    integers = lambda *shape: torch.randint(-1, 2, shape, generator=g).float()
    calls = []
    for rows, fin, fout in shapes:
        x, w, dy = integers(rows, fin), integers(fout, fin), integers(rows, fout)
        want = [t.to(dtype).to(device) for t in (dy @ w, dy.T @ x, dy.sum(0))]  # whole numbers: exact in any order of additions
        operands = [t.to(dtype).to(device) for t in (dy, x, w)]
        calls.append((operands, want, [torch.empty_like(t) for t in want]))
    stream, other = torch.cuda.Stream(), torch.cuda.Stream()

    def run(which):
        operands, _, outputs = calls[which]
        ops.linear_backward(*outputs, *operands)

    def check(which, call):
        for out in calls[which][2]:
            out.fill_(float("nan"))
        call()
        torch.cuda.synchronize()
        for name, got, exact in zip(("dX", "dW", "db"), calls[which][2], calls[which][1]):
            assert torch.equal(got, exact), name

    assert launches(lambda: run(0)) == 1 and launches(lambda: run(1)) == 1
    torch.cuda.synchronize()
    capi.call("cgptx_release_scratch")
    with torch.cuda.stream(stream):
        check(0, lambda: run(0))
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
            run(0)
        for _ in range(3):
            check(0, graph.replay)
            check(1, lambda: run(1))
    torch.cuda.synchronize()
    for _ in range(4):
        with torch.cuda.stream(other):
            graph.replay()
        with torch.cuda.stream(stream):
            run(1)
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        for _ in range(2):
            check(1, lambda: run(1))
            check(0, graph.replay)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("rows,k,n", [  # what the plan takes on 256 compute units
    (5005, 1024, 1024), (4833, 992, 1000),     # 160 x 128
    (7000, 2048, 768), (8999, 1728, 640),      # 192 x 128
    (8161, 4096, 1024),                        # 256 x 128 where nothing else fits better
    (5005, 1024, 2048), (10000, 1024, 1016),   # 160 x 256
    (11900, 1024, 1024), (11871, 352, 1024),   # 192 x 256
    (12500, 1024, 1024), (13001, 1024, 4096),  # 224 x 256, one round and four
])
def test_oblong_tiles_give_the_bits_of_square_ones(device, rows, k, n, dtype):
    """Results that do not start on 16 bytes run on square tiles of the general epilogue; others, with a bias or without, and as an
    input gradient, on whatever the plan takes: one sum over K each, in the same order. Integers small enough that all sums are exact
    check both."""
    g = torch.Generator().manual_seed(rows)
    x = torch.randint(-2, 3, (rows, k), generator=g).to(dtype).to(device)
    w = torch.randint(-1, 2, (n, k), generator=g).to(dtype).to(device)
    for scale in (1.0, 0.37):
        a, b = (x * scale).to(dtype), (w * 0.11 if scale != 1.0 else w).to(dtype)
        plain, biased, dx = (torch.full((rows, n), float("nan"), dtype=dtype, device=device) for _ in range(3))
        square = torch.full((rows * n + 4,), float("nan"), dtype=dtype, device=device)[4:].view(rows, n)
        bias = torch.randint(-9, 10, (n,), generator=g).to(dtype).to(device) * scale
        ops.linear_forward(biased, a, b, bias=bias)
        ops.linear_forward(square, a, b, bias=bias)
        assert torch.equal(biased, square)
        ops.linear_forward(plain, a, b)
        ops.linear_forward(square, a, b)
        assert torch.equal(plain, square)
        ops.linear_backward(dx, None, None, a, torch.empty_like(dx), b.t().contiguous())
        assert torch.equal(dx, square)
        if scale == 1.0:
            exact = a.float() @ b.float().t()
            assert torch.equal(plain, exact.to(dtype))
            assert torch.equal(biased, (exact + bias.float()).to(dtype))
            old = torch.randint(-8, 9, (rows, n), generator=g).to(dtype).to(device)
            added = old.clone()
            ops.linear_backward(added, None, None, a, torch.empty_like(dx), b.t().contiguous(),
                                options=ops.LinearBackwardOptions(accumulate_input=True))
            assert torch.equal(added, (exact + old.float()).to(dtype))


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("rows,k,n", [(1, 7, 8), (16, 1379, 256), (300, 517, 770), (257, 65, 3), (700, 4097, 64)])
def test_both_operands_of_odd_k_are_copied_in_one_launch(device, rows, k, n, dtype):
    """The copy of the input and that of the weight, and the product over them (in K slices: and their sum). Operands that start
    anywhere; integers small enough that all sums are exact."""
    g = torch.Generator().manual_seed(rows)
    x = torch.empty(rows * k + 1, dtype=dtype, device=device)[1:].view(rows, k)
    x.copy_(torch.randint(-1, 2, (rows, k), generator=g))
    w = torch.randint(-1, 2, (n, k), generator=g).to(dtype).to(device)
    y = torch.full((rows, n), float("nan"), dtype=dtype, device=device)
    ops.linear_forward(y, x, w)
    assert torch.equal(y, (x.float() @ w.float().t()).to(dtype))
    assert launches(lambda: ops.linear_forward(y, x, w)) <= 3


@pytest.mark.parametrize("dtype", DTYPES, ids=DTYPE_IDS)
@pytest.mark.parametrize("rows,fin,fout", [(1, 9, 8), (16, 1379, 256), (33, 517, 771), (257, 65, 40), (700, 1021, 200)])
@pytest.mark.parametrize("accumulate", [False, True], ids=["overwrite", "accumulate"])
def test_gradients_over_odd_rows_share_a_launch(device, rows, fin, fout, accumulate, dtype):
    """Weight and input of odd rows are copied together (an output gradient whose columns end inside a K tile in a launch of its own), and
    both gradients and the bias's come from one launch over the copies. A result on top of the input keeps the contractions' order: the
    weight gradient is that of what the input gradient left there. Integers small enough that all sums are exact."""
    g = torch.Generator().manual_seed(rows + fin)
    draw = lambda *shape: torch.randint(-1, 2, shape, generator=g).to(dtype).to(device)
    dy, x, w = draw(rows, fout), draw(rows, fin), draw(fout, fin)
    old = [draw(rows, fin), draw(fout, fin), draw(fout)]
    options = ops.LinearBackwardOptions(accumulate_input=accumulate, accumulate_weight=accumulate, accumulate_bias=accumulate)
    outputs = [t.clone() for t in old]
    ops.linear_backward(*outputs, dy, x, w, options=options)
    exact = [dy.float() @ w.float(), dy.float().t() @ x.float(), dy.float().sum(0)]
    for out, before, want in zip(outputs, old, exact):
        assert torch.equal(out, (want + before.float() if accumulate else want).to(dtype))
    assert launches(lambda: ops.linear_backward(*outputs, dy, x, w, options=options)) <= (3 if dtype != torch.float32 else 7)
    if not accumulate:
        lying = x.clone()
        ops.linear_backward(lying, outputs[1], None, dy, lying, w)
        assert torch.equal(lying, exact[0].to(dtype))
        want = dy.double().t() @ lying.double()
        assert (outputs[1].double() - want).abs().max() <= 2.0 ** -7 * max(1.0, want.abs().max().item())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("rows,fin,fout", [
    (5005, 1024, 2048), (6983, 760, 2048),   # dX on 224 x 256, dW in two and three slices; rows, columns and K end inside tiles
    (3000, 1024, 4096), (2993, 1016, 4064),  # dX on 192 x 128, dW one sum over K
])
@pytest.mark.parametrize("accumulate", [False, True], ids=["overwrite", "accumulate"])
def test_both_gradients_on_oblong_tiles_share_a_launch(device, rows, fin, fout, accumulate, dtype):
    test_both_gradients_on_large_tiles_share_a_launch(device, rows, fin, fout, accumulate, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("rows,fin,fout", [  # dX's tile and dW's slices as tests/cpp/gemm_plan_test.cpp holds them
    (732, 1368, 2208), (2419, 656, 3104), (3691, 400, 2208),    # 160 x 128 in 1, 2, 3
    (779, 3960, 1184), (3336, 1040, 1824), (2957, 720, 1184),   # 160 x 256 in 1, 2, 3
    (2323, 648, 3104), (3226, 600, 1632),                       # 192 x 128 in 1, 3
    (1080, 3624, 1056), (3963, 1040, 1632), (5180, 968, 1504),  # 192 x 256 in 1, 2, 3
    (1196, 3616, 1056), (3965, 1160, 1440), (4010, 1192, 1248),  # 224 x 256 in 1, 2, 3
    (2732, 776, 3232), (3004, 792, 1184),                       # 256 x 128 in 1, 3
])
@pytest.mark.parametrize("accumulate", [False, True], ids=["overwrite", "accumulate"])
def test_both_gradients_on_every_oblong_tile(device, rows, fin, fout, accumulate, dtype):
    """Rows, columns and K end inside tiles."""
    test_both_gradients_on_large_tiles_share_a_launch(device, rows, fin, fout, accumulate, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_oblong_tiles_of_192_x_256_end_anywhere(device, dtype):
    """Rows, columns and K end inside tiles."""
    test_oblong_tiles_give_the_bits_of_square_ones(device, 11871, 992, 1016, dtype)
