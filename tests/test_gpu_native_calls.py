"""Operator calls that host/dispatch.cpp makes by itself against the same calls through the functions of cgpt_amd/ops.py: what is
taken gives the same bits, what is refused is refused with the same words."""
import pytest
import torch

from cgpt_amd import ops
from tests.util import randn

pytestmark = pytest.mark.gpu


class _Declines:
    """A native side that takes nothing."""

    def __getattr__(self, name):
        return lambda *args: None


class _Counts:
    """The native side, and how many calls it took."""

    def __init__(self):
        self.taken = 0

    def __getattr__(self, name):
        function = getattr(_NATIVE, name)

        def call(*args):
            status = function(*args)
            self.taken += status is not None
            return status
        return call


_NATIVE = ops._native


def _calls(device, dtype):
    """name -> (function, tensors, keyword arguments): one call of each operator as programs make it."""
    def t(seed, *shape, of=dtype):
        return randn(shape, of, seed).to(device)
    ids = torch.tensor([3, 0, 5, 3, 1, 2], dtype=torch.int32, device=device)
    options = ops.FlashAttentionOptions(4, 2, 32)
    q, k, v, o = t(1, 2, 5, 4, 32), t(2, 2, 5, 2, 32), t(3, 2, 5, 2, 32), t(4, 2, 5, 4, 32)
    lse = t(5, 2, 5, 4, of=torch.float32).abs() + 2.0
    cos, sin = t(6, 5, 16), t(7, 5, 16)
    loss = torch.zeros(1, device=device)
    backward = ops.LinearBackwardOptions(accumulate_input=True, accumulate_bias=True)
    return {
        "rmsnorm_forward": (ops.rmsnorm_forward, [t(8, 6, 64), t(9, 6, 64), t(10, 64), 1e-5], {}),
        "rmsnorm_backward": (ops.rmsnorm_backward, [t(8, 6, 64), t(9, 64), t(10, 6, 64), t(11, 6, 64), t(12, 64), 1e-5], {}),
        "rope_forward": (ops.rope_forward, [q.clone(), k.clone(), cos, sin], {"rope_options": ops.RopeOptions(rotary_dim=32)}),
        "rope_backward": (ops.rope_backward, [q.clone(), k.clone(), o, v, cos, sin], {}),
        "swiglu_forward": (ops.swiglu_forward, [t(13, 3, 40), t(14, 3, 40), t(15, 3, 40)], {}),
        "swiglu_backward": (ops.swiglu_backward, [t(13, 3, 40), t(14, 3, 40), t(15, 3, 40), t(16, 3, 40), t(17, 3, 40)],
                            {"options": ops.SwiGLUBackwardOptions(accumulate_up=True)}),
        "linear_forward": (ops.linear_forward, [t(18, 2, 3, 24), t(19, 2, 3, 32), t(20, 24, 32)], {"bias": t(21, 24)}),
        "linear_backward": (ops.linear_backward, [t(18, 2, 3, 32), t(19, 24, 32), t(20, 24), t(21, 2, 3, 24), t(22, 2, 3, 32), t(23, 24, 32)],
                            {"options": backward}),
        "linear_backward_weight_only": (ops.linear_backward, [None, t(19, 24, 32), None, t(21, 6, 24), t(22, 6, 32), t(23, 24, 32)], {}),
        "add_tensors": (ops.add_tensors, [t(24, 7), t(25, 7), t(26, 7)], {}),
        "attention": (ops.flash_gqa_attention_forward, [o.clone(), q, k, v], {"options": options}),
        "attention_with_lse": (ops.flash_gqa_attention_forward_with_lse, [o.clone(), lse.clone(), q, k, v], {"options": options}),
        "attention_backward": (ops.flash_gqa_attention_backward, [q.clone(), k.clone(), v.clone(), o, q, k, v], {"options": options}),
        "attention_backward_with_lse": (ops.flash_gqa_attention_backward_with_lse, [q.clone(), k.clone(), v.clone(), o, o, lse, q, k, v],
                                        {"options": options, "accumulate_grads": True}),
        "embedding_forward": (ops.embedding_forward, [t(27, 6, 64), ids, 6, t(28, 9, 64)], {}),
        "embedding_backward": (ops.embedding_backward, [t(27, 9, 64), t(28, 6, 64), ids, 6],
                               {"options": ops.EmbeddingBackwardOptions(accumulate_weight=True)}),
        "cross_entropy_forward": (ops.cross_entropy_forward, [loss.clone(), t(29, 6, 33), ids, 6], {}),
        "cross_entropy_forward_backward": (ops.cross_entropy_forward_backward, [loss.clone(), t(30, 6, 33), t(31, 6, 33), ids, 6],
                                           {"gradient_scale": 64.0}),
        "cut_cross_entropy": (ops.cut_cross_entropy_forward_backward,
                              [loss.clone(), t(32, 6, 64), t(33, 33, 64), t(34, 6, 64), t(35, 33, 64), ids, 6], {"gradient_scale": 2.0}),
    }


def _outcome(monkeypatch, native, function, args, options):
    """The tensors after the call, or the kind and words of what it raised."""
    monkeypatch.setattr(ops, "_native", native)
    args = [a.clone(memory_format=torch.preserve_format) if type(a) is torch.Tensor else a for a in args]
    try:
        assert function(*args, **options) is None
    except Exception as error:  # noqa: BLE001 - compared
        return type(error), str(error)
    torch.cuda.synchronize()
    return [a for a in args if isinstance(a, torch.Tensor)]


def _bits(t):
    return torch.empty(t.numel(), dtype=t.dtype).copy_(t.detach().reshape(-1)).view(torch.uint8).numpy().tobytes()


def _same_outcome(monkeypatch, function, args, options, what):
    one = _outcome(monkeypatch, _NATIVE, function, args, options)
    other = _outcome(monkeypatch, _Declines(), function, args, options)
    if isinstance(one, tuple) or isinstance(other, tuple):
        assert one == other, what
        return False
    for a, b in zip(one, other):
        assert a.dtype == b.dtype and a.shape == b.shape and _bits(a) == _bits(b), what
    return True


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
def test_native_calls_give_what_the_functions_give(device, dtype, monkeypatch):
    for name, (function, args, options) in _calls(device, dtype).items():
        counts = _Counts()
        assert not isinstance(_outcome(monkeypatch, counts, function, args, options), tuple), name
        assert counts.taken == 1, f"{name} goes through Python"
        for stream in (None, torch.cuda.Stream(), torch.cuda.current_stream().cuda_stream):
            torch.cuda.synchronize()
            assert _same_outcome(monkeypatch, function, args, {**options, "stream": stream}, (name, stream)), name


def test_calls_of_another_form_are_taken_or_refused_as_before(device, monkeypatch):
    """Each argument in turn is replaced by what does not belong there, or what only the Python functions know."""
    refused = taken = 0
    for name, (function, args, options) in _calls(device, torch.bfloat16).items():
        forms = []
        for i, a in enumerate(args):
            if isinstance(a, torch.Tensor):
                other = torch.float16 if a.dtype != torch.float16 else torch.bfloat16
                wide = torch.zeros(*a.shape[:-1], 2 * a.shape[-1], dtype=a.dtype, device=device)
                padded = torch.zeros(*a.shape[:-1], a.shape[-1] + 1, dtype=a.dtype, device=device)
                forms += [(i, x) for x in (None, 1.0, a.cpu(), a.to(other), a.to(torch.float64), wide[..., ::2], padded, padded[..., :-1], a[:0], a[None],
                                           a.reshape(-1), torch.nn.Parameter(a, requires_grad=False) if a.is_floating_point() else a)]
            elif isinstance(a, float):
                forms += [(i, x) for x in (0, 1, 0.0, -1.0, float("nan"), float("inf"), 1e300, "x")]
            elif isinstance(a, int):
                forms += [(i, x) for x in (0, 1, 5, 7, -1, 2**65, 6.0)]
        for i, value in forms:
            changed = [*args[:i], value, *args[i + 1:]]
            if _same_outcome(monkeypatch, function, changed, options, (name, i, value)):
                taken += 1
            else:
                refused += 1
        for stream in ("x", 1.5, object()):
            refused += not _same_outcome(monkeypatch, function, args, {**options, "stream": stream}, (name, stream))
    assert taken > 40 and refused > 400, (taken, refused)


@pytest.mark.parametrize("field,value", [("num_query_heads", 3), ("num_kv_heads", 0), ("head_dim", 64), ("head_dim", None), ("attention_scale", float("nan")),
                                         ("attention_scale", 1), ("attention_scale", 0.3), ("causal", 1), ("causal", False), ("query_position_offset", 1),
                                         ("query_position_offset", -1), ("num_kv_heads", True)])
def test_attention_options_of_another_form(device, monkeypatch, field, value):
    for name, (function, args, options) in _calls(device, torch.float16).items():
        if "attention" not in name:
            continue
        changed = ops.FlashAttentionOptions(4, 2, 32)
        setattr(changed, field, value)
        _same_outcome(monkeypatch, function, args, {**options, "options": changed}, (name, field, value))
