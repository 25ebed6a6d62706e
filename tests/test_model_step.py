"""The composed train step: the float64 composition is pinned by finite differences (CPU), then
the GPU step (eager and hipGraph replay, dense and cut loss) is compared with it."""
import numpy as np
import pytest
import torch

from oracle import model64
from tests.util import to_np

TINY = dict(vocab=50, layers=2, hidden=32, inter=48, hq=4, hkv=2, d=8, eps=1e-5)


def random_params(cfg, rng, scale=0.3):
    H, I, QW, KW = cfg["hidden"], cfg["inter"], cfg["hq"] * cfg["d"], cfg["hkv"] * cfg["d"]
    layers = []
    for _ in range(cfg["layers"]):
        layers.append({
            "attention_norm": 1 + 0.1 * rng.normal(size=H), "q": scale * rng.normal(size=(QW, H)),
            "k": scale * rng.normal(size=(KW, H)), "q_norm": 1 + 0.1 * rng.normal(size=cfg["d"]),
            "k_norm": 1 + 0.1 * rng.normal(size=cfg["d"]), "v": scale * rng.normal(size=(KW, H)),
            "o": scale * rng.normal(size=(H, QW)), "ffn_norm": 1 + 0.1 * rng.normal(size=H),
            "gate": scale * rng.normal(size=(I, H)), "up": scale * rng.normal(size=(I, H)),
            "down": scale * rng.normal(size=(H, I)),
        })
    return {"embedding": scale * rng.normal(size=(cfg["vocab"], H)), "final_norm": 1 + 0.1 * rng.normal(size=H),
            "layers": layers}


def test_float64_composition_matches_finite_differences():
    """Pins oracle/model64.py: its analytic gradients equal central differences of its own loss,
    for a sample of entries of every parameter tensor (incl. the tied embedding, which receives
    both the classifier and the lookup gradient)."""
    cfg = dict(TINY, layers=2)
    rng = np.random.default_rng(0)
    params = random_params(cfg, rng)
    tokens = rng.integers(0, cfg["vocab"], size=(2, 5))
    targets = rng.integers(0, cfg["vocab"], size=(2, 5))
    tokens[0, 1] = tokens[0, 3]  # a repeated id
    loss, grads, _ = model64.forward_backward(params, tokens, targets, cfg)
    assert np.isfinite(loss)

    def check(array, grad, name):
        flat = array.reshape(-1)
        for idx in rng.choice(flat.size, size=min(6, flat.size), replace=False):
            old = flat[idx]
            flat[idx] = old + 1e-6
            hi = model64.loss_only(params, tokens, targets, cfg)
            flat[idx] = old - 1e-6
            lo = model64.loss_only(params, tokens, targets, cfg)
            flat[idx] = old
            fd = (hi - lo) / 2e-6
            assert abs(fd - grad.reshape(-1)[idx]) <= 1e-6 + 1e-5 * abs(fd), (name, idx, fd, grad.reshape(-1)[idx])

    check(params["embedding"], grads["embedding"], "embedding")
    check(params["final_norm"], grads["final_norm"], "final_norm")
    for l, (w, g) in enumerate(zip(params["layers"], grads["layers"])):
        for key in model64.LAYER_KEYS:
            check(w[key], g[key], f"layer{l}.{key}")
    # the embedding row of a token that is used twice and is also a target gets all three contributions
    used = tokens[0, 1]
    assert np.abs(grads["embedding"][used]).max() > 0


# --------------------------------------------------------------------------------- GPU
def torch_round(dtype):
    def rnd(a):
        return torch.from_numpy(np.asarray(a, dtype=np.float64)).to(torch.float32).to(dtype).to(torch.float64).numpy()
    return rnd


def build(device, dtype, batch, seq, cfg, seed=3):
    from cgpt_amd.model import Model, ModelConfig

    config = ModelConfig(vocabulary_size=cfg["vocab"], num_layers=cfg["layers"], hidden_size=cfg["hidden"],
                         intermediate_size=cfg["inter"], num_query_heads=cfg["hq"], num_kv_heads=cfg["hkv"],
                         head_dim=cfg["d"], rotary_dim=cfg["d"], rms_epsilon=cfg["eps"], dtype=dtype)
    return Model(config, batch, seq, seed=seed, device=device)


def params_from_model(model, cfg):
    """Reads the library's (rounded) weights back as the float64 parameter structure."""
    H, I, QW, KW, D = cfg["hidden"], cfg["inter"], cfg["hq"] * cfg["d"], cfg["hkv"] * cfg["d"], cfg["d"]
    shapes = {"attention_norm": (H,), "q": (QW, H), "k": (KW, H), "q_norm": (D,), "k_norm": (D,), "v": (KW, H),
              "o": (H, QW), "ffn_norm": (H,), "gate": (I, H), "up": (I, H), "down": (H, I)}
    names = {"input_layernorm.weight": "attention_norm", "self_attn.q_proj.weight": "q",
             "self_attn.k_proj.weight": "k", "self_attn.q_norm.weight": "q_norm", "self_attn.k_norm.weight": "k_norm",
             "self_attn.v_proj.weight": "v", "self_attn.o_proj.weight": "o",
             "post_attention_layernorm.weight": "ffn_norm", "mlp.gate_proj.weight": "gate",
             "mlp.up_proj.weight": "up", "mlp.down_proj.weight": "down"}
    params = {"layers": [dict() for _ in range(cfg["layers"])]}
    grads = {"layers": [dict() for _ in range(cfg["layers"])]}
    for name, p, g in model.parameters():
        if name == "model.embed_tokens.weight":
            params["embedding"], grads["embedding"] = to_np(p).reshape(cfg["vocab"], H), g
        elif name == "model.norm.weight":
            params["final_norm"], grads["final_norm"] = to_np(p), g
        else:
            _, _, layer, rest = name.split(".", 3)
            key = names[rest]
            params["layers"][int(layer)][key] = to_np(p).reshape(shapes[key])
            grads["layers"][int(layer)][key] = g
    return params, grads


def compare_gradients(got, want, tol, loss_scale):
    worst = [0.0, ""]

    def one(g, w, name):
        w = np.asarray(w).reshape(-1)
        scale = max(np.abs(w).max(), 1e-3 * loss_scale)
        got_flat = to_np(g).reshape(-1)
        err = np.abs(got_flat - w).max() / scale
        assert np.isfinite(got_flat).all(), name
        if err > worst[0]:
            worst[:] = [err, name]
        assert err <= tol, f"{name}: error {err:.3e} of the tensor's scale"
    one(got["embedding"], want["embedding"], "embedding")
    one(got["final_norm"], want["final_norm"], "final_norm")
    for l, (g, w) in enumerate(zip(got["layers"], want["layers"])):
        for key in model64.LAYER_KEYS:
            one(g[key], w[key], f"layer{l}.{key}")
    print(f"[parity] composed step: worst gradient error {worst[0]:.3e} of its tensor's scale ({worst[1]}; bound {tol:.1e})")


MODEL_CFG = dict(vocab=96, layers=2, hidden=64, inter=128, hq=2, hkv=1, d=32, eps=1e-5)


# Heads of 128 with 256-wide q and k/v projections, 64 rows: the shape class in which the step runs the
# q/k/v projections as one contraction over segmented operands and attention on its head_dim-128 kernels.
WIDE_CFG = dict(vocab=96, layers=1, hidden=256, inter=128, hq=2, hkv=2, d=128, eps=1e-5)


# Three layers with tile-aligned projections (256-wide q, k, v, hidden and [gate | up]) and 64 rows: the shape class in
# which the projections' weight gradients of all layers run as four launches at the end of the backward pass.
STACKED_CFG = dict(vocab=96, layers=3, hidden=256, inter=128, hq=2, hkv=2, d=128, eps=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
@pytest.mark.parametrize("loss_mode", [0, 1], ids=["dense", "cut"])
@pytest.mark.parametrize("shape", [(MODEL_CFG, 2, 24), (WIDE_CFG, 2, 32), (STACKED_CFG, 2, 32)],
                         ids=["heads32", "heads128-fused-qkv", "stacked-weight-gradients"])
def test_gpu_step_matches_float64_composition(device, dtype, loss_mode, shape):
    """Hidden 64, 2:1 heads of 32, T=24, B=2, two layers (and the wide-head variant above): every parameter
    gradient of the GPU step against the float64 composition that rounds each operator output to the storage
    dtype where the GPU stores it.
    Tolerance: 3e-2 of each tensor's largest gradient entry (the operators' own bar is 2e-2, and a gradient here has
    passed through several of them; the observed worst is printed)."""
    cfg, batch, seq = shape
    loss_scale = 64.0
    model = build(device, dtype, batch, seq, cfg)
    rng = np.random.default_rng(5)
    tokens = rng.integers(0, cfg["vocab"], size=(batch, seq))
    targets = rng.integers(0, cfg["vocab"], size=(batch, seq))
    tokens[1, 2] = tokens[1, 7]
    model.set_tokens(tokens, targets)
    model.forward_backward(loss_scale, loss_mode, use_graph=False)
    loss, _, _ = model.status()
    params, grads = params_from_model(model, cfg)
    want_loss, want, saved = model64.forward_backward(params, tokens, targets, cfg, loss_scale, torch_round(dtype))
    assert abs(loss - want_loss) <= 2e-2 * want_loss
    for l in range(cfg["layers"] + 1):
        hidden = to_np(model.activation(f"hidden.{l}")).reshape(batch * seq, cfg["hidden"])
        assert np.abs(hidden - saved["hidden"][l]).max() <= 4e-2 * max(1.0, np.abs(saved["hidden"][l]).max())
    compare_gradients(grads, want, 3e-2, loss_scale)
    model.close()


@pytest.mark.gpu
@pytest.mark.parametrize("seed", range(16))
def test_gpu_step_matches_float64_composition_on_random_configurations(device, seed):
    """Seeded random small models — 1 to 3 layers, 1 to 4 kv-heads with groups of 1 to 4, heads of 16 to 128, odd
    feed-forward widths, every storage dtype, both loss paths, eager and recorded — against the float64 composition:
    the shape classes in which the step falls back from its fused launches to the separate operators are exactly
    the ones fixed shape lists tend to miss."""
    rng = np.random.default_rng(700 + seed)
    dtype = [torch.bfloat16, torch.float16, torch.float32][int(rng.integers(0, 3))]
    hkv = int(rng.integers(1, 5))
    hq = hkv * int(rng.integers(1, 5))
    d = [16, 32, 64, 128][int(rng.integers(0, 4))]
    if hq * d > 1024:
        d = 32
    cfg = dict(vocab=int(rng.integers(40, 300)), layers=int(rng.integers(1, 4)), hidden=hq * d,
               inter=int(rng.integers(1, 40)) * 8 if rng.integers(0, 2) else int(rng.integers(8, 300)), hq=hq, hkv=hkv, d=d,
               eps=1e-5)
    batch, seq = int(rng.integers(1, 4)), int(rng.integers(2, 70))
    loss_mode, use_graph = int(rng.integers(0, 2)), bool(rng.integers(0, 2))
    loss_scale = 64.0
    print(f"model {cfg} batch={batch} seq={seq} loss_mode={loss_mode} graph={use_graph} {dtype}", flush=True)
    model = build(device, dtype, batch, seq, cfg, seed=seed)
    tokens = rng.integers(0, cfg["vocab"], size=(batch, seq))
    targets = rng.integers(0, cfg["vocab"], size=(batch, seq))
    model.set_tokens(tokens, targets)
    stream = torch.cuda.Stream(device=device)
    for _ in range(2 if use_graph else 1):  # the second call replays the recorded step
        model.forward_backward(loss_scale, loss_mode, use_graph=use_graph, stream=stream)
    loss, _, _ = model.status(stream)
    params, grads = params_from_model(model, cfg)
    want_loss, want, saved = model64.forward_backward(params, tokens, targets, cfg, loss_scale, torch_round(dtype))
    sixteen = dtype != torch.float32
    assert abs(loss - want_loss) <= (2e-2 if sixteen else 1e-4) * want_loss
    for l in range(cfg["layers"] + 1):
        hidden = to_np(model.activation(f"hidden.{l}")).reshape(batch * seq, cfg["hidden"])
        assert np.abs(hidden - saved["hidden"][l]).max() <= (4e-2 if sixteen else 1e-4) * max(1.0, np.abs(saved["hidden"][l]).max())
    compare_gradients(grads, want, 3e-2 if sixteen else 1e-3, loss_scale)
    model.close()


@pytest.mark.gpu
def test_graph_replay_equals_eager_and_losses_agree_between_modes(device):
    cfg = MODEL_CFG
    dtype = torch.bfloat16
    batch, seq = 2, 40
    rng = np.random.default_rng(6)
    tokens = rng.integers(0, cfg["vocab"], size=(batch, seq))
    targets = rng.integers(0, cfg["vocab"], size=(batch, seq))
    stream = torch.cuda.Stream(device=device)
    results = {}
    for mode in (0, 1):
        model = build(device, dtype, batch, seq, cfg)
        model.set_tokens(tokens, targets)
        model.forward_backward(1024.0, mode, use_graph=False, stream=stream)
        loss_eager = model.status(stream)[0]
        eager = [g.clone() for _, _, g in model.parameters()]
        model.forward_backward(1024.0, mode, use_graph=True, stream=stream)   # eager run + capture
        for replay in range(3):
            for _, _, g in model.parameters():
                g.zero_()
            torch.cuda.synchronize()
            model.forward_backward(1024.0, mode, use_graph=True, stream=stream)  # replay
            loss_graph = model.status(stream)[0]
            assert loss_graph == loss_eager
            for (name, _, g), e in zip(model.parameters(), eager):
                assert torch.equal(g, e), f"{name} differs on replay {replay}"
        results[mode] = (loss_eager, eager)
        model.close()
    assert abs(results[0][0] - results[1][0]) <= 1e-3 * results[0][0]
    for a, b in zip(results[0][1], results[1][1]):
        scale = max(float(a.float().abs().max()), 1e-3)
        assert float((a.float() - b.float()).abs().max()) <= 3e-2 * scale


@pytest.mark.gpu
def test_train_steps_reduce_the_loss_and_count_steps(device):
    cfg = MODEL_CFG
    from cgpt_amd.ops import AdamWOptions

    model = build(device, torch.bfloat16, 4, 32, cfg)
    rng = np.random.default_rng(7)
    tokens = rng.integers(0, cfg["vocab"], size=(4, 32))
    model.set_tokens(tokens, np.roll(tokens, -1, axis=1))
    options = AdamWOptions(learning_rate=1e-2, beta1=0.9, beta2=0.95, weight_decay=0.1, loss_scale=1024.0,
                           max_grad_norm=1.0)
    stream = torch.cuda.Stream(device=device)
    losses = []
    for _ in range(30):
        model.train_step(options, loss_mode=1, use_graph=True, stream=stream)
        losses.append(model.status(stream))
    assert all(finite for _, finite, _ in losses)
    assert losses[-1][2] == 30
    assert losses[-1][0] < 0.5 * losses[0][0]
    assert abs(losses[0][0] - np.log(cfg["vocab"])) < 0.5   # random init: loss starts near ln(vocab)
    model.close()


@pytest.mark.gpu
def test_recorded_train_step_follows_a_changing_learning_rate_and_skips_like_the_eager_one(device):
    """With use_graph the AdamW update is part of the recorded step and reads its options on the device. Two models
    from one seed take the same eight steps, one eagerly and one from the recording, with a learning rate, weight
    decay and clipping norm that change every step and one step whose gradients are made non-finite (both must skip
    it and count it): parameters, master copies and moments agree bit for bit after every step."""
    cfg = MODEL_CFG
    from cgpt_amd.ops import AdamWOptions

    batch, seq = 2, 24
    rng = np.random.default_rng(17)
    tokens = rng.integers(0, cfg["vocab"], size=(batch, seq))
    targets = rng.integers(0, cfg["vocab"], size=(batch, seq))
    stream = torch.cuda.Stream(device=device)
    models = [build(device, torch.bfloat16, batch, seq, cfg, seed=3) for _ in range(2)]
    for model in models:
        model.set_tokens(tokens, targets)
    saved = None
    for step in range(8):
        options = AdamWOptions(learning_rate=1e-2 / (1 + step), beta1=0.9, beta2=0.95, weight_decay=0.1 * (step % 3),
                               loss_scale=256.0, max_grad_norm=[1.0, float("inf"), 0.5][step % 3])
        if step == 4:  # a weight that overflows the forward pass: every gradient becomes non-finite
            saved = [models[i].parameters()[1][1].clone() for i in range(2)]
            for model in models:
                model.parameters()[1][1].fill_(float("inf"))
            torch.cuda.synchronize()
        for use_graph, model in zip((False, True), models):
            model.train_step(options, loss_mode=1, use_graph=use_graph, stream=stream)
        states = [model.status(stream) for model in models]
        assert states[0][1:] == states[1][1:], f"step {step}: {states}"
        assert states[0][1] == (step != 4), f"step {step}: finite flag {states[0][1]}"
        if step == 4:
            for i, model in enumerate(models):
                model.parameters()[1][1].copy_(saved[i])
            torch.cuda.synchronize()
        for index, ((name, p0, _), (_, p1, _)) in enumerate(zip(models[0].parameters(), models[1].parameters())):
            assert torch.equal(p0, p1), f"step {step}: {name} differs between the eager and the recorded step"
            for a, b in zip(models[0].optimizer_state(index), models[1].optimizer_state(index)):
                assert torch.equal(a, b), f"step {step}: optimizer state of {name} differs"
    assert models[0].status(stream)[2] == 7  # eight calls, one skipped
    for model in models:
        model.close()


@pytest.mark.gpu
def test_model_argument_errors(device):
    from cgpt_amd.model import Model, ModelConfig

    with pytest.raises(ValueError):
        Model(ModelConfig(num_query_heads=8, num_kv_heads=3), 1, 8, device=device)
    with pytest.raises(ValueError):
        Model(ModelConfig(hidden_size=1000), 1, 8, device=device)
    model = build(device, torch.bfloat16, 1, 8, MODEL_CFG)
    with pytest.raises(ValueError):
        model.forward_backward(0.0, 1)
    with pytest.raises(ValueError):
        model.forward_backward(1.0, 1, use_graph=True, stream=0)   # capture needs a real stream
    model.close()


def test_cpu_float32_step_matches_float64_composition():
    """oracle/cpu_model.py (the CPU baseline that bench.py times) against oracle/model64.py on a tiny model."""
    from oracle import cpu_model

    cfg = dict(TINY)
    w = cpu_model.make_weights(cfg, seed=1)
    for lw in w["layers"]:
        for key in lw:
            if lw[key].dim() == 2:
                lw[key].mul_(10.0)   # make the gradients large enough to compare
    w["embedding"].mul_(10.0)
    g = torch.Generator().manual_seed(2)
    tokens = torch.randint(0, cfg["vocab"], (2, 6), generator=g)
    targets = torch.randint(0, cfg["vocab"], (2, 6), generator=g)
    params = {"embedding": to_np(w["embedding"]), "final_norm": to_np(w["final_norm"]),
              "layers": [{k: to_np(v) for k, v in lw.items()} for lw in w["layers"]]}
    loss, grads = cpu_model.train_step(w, tokens, targets, cfg, 8.0)
    want_loss, want, _ = model64.forward_backward(params, tokens.numpy(), targets.numpy(), cfg, 8.0)
    assert abs(loss - want_loss) <= 1e-5 * want_loss
    compare_gradients(grads, want, 1e-4, 8.0)


@pytest.mark.gpu
@pytest.mark.parametrize("head_dim,rotary_dim,kv_heads,seq,dtype", [
    (64, 32, 2, 48, torch.bfloat16),     # the general row kernel, part of the head rotated
    (128, 128, 2, 48, torch.bfloat16),   # the kernel for head_dim 128; a group of four k rows spans two tokens
    (128, 128, 1, 333, torch.float16),   # the same with one kv head (four tokens per group), several trips per wavefront
    (128, 128, 4, 47, torch.bfloat16),   # 2 * 47 * 4 = 376 k rows and as many q rows per head group
], ids=["d64-r32", "d128-kv2", "d128-kv1-f16", "d128-kv4"])
def test_fused_qk_norm_rope_is_bit_identical_to_the_separate_operators(device, monkeypatch, head_dim, rotary_dim,
                                                                      kv_heads, seq, dtype):
    """Per-head RMSNorm + rotary embedding run as one pass (forward and backward) when head_dim is
    served by the row kernels; the pass keeps the separate operators' intermediate roundings, so a whole
    step gives the same bits either way. CGPTX_FUSE_QK=0 selects the separate operators."""
    from cgpt_amd.model import LOSS_DENSE, Model, ModelConfig
    config = ModelConfig(vocabulary_size=128, num_layers=2, hidden_size=4 * head_dim, intermediate_size=256,
                         num_query_heads=4, num_kv_heads=kv_heads, head_dim=head_dim, rotary_dim=rotary_dim, dtype=dtype)
    rng = np.random.default_rng(3)
    inputs = rng.integers(0, 128, size=2 * seq).astype(np.uint32)
    targets = rng.integers(0, 128, size=2 * seq).astype(np.uint32)
    results = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("CGPTX_FUSE_QK", fuse)
        model = Model(config, 2, seq, seed=4, device=device)
        model.set_tokens(inputs, targets)
        model.forward_backward(loss_scale=4.0, loss_mode=LOSS_DENSE)
        loss = model.status()[0]
        results.append((loss, [g.clone() for _, _, g in model.parameters()], model.activation("hidden.2").clone()))
    assert results[0][0] == results[1][0]
    assert torch.equal(results[0][2], results[1][2])
    for a, b in zip(results[0][1], results[1][1]):
        assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("head_dim,kv_heads", [(128, 3), (64, 1), (128, 6)], ids=["ragged-split", "general", "equal"])
def test_fused_qk_norm_rope_of_more_rows_than_the_chip_holds(device, monkeypatch, head_dim, kv_heads):
    """More rows than the chip holds at once: the separate norm, which fits more workgroups on it than the fused pass, groups the
    additions of the two norms' weight gradients otherwise. All else is that of the separate operators, bit for bit; those are fp32
    sums over up to 72000 rows, one rounding to bf16 (2^-9), beside sums of rounded terms whose error grows with the gradient's
    largest element."""
    from cgpt_amd.model import LOSS_DENSE, Model, ModelConfig
    config = ModelConfig(vocabulary_size=64, num_layers=1, hidden_size=6 * head_dim, intermediate_size=64, num_query_heads=6,
                         num_kv_heads=kv_heads, head_dim=head_dim, rotary_dim=head_dim, dtype=torch.bfloat16)
    batch, seq = 60, 200
    rng = np.random.default_rng(3)
    inputs, targets = (rng.integers(0, 64, size=batch * seq).astype(np.uint32) for _ in range(2))
    results = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("CGPTX_FUSE_QK", fuse)
        model = Model(config, batch, seq, seed=4, device=device)
        model.set_tokens(inputs, targets)
        model.forward_backward(loss_scale=4.0, loss_mode=LOSS_DENSE)
        results.append((model.status()[0], [(name, g.clone()) for name, _, g in model.parameters()]))
    assert results[0][0] == results[1][0]
    for (name, a), (_, b) in zip(results[0][1], results[1][1]):
        if "q_norm" in name or "k_norm" in name:
            a, b = a.float(), b.float()
            assert (a - b).abs().max() <= 2.0 ** -8 * b.abs().max()
        else:
            assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("kv_heads,rotary_dim", [(3, 64), (1, 64), (6, 32)], ids=["dense", "few-k-rows", "partly-rotated"])
def test_fused_qk_norm_rope_in_fp32_adds_as_the_separate_operators_do(device, monkeypatch, kv_heads, rotary_dim):
    """More rows than the chip holds at once, in fp32 storage, where no rounding hides another order of additions: q's and k's
    workgroups leave the partial sums of the weight gradients that launches of their own leave, so all gradients are
    bit-identical. (In 16-bit storage the separate norm fits more workgroups on a compute unit than the fused one.)"""
    from cgpt_amd.model import LOSS_DENSE, Model, ModelConfig
    config = ModelConfig(vocabulary_size=64, num_layers=1, hidden_size=6 * 64, intermediate_size=64, num_query_heads=6,
                         num_kv_heads=kv_heads, head_dim=64, rotary_dim=rotary_dim, dtype=torch.float32)
    batch, seq = 60, 200
    rng = np.random.default_rng(3)
    inputs, targets = (rng.integers(0, 64, size=batch * seq).astype(np.uint32) for _ in range(2))
    results = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("CGPTX_FUSE_QK", fuse)
        model = Model(config, batch, seq, seed=4, device=device)
        model.set_tokens(inputs, targets)
        model.forward_backward(loss_scale=4.0, loss_mode=LOSS_DENSE)
        results.append([(name, g.clone()) for name, _, g in model.parameters()])
    for (name, a), (_, b) in zip(*results):
        assert torch.equal(a, b), name


@pytest.mark.gpu
def test_norm_weight_gradients_reduced_at_the_end_of_the_backward_pass_are_bit_identical(device, monkeypatch):
    """The norm-backward passes of a step leave the reduction of their weight-gradient partial sums to one pair of
    launches at the end of the backward pass (same additions, same order); CGPTX_FUSE_DGAMMA=0 reduces after each
    pass. Eager passes (the first sizes the memory for the partial sums and still reduces at once, the later ones
    defer) and graph replays all give the same bits, with the block norms fused and separate."""
    from cgpt_amd.model import LOSS_CUT, Model, ModelConfig
    config = ModelConfig(vocabulary_size=512, num_layers=3, hidden_size=1024, intermediate_size=512, num_query_heads=8,
                         num_kv_heads=2, head_dim=128, rotary_dim=128, dtype=torch.bfloat16)
    batch, seq = 4, 512
    rng = np.random.default_rng(5)
    inputs = rng.integers(0, 512, size=batch * seq).astype(np.uint32)
    targets = rng.integers(0, 512, size=batch * seq).astype(np.uint32)
    stream = torch.cuda.Stream(device=device)

    def gradients(model):
        stream.synchronize()
        return [g.clone() for _, _, g in model.parameters()]

    for norms in ("1", "0"):
        monkeypatch.setenv("CGPTX_FUSE_NORMS", norms)
        monkeypatch.setenv("CGPTX_FUSE_DGAMMA", "0")
        model = Model(config, batch, seq, seed=6, device=device)
        model.set_tokens(inputs, targets)
        model.forward_backward(8.0, LOSS_CUT, use_graph=False, stream=stream)
        want = gradients(model)
        model.close()
        monkeypatch.setenv("CGPTX_FUSE_DGAMMA", "1")
        model = Model(config, batch, seq, seed=6, device=device)
        model.set_tokens(inputs, targets)
        for use_graph in (False, False, True, True, True, False):
            for _, _, g in model.parameters():
                g.zero_()
            torch.cuda.synchronize()
            model.forward_backward(8.0, LOSS_CUT, use_graph=use_graph, stream=stream)
            for (name, _, _), a, b in zip(model.parameters(), gradients(model), want):
                assert torch.equal(a, b), f"{name} (block norms fused: {norms}, graph: {use_graph})"
        model.close()


@pytest.mark.gpu
@pytest.mark.parametrize("batch,seq,together", [(3, 100, True), (16, 1024, False)], ids=["small", "large"])
def test_profile_times_the_launches_of_the_step(device, batch, seq, together):
    """The profiled pass makes the launches of every other pass, so it gives the same bits, and its labels tell what they were:
    a small model's gradients share launches, a large one's have their own."""
    from cgpt_amd.model import LOSS_CUT, Model, ModelConfig
    config = ModelConfig(vocabulary_size=503, num_layers=2, hidden_size=256, intermediate_size=704, num_query_heads=4,
                         num_kv_heads=2, head_dim=64, rotary_dim=64, dtype=torch.float16)
    rng = np.random.default_rng(5)
    inputs, targets = (rng.integers(0, 503, size=batch * seq).astype(np.uint32) for _ in range(2))
    model = Model(config, batch, seq, seed=6, device=device)
    model.set_tokens(inputs, targets)
    model.forward_backward(loss_scale=64.0, loss_mode=LOSS_CUT)
    torch.cuda.synchronize()
    want = [g.clone() for _, _, g in model.parameters()]
    labels = model.profile(64.0, LOSS_CUT)
    for (name, _, got), expected in zip(model.parameters(), want):
        assert torch.equal(got, expected), name
    assert all(ms > 0 for ms in labels.values())
    for projection in ("gate_up", "o", "qkv"):
        assert (f"gemm_dx_dw.{projection}" in labels) == together, labels
        assert (f"gemm_dx.{projection}" in labels) != together and (f"gemm_dw.{projection}" in labels) != together, labels
    model.close()


@pytest.mark.gpu
def test_swiglu_in_the_projection_epilogues_is_bit_identical_to_the_separate_operators(device, monkeypatch):
    """The SwiGLU product rides in the gate/up projection's epilogue and its gradient in the epilogue of the
    down projection's input gradient when the shapes fill the chip (here 4096 rows x 3328 feed-forward
    columns); both work from the rounded 16-bit values the separate operators would exchange, so a whole
    step gives the same bits either way. CGPTX_FUSE_SWIGLU=0 selects the separate operators."""
    from cgpt_amd.model import LOSS_DENSE, Model, ModelConfig
    config = ModelConfig(vocabulary_size=128, num_layers=2, hidden_size=256, intermediate_size=3328, num_query_heads=4,
                         num_kv_heads=2, head_dim=64, rotary_dim=64, dtype=torch.bfloat16)
    rng = np.random.default_rng(5)
    inputs = rng.integers(0, 128, size=4 * 1024).astype(np.uint32)
    targets = rng.integers(0, 128, size=4 * 1024).astype(np.uint32)
    results = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("CGPTX_FUSE_SWIGLU", fuse)
        model = Model(config, 4, 1024, seed=6, device=device)
        model.set_tokens(inputs, targets)
        model.forward_backward(loss_scale=4.0, loss_mode=LOSS_DENSE)
        loss = model.status()[0]
        results.append((loss, [g.clone() for _, _, g in model.parameters()], model.activation("hidden.2").clone()))
    assert np.isfinite(results[0][0]) and results[0][0] == results[1][0]
    assert torch.equal(results[0][2], results[1][2])
    for a, b in zip(results[0][1], results[1][1]):
        assert torch.equal(a, b)


@pytest.mark.gpu
def test_block_norms_in_one_pass_match_the_separate_operators(device, monkeypatch):
    """The attention and feed-forward norms of a block read the same input and run as one pass: forward
    bit-identical; backward adds the two branch gradients before the one rounding instead of rounding
    after each, so gradients agree to storage precision, not bit for bit. CGPTX_FUSE_NORMS=0 selects
    the separate operators."""
    from cgpt_amd.model import LOSS_DENSE, Model, ModelConfig
    config = ModelConfig(vocabulary_size=128, num_layers=2, hidden_size=256, intermediate_size=256, num_query_heads=4,
                         num_kv_heads=2, head_dim=64, rotary_dim=64, dtype=torch.bfloat16)
    rng = np.random.default_rng(5)
    inputs = rng.integers(0, 128, size=2 * 40).astype(np.uint32)
    targets = rng.integers(0, 128, size=2 * 40).astype(np.uint32)
    results = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("CGPTX_FUSE_NORMS", fuse)
        model = Model(config, 2, 40, seed=6, device=device)
        model.set_tokens(inputs, targets)
        model.forward_backward(loss_scale=4.0, loss_mode=LOSS_DENSE)
        loss = model.status()[0]
        results.append((loss, {n: g.float().cpu() for n, _, g in model.parameters()}, model.activation("hidden.2").clone()))
    assert results[0][0] == results[1][0]
    assert torch.equal(results[0][2], results[1][2])
    for name, fused in results[0][1].items():
        separate = results[1][1][name]
        scale = separate.abs().max().item() + 1e-12
        assert (fused - separate).abs().max().item() <= 2e-2 * scale, name


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16], ids=["bf16", "f16"])
def test_weight_gradients_of_all_layers_in_one_launch_agree_with_the_launches_per_layer(device, monkeypatch, dtype):
    """Tile-aligned models leave the projections' weight gradients to the end of the backward pass and compute
    them for all layers at once (CGPTX_STACK_DW=0 keeps one launch per layer and projection). Nothing else
    changes: loss, activations and every other gradient are bit-identical; the projections' weight gradients are
    the same sums over the rows taken in a different number of slices, equal to storage precision; eager and
    recorded passes of the stacked step give the same bits."""
    from cgpt_amd.model import LOSS_CUT, Model, ModelConfig
    config = ModelConfig(vocabulary_size=256, num_layers=4, hidden_size=512, intermediate_size=256, num_query_heads=4,
                         num_kv_heads=2, head_dim=128, rotary_dim=128, dtype=dtype)
    batch, seq = 2, 96
    rng = np.random.default_rng(9)
    inputs = rng.integers(0, 256, size=batch * seq).astype(np.uint32)
    targets = rng.integers(0, 256, size=batch * seq).astype(np.uint32)
    results = {}
    stream = torch.cuda.Stream(device=device)
    for stack in ("1", "0"):
        monkeypatch.setenv("CGPTX_STACK_DW", stack)
        model = Model(config, batch, seq, seed=8, device=device)
        model.set_tokens(inputs, targets)
        model.forward_backward(16.0, LOSS_CUT, use_graph=False, stream=stream)
        stream.synchronize()
        eager = {n: g.clone() for n, _, g in model.parameters()}
        for use_graph in (True, True):
            for _, _, g in model.parameters():
                g.zero_()
            torch.cuda.synchronize()
            model.forward_backward(16.0, LOSS_CUT, use_graph=use_graph, stream=stream)
            stream.synchronize()
            for n, _, g in model.parameters():
                assert torch.equal(g, eager[n]), f"{n}: recorded pass differs from the eager one (stack={stack})"
        results[stack] = (model.status(stream)[0], eager, model.activation(f"hidden.{config.num_layers}").clone())
        model.close()
    assert results["1"][0] == results["0"][0]
    assert torch.equal(results["1"][2], results["0"][2])
    projections = ("q_proj", "k_proj", "v_proj", "o_proj", "gate_proj", "up_proj", "down_proj")
    seen = 0
    for name, stacked in results["1"][1].items():
        separate = results["0"][1][name]
        if any(part in name for part in projections):
            seen += 1
            scale = separate.float().abs().max().item() + 1e-12
            assert (stacked.float() - separate.float()).abs().max().item() <= 1e-2 * scale, name
        else:
            assert torch.equal(stacked, separate), name
    assert seen == 7 * config.num_layers


HEADLINE = dict(vocabulary_size=32000, num_layers=8, hidden_size=1024, intermediate_size=2048, num_query_heads=8,
                num_kv_heads=2, head_dim=128, rotary_dim=128)
HEADLINE_CFG = dict(vocab=32000, layers=8, hidden=1024, inter=2048, hq=8, hkv=2, d=128, eps=1e-5)


# The 12-layer, 768-wide decoder with 12:4 heads of 64 that is named beside the preset as the 104m shape.
SECONDARY = dict(vocabulary_size=32000, num_layers=12, hidden_size=768, intermediate_size=2048, num_query_heads=12,
                 num_kv_heads=4, head_dim=64, rotary_dim=64)


@pytest.mark.gpu
@pytest.mark.parametrize("dims,batch,seq", [(HEADLINE, 32, 1024), (HEADLINE, 8, 4096), (SECONDARY, 32, 1024)],
                         ids=["b32-t1024", "long-context-b8-t4096", "12x768-b32-t1024"])
def test_headline_configuration_scales_exactly_replays_exactly_and_starts_at_the_closed_form_loss(device, dims, batch, seq):
    """The 104m preset at the benchmark's sizes (B=32, T=1024 and the long-context variant B=8, T=4096, bf16) and the
    12 x 768 shape at B=32, T=1024, where no CPU composition finishes in test time: properties that hold at any size.
    The backward pass is linear in the loss scale, and a factor of two is exact in binary floating point, so every
    gradient at scale 2048 is exactly twice the one at 1024; a hipGraph replay repeats the eager pass bit for bit; the
    two loss paths agree; a random-init model starts at the closed-form loss of Gaussian logits."""
    from cgpt_amd.model import LOSS_CUT, LOSS_DENSE, Model, ModelConfig

    config = ModelConfig(dtype=torch.bfloat16, **dims)
    model = Model(config, batch, seq, seed=0, device=device)
    assert model.num_parameters == (104_090_624 if dims is HEADLINE else 100_094_208)
    rng = np.random.default_rng(0)
    model.set_tokens(rng.integers(0, 32000, size=(batch, seq)), rng.integers(0, 32000, size=(batch, seq)))
    stream = torch.cuda.Stream(device=device)

    model.forward_backward(1024.0, LOSS_CUT, use_graph=False, stream=stream)
    loss, _, _ = model.status(stream)
    # Rows leave the final norm with unit RMS and the tied classifier is N(0, 0.02^2): logits are close to
    # N(0, H * 0.02^2) and independent of the target, so E[loss] = ln V + variance / 2.
    assert abs(loss - (np.log(32000.0) + 0.5 * dims["hidden_size"] * 0.02 ** 2)) < 0.02
    base = [g.clone() for _, _, g in model.parameters()]
    for (name, _, _), g in zip(model.parameters(), base):
        assert bool(torch.isfinite(g.float()).all()), name
        assert float(g.float().abs().max()) > 0.0, name

    model.forward_backward(2048.0, LOSS_CUT, use_graph=False, stream=stream)
    assert model.status(stream)[0] == loss
    for (name, _, g), b in zip(model.parameters(), base):
        assert torch.equal(g.float(), 2.0 * b.float()), f"{name}: not exactly twice the gradient at half the scale"

    model.forward_backward(1024.0, LOSS_CUT, use_graph=True, stream=stream)  # eager pass + capture
    for replay in range(2):
        for _, _, g in model.parameters():
            g.zero_()
        torch.cuda.synchronize()
        model.forward_backward(1024.0, LOSS_CUT, use_graph=True, stream=stream)
        assert model.status(stream)[0] == loss
        for (name, _, g), b in zip(model.parameters(), base):
            assert torch.equal(g, b), f"{name} differs on replay {replay}"

    model.forward_backward(1024.0, LOSS_DENSE, use_graph=False, stream=stream)
    assert abs(model.status(stream)[0] - loss) <= 1e-4 * loss
    for (name, _, g), b in zip(model.parameters(), base):
        scale = max(float(b.float().abs().max()), 1e-6)
        assert float((g.float() - b.float()).abs().max()) <= 3e-2 * scale, name
    model.close()


@pytest.mark.gpu
def test_adamw_over_all_104m_parameters_matches_the_float64_update(device):
    """Two full train steps of the 104m preset at B=32, T=1024 (hipGraph step + adamw_step_many_async over the 90
    tensors / 104,090,624 parameters: src/optim/adamw.cu:276-346). After each step the master copies, both
    moments and the 16-bit parameters of every tensor are compared with the float64 update
    (oracle64.adamw: unscale by the loss scale, one global norm over all tensors, clip to 1, bias correction)
    applied to the gradients the step left on the device."""
    from cgpt_amd.model import LOSS_CUT, Model, ModelConfig
    from cgpt_amd.ops import AdamWOptions
    from oracle import oracle64

    batch, seq = 32, 1024
    model = Model(ModelConfig(dtype=torch.bfloat16, **HEADLINE), batch, seq, seed=0, device=device)
    rng = np.random.default_rng(1)
    model.set_tokens(rng.integers(0, 32000, size=(batch, seq)), rng.integers(0, 32000, size=(batch, seq)))
    stream = torch.cuda.Stream(device=device)
    opt = dict(lr=3e-4, beta1=0.9, beta2=0.95, eps=1e-8, wd=0.1, loss_scale=1024.0, max_grad_norm=1.0)
    options = AdamWOptions(learning_rate=opt["lr"], beta1=opt["beta1"], beta2=opt["beta2"], epsilon=opt["eps"],
                           weight_decay=opt["wd"], loss_scale=opt["loss_scale"], max_grad_norm=opt["max_grad_norm"])
    tensors = model.parameters()
    assert len(tensors) == 90 and sum(p.numel() for _, p, _ in tensors) == 104_090_624
    state = [tuple(to_np(t) for t in model.optimizer_state(i)) for i in range(len(tensors))]
    for (name, p, _), (master, m, v) in zip(tensors, state):   # masters start as the 16-bit parameters, moments at 0
        assert np.array_equal(master, to_np(p)), name
        assert not m.any() and not v.any(), name
    step = 0
    eps32 = float(np.finfo(np.float32).eps)
    for _ in range(2):
        model.train_step(options, LOSS_CUT, use_graph=True, stream=stream)
        loss, finite, steps = model.status(stream)
        grads = [to_np(g) for _, _, g in tensors]
        norm = np.sqrt(sum(((g / opt["loss_scale"]) ** 2).sum() for g in grads))
        applied, masters, ms, vs, step = oracle64.adamw(
            None, grads, [s[0] for s in state], [s[1] for s in state], [s[2] for s in state], step, opt["lr"],
            opt["beta1"], opt["beta2"], opt["eps"], opt["wd"], opt["loss_scale"], opt["max_grad_norm"])
        assert applied and finite and steps == step, (loss, finite, steps)
        print(f"[parity] AdamW step {step}: loss {loss:.4f}, unscaled gradient norm {norm:.4f} "
              f"({'clipped' if norm > opt['max_grad_norm'] else 'not clipped'})")
        worst = dict(master=0.0, m=0.0, v=0.0)
        for i, (name, p, _) in enumerate(tensors):
            got_master, got_m, got_v = (to_np(t) for t in model.optimizer_state(i))
            # master: the update is lr-sized on parameters up to 1 (norm weights): a thousandth of lr plus the
            # fp32 representation of the value itself
            bound = 1e-3 * opt["lr"] + 2 * eps32 * np.abs(masters[i])
            err = np.abs(got_master - masters[i])
            assert (err <= bound).all(), f"{name}: master differs by {err.max():.3e}"
            worst["master"] = max(worst["master"], float(err.max()))
            for key, got, want in (("m", got_m, ms[i]), ("v", got_v, vs[i])):
                scale = max(float(np.abs(want).max()), 1e-30)
                rel = float(np.abs(got - want).max()) / scale
                assert rel <= 2e-5, f"{name}: {key} differs by {rel:.3e} of its largest entry"
                worst[key] = max(worst[key], rel)
            # the 16-bit parameter is the master copy rounded to nearest even
            assert torch.equal(p, model.optimizer_state(i)[0].to(torch.bfloat16)), name
            state[i] = (got_master, got_m, got_v)   # the next step starts from what the device holds
        print(f"[parity] AdamW step {step}: worst master error {worst['master']:.3e} (lr {opt['lr']:.0e}), "
              f"worst m {worst['m']:.3e}, v {worst['v']:.3e} of the tensor's largest entry")
    model.close()


def cpu_weights_from_model(model, cfg):
    """The library's weights as the float32 tensors oracle/cpu_model.py takes."""
    params, _ = params_from_model(model, cfg)
    as_f32 = lambda a: torch.from_numpy(np.ascontiguousarray(a)).float().contiguous()
    return {"embedding": as_f32(params["embedding"]), "final_norm": as_f32(params["final_norm"]),
            "layers": [{k: as_f32(v) for k, v in lw.items()} for lw in params["layers"]]}


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,tol", [(torch.bfloat16, 4e-2), (torch.float32, 1e-4)], ids=["bf16", "f32"])
def test_cpu_plumbing_configuration_forward_and_loss_against_the_cpu_port(device, dtype, tol):
    """The reference's CPU-runnable configuration: 104m dims, B=1, T=256, forward + cross-entropy loss in the
    order of src/core/generation_cpu.cpp:323-379 + cross_entropy_forward_cpu (oracle/cpu_model.forward_loss, the
    float32 port; about 40 s on one core, since linear_forward_cpu is serial for more than one row). The GPU
    forward runs on the same weights (the CPU side reads the library's rounded weights back): the hidden state
    entering every layer and leaving the last one, and the loss, must agree. bf16 rounds every operator output
    (2e-2 each, several operators deep: 4e-2 of the state's scale); fp32 storage accumulates in a different
    order only (1e-4 of the scale; 2e-6 observed)."""
    from cgpt_amd.model import LOSS_DENSE, Model, ModelConfig
    from oracle import cpu_model

    cfg, batch, seq = HEADLINE_CFG, 1, 256
    model = Model(ModelConfig(dtype=dtype, **HEADLINE), batch, seq, seed=0, device=device)
    g = torch.Generator().manual_seed(1)
    tokens = torch.randint(0, cfg["vocab"], (batch, seq), generator=g)
    targets = torch.randint(0, cfg["vocab"], (batch, seq), generator=g)
    model.set_tokens(tokens.numpy(), targets.numpy())
    model.forward_backward(1.0, LOSS_DENSE, use_graph=False)
    loss, _, _ = model.status()
    want_loss, want_hidden, want_checksum = cpu_model.forward_loss(cpu_weights_from_model(model, cfg), tokens, targets, cfg)
    print(f"[parity] configuration 1 ({dtype}): GPU loss {loss:.6f}, CPU port {want_loss:.6f}, logits checksum {want_checksum:.4f}")
    assert abs(loss - want_loss) <= (5e-3 if dtype == torch.bfloat16 else 1e-4) * want_loss
    for l, want in enumerate(want_hidden):
        got = to_np(model.activation(f"hidden.{l}")).reshape(batch * seq, cfg["hidden"])
        scale = max(1.0, float(want.abs().max()))
        err = float(np.abs(got - to_np(want)).max()) / scale
        print(f"[parity] hidden.{l}: {err:.3e} of scale {scale:.3g}")
        assert err <= tol, f"hidden state {l}: {err:.3e}"
    # the checksum follows from logits that agree element by element: N*V terms with errors below tol each
    logits = to_np(model.activation("logits"))
    assert abs(logits.sum() - want_checksum) <= tol * np.abs(logits).sum()
    model.close()


@pytest.mark.gpu
def test_graph_is_recorded_again_after_the_scratch_arena_moves(device):
    """A recorded step holds addresses inside the stream's scratch arena. Releasing the arena
    (cgptx_release_scratch), or an operator on the same stream that needs a larger one, frees that block: the
    next graph step must notice, run eagerly and record again, and give the same bits as before."""
    from cgpt_amd import capi, ops

    cfg, dtype, batch, seq = MODEL_CFG, torch.bfloat16, 2, 40
    rng = np.random.default_rng(8)
    model = build(device, dtype, batch, seq, cfg)
    model.set_tokens(rng.integers(0, cfg["vocab"], size=(batch, seq)), rng.integers(0, cfg["vocab"], size=(batch, seq)))
    stream = torch.cuda.Stream(device=device)

    def step():
        for _, _, g in model.parameters():
            g.zero_()
        torch.cuda.synchronize()
        model.forward_backward(64.0, 1, use_graph=True, stream=stream)
        return model.status(stream)[0], [g.clone() for _, _, g in model.parameters()]

    step()                      # eager + capture
    want = step()               # replay
    capi.call("cgptx_release_scratch")
    # fill the freed block with other data so that a stale replay could not pass by accident
    junk = [torch.full((1 << 20,), 1e30, device=device) for _ in range(8)]
    after_release = step()
    with torch.cuda.stream(stream):   # a larger request on the same stream reallocates the arena
        big_rows = 1 << 16
        x = torch.randn(big_rows, 1024, device=device).to(dtype)
        dx, dw = torch.empty_like(x), torch.empty(1024, dtype=dtype, device=device)
        ops.rmsnorm_backward(dx, dw, x, x, torch.ones(1024, dtype=dtype, device=device), 1e-5, stream=stream)
    torch.cuda.synchronize()
    after_growth = step()
    replay = step()
    del junk
    for name, (loss, grads) in (("release", after_release), ("growth", after_growth), ("replay", replay)):
        assert loss == want[0], name
        for a, b in zip(grads, want[1]):
            assert torch.equal(a, b), name
    model.close()


@pytest.mark.gpu
def test_step_as_the_reference_call_sequence_agrees_with_the_fused_step(device, monkeypatch):
    """CGPTX_FUSE=0 runs the step as the reference's own call sequence (one public operator per call: separate
    q / k / v and gate / up projections with accumulating input gradients, separate SwiGLU, RoPE and residual
    additions). The default step fuses across those boundaries and rounds less often: the two agree to storage
    precision, the loss almost exactly."""
    from cgpt_amd.model import LOSS_CUT, Model, ModelConfig
    config = ModelConfig(vocabulary_size=512, num_layers=2, hidden_size=256, intermediate_size=512, num_query_heads=2,
                         num_kv_heads=2, head_dim=128, rotary_dim=128, dtype=torch.bfloat16)
    rng = np.random.default_rng(9)
    inputs, targets = rng.integers(0, 512, size=(2, 64)), rng.integers(0, 512, size=(2, 64))
    results = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("CGPTX_FUSE", fuse)
        model = Model(config, 2, 64, seed=6, device=device)
        model.set_tokens(inputs, targets)
        model.forward_backward(loss_scale=64.0, loss_mode=LOSS_CUT)
        results.append((model.status()[0], {n: g.float().cpu() for n, _, g in model.parameters()},
                        model.activation("hidden.2").float().cpu()))
        model.close()
    assert abs(results[0][0] - results[1][0]) <= 1e-3 * results[1][0]
    assert (results[0][2] - results[1][2]).abs().max().item() <= 4e-2 * max(1.0, results[1][2].abs().max().item())
    for name, fused in results[0][1].items():
        separate = results[1][1][name]
        scale = separate.abs().max().item() + 1e-12
        assert (fused - separate).abs().max().item() <= 3e-2 * scale, name


@pytest.mark.gpu
@pytest.mark.parametrize("batch,seq", [(16, 313), (8, 1024), (32, 1024)], ids=["ragged", "8192", "32768"])
def test_block_output_is_the_residual_sum_of_its_parts(device, batch, seq):
    """hidden[1] = x + attention_output Wo + activated Wdown over every element, at row counts whose output projections run on
    128- and 256-wide tiles: the two sums are rounded once each, so no element may be off by more than a few roundings
    (8 bits of mantissa: 2^-8 of the larger sum each, four times that is allowed). A store that goes wrong in one element of
    thousands shows here and in no norm."""
    from cgpt_amd.model import LOSS_CUT, Model, ModelConfig

    config = ModelConfig(vocabulary_size=512, num_layers=1, hidden_size=768, intermediate_size=2048, num_query_heads=12,
                         num_kv_heads=4, head_dim=64, rotary_dim=64, dtype=torch.bfloat16)
    model = Model(config, batch, seq, seed=3, device=device)
    rng = np.random.default_rng(3)
    model.set_tokens(rng.integers(0, 512, size=(batch, seq)), rng.integers(0, 512, size=(batch, seq)))
    stream = torch.cuda.Stream(device=device)
    weights = {name: p.float() for name, p, _ in model.parameters()}
    o, down = (weights[f"model.layers.0.{name}.weight"].view(768, -1).T.contiguous() for name in ("self_attn.o_proj", "mlp.down_proj"))
    for _ in range(3):
        model.forward_backward(1024.0, LOSS_CUT, use_graph=False, stream=stream)
        torch.cuda.synchronize()
        read = lambda name, width: model.activation(name).view(-1, width).float()
        first = read("hidden.0", 768) + read("layer.0.attention_output", 768) @ o
        want = first + read("layer.0.activated", 2048) @ down
        error = (read("hidden.1", 768) - want).abs()
        assert torch.isfinite(error).all()
        assert (error <= 4 * 2.0 ** -8 * torch.maximum(first.abs(), want.abs()) + 1e-3).all(), error.max().item()
    model.close()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16], ids=["f32", "f16", "bf16"])
@pytest.mark.parametrize("batch,seq,heads,kv_heads,head_dim,inter,layers", [
    (3, 100, 4, 2, 64, 704, 2),   # one weight gradient per layer and projection
    (1, 33, 2, 2, 128, 520, 2),   # all dimensions multiples of 256 but the last: stacked weight gradients in 16-bit storage
    (2, 16, 3, 1, 32, 72, 1),
])
def test_branches_of_a_small_step_share_launches(device, monkeypatch, dtype, batch, seq, heads, kv_heads, head_dim, inter, layers):
    """A few hundred tokens: the attention and the feed-forward branch's first projections run in one launch, so do the gradients
    of their last and of their first ones, and the SwiGLU product and its gradient ride beside q's and k's norms.
    CGPTX_FUSE_SWIGLU=0 keeps the branches apart: more launches and the same step, in 16-bit storage to the bit (fp32 steps share
    launches also where that changes the order of a sum)."""
    from cgpt_amd.model import LOSS_DENSE, Model, ModelConfig
    from tests.util import STOL, assert_scaled_close, launches
    config = ModelConfig(vocabulary_size=203, num_layers=layers, hidden_size=heads * head_dim, intermediate_size=inter,
                         num_query_heads=heads, num_kv_heads=kv_heads, head_dim=head_dim, rotary_dim=head_dim, dtype=dtype)
    rng = np.random.default_rng(batch + seq)
    inputs, targets = (rng.integers(0, 203, size=batch * seq).astype(np.uint32) for _ in range(2))
    results, counts = [], []
    for fuse in ("1", "0"):
        monkeypatch.setenv("CGPTX_FUSE_SWIGLU", fuse)
        model = Model(config, batch, seq, seed=4, device=device)
        model.set_tokens(inputs, targets)
        model.forward_backward(loss_scale=4.0, loss_mode=LOSS_DENSE)
        results.append([(name, g.clone()) for name, _, g in model.parameters()])
        counts.append(launches(lambda: model.forward_backward(4.0, LOSS_DENSE, use_graph=False, stream=torch.cuda.current_stream())))
        model.close()
    assert counts[0] <= counts[1] - 3 * layers, counts
    for (name, a), (_, b) in zip(*results):
        if dtype == torch.float32:
            assert_scaled_close(a, b, STOL[dtype], name)
        else:
            assert torch.equal(a, b), name


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16], ids=["f16", "bf16"])
@pytest.mark.parametrize("batch,seq,heads,kv_heads,head_dim,inter,layers", [
    (21, 112, 16, 4, 32, 1024, 1), (32, 140, 8, 4, 64, 1024, 2), (7, 22, 8, 4, 128, 2752, 2), (32, 111, 6, 2, 32, 512, 2),
    (8, 255, 7, 7, 128, 576, 1),  # q, k and v too wide for a group of their own: their input gradients are added up in storage
])
def test_sharing_launches_changes_no_sum(device, monkeypatch, dtype, batch, seq, heads, kv_heads, head_dim, inter, layers):
    """Steps some of whose projections, by themselves, run on large tiles or in K slices: those stay apart, since a group would add
    them up in another order, and the gradients are those of a step whose branches share nothing, bit for bit."""
    from cgpt_amd.model import LOSS_DENSE, Model, ModelConfig
    config = ModelConfig(vocabulary_size=203, num_layers=layers, hidden_size=heads * head_dim, intermediate_size=inter,
                         num_query_heads=heads, num_kv_heads=kv_heads, head_dim=head_dim, rotary_dim=head_dim, dtype=dtype)
    rng = np.random.default_rng(batch + seq)
    inputs, targets = (rng.integers(0, 203, size=batch * seq).astype(np.uint32) for _ in range(2))
    results = []
    for fuse in ("1", "0"):
        monkeypatch.setenv("CGPTX_FUSE_SWIGLU", fuse)
        model = Model(config, batch, seq, seed=4, device=device)
        model.set_tokens(inputs, targets)
        model.forward_backward(loss_scale=4.0, loss_mode=LOSS_DENSE)
        results.append([(name, g.clone()) for name, _, g in model.parameters()])
        model.close()
    for (name, a), (_, b) in zip(*results):
        assert torch.equal(a, b), name


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("batch,seq,vocab", [(1, 33, 203), (3, 100, 1000), (64, 128, 517), (64, 129, 517)])
@pytest.mark.parametrize("use_graph", [False, True], ids=["eager", "recorded"])
def test_launches_that_a_step_shares_give_what_the_operators_give(device, dtype, batch, seq, vocab, use_graph):
    """The rows' losses are averaged beside the norms' reductions, up to 8192 tokens are grouped beside their lookup, and the dense
    loss leaves an odd vocabulary's gradient in padded rows: the loss is that of the operator on the step's logits, the classifier's and
    the table's gradient what the operators make of the step's tensors (sums of 16-bit products in another order: STOL of the scale;
    fp32 1e-4), with ids so unlike that both kinds of segments occur."""
    from cgpt_amd import ops
    from cgpt_amd.model import LOSS_DENSE, Model, ModelConfig
    from tests.util import STOL

    config = ModelConfig(vocabulary_size=vocab, num_layers=2, hidden_size=128, intermediate_size=192, num_query_heads=4, num_kv_heads=2,
                         head_dim=32, rotary_dim=32, dtype=dtype)
    model = Model(config, batch, seq, seed=11, device=device)
    rows, rng, stream = batch * seq, np.random.default_rng(batch + seq), torch.cuda.Stream(device=device)
    for call in range(3 if use_graph else 1):
        tokens = np.minimum(rng.geometric(0.02, size=(batch, seq)) - 1, vocab - 1)
        tokens[:, ::3] = 7
        targets = rng.integers(0, vocab, size=(batch, seq))
        model.set_tokens(tokens, targets)
        torch.cuda.synchronize()
        model.forward_backward(32.0, LOSS_DENSE, use_graph=use_graph, stream=stream)
        loss, _, _ = model.status(stream)
        logits = model.activation("logits").view(rows, vocab)
        normalized, d_hidden = (model.activation(name).view(rows, 128) for name in ("normalized", "grad.hidden.0"))
        ids, wanted = (torch.from_numpy(a.reshape(-1).astype(np.int32)).to(device) for a in (tokens, targets))
        want_loss, gradient = torch.empty(1, device=device), torch.empty_like(logits)
        ops.cross_entropy_forward_backward(want_loss, gradient, logits, wanted, rows, gradient_scale=32.0)
        assert loss == want_loss.item()
        table = {name: gradient for name, _, gradient in model.parameters()}["model.embed_tokens.weight"].view(vocab, 128)
        want = torch.empty_like(table)
        ops.linear_backward(None, want, None, gradient, normalized, torch.zeros(vocab, 128, dtype=dtype, device=device))
        ops.embedding_backward(want, d_hidden, ids, rows, options=ops.EmbeddingBackwardOptions(accumulate_weight=True))
        scale = want.float().abs().max().item()
        assert (table.float() - want.float()).abs().max().item() <= STOL[dtype] * scale
    model.close()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,vocab", [(torch.bfloat16, 131083), (torch.float16, 131080), (torch.float32, 65541)], ids=["bf16", "f16", "f32"])
def test_a_dense_step_over_longer_rows_than_registers_hold_gives_what_the_operators_give(device, dtype, vocab):
    """The loss's gradient keeps rows like the logits' there, and the classifier's gradients read a copy in padded ones."""
    test_launches_that_a_step_shares_give_what_the_operators_give(device, dtype, 1, 33, vocab, False)
