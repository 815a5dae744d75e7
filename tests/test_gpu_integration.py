"""GPU: the torch integration paths run the HIP kernels end to end on a tiny bf16 Llama
(enable_flash_attention + make_loss_fn / make_packed_loss_fn), checked against eager attention and
the plain-torch loss contract."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu
transformers = pytest.importorskip("transformers")


def _model():
    torch.manual_seed(0)
    cfg = transformers.LlamaConfig(vocab_size=512, hidden_size=256, intermediate_size=512, num_hidden_layers=2,
                                   num_attention_heads=4, num_key_value_heads=2, head_dim=64,
                                   max_position_embeddings=512)
    m = transformers.LlamaForCausalLM(cfg).to("cuda", torch.bfloat16).eval()
    m.config._attn_implementation = "eager"
    m.lm_head.weight.requires_grad_(False)
    return m


def test_flash_attention_kernel_matches_eager_logits():
    from mlx_train_perf.attention import enable_flash_attention
    from mlx_train_perf.attention.api import VJP_CALLS

    m = _model()
    x = torch.randint(0, 512, (2, 130), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    with torch.no_grad():
        ref = m(input_ids=x).logits.float()
    enable_flash_attention(m, impl="kernel", seq_len=130, batch_size=2)
    with torch.no_grad():
        out = m(input_ids=x).logits.float()
    assert float((out - ref).norm() / ref.norm()) < 2e-2
    before = VJP_CALLS.get("flash_attention_kernel_bwd", 0)
    m(input_ids=x).logits.float().sum().backward()
    assert VJP_CALLS.get("flash_attention_kernel_bwd", 0) > before


def _default_loss_by_hand(m, batch, lengths):
    """The mlx-lm trainer's `default_loss` written out independently of the adapter: the model's own
    trunk, fp64 logits against its lm_head, and the (offset, length) window walked token by token
    (inputs = batch[:, :-1], targets = batch[:, 1:], step j + 1 counted iff offset <= j + 1 <= length;
    loss = summed NLL / counted tokens)."""
    with torch.no_grad():
        hid = m.model(input_ids=batch[:, :-1]).last_hidden_state.double().cpu()
    w = m.lm_head.weight.double().cpu()
    logp = torch.log_softmax(hid @ w.T, dim=-1)
    tg = batch[:, 1:].cpu()
    total, count = 0.0, 0
    for r in range(batch.shape[0]):
        off, length = (int(x) for x in lengths[r])
        for j in range(tg.shape[1]):
            if off <= j + 1 <= length:
                total -= float(logp[r, j, tg[r, j]])
                count += 1
    return total / count, count


def test_loss_fn_kernel_matches_default_loss_by_hand():
    """make_loss_fn on the kernel impl against the documented trainer contract computed without the
    adapter (a mask or normalization bug in the adapter cannot cancel here)."""
    from mlx_train_perf.adapters.transformers_lm import make_loss_fn

    m = _model()
    g = torch.Generator(device="cuda").manual_seed(2)
    batch = torch.randint(0, 512, (3, 65), device="cuda", generator=g)
    lengths = torch.tensor([[1, 64], [5, 40], [64, 64]], device="cuda")
    want, count = _default_loss_by_hand(m, batch, lengths)
    lk, nk = make_loss_fn(m, impl="kernel")(m, batch, lengths)
    assert int(nk) == count == 64 + 36 + 1
    assert abs(lk.item() - want) < 2e-3 * abs(want), (lk.item(), want)


def test_mlx_style_wrapper_on_kernel_matches_stock():
    """FlashAttentionWrapper (the mlx-lm-shaped module surgery) with impl="kernel" on the GPU: output
    and input gradient against the stock block, computed in fp32 on the CPU; the kernel backward runs."""
    from test_adapters import _mlx_style_model

    from mlx_train_perf.attention import FlashAttentionWrapper, enable_flash_attention
    from mlx_train_perf.attention.api import VJP_CALLS

    print("[mlx-style FlashAttentionWrapper impl=kernel]", flush=True)
    stock = _mlx_style_model(layers=1).float()
    gpu = _mlx_style_model(layers=1).to("cuda", torch.bfloat16)
    x = torch.randn(2, 130, 64, generator=torch.Generator().manual_seed(6)).to(torch.bfloat16)
    xr = x.float().requires_grad_(True)
    ref = stock.model.layers[0].self_attn(xr)
    ref.backward(torch.ones_like(ref))
    enable_flash_attention(gpu, impl="kernel", seq_len=130, batch_size=2)
    wrap = gpu.model.layers[0].self_attn
    assert isinstance(wrap, FlashAttentionWrapper)
    xg = x.cuda().requires_grad_(True)
    before = VJP_CALLS.get("flash_attention_kernel_bwd", 0)
    out = wrap(xg, mask="causal")
    out.backward(torch.ones_like(out))
    assert VJP_CALLS.get("flash_attention_kernel_bwd", 0) == before + 1
    e_out = float((out.float().cpu() - ref.detach()).norm() / ref.detach().norm())
    e_dx = float((xg.grad.float().cpu() - xr.grad).norm() / xr.grad.norm())
    assert e_out < 2e-2 and e_dx < 3e-2, (e_out, e_dx)


def test_enable_prewarms_causal_and_packed_kernels():
    """enable_flash_attention(seq_len=, packed=True) runs the causal and the packed kernels once at the
    hinted shape (forward and backward), as the reference pre-warms its packed-keyed rate slots."""
    from mlx_train_perf.attention import enable_flash_attention
    from mlx_train_perf.attention.api import VJP_CALLS

    m = _model()
    before = VJP_CALLS.get("flash_attention_kernel_bwd", 0)
    enable_flash_attention(m, impl="kernel", seq_len=96, batch_size=2, packed=True)
    assert VJP_CALLS.get("flash_attention_kernel_bwd", 0) == before + 2
    enable_flash_attention(m, impl="kernel", seq_len=96, batch_size=2)
    assert VJP_CALLS.get("flash_attention_kernel_bwd", 0) == before + 3


def test_packed_loss_kernel_path_runs_and_matches_reference_attention():
    from mlx_train_perf.adapters.transformers_lm import make_packed_loss_fn
    from mlx_train_perf.attention import enable_flash_attention
    from mlx_train_perf.data.packing import build_row

    m = _model()
    g = torch.Generator().manual_seed(3)
    docs = [(torch.randint(1, 512, (n,), generator=g).tolist(), 1) for n in (40, 3, 70)]
    row, sid, sst, lm = build_row(docs, pack_len=128)
    args = [torch.tensor([x], device="cuda") for x in (row, sid, sst, lm)]
    enable_flash_attention(m, impl="kernel")
    lk, _ = make_packed_loss_fn(m, impl="kernel")(m, *args)
    lk.backward()
    m.zero_grad()
    m.config._mtp_flash_impl = "reference"
    lr, _ = make_packed_loss_fn(m, impl="naive")(m, *args)
    assert abs(lk.item() - lr.item()) < 2e-2 * abs(lr.item())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("mask", ["causal", "full", "packed"])
def test_attention_node_equals_the_python_function(dtype, mask):
    """flash_attention's C++ node against the Python Function it stands for, bit for bit: strided inputs,
    a strided and a missing output gradient, inputs without gradients, hooks on the saved tensors, two
    backwards through one graph, evaluation, and the counters."""
    from mlx_train_perf.attention import PackedMask, api, flash_attention

    g = torch.Generator().manual_seed(5)

    def strided(h):
        return torch.randn(2, 130, h, 64, generator=g).to("cuda", dtype).transpose(1, 2)

    q, do = strided(4), strided(4)
    k, v = strided(2), strided(2)
    seg = args = None
    if mask == "packed":
        sid = torch.tensor([[0] * 50 + [1] * 80] * 2)
        sst = torch.tensor([[0] * 50 + [50] * 80] * 2)
        seg = PackedMask(seg_id=sid.cuda(), seg_start=sst.cuda())
        args = (seg.seg_id.int(), seg.seg_start.int())
    leaves = [x.clone().detach().requires_grad_(True) for x in (q, k, v)]

    def node(a, b, c):
        return flash_attention(a, b, c, scale=0.125, causal=mask != "full", segments=seg)

    def function(a, b, c):
        return api._KernelAttention.apply(a.contiguous(), b.contiguous(), c.contiguous(), *(args or (None, None)), 0.125,
                                          mask != "full")[0]

    o, ref = node(*leaves), function(*leaves)
    assert type(o.grad_fn) is not type(ref.grad_fn)
    assert torch.equal(o, ref)
    before = dict(api.VJP_CALLS)
    want = torch.autograd.grad(ref, leaves, do)
    got = torch.autograd.grad(o, leaves, do, retain_graph=True)
    again = torch.autograd.grad(o, leaves, do)
    assert all(torch.equal(a, w) and torch.equal(b, w) for a, b, w in zip(got, again, want))
    assert all(api.VJP_CALLS[n] == before.get(n, 0) + 3 for n in ("flash_attention", "flash_attention_kernel_bwd"))
    with pytest.raises(RuntimeError):   # freed by the second backward
        torch.autograd.grad(o, leaves, do)
    (dk,) = torch.autograd.grad(node(q, leaves[1], v), leaves[1], do)   # only k asks for a gradient
    assert torch.equal(dk, want[1])
    counts = []
    for f in (node, function):
        packed = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.shape) or t.cpu(), lambda t: t.cuda()):
            out = f(*leaves)
        assert all(torch.equal(a, w) for a, w in zip(torch.autograd.grad(out, leaves, do), want))
        counts.append(sorted(packed))
    assert counts[0] == counts[1]
    with torch.no_grad():
        assert torch.equal(node(q, k, v), o) and not node(q, k, v).requires_grad
    with torch.inference_mode():
        assert torch.equal(node(q, k, v), o)


def test_attention_refuses_what_the_python_function_refuses():
    """Function transforms and forward-mode gradients raise, as they do for the Python Function."""
    from mlx_train_perf.attention import flash_attention

    q = torch.randn(1, 2, 32, 64, device="cuda", dtype=torch.bfloat16)

    def f(x):
        return flash_attention(x, q, q, scale=0.125).float().sum()

    with pytest.raises(RuntimeError):
        torch.func.grad(f)(q)
    with pytest.raises(RuntimeError):
        torch.func.vmap(f)(q[None])
    with torch.autograd.forward_ad.dual_level(), pytest.raises(RuntimeError):
        f(torch.autograd.forward_ad.make_dual(q, q))


LOSS_MODES = [{}, {"MTP_LCE_TRANSPOSED_HEAD": "0"}, {"MTP_LCE_TRANSPOSED_HEAD": "1"},
              {"MTP_LCE_TRANSPOSED_HEAD": "0", "MTP_LCE_STAGE_HEAD": "0"}, {"MTP_LCE_BWD_BUDGET": "300000"}]


@pytest.mark.parametrize("env", LOSS_MODES, ids=lambda e: ",".join(f"{k[8:]}={v}" for k, v in e.items()) or "default")
@pytest.mark.parametrize(("kind", "dtype", "d"), [("frozen", torch.bfloat16, 128), ("frozen", torch.bfloat16, 72),
                                                  ("trainable", torch.bfloat16, 128), ("q4", torch.bfloat16, 128),
                                                  ("trainable", torch.float32, 36), ("q4", torch.float32, 64)])
def test_loss_node_equals_the_python_function(kind, dtype, d, env, monkeypatch):
    """linear_cross_entropy's C++ node against the Python Function it stands for, bit for bit, in every head
    mode: both reductions, a strided gradient, an explicit chunk, hooks on the saved tensors, the counter,
    two backwards, evaluation."""
    from mlx_train_perf import DenseHead, QuantizedHead, _native, linear_cross_entropy
    from mlx_train_perf.core import loss as L
    from mlx_train_perf.core.quant import quantize

    for name in ("MTP_LCE_TRANSPOSED_HEAD", "MTP_LCE_STAGE_HEAD", "MTP_LCE_BWD_BUDGET"):
        monkeypatch.delenv(name, raising=False)
    for name, value in env.items():
        monkeypatch.setenv(name, value)
    g = torch.Generator().manual_seed(9)
    n, v = 321, 700
    hidden = torch.randn(n, d, generator=g).to("cuda", dtype).requires_grad_(True)
    w = (torch.randn(v, d, generator=g) * 0.05).to("cuda", dtype)
    t = torch.randint(0, v, (n,), generator=g).cuda()
    t[::7] = -100
    wrt = [hidden]
    if kind == "q4":
        head = QuantizedHead(**dict(zip(("w_q", "scales", "biases"), quantize(w))))
    else:
        head = DenseHead(weight=w.requires_grad_(kind == "trainable"), trainable=kind == "trainable")
        wrt += [w] if kind == "trainable" else []
    ct = torch.rand(n, 2, generator=g).cuda()[:, 0]

    def calls():
        out = []
        for kw in ({"reduction": "none"}, {"reduction": "mean"}, {"reduction": "none", "chunk_size": 256}):
            loss = linear_cross_entropy(hidden, head, t, **kw)
            grad = ct if kw["reduction"] == "none" else torch.tensor(0.5, device="cuda")
            before = L.VJP_CALLS.get("kernel", 0)
            first = torch.autograd.grad(loss, wrt, grad, retain_graph=True)
            out += [loss.detach(), *first, *torch.autograd.grad(loss, wrt, grad)]
            assert L.VJP_CALLS["kernel"] == before + 2
        packed = []
        with torch.autograd.graph.saved_tensors_hooks(lambda x: packed.append(x.shape) or x.cpu(), lambda x: x.cuda()):
            loss = linear_cross_entropy(hidden, head, t)
        out += torch.autograd.grad(loss, wrt)
        with torch.no_grad():
            out.append(linear_cross_entropy(hidden, head, t))
            assert not out[-1].requires_grad
        return out, sorted(packed), type(loss.grad_fn)

    L.clear_transposed_head_cache()
    got, packed, node = calls()
    monkeypatch.setattr(_native, "plain", lambda *a: False)
    want, packed_f, function = calls()
    assert node is not function and packed == packed_f
    assert len(got) == len(want) and all(torch.equal(a, b) for a, b in zip(got, want))
    L.clear_transposed_head_cache()


@pytest.mark.parametrize("reduction", ["none", "mean", "sum"])
@pytest.mark.parametrize("which", ["hidden", "trainable w", "frozen w", "scales", "biases"])
def test_loss_refuses_forward_mode_tangents(which, reduction):
    """No loss without its tangent: a dual tensor in any place is refused as the Python Function refuses it."""
    from torch.autograd import forward_ad

    from mlx_train_perf import DenseHead, QuantizedHead, linear_cross_entropy
    from mlx_train_perf.core.quant import quantize

    g = torch.Generator().manual_seed(3)
    hidden, w = (torch.randn(n, 64, generator=g).to("cuda", torch.bfloat16) for n in (40, 300))
    t = torch.randint(0, 300, (40,), generator=g).cuda()
    q = dict(zip(("w_q", "scales", "biases"), quantize(w)))
    with forward_ad.dual_level():
        def dual(x):
            return forward_ad.make_dual(x, torch.ones_like(x))

        if which in q:
            head = QuantizedHead(**{**q, which: dual(q[which])})
        else:
            head = DenseHead(weight=dual(w) if which.endswith("w") else w, trainable=which == "trainable w")
        with pytest.raises(NotImplementedError):
            linear_cross_entropy(dual(hidden) if which == "hidden" else hidden, head, t, reduction=reduction)


@pytest.mark.parametrize("which", ["q", "k", "v"])
def test_attention_refuses_forward_mode_tangents(which):
    from torch.autograd import forward_ad

    from mlx_train_perf.attention import flash_attention

    x = {n: torch.randn(1, 2, 32, 64, device="cuda", dtype=torch.bfloat16) for n in "qkv"}
    with forward_ad.dual_level():
        x[which] = forward_ad.make_dual(x[which], torch.ones_like(x[which]))
        with pytest.raises(NotImplementedError):
            flash_attention(**x, scale=0.125)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("which", ["frozen w", "scales", "biases"])
def test_loss_node_keeps_inputs_without_gradients_in_the_graph(which, dtype):
    """A frozen weight, scales or biases that ask for a gradient are inputs of the loss, as they are of the
    Python Function: the loss asks for one although hidden does not, and their accumulation hooks run (with
    no gradient)."""
    from mlx_train_perf import DenseHead, QuantizedHead, linear_cross_entropy
    from mlx_train_perf.core.quant import quantize

    g = torch.Generator().manual_seed(4)
    hidden, w = (torch.randn(n, 64, generator=g).to("cuda", dtype) for n in (40, 300))
    t = torch.randint(0, 300, (40,), generator=g).cuda()
    q = dict(zip(("w_q", "scales", "biases"), quantize(w)))
    x = (w if which == "frozen w" else q[which]).requires_grad_(True)
    head = DenseHead(weight=w, trainable=False) if which == "frozen w" else QuantizedHead(**q)
    calls = []
    x.register_post_accumulate_grad_hook(lambda p: calls.append(p.grad))
    for h in (hidden, hidden.clone().requires_grad_(True)):
        for reduction in ("none", "mean", "sum"):
            calls.clear()
            loss = linear_cross_entropy(h, head, t, reduction=reduction)
            assert loss.requires_grad
            loss.sum().backward()
            assert calls == [None] and x.grad is None
            assert (h.grad is not None) == h.requires_grad
    with torch.no_grad():
        assert not linear_cross_entropy(hidden, head, t).requires_grad


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_loss_arguments_past_64_bits(dtype):
    """Any chunk above the vocabulary is the whole vocabulary and any below a tile one tile, bit for bit; an
    ignore_index that no target can hold, or that is no whole number, is taken as torch's operators take it."""
    import sys

    from mlx_train_perf import DenseHead, linear_cross_entropy

    g = torch.Generator().manual_seed(6)
    hidden, w = (torch.randn(n, 128, generator=g).to("cuda", dtype) for n in (300, 1000))
    hidden.requires_grad_(True)
    head = DenseHead(weight=w * 0.05, trainable=False)
    t = torch.randint(0, 1000, (300,), generator=g).cuda()

    def step(**kw):
        loss = linear_cross_entropy(hidden, head, t, **kw)
        return loss.detach(), *torch.autograd.grad(loss, hidden)

    whole, tile = step(chunk_size=1000), step(chunk_size=1)
    assert not torch.equal(whole[1], tile[1])   # another order of sums
    for size, want in ((sys.maxsize, whole), (2 ** 70, whole), (-5, tile), (-2 ** 70, tile)):
        assert all(torch.equal(a, b) for a, b in zip(step(chunk_size=size), want)), size
    none, count = linear_cross_entropy(hidden, head, t, reduction="none"), torch.tensor(300.0, device="cuda")
    for index in (2 ** 63, 2 ** 64 - 100):
        assert torch.equal(linear_cross_entropy(hidden, head, t, reduction="none", ignore_index=index), none)
    assert torch.equal(linear_cross_entropy(hidden, head, t, ignore_index=2 ** 63), none.sum() / count)
    t[:3] = 3
    got = linear_cross_entropy(hidden, head, t, ignore_index=3.5)   # read as 3 by the loss, no target's equal
    none = linear_cross_entropy(hidden, head, t, reduction="none", ignore_index=3)
    assert torch.equal(got, none.sum() / count)


def test_calls_without_the_autograd_nodes(monkeypatch):
    """An installation with the C-ABI library alone: the Python Functions serve every call, the same bits."""
    import sys

    import mlx_train_perf
    from mlx_train_perf import DenseHead, _native, linear_cross_entropy
    from mlx_train_perf.attention import flash_attention

    g = torch.Generator().manual_seed(8)
    x, w = (torch.randn(n, 64, generator=g).to("cuda", torch.bfloat16).requires_grad_(True) for n in (40, 300))
    q = torch.randn(1, 2, 70, 64, generator=g).to("cuda", torch.bfloat16).requires_grad_(True)
    t = torch.randint(0, 300, (40,), generator=g).cuda()

    def calls():
        loss = linear_cross_entropy(x, DenseHead(weight=w), t)
        o = flash_attention(q, q, q, scale=0.125)
        grads = torch.autograd.grad(loss, (x, w)) + torch.autograd.grad(o.float().square().sum(), q)
        return (loss.detach(), o.detach(), *grads), (type(loss.grad_fn).__name__, type(o.grad_fn).__name__)

    want, built = calls()
    monkeypatch.setattr(_native, "_nodes", None)
    monkeypatch.delattr(mlx_train_perf, "_mtp_torch", raising=False)
    monkeypatch.setitem(sys.modules, "mlx_train_perf._mtp_torch", None)   # its import fails
    with pytest.warns(UserWarning, match="cannot be loaded"):
        got, names = calls()
    assert names == ("_KernelLCEBackward", "_KernelAttentionBackward") and not set(names) & set(built)
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_loss_node_reads_the_environment_as_python_does():
    """A switch set in the C environment alone (os.putenv) is none to os.environ, nor to the node's backward."""
    import os

    from mlx_train_perf import DenseHead, linear_cross_entropy
    from mlx_train_perf.core import loss as L

    assert "MTP_LCE_TRANSPOSED_HEAD" not in os.environ
    g = torch.Generator().manual_seed(5)
    x, w = (torch.randn(n, 64, generator=g).to("cuda", torch.bfloat16).requires_grad_(True) for n in (40, 300))
    L.clear_transposed_head_cache()
    os.putenv("MTP_LCE_TRANSPOSED_HEAD", "1")   # would keep a trainable head's transposed copy
    try:
        linear_cross_entropy(x, DenseHead(weight=w), torch.zeros(40, dtype=torch.int64, device="cuda")).backward()
    finally:
        os.unsetenv("MTP_LCE_TRANSPOSED_HEAD")
    assert L.transposed_head_cache_bytes() == 0
