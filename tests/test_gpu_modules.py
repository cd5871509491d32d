"""Module-level parity on the GPU: FlashAttention / FlashAttentionOp as schedules install them,
against an oracle composite built from the same weights (restates tests/test_op.py::test_attention,
whose bar is atol = rtol = 5e-2 in fp16)."""
import pytest
import torch

from oracle import attention as OA
from slapo_amd import op
from tests.conftest import assert_parity

pytestmark = pytest.mark.gpu


def _oracle_block(m, x, mask):
    """QKV GEMM with the head-interleaved [H, 3, D] packing, oracle attention, out_proj."""
    w = {n: p.detach().cpu().double() for n, p in m.named_parameters()}
    b, s, _ = x.shape
    h, d = m.num_attention_heads, m.attention_head_size
    if m.fused_qkv:
        packed = (x @ w["qkv.weight"].t() + w["qkv.bias"]).view(b, s, h, 3 * d)
        q, k, v = packed.split(d, dim=-1)
    else:
        q, k, v = ((x @ w[f"{n}.weight"].t() + w[f"{n}.bias"]).view(b, s, h, d)
                   for n in ("query", "key", "value"))
    ctx = OA.xformers_ref(q, k, v, mask, m.output_proj, compute_dtype=torch.float64)
    ctx = ctx.reshape(b, s, h * d)
    if m.output_proj:
        ctx = ctx @ w["out_proj.weight"].t() + w["out_proj.bias"]
    return ctx


@pytest.mark.parametrize("fused_qkv,output_proj", [(True, True), (False, True), (False, False)])
def test_flash_attention_module_fwd_bwd(fused_qkv, output_proj):
    torch.manual_seed(0)
    b, s, hidden, heads = 2, 256, 512, 8
    m = op.FlashAttention(hidden_size=hidden, num_attention_heads=heads, output_proj=output_proj,
                          attn_pdrop=0.0, resid_pdrop=0.0, attn_op_name="hip_cdna4",
                          fused_qkv=fused_qkv).half().cuda()
    x = torch.randn(b, s, hidden, dtype=torch.float16, device="cuda", requires_grad=True)
    mask = torch.randn(b, 1, 1, s, dtype=torch.float16, device="cuda", requires_grad=True)
    out, present = m(x, mask, None)
    assert present is None and out.shape == (b, s, hidden)
    out.backward(torch.ones_like(out))
    xr = x.detach().cpu().double().requires_grad_(True)
    ref = _oracle_block(m, xr, mask.detach().cpu().double())
    ref.backward(torch.ones_like(ref))
    torch.testing.assert_close(out.detach().cpu().double(), ref.detach(), atol=5e-2, rtol=5e-2)
    torch.testing.assert_close(x.grad.cpu().double(), xr.grad, atol=5e-2, rtol=5e-2)
    assert mask.grad is None  # bias gradient is not produced (as in the reference)
    out2, present = m(x, mask, None, use_cache=True)
    assert present[0].shape == (b, s, heads, hidden // heads)


def test_flash_attention_op_replacement_call():
    """The tutorial's subgraph replacement calls the op with concrete_args attention_mask=None,
    p=0.1 (docs/source/scripts/attention-single-gpu.py:279-282)."""
    core = op.FlashAttentionOp("hip_cdna4", apply_causal_mask=False)
    q, k, v = (torch.randn(2, 64, 4, 64, device="cuda", dtype=torch.bfloat16) for _ in range(3))
    out = core(q, k, v, None, 0.0)
    ref = OA.xformers_ref(q.cpu(), k.cpu(), v.cpu(), None, False, compute_dtype=torch.float64)
    assert_parity(out, ref, torch.bfloat16, "op forward")
    assert core(q, k, v, None, 0.1).shape == q.shape


def test_window_kwarg_local_attention_module():
    m = op.FlashAttention(128, 2, attn_op_name="hip_cdna4", fused_qkv=True, window=16).half().cuda()
    x = torch.randn(1, 96, 128, dtype=torch.float16, device="cuda")
    out, _ = m(x)
    mg = op.FlashAttention(128, 2, attn_op_name="hip_cdna4", fused_qkv=True).half().cuda()
    mg.load_state_dict(m.state_dict())
    out_g, _ = mg(x)
    # the first `window` positions see the same keys under both masks, later ones do not
    assert torch.equal(out[:, :16], out_g[:, :16]) and not torch.equal(out[:, 16:], out_g[:, 16:])


def _attention_with_dropout_tail():
    torch.manual_seed(3)
    m = op.FlashAttention(hidden_size=256, num_attention_heads=4, output_proj=True,
                          attn_pdrop=0.0, resid_pdrop=0.1, attn_op_name="hip_cdna4",
                          fused_qkv=True).half().cuda()
    x = torch.randn(2, 128, 256, dtype=torch.float16, device="cuda")
    return m, x


def _same_mask_close_values(a, b):
    assert ((a == 0) != (b == 0)).float().mean().item() < 5e-4  # exact zeros of the GEMM aside
    assert 0.08 < (a == 0).float().mean().item() < 0.12
    torch.testing.assert_close(a.float(), b.float(), atol=1e-2, rtol=1e-2)


def test_hooks_on_out_proj_fire_and_their_result_is_used():
    """Schedules hang the tensor-parallel all-reduce on `out_proj` as a forward hook
    (`.sync(mode="fwd_post")`: slapo/sharding/shard_ops.py:436-440, model_schedule/gpt2.py:482-485)
    and `.replace` carries hooks over (primitives/replace.py:254).  With a hook on either child the
    block calls the children as the reference does (attention.py:514-516): the hook runs once per
    forward and what it returns is what `resid_dropout` sees.  Without hooks the fused pass runs
    and draws the same mask as `nn.Dropout`."""
    m, x = _attention_with_dropout_tail()
    torch.cuda.manual_seed(77)
    plain, _ = m(x)

    calls = []

    def post(mod, inp, out):
        calls.append(tuple(out.shape))
        return out * 2

    h = m.out_proj.register_forward_hook(post)
    torch.cuda.manual_seed(77)
    hooked, _ = m(x)
    assert calls == [(2, 128, 256)]
    # the same draw masks both paths; values differ by the roundings of GEMM-with-bias then
    # dropout against GEMM then bias + dropout in one pass
    _same_mask_close_values(hooked, plain * 2)
    h.remove()

    pre_calls = []
    h = m.out_proj.register_forward_pre_hook(lambda mod, inp: pre_calls.append(1))
    torch.cuda.manual_seed(77)
    again, _ = m(x)
    assert pre_calls == [1]
    _same_mask_close_values(again, plain)
    h.remove()

    grads = []
    h = m.out_proj.register_full_backward_hook(lambda mod, gi, go: grads.append(go[0].shape))
    xg = x.clone().requires_grad_(True)
    m(xg)[0].sum().backward()
    assert len(grads) == 1
    h.remove()


def test_replaced_children_of_the_tail_are_called_as_modules():
    """A `resid_dropout` replaced by Identity (no `.p`) or an `out_proj` wrapped in another module
    type must keep working: the block then calls them as the reference does."""
    m, x = _attention_with_dropout_tail()
    torch.cuda.manual_seed(5)
    fused, _ = m(x)
    m.resid_dropout = torch.nn.Identity()
    no_drop, _ = m(x)
    kept = fused != 0
    assert torch.allclose(fused[kept].float(), no_drop[kept].float() / 0.9, atol=2e-3, rtol=2e-3)

    class Wrapped(torch.nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner = inner

        def forward(self, t):
            return self.inner(t) + 1

    m.out_proj = Wrapped(m.out_proj)
    assert torch.equal(m(x)[0], no_drop + 1)


def test_ops_on_side_streams_from_two_threads():
    """The entry points take the caller's stream and keep no state between calls: two host
    threads, each on a stream of its own (default priority), run attention forward + backward and
    the LayerNorm epilogue at the same time and get what a single-threaded run on the default
    stream gets, bit for bit."""
    import threading

    from slapo_amd import op

    g = torch.Generator().manual_seed(21)
    mk = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16).cuda()
    cases = []
    for d in (64, 128):
        q, k, v, do = (mk(2, 384, 4, d) for _ in range(4))
        x, res, gy, w, b = mk(384, 512), mk(384, 512), mk(384, 512), mk(512), mk(512)
        cases.append((q, k, v, do, x, res, gy, w, b))

    def run(case):
        q, k, v, do, x, res, gy, w, b = case
        ql, kl, vl, xl = (t.clone().requires_grad_(True) for t in (q, k, v, x))
        out = op.hip_attention(ql, kl, vl, None, causal=True)
        y = op.bias_dropout_residual_layer_norm(xl, b, res, w, b, 0.0, 1e-5, True)
        grads = torch.autograd.grad((out, y), (ql, kl, vl, xl), (do, gy))
        return (out, y) + tuple(grads)

    want = [run(c) for c in cases]
    torch.cuda.synchronize()
    got, errors = [None, None], []

    def worker(i):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                for _ in range(5):
                    res_ = run(cases[i])
                stream.synchronize()
            got[i] = res_
        except Exception as exc:  # pylint: disable=broad-except
            errors.append(exc)

    threads = [threading.Thread(target=worker, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not errors, errors
    for i in range(2):
        for a, b_ in zip(got[i], want[i]):
            assert torch.equal(a, b_)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("tokens,heads,head_size", [(5, 3, 8), (33, 2, 20), (7, 1, 3)])
def test_fused_qkv_layout_and_gradient(dtype, tokens, heads, head_size):
    """One pass in each direction, 16-byte runs and element by element, against torch's own
    splitting of the same projection output; a result that is not used gives no gradient."""
    m = op.FusedQKV(heads * head_size, heads, 1).to(device="cuda", dtype=dtype)
    x = torch.randn(2, tokens, heads * head_size, device="cuda", dtype=dtype, requires_grad=True)
    go = [torch.randn(2, tokens, heads, head_size, device="cuda", dtype=dtype) for _ in range(3)]
    packed = m.fused_linear(x)
    ref = [t.squeeze(-1) for t in m.reshape_for_scores(packed).split(1, dim=-1)]
    out = m(x)
    for used in (3, 2):
        for a, r in zip(out, ref):
            assert a.shape == r.shape and a.is_contiguous() and torch.equal(a, r)
        ga, = torch.autograd.grad(out[:used], x, go[:used], retain_graph=True)
        gr, = torch.autograd.grad(ref[:used], x, go[:used], retain_graph=True)
        assert torch.equal(ga, gr)


@pytest.mark.parametrize("dtype,head_dim,p", [(torch.float16, 64, 0.0), (torch.bfloat16, 80, 0.1),
                                              (torch.float32, 12, 0.1)])
def test_packed_attention_equals_the_split_call(dtype, head_dim, p):
    """FlashAttention hands the fused projection to the kernel in one piece: same output and the
    same gradient, bit for bit, as splitting it and calling the op."""
    torch.manual_seed(4)
    heads, b, s = 3, 2, 75
    m = op.FlashAttention(heads * head_dim, heads, attn_pdrop=p, output_proj=True, fused_qkv=True,
                          attn_op_name="hip_cdna4").to(device="cuda", dtype=dtype)
    x = torch.randn(b, s, heads * head_dim, device="cuda", dtype=dtype, requires_grad=True)
    mask = torch.zeros(b, 1, 1, s, device="cuda", dtype=dtype)
    mask[1, ..., 50:] = torch.finfo(dtype).min
    results = []
    for use_cache in (False, True):  # the cache asks for k and v: the split form
        torch.cuda.manual_seed(9)
        out, _ = m(x, mask, use_cache=use_cache)
        results.append([out, *torch.autograd.grad(out, [x, *m.qkv.parameters()],
                                                  torch.ones_like(out))])
    for a, r in zip(*results):
        assert torch.equal(a, r)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("layout", ["expanded", "sliced"])
def test_attention_backward_with_saved_tensors_kept_on_the_host(dtype, layout):
    # the hooks bring a saved mask back dense, whatever its strides were in the forward
    torch.manual_seed(0)
    b, s, h, d = 2, 96, 2, 64
    q, k, v = (torch.randn(b, s, h, d, dtype=dtype, device="cuda", requires_grad=True)
               for _ in range(3))
    if layout == "expanded":
        mask = torch.randn(1, 1, 1, s, device="cuda").expand(b, h, 1, s)
    else:
        mask = torch.randn(b, h, s, 2 * s, device="cuda")[..., ::2]
    g = torch.randn(b, s, h, d, dtype=dtype, device="cuda")
    plain = torch.autograd.grad(op.hip_attention(q, k, v, mask, causal=True), (q, k, v), g)
    with torch.autograd.graph.save_on_cpu():
        out = op.hip_attention(q, k, v, mask, causal=True)
    for a, r in zip(torch.autograd.grad(out, (q, k, v), g), plain):
        assert torch.equal(a, r)


def test_fused_qkv_where_its_operations_are_watched():
    torch.manual_seed(0)
    m = op.FusedQKV(32, 4, 1).cuda().double()
    x = torch.randn(2, 6, 32, device="cuda", dtype=torch.float64)

    def ref(x):
        packed = m.fused_linear(x).view(*x.shape[:-1], 4, 8, 3)
        return [t.squeeze(-1) for t in packed.split(1, dim=-1)]

    def check(got, want):
        for a, r in zip(got, want):
            assert torch.equal(a, r)

    check(m(x), ref(x))  # a type that the kernel does not move
    m, x = m.float(), x.float()
    check(m(x), ref(x))
    batched = torch.func.vmap(lambda t: tuple(m(t)))(x)
    assert all(a.shape == (2, 6, 4, 8) for a in batched)
    _, tangents = torch.func.jvp(lambda t: tuple(m(t)), (x,), (x,))
    _, wanted = torch.func.jvp(lambda t: tuple(ref(t)), (x,), (x,))
    check(tangents, wanted)
    x = x.requires_grad_()  # a second derivative reaches the incoming gradient
    g = torch.randn(2, 6, 4, 8, device="cuda", requires_grad=True)
    seconds = []
    for f in (m, ref):
        first, = torch.autograd.grad(f(x)[1], x, g, create_graph=True)
        seconds.append(torch.autograd.grad(first.square().sum(), g)[0])
    torch.testing.assert_close(*seconds)


class _AmongTorchOperations(torch.nn.Module):
    """An op of [2, 24, 64] values between two torch operations."""

    def __init__(self, name):
        super().__init__()
        self.name = name
        vec = lambda: torch.nn.Parameter(torch.randn(64))
        self.bias, self.weight, self.shift = vec(), vec(), vec()
        self.register_buffer("mask", torch.randn(2, 1, 1, 24))
        self.register_buffer("target", torch.randint(0, 64, (2, 24)))
        if name == "flash_attention":
            self.child = op.FlashAttention(64, 4, 0.1, 0.1, "hip_cdna4", fused_qkv=True)
        elif name == "fused_mlp":
            self.child = op.FusedMLP(64, 64, "gelu_new", 0.1)

    def forward(self, x):
        x = x * 1.5
        if self.name == "attention":
            q = x.view(2, 24, 4, 16)
            y = op.hip_attention(q, q.flip(1), q - 1, self.mask, causal=True, p=0.1).flatten(2)
        elif self.name == "flash_attention":
            y = self.child(x, self.mask)[0]
        elif self.name == "fused_mlp":
            y = self.child(x)
        elif self.name == "bias_gelu":
            y = op.bias_gelu(x, self.bias)
        elif self.name == "new_gelu":
            y = op.new_gelu(x)
        elif self.name == "bias_dropout":
            y = op.bias_dropout(x, self.bias, 0.1)
        elif self.name == "bias_dropout_residual":
            y = op.bias_dropout_residual(x, self.bias, x.flip(1), 0.1)
        elif self.name == "layer_norm":
            y = op.bias_dropout_residual_layer_norm(x, self.bias, x.flip(1), self.weight,
                                                    self.shift, 0.1)
        else:
            y = op.vocab_parallel_cross_entropy(x, self.target, 0.1)
        return y * 0.5 + 1


@pytest.mark.parametrize("grad", [True, False])
@pytest.mark.parametrize("name", ["attention", "flash_attention", "fused_mlp", "bias_gelu",
                                  "new_gelu", "bias_dropout", "bias_dropout_residual",
                                  "layer_norm", "cross_entropy"])
def test_traced_ops_compute_on_their_inputs(name, grad):
    """`torch.jit.trace` keeps an op as an operation: the traced module gives what the module gives
    on other inputs than the example, its dropout draws again, and gradients flow through it."""
    m = _AmongTorchOperations(name).cuda()
    with torch.set_grad_enabled(grad):
        traced = torch.jit.trace(m, torch.randn(2, 24, 64, device="cuda"), check_trace=False)
        x = torch.randn(2, 24, 64, device="cuda", requires_grad=grad)
        torch.cuda.manual_seed(3)
        wanted = m(x)
        torch.cuda.manual_seed(3)
        got = traced(x)
    assert torch.equal(got, wanted)
    if grad:
        into = [x, *m.parameters()]
        up = torch.randn_like(wanted)
        for a, r in zip(torch.autograd.grad(got, into, up, allow_unused=True),
                        torch.autograd.grad(wanted, into, up, allow_unused=True)):
            assert (a is None) == (r is None) and (a is None or torch.equal(a, r))
