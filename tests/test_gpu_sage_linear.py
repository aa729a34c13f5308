"""The dense part of the GraphSAGE layer as one kernel each way, against float64; and which calls keep the module's own
operators."""
import pytest

torch = pytest.importorskip("torch")

if torch.cuda.is_available():
    import f2cgt_amd
    from f2cgt_amd import pipeline

pytestmark = pytest.mark.gpu


def _inputs(m, k0, k1, n, seed=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed + m + 7 * n)
    x0, x1 = torch.randn((m, k0), generator=g, device="cuda"), torch.randn((m, k1), generator=g, device="cuda")
    w0 = (torch.randn((n, k0), generator=g, device="cuda") / k0 ** 0.5).requires_grad_()
    w1 = (torch.randn((n, k1), generator=g, device="cuda") / k1 ** 0.5).requires_grad_()
    b = torch.randn((n,), generator=g, device="cuda").requires_grad_()
    return x0, x1, w0, w1, b, torch.randn((m, n), generator=g, device="cuda")


@pytest.mark.parametrize("m,k0,k1,n", [(1, 4, 4, 1), (31, 32, 36, 33), (32, 4, 100, 32), (33, 64, 28, 70), (1024, 128, 128, 256),
                                       (1025, 100, 100, 5), (2500, 12, 200, 31), (4000, 260, 36, 64)])
@pytest.mark.parametrize("relu", [True, False])
def test_output_and_gradients_against_float64(m, k0, k1, n, relu):
    lib = f2cgt_amd.load()
    x0, x1, w0, w1, b, g = _inputs(m, k0, k1, n)
    out = lib.sage_linear(x0, x1, w0, w1, b, relu)
    out.backward(g)
    X0, X1, W0, W1, B, G = (t.detach().double() for t in (x0, x1, w0, w1, b, g))
    z = X0 @ W0.t() + X1 @ W1.t() + B
    unit = 2.0 ** -24
    # a sum of k products, each rounded, partial sums within the sum of the magnitudes; any order
    size = X0.abs() @ W0.abs().t() + X1.abs() @ W1.abs().t() + B.abs()
    assert bool(((out.double() - (z.clamp(min=0) if relu else z)).abs() <= (k0 + k1 + 4) * unit * size).all())
    if relu:
        G = torch.where(out.detach() <= 0, 0.0, G)
    for got, want, size in ((w0.grad, G.t() @ X0, G.abs().t() @ X0.abs()), (w1.grad, G.t() @ X1, G.abs().t() @ X1.abs()),
                            (b.grad, G.sum(0), G.abs().sum(0))):
        assert bool(((got.double() - want).abs() <= (m + 4) * unit * size).all())


def test_special_values_and_absent_parts():
    lib = f2cgt_amd.load()
    x0, x1, w0, w1, b, g = _inputs(40, 8, 12, 6)
    x0[3, 2], x0[5, 0] = float("nan"), float("inf")
    out = lib.sage_linear(x0, x1, w0, w1, b, True)
    want = torch.relu(torch.nn.functional.linear(x0, w0, b) + torch.nn.functional.linear(x1, w1))
    assert torch.equal(out.isnan(), want.isnan()) and bool(out[3].isnan().all())
    assert torch.equal(out.isinf(), want.isinf())
    w1.requires_grad_(False)
    out = lib.sage_linear(x0[10:], x1[10:], w0, w1, None, False)     # no bias; a weight without a gradient
    out.backward(g[10:])
    assert w0.grad is not None and w1.grad is None and b.grad is None
    torch.testing.assert_close(w0.grad, g[10:].t() @ x0[10:], rtol=1e-5, atol=1e-4)
    with torch.no_grad():
        assert not lib.sage_linear(x0, x1, w0, w1, b, True).requires_grad


# columns with and without a rest of sixteen, and past what the kernel takes; a minibatch's rows
@pytest.mark.parametrize("k0,k1", [(128, 128), (96, 96), (100, 100), (64, 28), (36, 48), (260, 36), (256, 256)])
@pytest.mark.parametrize("m,n", [(500, 128), (1024, 256), (3001, 128), (4096, 64)])
@pytest.mark.parametrize("relu", [True, False])
@pytest.mark.parametrize("with_bias", [True, False])
def test_a_pass_that_is_differentiated_has_the_operators_values(m, k0, k1, n, relu, with_bias):
    """Bit for bit: next to zero another last bit would be another mask of the gradient."""
    x0, x1, w0, w1, b, _ = _inputs(m, k0, k1, n)
    got = f2cgt_amd.load().sage_linear(x0, x1, w0, w1, b if with_bias else None, relu)
    want = torch.nn.functional.linear(x0, w0, b if with_bias else None) + torch.nn.functional.linear(x1, w1)
    assert torch.equal(got, torch.relu(want) if relu else want)


def test_passes_of_many_rows_are_differentiated_by_the_operators():
    x0, x1, w0, w1, b, _ = _inputs(4097, 8, 8, 4)
    lib = f2cgt_amd.load()
    assert lib.sage_linear(x0, x1, w0, w1, b, True) is None and lib.sage_linear(x0[1:], x1[1:], w0, w1, b, True) is not None
    with torch.no_grad():
        out = lib.sage_linear(x0, x1, w0, w1, b, True)
    torch.testing.assert_close(out, torch.relu(torch.nn.functional.linear(x0, w0, b) + torch.nn.functional.linear(x1, w1)),
                               rtol=1e-5, atol=1e-5)


def test_gradient_of_the_gradient():
    lib = f2cgt_amd.load()
    x0, x1, w0, w1, b, g = _inputs(50, 8, 8, 7)
    g.requires_grad_()
    got = torch.autograd.grad(lib.sage_linear(x0, x1, w0, w1, b, True), (w0, b), g, create_graph=True)
    want = torch.autograd.grad(torch.relu(torch.nn.functional.linear(x0, w0, b) + torch.nn.functional.linear(x1, w1)), (w0, b), g,
                               create_graph=True)
    for a, c in zip(got, want):
        torch.testing.assert_close(a, c, rtol=1e-5, atol=1e-4)
    (gg,) = torch.autograd.grad(got[0].square().sum(), g)
    (ww,) = torch.autograd.grad(want[0].square().sum(), g)
    torch.testing.assert_close(gg, ww, rtol=1e-4, atol=1e-2)


def test_calls_left_to_the_modules_operators():
    """Each is what the layer did without the kernel: the layer's result is that of its two Linears."""
    lib = f2cgt_amd.load()
    x0, x1, w0, w1, b, _ = _inputs(64, 16, 16, 8)
    take = lambda *a: lib.sage_linear(*a) is not None
    assert take(x0, x1, w0, w1, b, True)
    assert not take(x0.double(), x1.double(), w0.double(), w1.double(), b.double(), True)
    assert not take(x0.cpu(), x1.cpu(), w0.cpu(), w1.cpu(), b.cpu(), True)
    assert not take(x0.clone().requires_grad_(), x1, w0, w1, b, True)         # the input is differentiated
    assert not take(x0.t().contiguous().t(), x1, w0, w1, b, True)             # not dense rows
    assert not take(x0[:0], x1[:0], w0, w1, b, True)
    assert not take(x0[:, :15].contiguous(), x1, w0[:, :15].contiguous(), w1, b, True)
    assert not take(x0.reshape(-1)[1:1 + 63 * 16].view(63, 16), x1[:63], w0, w1, b, True)   # 4 bytes off
    assert not take(x0, x1[:63], w0, w1, b, True) and not take(x0, x1, w0[:7], w1, b, True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not take(x0, x1, w0, w1, b, True)
    with torch.autograd.forward_ad.dual_level():
        assert not take(x0, x1, w0, w1, b, True)
    seen = []
    torch.func.grad(lambda w: (seen.append(take(x0, x1, w, w1, b, True)), w.sum())[1])(w0.detach())
    torch.func.vmap(lambda w: (seen.append(take(x0, x1, w, w1, b, True)), w)[1])(w0.detach()[None])
    assert seen == [False, False]
    from torch.utils.flop_counter import FlopCounterMode
    with FlopCounterMode(display=False):
        assert not take(x0, x1, w0, w1, b, True)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t.shape) or t.cpu(), lambda t: t.cuda()):
        out = lib.sage_linear(x0, x1, w0, w1, b, True)
    out.sum().backward()                                                      # the saved tensors went through the hooks
    assert len(seen) == 5 and torch.allclose(b.grad, (out > 0).sum(0).float())


def test_layer_equals_its_linears_with_hooks_and_without():
    torch.manual_seed(0)
    conv = pipeline.MySAGEConv(16, 8, "mean", None, activation=torch.relu).cuda()
    h = torch.randn((300, 16), device="cuda")
    indptr = torch.arange(0, 301, 3, device="cuda")
    indices = torch.randint(0, 300, (300,), device="cuda")
    plain = conv((indptr, indices), (h[:100], h))
    assert type(plain.grad_fn).__name__.startswith("CppNode") or "Sage" in plain.grad_fn.name()
    calls = []
    handle = conv.fc_neigh.register_forward_hook(lambda *a: calls.append(1))
    hooked = conv((indptr, indices), (h[:100], h))
    handle.remove()
    assert calls == [1]
    torch.testing.assert_close(plain, hooked, rtol=1e-5, atol=1e-5)
    scaled = torch.nn.utils.parametrizations.weight_norm(conv.fc_self)
    assert scaled is conv.fc_self
    torch.testing.assert_close(conv((indptr, indices), (h[:100], h)), plain, rtol=1e-5, atol=1e-5)
    conv.activation = torch.tanh
    out = conv((indptr, indices), (h[:100], h))
    assert float(out.detach().min()) < 0


def _against_the_operators(run, relu=True):
    """`run(out, parameters)` on the kernel's output and on the two Linears': the same gradients."""
    x0, x1, w0, w1, b, g = _inputs(300, 16, 24, 40)
    got = run(f2cgt_amd.load().sage_linear(x0, x1, w0, w1, b, relu), (w0, w1, b), g)
    z = torch.nn.functional.linear(x0, w0, b) + torch.nn.functional.linear(x1, w1)
    want = run(torch.relu(z) if relu else z, (w0, w1, b), g)
    for a, c in zip(got, want):
        assert a.shape == c.shape
        torch.testing.assert_close(a, c, rtol=1e-5, atol=1e-4)


@pytest.mark.parametrize("relu", [True, False])
def test_batched_gradients(relu):
    _against_the_operators(lambda out, p, g: torch.autograd.grad(out, p, torch.stack([g, 2 * g, g.flip(0)]), is_grads_batched=True), relu)


def test_gradients_that_are_not_plain_memory():
    """A view that negates, rows that are one row, columns apart: what an operator in between may hand on."""
    for form in (torch._neg_view, lambda g: g[:1].expand_as(g), lambda g: g.t().contiguous().t()):
        _against_the_operators(lambda out, p, g: torch.autograd.grad(out, p, form(g)))
    zero = torch._efficientzerotensor((300, 40), device="cuda")
    _against_the_operators(lambda out, p, g: torch.autograd.grad(out, p, zero))


def test_a_mode_around_the_backward_pass_sees_its_operators():
    from torch.utils._python_dispatch import TorchDispatchMode
    seen = []

    class Seen(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))

    def run(out, p, g):
        with Seen():
            return torch.autograd.grad(out, p, g)
    x0, x1, w0, w1, b, g = _inputs(300, 16, 24, 40)
    run(f2cgt_amd.load().sage_linear(x0, x1, w0, w1, b, True), (w0, w1, b), g)
    assert sum("mm" in name for name in seen) == 2 and any("threshold_backward" in name for name in seen)
    _against_the_operators(run)


def test_saved_tensors_that_come_back_in_another_layout():
    x0, x1, w0, w1, b, g = _inputs(300, 16, 24, 40)
    want = torch.autograd.grad(f2cgt_amd.load().sage_linear(x0, x1, w0, w1, b, True), (w0, w1, b), g)
    for unpack in (lambda t: t.t().contiguous().t(), lambda t: torch.cat([t.new_zeros(1), t.reshape(-1)])[1:].view(t.shape)):
        with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
            out = f2cgt_amd.load().sage_linear(x0, x1, w0, w1, b, True)
        for a, c in zip(torch.autograd.grad(out, (w0, w1, b), g), want):
            torch.testing.assert_close(a, c, rtol=1e-5, atol=1e-4)


def test_subclasses_with_operators_of_their_own_keep_them():
    calls = []

    class Tagged(torch.Tensor):
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            calls.append(getattr(func, "__name__", str(func)))
            return super().__torch_function__(func, types, args, kwargs or {})

    class Bare(torch.Tensor):        # results of its operators are of its class
        pass

    lib = f2cgt_amd.load()
    x0, x1, w0, w1, b, _ = _inputs(300, 16, 16, 40)
    for kind in (Tagged, Bare):
        for at in range(5):
            args = [x0, x1, w0, w1, b]
            args[at] = args[at].detach().as_subclass(kind)
            assert lib.sage_linear(*args, True) is None, (kind, at)
    conv = pipeline.MySAGEConv(16, 40, "mean", None, activation=torch.relu).cuda()
    indptr, indices = torch.arange(0, 301, device="cuda"), torch.arange(0, 300, device="cuda")
    plain = conv((indptr, indices), (x0, x1))
    del calls[:]
    got = conv((indptr, indices), (x0.as_subclass(Tagged), x1))
    assert isinstance(got, Tagged) and "linear" in calls and type(plain) is torch.Tensor
    torch.testing.assert_close(got.as_subclass(torch.Tensor), plain, rtol=1e-5, atol=1e-5)
    parameter = torch.nn.Parameter(w0.detach())      # (a class of its own without operators)
    assert lib.sage_linear(x0, x1, parameter, w1, b, True) is not None


# few rows, few outputs, class counts and outputs of no whole tile, more columns than the kernel takes, many rows
_SHAPES = [(m, k0, k1, n) for m in (1, 2, 33, 100, 256, 257, 300, 1000, 2049, 4096)
           for n in (1, 5, 16, 17, 40, 41, 47, 128, 172, 256, 349, 600)
           for k0, k1 in ((128, 128), (116, 84), (100, 4), (52, 96), (36, 16), (8, 12), (132, 64))]
_MANY = [(m, k, k, n) for m in (4097, 8192, 20000, 30840, 30841, 70000) for n in (8, 17, 47, 64, 128, 256) for k in (128, 100, 36, 600)]


@pytest.mark.parametrize("relu", [True, False])
def test_values_are_the_operators_at_any_size(relu):
    """Bit for bit, with gradients (where the pass is taken) and without: a kernel that adds in another order than the
    library's at some size, or a library that does, shows here."""
    lib = f2cgt_amd.load()
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    pool = [torch.randn(max(m * k for m, k, *_ in _MANY), generator=g, device="cuda") for _ in range(2)]
    weights = [torch.randn(600 * 600, generator=g, device="cuda") / 10 for _ in range(2)]
    bias = torch.randn(600, generator=g, device="cuda")
    bad = []
    for m, k0, k1, n in _SHAPES + _MANY:
        x0, x1 = pool[0][:m * k0].view(m, k0), pool[1][:m * k1].view(m, k1)
        w0, w1, b = weights[0][:n * k0].view(n, k0), weights[1][:n * k1].view(n, k1), bias[:n]
        want = torch.nn.functional.linear(x0, w0, b) + torch.nn.functional.linear(x1, w1)
        want = torch.relu(want) if relu else want
        if not torch.equal(lib.sage_linear(x0, x1, w0, w1, b, relu), want):
            bad.append((m, k0, k1, n))
        if m <= 4096:
            out = lib.sage_linear(x0, x1, w0.requires_grad_(), w1, b, relu)
            if out is not None and not torch.equal(out.detach(), want):
                bad.append((m, k0, k1, n, "differentiated"))
    assert not bad


@pytest.mark.parametrize("m", [100, 300, 1024, 2000, 4096])
def test_gradients_are_as_close_to_float64_as_the_operators(m):
    """Relative error (2-norm), the mean of forty inputs: of the bias's 256 sums and of the weights'."""
    lib = f2cgt_amd.load()
    err = torch.zeros((2, 2), dtype=torch.float64, device="cuda")
    for seed in range(40):
        x0, x1, w0, w1, b, g = _inputs(m, 8, 8, 256, seed)
        exact = (g.double().t() @ x0.double(), g.double().sum(0))
        for i, out in enumerate((lib.sage_linear(x0, x1, w0, w1, b, False),
                                 torch.nn.functional.linear(x0, w0, b) + torch.nn.functional.linear(x1, w1))):
            for j, (a, e) in enumerate(zip(torch.autograd.grad(out, (w0, b), g), exact)):
                err[i, j] += (a.double() - e).norm() / e.norm()
    # the mean of forty such errors is itself known to about 1 % (256 values each, of spread 1 about their size: 1 / sqrt(2 * 256 * 40))
    assert bool((err[0] <= 1.01 * err[1]).all()), (err / 40).tolist()


def test_several_threads_with_hooks():
    """The call runs without the interpreter's lock; hooks on saved tensors take it for themselves."""
    import threading
    lib = f2cgt_amd.load()
    x0, x1, w0, w1, b, g = _inputs(300, 16, 24, 40)
    want = torch.autograd.grad(lib.sage_linear(x0, x1, w0, w1, b, True), (w0, w1, b), g)
    torch.cuda.synchronize()
    same = []

    def work():
        with torch.cuda.stream(torch.cuda.Stream()):
            mine = [p.detach().clone().requires_grad_() for p in (w0, w1, b)]
            for _ in range(20):
                with torch.autograd.graph.saved_tensors_hooks(lambda t: [t], lambda kept: kept[0]):
                    out = lib.sage_linear(x0, x1, *mine, True)
                same.append(all(torch.equal(p, q) for p, q in zip(torch.autograd.grad(out, mine, g), want)))
            torch.cuda.current_stream().synchronize()
    threads = [threading.Thread(target=work) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert same == [True] * 80
