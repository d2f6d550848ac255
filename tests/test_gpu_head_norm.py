"""The head norms of q and k in one launch: against LayerNorm in 64 bits, and where the library's own modules keep the work."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _norm(D, dtype, dev, affine, seed, eps=1e-5):
    n = torch.nn.LayerNorm(D, eps=eps, elementwise_affine=affine).to(dev, dtype).requires_grad_(False)
    if affine:
        g = torch.Generator(device=dev).manual_seed(seed)
        n.weight.copy_(torch.randn(D, generator=g, device=dev) + 1)
        n.bias.copy_(torch.randn(D, generator=g, device=dev))
    return n


def _exact(n, x):
    w, b = (None, None) if n.weight is None else (n.weight.double(), n.bias.double())
    return torch.nn.functional.layer_norm(x.double(), n.normalized_shape, w, b, n.eps)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,N,H,D", [(1, 1, 1, 64), (1, 1, 1, 128), (1, 31, 1, 64), (1, 127, 1, 64), (1, 129, 1, 64), (2, 21, 3, 64),
                                     (1, 63, 1, 128), (1, 65, 1, 128), (2, 1001, 4, 64), (1, 777, 5, 128)])
@pytest.mark.parametrize("affine", [True, False])
def test_head_norms_against_64_bits(dev, dtype, B, N, H, D, affine):
    """Edges of the rows a workgroup takes (128 of 64 channels, 64 of 128).  Half a unit in the last place of the result, and
    of the sums in fp32 2^-20 of its terms' size: |x - mean| / std * |w| + |b|, below 2^4 here."""
    from paroatten_amd import _lib
    from paroatten_amd.cogvideox import _head_norms
    g = torch.Generator(device=dev).manual_seed(N + D)
    q, k = ((torch.randn(B, N, H, D, generator=g, device=dev) * s + m).to(dtype).transpose(1, 2) for s, m in ((1, 0), (0.3, 2)))
    nq, nk = _norm(D, dtype, dev, affine, 1), _norm(D, dtype, dev, affine, 2, eps=1e-3)
    assert _lib.ops().head_norm(q, k, nq.weight, nq.bias, nq.eps, nk.weight, nk.bias, nk.eps)
    ulp = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    for got, n, x in zip(_head_norms(nq, nk, q, k), (nq, nk), (q, k)):
        want = _exact(n, x)
        assert got.shape == x.shape and got.stride() == x.stride() and got.dtype == dtype
        assert ((got.double() - want).abs() <= ulp * want.abs() + 2.0 ** -16).all()
        library = n(x.transpose(1, 2)).transpose(1, 2)
        assert (got.double() - want).norm() <= 1.001 * (library.double() - want).norm() + 1e-12


def test_rows_without_variance_and_non_finite_rows(dev):
    from paroatten_amd.cogvideox import _head_norms
    D = 64
    q = torch.zeros(1, 5, 1, D, dtype=torch.float16, device=dev)
    q[0, 1] = 7.0
    q[0, 2, 0, 3] = float("nan")
    q[0, 3, 0, 3] = float("inf")
    q[0, 4] = torch.linspace(-60000, 60000, D)
    q = q.transpose(1, 2)
    n = _norm(D, torch.float16, dev, True, 3)
    got, same = _head_norms(n, n, q, q)
    want = n(q.transpose(1, 2)).transpose(1, 2)
    assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got.isnan(), same.isnan())
    assert torch.allclose(got[:, :, [0, 1, 4]].float(), want[:, :, [0, 1, 4]].float(), atol=2e-3, rtol=2e-3)


@pytest.mark.parametrize("ctypes", [False, True])
@pytest.mark.parametrize("kind", ["grad_of_the_input", "grad_of_the_weight", "autocast", "hook", "other_dtype", "strides", "one_norm",
                                  "mode", "width"])
def test_where_the_modules_keep_the_work(dev, kind, ctypes, monkeypatch):
    from torch.utils._python_dispatch import TorchDispatchMode

    from paroatten_amd import _lib
    from paroatten_amd import _ops as mirror
    from paroatten_amd import cogvideox as C
    D = 32 if kind == "width" else 64
    x = torch.randn(2, 9, 3, D, device=dev, dtype=torch.bfloat16)
    q, k = x.transpose(1, 2), (x * 2).transpose(1, 2)
    nq, nk, seen = _norm(D, torch.bfloat16, dev, True, 1), _norm(D, torch.bfloat16, dev, True, 2), []

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))
    if kind == "grad_of_the_input":
        q = x.clone().requires_grad_().transpose(1, 2)
    elif kind == "grad_of_the_weight":
        nk.requires_grad_(True)
    elif kind == "hook":
        nk.register_forward_hook(lambda *a: seen.append("hook"))
    elif kind == "other_dtype":
        nq, nk = nq.float(), nk.float()
        q, k = q.float(), k.float()
    elif kind == "strides":
        k = (x * 2).transpose(1, 2).contiguous()
    elif kind == "one_norm":
        nk = None
    class Ops:   # either form of the entry says no
        @staticmethod
        def head_norm(*args):
            r = (mirror if ctypes else compiled).head_norm(*args)
            return pytest.fail("the kernel was called") if r else r
    compiled = _lib.ops()
    monkeypatch.setattr(_lib, "ops", lambda: Ops)
    with torch.autocast("cuda", torch.bfloat16, enabled=kind == "autocast"):
        if kind == "mode":
            with Mode():
                got = C._head_norms(nq, nk, q, k)
        else:
            got = C._head_norms(nq, nk, q, k)
        want = nq(q), k if nk is None else nk(k)
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert got[0].requires_grad == (kind == "grad_of_the_input") and got[1].requires_grad == (kind == "grad_of_the_weight")
    assert bool(seen) == (kind in ("hook", "mode"))


@pytest.mark.parametrize("ctypes", [False, True])
@pytest.mark.parametrize("kind", ["tangent_of_the_input", "tangent_of_the_weight", "subclass", "subclass_of_the_weight", "negated_view",
                                  "vmap"])
def test_what_rides_on_a_tensor_is_kept(dev, kind, ctypes, monkeypatch):
    """With gradients off: forward-mode tangents, subclasses of tensors that know no dispatch, lazily negated views and batched tensors
    come out of the modules as they always did."""
    import torch.autograd.forward_ad as fw

    from paroatten_amd import _lib
    from paroatten_amd import _ops as mirror
    from paroatten_amd import cogvideox as C
    if ctypes:
        monkeypatch.setattr(_lib, "ops", lambda: mirror)
    D = 64
    x = torch.randn(2, 9, 3, D, device=dev, dtype=torch.float16)
    dx = torch.randn_like(x)
    nq, nk, seen = _norm(D, torch.float16, dev, True, 1), _norm(D, torch.float16, dev, True, 2), []

    class Sub(torch.Tensor):
        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            seen.append(func)
            return super().__torch_function__(func, types, args, kwargs or {})

    with torch.no_grad(), fw.dual_level():
        q, k = x.transpose(1, 2), (x * 2).transpose(1, 2)
        if kind == "tangent_of_the_input":
            k = fw.make_dual(x * 2, dx).transpose(1, 2)
        elif kind == "tangent_of_the_weight":
            del nq.weight
            nq.register_parameter("weight", None)
            nq.__dict__["_parameters"]["weight"] = fw.make_dual(torch.ones(D, device=dev, dtype=torch.float16), dx[0, 0, 0])
        elif kind == "subclass":
            q = q.as_subclass(Sub)
        elif kind == "subclass_of_the_weight":
            nk.__dict__["_parameters"]["weight"] = nk.weight.data.as_subclass(Sub)
        elif kind == "negated_view":
            q = torch._neg_view(x).transpose(1, 2)
        seen.clear()
        if kind == "vmap":
            got = torch.vmap(lambda a, b: C._head_norms(nq, nk, a, b))(q[None].repeat(2, 1, 1, 1, 1), k[None].repeat(2, 1, 1, 1, 1))
            got = [g[1] for g in got]
        else:
            got = C._head_norms(nq, nk, q, k)
        called = len(seen)
        want = [n(t.transpose(1, 2)).transpose(1, 2) for n, t in ((nq, q), (nk, k))]
        for g, w in zip(got, want):
            assert type(g) is type(w) and torch.allclose(g.as_subclass(torch.Tensor).float(), w.as_subclass(torch.Tensor).float(), atol=2e-3, rtol=2e-3)
            gt, wt = fw.unpack_dual(g.as_subclass(torch.Tensor)).tangent, fw.unpack_dual(w.as_subclass(torch.Tensor)).tangent
            assert (gt is None) == (wt is None) and (gt is None or torch.allclose(gt.float(), wt.float(), atol=2e-3, rtol=2e-3))
        assert any(fw.unpack_dual(w.as_subclass(torch.Tensor)).tangent is not None for w in want) == kind.startswith("tangent")
    assert (called > 0) == kind.startswith("subclass")
