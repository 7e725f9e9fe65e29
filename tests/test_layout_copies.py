"""layout.clone and step() over every form of State they take: one buffer (any pitch), one buffer per leaf, a leaf that
lies elsewhere, tensors in another order or on the CPU. The copy must hold the same words in memory of its own."""
import numpy as np
import pytest

from util import b2, leaf_mismatches, wd

torch = pytest.importorskip("torch")


def _host_state(n):
    return b2.scenes.make_config(1, n)


def _copies(state, host):
    out = b2.layout.clone(state)
    assert leaf_mismatches(host, b2.layout.to_host(out)) == []
    src = {t.untyped_storage().data_ptr() for t in wd.leaves(state)} - {0}  # 0: no worlds, no memory
    assert not src & {t.untyped_storage().data_ptr() for t in wd.leaves(out)}
    assert [tuple(t.shape) for t in wd.leaves(out)] == [tuple(t.shape) for t in wd.leaves(state)]
    return out


@pytest.mark.parametrize("n,pitch,packed", [(1, None, True), (3, None, True), (64, None, True), (50, 64, True),
                                            (5, 9, False), (0, None, True)])
def test_clone_on_the_cpu(n, pitch, packed):
    _, _, st, _ = _host_state(max(n, 1))
    if n == 0:
        st = wd.from_leaves([x[:0] for x in wd.leaves(st)])
    _copies(b2.layout.to_device(st, "cpu", pitch, packed), st)


def _grad_flows(device, n):
    """A leaf that requires grad is the source of its copy's gradient, and the leaves are separate to autograd."""
    _, _, st, _ = _host_state(n)
    dev = b2.layout.to_device(st, device)
    x = torch.ones_like(dev.bodies.v).requires_grad_()
    dev.bodies.v.copy_(x)
    dev.bodies.w.zero_()
    assert dev.bodies.v.requires_grad and not dev.bodies.w.requires_grad
    out = b2.layout.clone(dev)
    assert not out.bodies.w.requires_grad
    (g,) = torch.autograd.grad(out.bodies.v.sum(), x)
    assert bool((g == 1).all())


@pytest.mark.parametrize("n", [3, 64])
def test_clone_keeps_autograd(n):
    _grad_flows("cpu", n)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [3, 64])
def test_clone_keeps_autograd_on_the_gpu(n):
    _grad_flows("cuda", n)


@pytest.mark.parametrize("n,k,whole", [(4096, 16, False), (4096, 2047, False), (4096, 2048, True), (64, 1, True)])
def test_clone_of_the_first_worlds(n, k, whole):
    """A State narrowed to its first worlds: the copy holds what those need, not the State that they are part of (whose
    padding is copied along where it is no more than the worlds, or small)."""
    one = _host_state(1)[2]
    dev = b2.layout.empty_device_state(n, wd.dims(one), "cpu")
    for dst, src in zip(wd.leaves(dev), wd.leaves(one)):
        dst.copy_(torch.from_numpy(np.ascontiguousarray(src)).expand(dst.shape))
    out = _copies(wd.from_leaves([t[:k] for t in wd.leaves(dev)]), wd.batch(wd.from_leaves([x[0] for x in wd.leaves(one)]), k))
    held = sum({t.untyped_storage().data_ptr(): t.untyped_storage().nbytes() for t in wd.leaves(out)}.values())
    need = 4 * b2.layout.packed_words(wd.dims(one))[-1]
    assert held == need * (n if whole else k)


@pytest.mark.parametrize("n", [3, 64])
@pytest.mark.parametrize("copied", [False, True])
def test_a_write_into_a_leaf_leaves_the_others(n, copied):
    """A backward pass may use what it saved of a leaf (a mask, an index, a factor) after another leaf was written."""
    dev = b2.layout.to_device(_host_state(n)[2], "cpu")
    dev = b2.layout.clone(dev) if copied else dev
    x = torch.ones(n, dev.contacts.touching.shape[1], requires_grad=True)
    mask, at, by = dev.contacts.touching, dev.contacts.count, dev.contacts.friction
    versions = [t._version for t in wd.leaves(dev)]
    loss = (torch.where(mask, x, 2 * x) + x[torch.arange(n)[:, None], at.long()] + x * by).sum()
    for leaf in (dev.new_fixture, dev.next_key, dev.bodies.v):
        leaf.zero_()
    loss.backward()
    assert x.grad is not None
    written = {k for k, t in enumerate(wd.leaves(dev)) if t._version != versions[k]}
    assert written == {k for k, t in enumerate(wd.leaves(dev)) if any(t is w for w in (dev.new_fixture, dev.next_key,
                                                                                       dev.bodies.v))}


def test_leaves_in_inference_mode():
    with torch.inference_mode():
        _copies(b2.layout.to_device(_host_state(3)[2], "cpu"), _host_state(3)[2])


@pytest.mark.parametrize("n,pitch", [(3, None), (64, None), (5, 9)])
def test_clone_keeps_a_tangent(n, pitch):
    """Inside a forward-mode level a leaf's tangent is copied with it."""
    _, _, st, _ = _host_state(n)
    dev = b2.layout.to_device(st, "cpu", pitch)
    with torch.autograd.forward_ad.dual_level():
        v = torch.autograd.forward_ad.make_dual(dev.bodies.v, torch.full_like(dev.bodies.v, 2.0))
        out = b2.layout.clone(dev._replace(bodies=dev.bodies._replace(v=v)))
        got = torch.autograd.forward_ad.unpack_dual(out.bodies.v)
        assert got.tangent is not None and bool((got.tangent == 2.0).all())
        assert torch.equal(got.primal, dev.bodies.v)


@pytest.mark.parametrize("n", [3, 64])
@pytest.mark.parametrize("how", ["make_fx", "functionalize", "jit", "compile"])
def test_clone_is_traced(n, how):
    """A traced clone copies its inputs at every call, not those that it was traced with."""
    from torch.fx.experimental.proxy_tensor import make_fx

    def ones(k):
        return [t.fill_(k) for t in wd.leaves(b2.layout.to_device(_host_state(n)[2], "cpu"))]  # parts of one buffer

    def copy(*leaves):
        return tuple(wd.leaves(b2.layout.clone(wd.from_leaves(list(leaves)))))

    traced = {"make_fx": lambda: make_fx(copy)(*ones(0)), "functionalize": lambda: torch.func.functionalize(copy),
              "jit": lambda: torch.jit.trace(copy, tuple(ones(0)), check_trace=False),
              "compile": lambda: torch.compile(copy, backend="eager")}[how]()
    given = ones(1)
    got = traced(*given)
    assert all(torch.equal(a, b) and a.data_ptr() != b.data_ptr() for a, b in zip(got, given))


def test_clone_of_a_subclass():
    """A leaf of a tensor subclass sees its copy."""
    class Seen(torch.Tensor):
        calls = []

        @classmethod
        def __torch_function__(cls, func, types, args=(), kwargs=None):
            cls.calls.append(func.__name__)
            return super().__torch_function__(func, types, args, kwargs or {})

    dev = b2.layout.to_device(_host_state(3)[2], "cpu")
    b2.layout.clone(dev._replace(bodies=dev.bodies._replace(v=dev.bodies.v.as_subclass(Seen))))
    assert "copy_" in Seen.calls


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["one", "odd", "pitch", "leaves", "elsewhere", "batch_major", "double"])
def test_clone_and_step_on_the_gpu(oracle, case):
    n = {"one": 1, "odd": 37, "pitch": 50}.get(case, 64)
    s, m, st, cfg = _host_state(n)
    dev = b2.layout.to_device(st, "cuda", 64 if case == "pitch" else None, case != "leaves")
    if case == "elsewhere":  # one leaf replaced by a tensor of its own, in the same layout
        key = dev.contacts.key
        dev = dev._replace(contacts=dev.contacts._replace(key=torch.empty_strided(key.shape, key.stride(), dtype=key.dtype,
                                                                                  device="cuda").copy_(key)))
    elif case == "batch_major":  # state_view refuses it, a copy lays it out afresh
        dev = wd.from_leaves([t.contiguous() for t in wd.leaves(dev)])
        with pytest.raises(ValueError):
            b2.layout.state_view(dev)
    elif case == "double":
        dev = dev._replace(bodies=dev.bodies._replace(w=dev.bodies.w.double()))
        with pytest.raises(TypeError):
            b2.layout.state_view(dev)
    out = _copies(dev, st) if case != "double" else b2.layout.clone(dev)
    if case == "pitch":
        assert b2.layout.pitch_of(out) == 64
    ref = oracle.step(m, st, s, cfg.dt)
    stepped = b2.step(m, dev, s, cfg.dt)
    assert leaf_mismatches(ref, b2.layout.to_host(stepped)) == []
    b2.step_(m, out, s, cfg.dt)
    assert leaf_mismatches(ref, b2.layout.to_host(out)) == []
    if case != "double":
        assert leaf_mismatches(st, b2.layout.to_host(dev)) == []  # the input as it was
