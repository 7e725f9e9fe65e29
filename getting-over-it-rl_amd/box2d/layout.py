"""Batches of States on the GPU in the kernels' worlds-minor layout, and back.

A device State has the reference's field names and logical shapes (N, *inner) (goi_jax/box2d/world.py:70-174), as
torch tensors whose storage is worlds-minor: leaf L with inner shape S is one contiguous (prod(S), pitch) buffer
viewed as (N, *S) with stride 1 on the world axis. `state_view` hands those buffers to the C ABI without copies.
"""
import array
import ctypes
import functools
import operator

import numpy as np
import torch
from torch.autograd import forward_ad

from . import world as wd
from ._abi import GoiStateView

_TORCH = {np.dtype(np.float32): torch.float32, np.dtype(np.int32): torch.int32, np.dtype(bool): torch.bool}


def _dtype(dt):
    return _TORCH[np.dtype(dt)]


def packed_words(dims):
    """The packed layout of capacities dims = (B, R, J, C): words[l] = 4-byte words per unit of pitch before leaf l
    (each leaf's per-world bytes rounded up to a multiple of 4), words[-1] the whole; the library's goi_packed_layout
    gives the same table."""
    words = [0]
    for _, _, dt, inner in wd.LEAVES:
        nbytes = int(np.prod(wd.leaf_shape(inner, dims), dtype=np.int64)) * np.dtype(dt).itemsize
        words.append(words[-1] + (nbytes + 3) // 4)
    return words


@functools.lru_cache(maxsize=64)
def _spec(n, dims, pitch):
    """What the leaves of n worlds of capacities dims with a pitch look like, in ABI order: dtypes, shapes, strides
    (worlds-minor), and their byte offsets as the consecutive parts of one buffer, with that buffer's bytes, and the
    offsets in elements."""
    dtypes, shapes, strides = [], [], []
    for _, _, dt, inner in wd.LEAVES:
        shape = wd.leaf_shape(inner, dims)
        want, acc = [], pitch
        for d in reversed(shape):
            want.insert(0, acc)
            acc *= d
        dtypes.append(_dtype(dt))
        shapes.append((n,) + shape)
        strides.append((1, *want))
    offsets = [4 * w * pitch for w in packed_words(dims)]
    at = [o // dt.itemsize for o, dt in zip(offsets, dtypes)]
    return dtypes, shapes, strides, offsets[:-1], offsets[-1], at


def _traced():
    """Whether the operations are recorded or rewritten (a dispatch mode, a functorch transform, torch.jit.trace,
    torch.compile): one buffer's leaves alias it in ways those do not follow, so each leaf is then a tensor by itself."""
    return (torch.compiler.is_compiling() or torch.jit.is_tracing() or torch._C._len_torch_dispatch_stack() > 0
            or torch._C._functorch.peek_interpreter_stack() is not None)


def _carve(buf, n, dims, pitch):
    """The State whose leaves are the consecutive parts of the byte buffer buf. Each leaf is a tensor of its own to autograd
    (.data, then set to its part): as views of one tensor they would share its version counter and its graph, so that a
    write into one leaf spoiled what a backward pass saved of another."""
    dtypes, shapes, strides, _, _, at = _spec(n, dims, pitch)
    store = buf.untyped_storage()
    typed = {dt: buf.view(dt) for dt in (torch.float32, torch.int32, torch.bool)}
    return wd.from_leaves([typed[dt].data.set_(store, o, sh, st) for dt, o, sh, st in zip(dtypes, at, shapes, strides)])


def empty_device_state(n, dims, device="cuda", pitch=None, packed=True):
    """An uninitialised device State of n worlds with capacities dims = (B, R, J, C), pitch n by default. The leaves
    are by default the consecutive parts of one buffer, which a clone copies whole; with a pitch that is a multiple of
    64 that is the packed layout, which lets the step address every leaf from one base pointer. A leaf that a program
    keeps then keeps the State's whole buffer, and torch.save of a leaf writes all of it: keep or save a clone() of the
    leaf. packed=False gives one buffer per leaf, and so does code that is traced (_traced)."""
    pitch = n if pitch is None else pitch
    dims = tuple(dims)
    if packed and pitch > 0 and not _traced():
        return _carve(torch.empty(_spec(n, dims, pitch)[4], dtype=torch.uint8, device=device), n, dims, pitch)
    vals = []
    for _, _, dt, inner in wd.LEAVES:
        shape = wd.leaf_shape(inner, dims)
        buf = torch.empty(tuple(shape) + (pitch,), dtype=_dtype(dt), device=device)
        vals.append(buf[..., :n].movedim(-1, 0))
    return wd.from_leaves(vals)


def to_device(state, device="cuda", pitch=None, packed=True):
    """A batched numpy State (leading world axis) to a device State (packed by default, as empty_device_state)."""
    leaves = wd.leaves(state)
    n = np.asarray(leaves[0]).shape[0]
    dims = wd.dims(state)
    out = empty_device_state(n, dims, device, pitch, packed)
    for dst, src in zip(wd.leaves(out), leaves):
        src = np.asarray(src)
        dst.copy_(torch.from_numpy(np.ascontiguousarray(src)).to(device))
    return out


def to_host(state):
    """A device State to a batched numpy State (contiguous, batch-major)."""
    return wd.from_leaves([np.ascontiguousarray(t.detach().cpu().numpy()) for t in wd.leaves(state)])


def clone(state):
    """A deep copy of a device State in the same layout."""
    return clone_view(state)[1]()


def clone_view(state):
    """A State's copy as (its GoiStateView, a function that returns the State): a caller that launches work on the copy
    does so before the copy's 71 tensors are made. The view is None for a State that state_view would not take."""
    leaves = wd.leaves(state)
    n = leaves[0].shape[0]
    dims = wd.dims(state)
    found = _match(state, leaves, n, dims) if _memory_is_all(leaves) else None
    buf = None if found is None else _copy_buffer(leaves, n, dims, *found)
    if buf is not None:
        pitch, base = found[0], buf.data_ptr()
        view = _view(n, dims, pitch, [base + o for o in _spec(n, dims, pitch)[3]]) if buf.is_cuda else None
        return view, lambda: _carve(buf, n, dims, pitch)
    out = empty_device_state(n, dims, leaves[0].device)
    for dst, src in zip(wd.leaves(out), leaves):
        dst.copy_(src)
    return None, lambda: out


def _memory_is_all(leaves):
    """Whether a copy of the leaves' memory copies all they are. A leaf that requires grad is copied as a leaf, so that its
    copy has it as its gradient's source, and so is every leaf inside a forward-mode level, where it may have a tangent,
    of a tensor subclass, which may see the copy, and in traced code."""
    return (not _traced() and forward_ad._current_level < 0 and not any(map(_REQUIRES_GRAD, _FLOATS(leaves)))
            and list(map(type, leaves)) == _PLAIN)


def _copy_buffer(leaves, n, dims, pitch, ptrs):
    """A copy of the one buffer whose consecutive parts the (checked) leaves are, by a single device copy, or None where
    the leaves are not laid out so, or are the first few worlds of a much larger buffer: the copy holds all of it, so more
    padding than worlds is copied only up to 1 MiB (16 of 65,536 rig worlds would hold 373 MB)."""
    if pitch <= 0:
        return None
    _, _, _, offsets, nbytes, _ = _spec(n, dims, pitch)
    if pitch > 2 * n and nbytes > 1 << 20:
        return None
    base = ptrs[0]
    if ptrs != [base + o for o in offsets]:
        return None
    store = leaves[0].untyped_storage()
    start = base - store.data_ptr()
    if store.nbytes() - start < nbytes:
        return None
    src = torch.empty(0, dtype=torch.uint8, device=leaves[0].device).set_(store, start, (nbytes,))
    return torch.empty_like(src).copy_(src)


def pitch_of(state):
    """The worlds-minor pitch of a device State's leaves."""
    t = state.bodies.xf_p
    return t.stride(-1) if t.dim() > 1 else t.shape[0]


_PLAIN = [torch.Tensor] * len(wd.LEAVES)
_FLOATS = operator.itemgetter(*[k for k, leaf in enumerate(wd.LEAVES) if np.dtype(leaf[2]) == np.float32])
_SHAPE, _DTYPE, _DEVICE, _REQUIRES_GRAD = map(operator.attrgetter, ("shape", "dtype", "device", "requires_grad"))


def _match(state, leaves, n, dims):
    """(pitch, leaf addresses) of a State in the worlds-minor layout on one device, None for anything else. The leaves'
    types, shapes, strides and devices are compared as whole lists."""
    try:
        pitch, device = state.bodies.xf_p.stride(-1), leaves[0].device
        if pitch < n:
            return None
        dtypes, shapes, strides, _, _, _ = _spec(n, dims, pitch)
        if (list(map(_DTYPE, leaves)) == dtypes and list(map(_SHAPE, leaves)) == shapes
                and list(map(torch.Tensor.stride, leaves)) == strides
                and list(map(_DEVICE, leaves)) == [device] * len(leaves)):
            return pitch, list(map(torch.Tensor.data_ptr, leaves))
    except (AttributeError, TypeError, RuntimeError):  # not all tensors, or tensors without memory
        pass
    return None


def _check(state, leaves, n, dims):
    """_match on a GPU, or what is wrong: the leaves walked one by one for the message."""
    found = _match(state, leaves, n, dims)
    return found if found and leaves[0].device.type == "cuda" else _check_leaves(leaves, n, dims)


def _check_leaves(leaves, n, dims):
    pitch = None
    device = None
    for t, (_, name, dt, inner) in zip(leaves, wd.LEAVES):
        if not isinstance(t, torch.Tensor) or not t.is_cuda:
            raise ValueError(f"leaf {name}: not a GPU tensor (move the State with layout.to_device)")
        if device is not None and t.device != device:
            raise ValueError(f"leaf {name}: on {t.device}, other leaves on {device}")
        device = t.device
        if t.dtype != _dtype(dt):
            raise TypeError(f"leaf {name}: dtype {t.dtype}, expected {_dtype(dt)}")
        shape = (n,) + wd.leaf_shape(inner, dims)
        if tuple(t.shape) != shape:
            raise ValueError(f"leaf {name}: shape {tuple(t.shape)}, expected {shape}")
        if t.dim() > 1:
            p = t.stride(-1)
            want, acc = [1], p
            for d in reversed(shape[1:]):
                want.insert(1, acc)
                acc *= d
            if tuple(t.stride()) != tuple(want) or p < n or (pitch is not None and p != pitch):
                raise ValueError(f"leaf {name}: not in the worlds-minor layout (strides {t.stride()})")
            pitch = p
        elif t.stride(0) != 1:
            raise ValueError(f"leaf {name}: world stride must be 1")
    return n if pitch is None else pitch, [t.data_ptr() for t in leaves]


def _view(n, dims, pitch, ptrs):
    v = GoiStateView()
    v.n_worlds = n
    v.pitch = pitch
    v.B, v.R, v.J, v.C = dims
    words = array.array("Q", ptrs)
    ctypes.memmove(v.leaf, words.buffer_info()[0], 8 * len(ptrs))
    return v


def state_view(state):
    """GoiStateView over a device State; checks the worlds-minor layout."""
    leaves = wd.leaves(state)
    n = leaves[0].shape[0]
    dims = wd.dims(state)
    pitch, ptrs = _check(state, leaves, n, dims)
    return _view(n, dims, pitch, ptrs)
