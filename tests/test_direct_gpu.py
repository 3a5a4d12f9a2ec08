"""The native layer call (_direct.so) that Int8Linear.forward tries first: bit-identical to the Python paths, and it
steps aside (None) or refuses exactly where they decide."""
import gc
import threading

import pytest
import torch

pytestmark = pytest.mark.gpu


def _general(q, x):
    from pyraquant_amd import int8_exec as E

    E.DIRECT_CALLS = False
    try:
        return q(x)
    finally:
        E.DIRECT_CALLS = True


def _layer(cuda, K=1280, N=640, group=0, bias=True, rank=0):
    from pyraquant_amd import int8_exec as E
    from pyraquant_amd.workloads import make_linear

    return E.Int8Linear(make_linear(K, N, rank, bias), device=cuda, group_size=group)


@pytest.mark.parametrize("group", [0, 32])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(0, 1280), (1, 1280), (77, 1280), (2000, 1280), (1280,), (2, 3, 1280), (0, 3, 1280)])
def test_native_call_equals_python_paths(cuda, group, dtype, shape):
    from pyraquant_amd import _lib

    q = _layer(cuda, group=group)
    x = torch.randn(*shape, device=cuda).to(dtype)
    y = _lib.load_direct()(q.__dict__, q._buffers, x)
    assert isinstance(y, torch.Tensor) and y.shape == (*shape[:-1], 640) and y.dtype == dtype
    assert not y.requires_grad and y.is_contiguous()
    if x.numel():
        assert torch.equal(y, _general(q, x)) and torch.equal(q(x), y)


def test_native_call_steps_aside(cuda):
    """Views with other strides and alignments, other dtypes, devices and widths, tensor subclasses, layers with a
    low-rank branch, and buffers in a state the kernels do not read: None, and forward() answers (or raises) as the
    Python paths do."""
    from pyraquant_amd import _lib

    native = _lib.load_direct()
    q = _layer(cuda)
    wide = torch.randn(64, 2600, device=cuda).bfloat16()
    for x in (wide[:, :1280], wide[:, 8:1288]):                           # aligned slices are taken
        assert torch.equal(native(q.__dict__, q._buffers, x), _general(q, x))
    for x in (wide[:, 1:1281], wide[:, ::2][:, :1280], torch.randn(1280, 64, device=cuda).bfloat16().t(),
              torch.randn(4, 1288, device=cuda).bfloat16()[:, :1280][:, :].as_strided((4, 1280), (1284, 1))):
        assert native(q.__dict__, q._buffers, x) is None
        assert torch.equal(q(x), _general(q, x.contiguous()))
    for x, err in ((torch.randn(4, 1280, device=cuda), ValueError), (torch.randn(4, 1280).bfloat16(), AssertionError)):
        assert native(q.__dict__, q._buffers, x) is None
        with pytest.raises(err):
            q(x)
    assert native(q.__dict__, q._buffers, torch.randn(4, 1344, device=cuda).bfloat16()) is None

    class Sub(torch.Tensor):
        pass

    x = torch.randn(8, 1280, device=cuda).bfloat16()
    assert native(q.__dict__, q._buffers, x.as_subclass(Sub)) is None
    assert native(q.__dict__, q._buffers, None) is None
    r = _layer(cuda, rank=32)
    assert native(r.__dict__, r._buffers, x) is None and torch.equal(r(x), _general(r, x))
    for name, bad in (("w_scale", q.w_scale.double()), ("bias", q.bias.half()), ("weight_packed", None),
                      ("w_scale", q.w_scale.cpu()), ("bias", torch.zeros(1280, device=cuda)[::2])):
        p = _layer(cuda)
        p._buffers[name] = bad
        assert native(p.__dict__, p._buffers, x) is None, name
    with pytest.raises(RuntimeError):                                     # no storage: as data_ptr() raises in Python
        torch.func.vmap(q)(x.reshape(2, 4, 1280))


def test_native_call_reads_the_buffers_of_this_call(cuda):
    """Nothing is kept between calls: replaced buffers, swapped storage, and an attribute set on the instance."""
    q = _layer(cuda)
    x = torch.randn(100, 1280, device=cuda).bfloat16()
    y = q(x)
    q.w_scale.data = q.w_scale.data * 2                                   # the same object, another storage
    assert torch.equal(q(x), _general(q, x)) and not torch.equal(q(x), y)
    q.bias = None
    assert torch.equal(q(x), _general(q, x))
    x.requires_grad_(True)
    assert not q(x).requires_grad


def test_native_call_streams_threads_and_graphs(cuda):
    """Calls from several threads on streams of their own, each with its own allocations, and a captured call replayed
    between eager ones."""
    q = _layer(cuda)
    xs = [torch.randn(300 + 700 * i, 1280, device=cuda).bfloat16() for i in range(4)]
    refs = [_general(q, x) for x in xs]
    torch.cuda.synchronize()
    bad = []

    def work(i):
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            for _ in range(50):
                if not torch.equal(q(xs[i]), refs[i]):
                    bad.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    [t.start() for t in threads]
    [t.join() for t in threads]
    assert not bad
    for x, ref in ((xs[0][:20].clone(), refs[0][:20]), (xs[1], refs[1])):   # one kernel, and two
        g = torch.cuda.CUDAGraph()
        q(x)
        torch.cuda.synchronize()
        with torch.cuda.graph(g):
            y = q(x)
        for _ in range(3):
            y.zero_()
            g.replay()
            eager = q(x)
            torch.cuda.synchronize()
            assert torch.equal(y, ref) and torch.equal(eager, ref)


@pytest.mark.parametrize("M,swap_at", [(20, 0), (1500, 0), (1500, 1)])   # one kernel; two, and a workspace
def test_native_call_holds_its_tensors(cuda, M, swap_at):
    """A module given other buffers during the call (here by a dispatch mode, at one of the call's own allocations) does
    not take the old ones away from it: their memory is still theirs when the kernels are launched."""
    from torch.utils._python_dispatch import TorchDispatchMode

    q = _layer(cuda)
    names = ("weight_packed", "w_scale", "bias")
    x = torch.randn(M, 1280, device=cuda).bfloat16()
    ref = q(x)
    torch.cuda.synchronize()
    new = {n: torch.zeros_like(q._buffers[n]) for n in names}
    poison = []

    class Swap(TorchDispatchMode):
        calls = 0

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            out = func(*args, **(kwargs or {}))
            if func is torch.ops.aten.empty.memory_format:
                if self.calls == swap_at:
                    before = torch.cuda.memory_allocated()
                    q._buffers.update(new)
                    assert torch.cuda.memory_allocated() == before, "the call's tensors have been freed"
                    poison.extend(torch.full_like(t, 7) for t in new.values())
                self.calls += 1
            return out

    gc.collect()   # (other tests' cycles would count as freed here)
    with Swap() as mode:
        y = q(x)
    assert mode.calls == (1 if M < 100 else 2) and len(poison) == 3
    assert torch.equal(y, ref) and torch.equal(q(x), torch.zeros_like(ref))


@pytest.mark.parametrize("rank", [0, 32])
def test_buffers_made_parameters(cuda, rank):
    """A bias, or a low-rank factor, that the user has made an nn.Parameter is no longer a buffer and still counts."""
    from pyraquant_amd import _lib

    q = _layer(cuda, rank=rank)
    x = torch.randn(64, 1280, device=cuda).bfloat16()
    y = q(x)
    q.bias = torch.nn.Parameter(q.bias + 1)
    assert _lib.load_direct()(q.__dict__, q._buffers, x) is None
    assert torch.equal(q(x), _general(q, x)) and not torch.equal(q(x), y)
    if rank:
        p = _layer(cuda, rank=rank)
        p.lr_A = torch.nn.Parameter(p.lr_A)
        assert _lib.load_direct()(p.__dict__, p._buffers, x) is None
        assert torch.equal(p(x), y) and torch.equal(_general(p, x), y)


def test_native_call_is_loaded_for_its_own_layers_only(cuda, monkeypatch):
    """Where _direct.so does not load, layers it cannot take (a low-rank branch, no packed weights) run as ever; one it
    takes says so."""
    from pyraquant_amd import _lib
    from pyraquant_amd import int8_exec as E

    def missing():
        raise _lib.LibraryMissing("not built")

    monkeypatch.setattr(_lib, "load_direct", missing)
    monkeypatch.setattr(E, "_direct_linear", None)
    x = torch.randn(64, 1280, device=cuda).bfloat16()
    unpacked = _layer(cuda)
    unpacked.weight_packed = None
    for q in (_layer(cuda, rank=32), unpacked):
        assert torch.equal(q(x), _general(q, x))
    with pytest.raises(_lib.LibraryMissing):
        _layer(cuda)(x)


def test_native_call_allocates_as_the_python_path(cuda):
    """The workspace before the output, so that consecutive calls take the same workspace and outputs of their own; a
    layer of few rows allocates its output alone."""
    from torch.utils._python_dispatch import TorchDispatchMode

    class Sizes(TorchDispatchMode):
        def __init__(self):
            super().__init__()
            self.seen = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            out = func(*args, **(kwargs or {}))
            if func is torch.ops.aten.empty.memory_format:
                self.seen.append((out.dtype, out.numel()))
            return out

    for group, M in ((0, 20), (0, 1500), (32, 20), (32, 1500)):
        q = _layer(cuda, group=group)
        x = torch.randn(M, 1280, device=cuda).bfloat16()
        with Sizes() as native:
            q(x)
        with Sizes() as python:
            q._forward_direct(x)
        assert [d for d, _ in python.seen] == [torch.uint8, torch.bfloat16]
        assert native.seen == (python.seen[1:] if group == 0 and M < 100 else python.seen)
