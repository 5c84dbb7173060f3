"""The native host path of the frequent calls takes plain arguments only: everything else comes back as
"not taken" and meets the checks in Python, with the same errors as before."""
import pytest
import torch

from wmma_extension_amd import _lib, tcec
from wmma_extension_amd._lib import WmmaeError

NOT_TAKEN = 1


def test_what_is_not_plain_is_not_taken():
    calls = tcec._native()
    A = torch.zeros(8, 8)
    for name in ("sgemm", "sgemm_strided_batched", "sgemm_batched", "matmul_tn", "pack", "gemm_packed", "api_gemm",
                 "primitive_tiles"):
        assert getattr(calls, name)() == NOT_TAKEN
        assert getattr(calls, name)(*[None] * 17) == NOT_TAKEN
    ok = ["T", "N", 8, 8, 8, 1.0, A, 8, A, 8, 0.0, A, 8, 0, 0, None, 0]
    assert calls.sgemm(*ok) == NOT_TAKEN                      # tensors of the host
    for i, v in ((0, "TT"), (0, ""), (0, b"T"), (0, "Τ"), (2, 8.0), (2, 1 << 70), (3, 1 << 40), (5, "1"), (6, 5),
                 (15, [1]), (16, None), (16, 1.5)):
        assert calls.sgemm(*(ok[:i] + [v] + ok[i + 1:])) == NOT_TAKEN, (i, v)
    with pytest.raises(ValueError, match="device tensors"):
        tcec.sgemm(*ok[:13])
    with pytest.raises(ValueError, match="device tensors"):
        tcec.matmul_tn(A, A)


@pytest.fixture
def no_module(monkeypatch):
    """A package whose module was built for another torch, or not at all."""
    monkeypatch.setattr(torch, "__version__", torch.__version__ + ".other")
    monkeypatch.setattr(tcec, "_calls", None)


def test_a_package_without_the_module(no_module):
    """(built by the hipcc line alone): every call goes through the checks in Python, warned of once."""
    assert _lib.host_calls_path() != _lib.host_calls_path().replace(".other", "")
    A = torch.zeros(8, 8)
    with pytest.warns(RuntimeWarning, match="ctypes"):
        calls = tcec._native()
    assert tcec._native() is calls
    for name in ("sgemm", "sgemm_strided_batched", "sgemm_batched", "matmul_tn", "pack", "gemm_packed", "api_gemm",
                 "primitive_tiles"):
        assert getattr(calls, name)(A, 1) == NOT_TAKEN
    with pytest.raises(ValueError, match="device tensors"):
        tcec.sgemm("T", "N", 8, 8, 8, 1.0, A, 8, A, 8, 0.0, A, 8)
    with pytest.raises(ValueError, match="device tensors"):
        tcec.matmul_tn(A, A)


@pytest.mark.gpu
@pytest.mark.filterwarnings("ignore:.*ctypes.*:RuntimeWarning")
def test_results_without_the_module(tc, dev, monkeypatch):
    m, n, k = 96, 80, 160
    A, B, C = torch.rand((m, k), device=dev), torch.rand((n, k), device=dev), torch.zeros((n, m), device=dev)
    want = tc.matmul_tn(A, B)
    monkeypatch.setattr(torch, "__version__", torch.__version__ + ".other")
    monkeypatch.setattr(tcec, "_calls", None)
    assert torch.equal(tc.matmul_tn(A, B), want)
    tc.sgemm("T", "N", m, n, k, 1.0, A, k, B, k, 0.0, C, m)
    assert torch.equal(C, want)


@pytest.mark.gpu
def test_the_same_results_and_errors_on_either_path(tc, dev):
    m, n, k = 96, 80, 160
    A, B = torch.rand((m, k), device=dev), torch.rand((n, k), device=dev)
    want = tc.matmul_tn(A, B, out=torch.empty((n, m), device=dev))      # (an output of the caller: checked in Python)
    assert torch.equal(tc.matmul_tn(A, B), want)
    C = torch.zeros((n, m), device=dev)
    tc.sgemm("T", "N", m, n, k, 1, A, k, B, k, 0, C, m)
    assert torch.equal(C, want)
    # views that are not contiguous, numbers that are no plain floats, a parameter
    wide = torch.rand((m, k + 12), device=dev)
    view = wide[:, :k].copy_(A)
    C.zero_()
    tc.sgemm("T", "N", m, n, k, torch.tensor(1.0), view, k + 12, torch.nn.Parameter(B), k, 0.0, C, m)
    assert torch.equal(C, want)
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        stream.wait_stream(torch.cuda.default_stream())
        got = tc.matmul_tn(A, B)
    stream.synchronize()
    assert torch.equal(got, want)

    class Seen(torch.utils._python_dispatch.TorchDispatchMode):
        ops = ()

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.ops += (str(func),)
            return func(*args, **(kwargs or {}))
    with Seen() as seen:
        got = tc.matmul_tn(A, B)
    assert torch.equal(got, want) and any("empty" in o for o in seen.ops)
    with pytest.raises(ValueError, match="float32"):
        tc.sgemm("T", "N", m, n, k, 1.0, A.double(), k, B, k, 0.0, C, m)
    with pytest.raises(ValueError, match="bytes from its first element"):
        tc.sgemm("T", "N", m, n, k + 1, 1.0, A, k + 1, B, k + 1, 0.0, C, m)
    with pytest.raises(ValueError, match="device tensors"):
        tc.sgemm("T", "N", m, n, k, 1.0, A.cpu(), k, B, k, 0.0, C, m)
    with pytest.raises(AssertionError):
        tc.matmul_tn(A, B[:, :-1])
    for flags in (64, 2 | 8):
        with pytest.raises(WmmaeError) as e:
            tc.sgemm("T", "N", m, n, k, 1.0, A, k, B, k, 0.0, C, m, 0, flags)
        assert e.value.status == -1
    with pytest.raises(WmmaeError) as e:
        tc.api_gemm(0, 1, 100, n, k, 1.0, A[:, :128].contiguous(), 128, B, k, 0.0, C, m)
    assert e.value.status in (-3, -4)
    # gradients and transforms: raw pointers of wrapped tensors are refused as before
    with pytest.raises(RuntimeError):
        torch.func.vmap(lambda a: tc.matmul_tn(a, B))(A.expand(2, m, k).contiguous())


@pytest.mark.gpu
@pytest.mark.parametrize("policy", [0, 2])
def test_plain_arguments_are_taken(tc, dev, policy, monkeypatch):
    """Each function itself, so that one that turns every call away is seen, and its output against the
    same call through the checks in Python."""
    m, n, k, batch = 128, 256, 160, 3
    calls, stream = tcec._native(), tcec._native_stream()
    assert not isinstance(calls, tcec._NoNativeCalls) and stream is not None
    A, B = (torch.rand((batch, x, k), device=dev) - 0.5 for x in (m, n))
    C0 = torch.rand((batch, n, m), device=dev)
    ws = torch.empty(tc.workspace_bytes(m, n, k, batch, policy), dtype=torch.uint8, device=dev)
    pa, pb = (torch.empty(tc.pack_bytes(x, k, 1, policy), dtype=torch.uint8, device=dev) for x in (m, n))
    tiles = torch.rand((5, 256), device=dev)
    api = {0: (0, 1), 2: (2, 1)}[policy]
    rows = [("sgemm", lambda C: ("T", "N", m, n, k, 0.5, A, k, B, k, 1, C, m, policy, 0, ws)),
            ("sgemm_strided_batched", lambda C: ("T", "N", m, n, k, 0.5, A, k, m * k, B, k, n * k, 1.5, C, m, m * n, batch,
                                                 tc.Policy(policy), 0, ws)),
            ("sgemm_batched", lambda C: ("T", "N", m, n, k, 0.5, *sum(([p, ld] for p, ld in zip(
                [torch.tensor([e.data_ptr() for e in X], device=dev) for X in (A, B)], (k, k))), []), 1.5,
                torch.tensor([e.data_ptr() for e in C], device=dev), m, batch, policy, 0, None)),
            ("gemm_packed", lambda C: (policy, m, n, k, 1.0, pa, pb, 1.0, C, m, 1, 0, 0, None)),
            ("api_gemm", lambda C: (*api, m, n, k, 1.0, A, k, B, k, 1.0, C, m))]
    for X, x, out in ((A, m, pa), (B, n, pb)):
        args = (policy, x, k, X, k, 1, out, 1, 0)
        assert calls.pack(*args, stream) == 0
        got = out.clone()
        with monkeypatch.context() as mp:
            mp.setattr(tcec, "_calls", tcec._NoNativeCalls())
            out.zero_()
            tc.pack(*args)
        assert torch.equal(got, out)
    for name, args in rows:
        C = C0.clone()
        assert getattr(calls, name)(*args(C), stream) == 0, name
        D = C0.clone()
        with monkeypatch.context() as mp:
            mp.setattr(tcec, "_calls", tcec._NoNativeCalls())
            getattr(tc, name)(*args(D))
        assert torch.equal(C, D) and not torch.equal(C, C0), name
    got, dicts = calls.matmul_tn(A[0], B[0], policy, 0, ws, stream), calls.primitive_tiles(tiles, stream)
    assert isinstance(got, torch.Tensor) and isinstance(dicts, dict)
    with monkeypatch.context() as mp:
        mp.setattr(tcec, "_calls", tcec._NoNativeCalls())
        assert torch.equal(got, tc.matmul_tn(A[0], B[0], policy, 0, ws))
        want = tc.primitive_tiles(tiles)
    assert set(want) == set(dicts) and all(torch.equal(want[x], dicts[x]) for x in want)
