"""The Python calls' native launcher against the ctypes way it stands in for: same results, same refusals."""
import ctypes

import pytest


def test_launcher_is_loaded_and_leaves_other_operands_alone(hgemm_lib):
    """No GPU: CPU tensors, wrong types, negative and fractional sizes go to the method in Python, which says what is wrong."""
    import gc
    import weakref
    import torch
    from cuda_hgemm_amd import binding
    if hgemm_lib._native_product is None:
        pytest.skip("library loaded before torch")
    native = binding._native_calls()
    assert type(hgemm_lib.call) is native.Caller
    A, B, C = torch.ones(4, 8).half(), torch.ones(5, 8).half(), torch.empty(4, 5).half()
    assert hgemm_lib._run_address == ctypes.cast(hgemm_lib.dll.hgemm_variant_run, ctypes.c_void_p).value
    seen = []
    caller = native.Caller(hgemm_lib._run_address, {"hgemm_auto": 21}, lambda *a, **k: seen.append((a, k)) or "method")
    calls = [((A, B, C, 4, 5, 8), {}), ((A, B, None, 4, 5, 8), {}), ((A, [1.0], C, 4, 5, 8), {}), ((A, B, C, -4, 5, 8), {}),
             ((A, B, C, 4.0, 5, 8), {}), ((A, B, C, 4, 5, 1 << 70), {}), ((A, B, C, True, 5, 8), {}), ((A, B), {}), ((A, B, C, 4, 5), {"K": 8})]
    for args, named in calls:
        assert caller("hgemm_auto", *args, **named) == "method"
    assert caller("no such", A, B, C, 4, 5, 8) == caller(["hgemm_auto"], A, B, C, 4, 5, 8) == "method" and len(seen) == len(calls) + 2
    assert seen[-3] == (("hgemm_auto", A, B, C, 4, 5), {"K": 8})
    for name, error in [("hgemm_auto", ValueError), ("no such", (ValueError, KeyError))]:
        with pytest.raises(error):
            hgemm_lib.call(name, A, B, C, 4, 5, 8)
    assert hgemm_lib._native_product(hgemm_lib._run_address, 21, A, B) is None
    assert hgemm_lib._native_product(hgemm_lib._run_address, 21, A, "B") is None

    class Owner:                       # an owner and its caller refer to each other
        def method(self):
            pass
    owner = Owner()
    owner.call, gone = native.Caller(hgemm_lib._run_address, {}, owner.method), weakref.ref(owner)
    del owner
    gc.collect()
    assert gone() is None


def test_a_module_that_does_not_fit_is_left_out(hgemm_lib, monkeypatch, tmp_path):
    """A launcher that does not load, or was built against another torch: a warning, and calls go through ctypes."""
    import torch
    from cuda_hgemm_amd import binding
    A, B, C = torch.ones(4, 8).half(), torch.ones(5, 8).half(), torch.empty(4, 5).half()

    def library_without_it():
        monkeypatch.setattr(binding, "_call_module", None)
        with pytest.warns(RuntimeWarning, match="is not used"):
            lib = binding.HgemmLibrary(hgemm_lib.path)
        assert lib._native_product is None and "call" not in vars(lib)
        with pytest.raises(ValueError, match="GPU"):
            lib.call("hgemm_auto", A, B, C, 4, 5, 8)

    with monkeypatch.context() as m:
        broken = tmp_path / "_call.so"
        broken.write_bytes(b"not a shared object")
        m.setattr(binding, "call_module_path", lambda: str(broken))
        library_without_it()
    if binding._native_calls() is not None:
        with monkeypatch.context() as m:
            m.setattr(torch, "__version__", "1.13.1")
            library_without_it()


def test_a_subclass_keeps_its_own_call(hgemm_lib):
    from cuda_hgemm_amd import binding

    class Counted(binding.HgemmLibrary):
        def call(self, *args):
            return "counted", args

    lib = Counted(hgemm_lib.path)
    assert lib.call("hgemm_auto", 1) == ("counted", ("hgemm_auto", 1)) and lib._native_product is None


@pytest.mark.gpu
def test_products_and_refusals(hgemm_lib, gpu):
    import torch
    import cuda_hgemm_amd
    A, B = torch.randint(-1, 2, (48, 64), device=gpu).half(), torch.randint(-1, 2, (40, 64), device=gpu).half()
    exact = (A.float() @ B.float().t()).half()
    for _ in range(2):      # the first call of a variant goes through ctypes
        out = cuda_hgemm_amd.hgemm(A, B)
        assert out.shape == (48, 40) and out.dtype == torch.float16 and out.is_contiguous() and not out.requires_grad
        assert torch.equal(out, exact)
        assert torch.equal(cuda_hgemm_amd.hgemm(torch.nn.Parameter(A), B), exact)
        into = torch.empty_like(exact)
        assert cuda_hgemm_amd.hgemm(A, B, out=into) is into and torch.equal(into, exact)
        with torch.inference_mode():
            assert cuda_hgemm_amd.hgemm(A, B).is_inference()

        class Named(torch.Tensor):
            pass
        assert torch.equal(cuda_hgemm_amd.hgemm(A.as_subclass(Named), B).as_subclass(torch.Tensor), exact)
        shifted = torch.ones(48 * 64 + 1, dtype=torch.float16, device=gpu)[1:].view(48, 64)
        for bad, error in [(A.float(), TypeError), (A.cpu(), (TypeError, ValueError)), (A[:, :32], ValueError), (A.t().contiguous().t(), ValueError),
                           (shifted, ValueError), (A[0], ValueError), (torch.empty((0, 64), device=gpu).half(), ValueError)]:
            with pytest.raises(error):
                cuda_hgemm_amd.hgemm(bad, B)
        with pytest.raises(ValueError, match="cannot run"):
            cuda_hgemm_amd.hgemm(A, B, variant="hgemm_mfma_base")
        with pytest.raises(RuntimeError):      # a batched tensor has no memory of its own
            torch.func.vmap(lambda a: cuda_hgemm_amd.hgemm(a, B))(A[None])
