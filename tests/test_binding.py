"""The native marshalling of the Python mirror's calls (csrc/py/q4_binding.cpp):
it declines (None) whatever is not the plain accepted call, so that errors stay
those of the Python checks, and where it makes the call the result is that of
the ctypes route, bit for bit."""
import pytest

from helpers import gpu_inputs


@pytest.fixture
def native(pkg):
    if not pkg._native_tried:
        pkg._load_binding()
    assert pkg._native is not None, "lib/_q4_binding.*.so is not built"
    return pkg._native


@pytest.mark.parametrize("attr,value", [("__version__", "9.9.0"), ("git_version", "0" * 40)])
def test_another_torchs_binding_is_not_loaded(pkg, native, monkeypatch, attr, value):
    """Its inlined reads of a tensor may not fit: ctypes serves the calls."""
    import torch
    monkeypatch.setattr(torch.version, attr, value)
    monkeypatch.setattr(pkg, "_native", None)
    with pytest.warns(UserWarning, match="another Python or torch"):
        pkg._load_binding()
    assert pkg._native is None


def test_declines_host_tensors_and_other_types(pkg, native):
    import torch
    x = torch.zeros(1, 64, dtype=torch.float16)
    w = torch.zeros(4, 8, dtype=torch.int32)
    s = torch.zeros(4, 1, dtype=torch.float16)
    W = pkg.Q4Weight(w, s, s, 64, 64)
    for a in ((x, w, s, s, 1, 64, 4, 64, None, None), (None, w, s, s, 1, 64, 4, 64, None, None),
              (x, w, s, s, 1.0, 64, 4, 64, None, None), (x, w, s, s, 2**40, 64, 4, 64, None, None),
              (x, w), ()):
        assert native.matmul_q4(*a) is None
    assert native.linear(x, W, 1, 64, 4, False, None, None) is None
    assert native.linear(x, (w, s, s), 1, 64, 4, False, None, None) is None
    assert native.embedding_q4(W, 4, torch.zeros(2, dtype=torch.int32), None, None) is None
    with pytest.raises(ValueError, match="device tensor"):
        pkg.matmul_q4(x, w, s, s, 1, 64, 4, 64)


def _calls(pkg, dev):
    """(name, call) over every bound function, on fresh inputs."""
    import torch
    M, N, K, g = 3, 256, 512, 64
    x, sets = gpu_inputs(M, N, K, g, seed=1, dev=dev, n_weights=2)
    W, U = (pkg.Q4Weight(*t, K, g) for t in sets)
    (w, s, b) = sets[0]
    gen = torch.Generator(device=dev).manual_seed(2)
    r = torch.randn(M, N, generator=gen, device=dev).half()
    nk, nn = torch.rand(K, generator=gen, device=dev), torch.rand(N, generator=gen, device=dev)
    logits = torch.randn(5000, generator=gen, device=dev)
    seen = torch.arange(7, dtype=torch.int32, device=dev)
    yield "matmul_q4", lambda: pkg.matmul_q4(x, w, s, b, M, K, N, g)
    yield "matmul_q4_fast", lambda: pkg.matmul_q4_fast(x, w, s, b, M, K, N, g)
    yield "matmul_q4_fast_f32", lambda: pkg.matmul_q4_fast_f32(x, w, s, b, M, K, N, g)
    yield "linear", lambda: pkg.linear(x, W, M, K, N, True)
    yield "silu_mul", lambda: pkg.silu_mul(r, r)
    yield "matmul_q4_silu_mul", lambda: pkg.matmul_q4_silu_mul(x, W, U, M, K, N)
    yield "matmul_q4_geglu", lambda: pkg.matmul_q4_geglu(x, W, U, M, K, N)
    yield "matmul_q4_ex", lambda: pkg.matmul_q4_ex(x.bfloat16(), W, M, N, torch.bfloat16, nn,
                                                   pkg.SLTX_EPI_GELU_TANH)
    yield "matmul_q4_ex f32", lambda: pkg.matmul_q4_ex(x.float(), W, M, N)
    yield "rms_norm", lambda: pkg.rms_norm(x, nk, 1e-5, M, K)
    yield "residual_rms_norm", lambda: pkg.residual_rms_norm(x, x, nk, 1e-5, M, K)
    yield "rmsnorm_matmul_q4", lambda: pkg.rmsnorm_matmul_q4(x[:1], nk, 1e-5, W, N)
    yield "residual_rmsnorm_matmul_q4_silu_mul", lambda: pkg.residual_rmsnorm_matmul_q4_silu_mul(
        x[:1], x[1:2], nk, 1e-5, W, U, N)
    yield "matmul_q4_residual", lambda: pkg.matmul_q4_residual(x, W, r, M, N)
    yield "matmul_q4_residual_rms_norm", lambda: pkg.matmul_q4_residual_rms_norm(
        x, W, r, nn, 1e-5, M, N, True)
    yield "embedding_q4", lambda: pkg.embedding_q4(W, N, seen)
    yield "argmax", lambda: pkg.argmax(logits)
    yield "sample", lambda: pkg.sample(logits, 0.7, 0.9, 1.1, seen, 0.25)


@pytest.mark.gpu
def test_same_results(pkg, dev, native, monkeypatch):
    import torch
    for name, call in _calls(pkg, dev):
        made = []
        bound = getattr(native, name.split()[0])
        monkeypatch.setattr(pkg, "_native", type("N", (), {name.split()[0]: staticmethod(
            lambda *a: made.append(bound(*a)) or made[-1])}))
        got = call()
        assert made and made[0] is got, f"{name}: declined"
        monkeypatch.setattr(pkg, "_native", None)
        want = call()
        torch.cuda.synchronize()
        for a, b in zip(*((v if isinstance(v, tuple) else (v,)) for v in (got, want))):
            assert a.dtype == b.dtype and a.shape == b.shape and torch.equal(a, b), name


@pytest.mark.gpu
def test_streams_outputs_and_errors(pkg, dev, native):
    import torch
    M, N, K, g = 2, 128, 256, 64
    x, [(w, s, b)] = gpu_inputs(M, N, K, g, seed=4, dev=dev)
    want = pkg.matmul_q4(x, w, s, b, M, K, N, g)
    st = torch.cuda.Stream()
    out = torch.empty_like(want)
    torch.cuda.synchronize()
    for stream in (st, st.cuda_stream, None):
        with torch.cuda.stream(st):
            assert pkg.matmul_q4(x, w, s, b, M, K, N, g, out=out, stream=stream) is out
        st.synchronize()
        assert torch.equal(out, want)
        out.zero_()
        torch.cuda.synchronize()
    # what the Python checks and the library refuse stays refused
    for bad in (dict(x=x[:, ::2]), dict(x=x.float()), dict(out=torch.empty(1, device=dev).half()),
                dict(w=w[:64]), dict(s=s.float())):
        a = dict(x=x, w=w, s=s, out=None) | bad
        with pytest.raises(ValueError):
            pkg.matmul_q4(a["x"], a["w"], a["s"], b, M, K, N, g, out=a["out"])
    with pytest.raises(pkg.SltxError) as e:
        pkg.matmul_q4(x, w, s, b, M, K, N, g, out=x.view(-1)[: M * N].view(M, N))
    assert e.value.code == pkg.SLTX_ERR_INVALID and "overlaps" in str(e.value)


@pytest.mark.gpu
def test_other_threads_run_while_an_output_is_allocated(pkg, dev, native):
    """Within a limit that holds either a cached block or the new output, the
    allocator gives the block back, which waits for the GPU's queued work: about a
    second here.  Another Python thread goes on meanwhile."""
    import threading
    import time
    import torch
    a = torch.zeros(48 << 20, device=dev, dtype=torch.float16)
    m = torch.zeros(8192, 8192, device=dev, dtype=torch.float16)
    r = torch.empty_like(m)
    torch.mm(m, m, out=r)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    cached = torch.empty(64 << 20, device=dev, dtype=torch.uint8)
    del cached   # 64 MB kept by the allocator; the output takes 96 MB
    total = torch.cuda.get_device_properties(dev).total_memory
    gap, stop = [0.0], threading.Event()

    def tick():
        last = time.perf_counter()
        while not stop.is_set():
            time.sleep(0.001)
            now = time.perf_counter()
            gap[0] = max(gap[0], now - last)
            last = now

    t = threading.Thread(target=tick)
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + (48 << 20)) / total)
    try:
        for _ in range(800):
            torch.mm(m, m, out=r)
        t.start()
        begin = time.perf_counter()
        out = pkg.silu_mul(a, a)
        took = time.perf_counter() - begin
    finally:
        stop.set()
        if t.ident is not None:
            t.join()
        torch.cuda.set_per_process_memory_fraction(1.0)
        torch.cuda.synchronize()
    assert not out.any()
    assert took > 0.2, f"the allocator did not wait ({took:.3f} s)"
    assert gap[0] < took / 2, f"another thread stood still for {gap[0]:.3f} of {took:.3f} s"
