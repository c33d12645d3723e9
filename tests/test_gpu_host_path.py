"""The C++ host path (csrc/host/torch_host.cpp) against the Python path of the
same operators: the same kernels with the same arguments, so outputs and
gradients are bitwise equal for every form it accepts, and what it does not
accept is handled (or refused) by Python as before."""

import math

import pytest
import torch


@pytest.fixture
def python_path(monkeypatch):
    """Runs a function with the extension out of reach."""
    from openfold3_triangle_kernel_amd import _native

    def run(fn):
        with monkeypatch.context() as m:
            m.setattr(_native, "_HOST", False)
            return fn()

    return run


def test_host_path_declines_cpu_tensors():
    from openfold3_triangle_kernel_amd import _native

    host = _native.host()
    assert host is not None, "the host extension is built beside the library"
    t = torch.zeros(1, 2, 1, 8, 8, dtype=torch.bfloat16)
    assert host.attention(t, t, t, torch.zeros(1, 2, 1, 1, 8), torch.zeros(1, 1, 1, 8, 8)) is None
    w = [torch.zeros(64, 32)] * 2 + [torch.zeros(32, 32)] * 2 + [torch.zeros(32)] * 4
    assert host.trimul(torch.zeros(1, 4, 4, 32, dtype=torch.bfloat16), None, w, True) is None


ATTENTION = [
    # prefix, O, H, N, D, seq_major, bias prefix, bias dtype, transposed, mask prefix, mask dtype
    ((1,), 3, 2, 64, 32, False, (1,), torch.bfloat16, False, (1,), torch.float32),
    ((1,), 3, 2, 70, 32, True, (1,), torch.bfloat16, True, (1,), torch.float32),
    ((2,), 2, 1, 33, 64, False, (2,), torch.float32, False, (1,), torch.bfloat16),
    ((2, 2), 2, 2, 40, 16, True, (1, 1), torch.bfloat16, True, (2, 1), torch.float32),
    ((2, 1), 2, 1, 64, 8, False, (), torch.float32, True, (), torch.float16),
    ((2, 2), 2, 1, 20, 8, False, (2, 1), torch.bfloat16, False, (2, 2), torch.float32),  # Python
    ((1,), 2, 2, 24, 12, False, (1,), torch.bfloat16, False, (1,), torch.float32),       # Python
]


@pytest.mark.gpu
@pytest.mark.parametrize("needs", ["all", "v", "bias", "none"])
@pytest.mark.parametrize("case", ATTENTION, ids=[str(i) for i in range(len(ATTENTION))])
def test_attention_host_path_equals_python_path(gpu, python_path, case, needs):
    from openfold3_triangle_kernel_amd import _native, attention

    prefix, O, H, N, D, seq, bp, bdt, transposed, mp, mdt = case
    print(f"[host path attention] {case} {needs}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(N + D)
    shape = (*prefix, O, N, H, D) if seq else (*prefix, O, H, N, D)
    qkv = [torch.randn(shape, device=gpu, generator=g).bfloat16() for _ in range(3)]
    if seq:
        qkv = [t.transpose(-2, -3) for t in qkv]
    bias = torch.randn((*bp, 1, H, N, N), device=gpu, generator=g).to(bdt)
    if transposed:
        bias = bias.transpose(-1, -2)
    mask = torch.zeros((*mp, O, 1, 1, N), device=gpu, dtype=mdt)
    mask[..., -3:] = float("-inf")
    dout = torch.randn((*prefix, O, N, H, D), device=gpu, generator=g)
    served = D % 8 == 0 and (math.prod(bp) == 1 or bp == prefix)

    def run():
        xs = [t.detach().requires_grad_(needs in ("all", n))
              for n, t in zip(("q", "k", "v", "bias"), (*qkv, bias))]
        before = attention.invocation_count()
        out = attention.turbopairformer_triangle_attention(*xs[:3], mask, xs[3])
        assert attention.invocation_count() == before + 1
        want = [x for x in xs if x.requires_grad]
        return [out, *(torch.autograd.grad(out, want, dout) if want else ())]

    xs = [t.detach() for t in (*qkv, bias)]
    assert (_native.host().attention(*xs[:3], mask, xs[3]) is not None) == served
    for a, b in zip(run(), python_path(run)):
        assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.gpu
def test_attention_host_path_leaves_refusals_and_transforms_to_python(gpu, monkeypatch):
    from openfold3_triangle_kernel_amd import _native, turbopairformer_triangle_attention as attn

    host = _native.host()
    q = torch.randn(1, 2, 1, 16, 8, device=gpu).bfloat16()
    mask, bias = torch.zeros(1, 2, 1, 1, 16, device=gpu), torch.zeros(1, 1, 1, 16, 16, device=gpu)
    assert host.attention(q, q, q, mask, bias) is not None
    off = torch.empty(q.numel() + 1, device=gpu, dtype=q.dtype)[1:].view(q.shape).copy_(q)
    for args in ((q, q[:, :1], q, mask, bias), (q, q, q, mask[..., :8], bias),
                 (q, q, q, mask, bias[..., :8]), (q.float(), q, q, mask, bias),
                 (q, q, q, mask.requires_grad_(), bias), (off, q, q, mask.detach(), bias)):
        assert host.attention(*args) is None
    mask = mask.detach()
    assert torch.equal(attn(off, q, q, mask, bias), attn(q, q, q, mask, bias))
    seen = []
    torch.func.vmap(lambda x: seen.append(host.attention(x, x, x, mask, bias)) or x)(q[None])
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(q, q)
        seen.append(host.attention(dual, q, q, mask, bias))
    assert seen == [None, None]
    monkeypatch.setenv("TURBOPAIRFORMER_SR_BACKWARD", " 0 ")
    assert host.attention(q, q, q, mask, bias) is None
    with pytest.raises(ValueError, match="SR_BACKWARD"):
        attn(q, q, q, mask, bias)
    monkeypatch.setenv("TURBOPAIRFORMER_SR_BACKWARD", "1")
    monkeypatch.setenv("OPENFOLD3_SR_SHADOW", "2")
    with pytest.raises(ValueError, match="SR_SHADOW"):
        attn(q, q, q, mask, bias)


@pytest.mark.gpu
@pytest.mark.parametrize("needs", ["all", "z", "p_out_weight", "none"])
@pytest.mark.parametrize("prefix,N,C,mask_dtype,param_dtype", [
    ((1,), 24, 32, torch.float32, torch.float32), ((), 17, 64, torch.bfloat16, torch.float32),
    ((2, 1), 9, 128, None, torch.float32), ((1,), 16, 32, torch.float32, torch.bfloat16)])
def test_trimul_host_path_equals_python_path(gpu, python_path, prefix, N, C, mask_dtype,
                                             param_dtype, needs):
    from openfold3_triangle_kernel_amd import turbo_trimul

    print(f"[host path trimul] {prefix} N={N} C={C} {mask_dtype} {param_dtype} {needs}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(N)
    z = torch.randn(*prefix, N, N, C, device=gpu, generator=g).bfloat16()
    mask = None if mask_dtype is None else (
        torch.rand(*prefix, N, N, device=gpu, generator=g) > 0.2).to(mask_dtype)
    shapes = dict(norm_in_weight=(C,), norm_in_bias=(C,), p_in_weight=(2 * C, C),
                  g_in_weight=(2 * C, C), norm_out_weight=(C,), norm_out_bias=(C,),
                  p_out_weight=(C, C), g_out_weight=(C, C))
    w = {n: (torch.randn(s, device=gpu, generator=g) / C ** 0.5).to(param_dtype)
         for n, s in shapes.items()}
    dout = torch.randn_like(z)

    def run():
        xs = {n: t.detach().clone().requires_grad_(needs in ("all", n))
              for n, t in dict(w, z=z).items()}
        outs = []
        for direction in ("outgoing", "incoming"):
            out = turbo_trimul(xs["z"], direction, mask, **{n: xs[n] for n in w})
            want = [x for x in xs.values() if x.requires_grad]
            outs += [out, *(torch.autograd.grad(out, want, dout) if want else ())]
        return outs

    for a, b in zip(run(), python_path(run)):
        assert a.shape == b.shape and a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.gpu
def test_host_path_saved_tensor_hooks_and_checkpoint(gpu):
    """Saved tensors go through autograd's hooks, so activation offloading and
    non-reentrant checkpointing see them."""
    from torch.utils.checkpoint import checkpoint

    from openfold3_triangle_kernel_amd import turbopairformer_triangle_attention as attn

    q = torch.randn(1, 2, 2, 48, 16, device=gpu).bfloat16().requires_grad_(True)
    mask = torch.zeros(1, 2, 1, 1, 48, device=gpu)
    bias = torch.randn(1, 1, 2, 48, 48, device=gpu).bfloat16().requires_grad_(True)
    ref = torch.autograd.grad(attn(q, q, q, mask, bias).float().sum(), (q, bias))
    packed = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(1) or t.cpu(),
                                                  lambda t: t.to(gpu)):
        got = attn(q, q, q, mask, bias).float().sum()
    assert len(packed) >= 7
    for a, b in zip(ref, torch.autograd.grad(got, (q, bias))):
        assert torch.equal(a, b)
    got = checkpoint(lambda x, b: attn(x, x, x, mask, b).float().sum(), q, bias, use_reentrant=False)
    for a, b in zip(ref, torch.autograd.grad(got, (q, bias))):
        assert torch.equal(a, b)


def _misaligned(t):
    """t's values, contiguous, starting 2 bytes past a 16-byte boundary."""
    out = torch.empty(t.numel() + 1, device=t.device, dtype=t.dtype)[1:].view(t.shape).copy_(t)
    assert out.is_contiguous() and out.data_ptr() % 16 == 2
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("N,D", [(33, 32), (64, 32), (33, 64), (64, 64)])
def test_attention_misaligned_upstream_gradient(gpu, python_path, N, D):
    """The kernels load 16 bytes at a time: an upstream gradient that starts
    off that boundary gives the bits of the aligned one on both host paths."""
    from openfold3_triangle_kernel_amd import turbopairformer_triangle_attention as attn

    print(f"[misaligned dO] N={N} D={D}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(N)
    xs = [torch.randn(1, 5, 2, N, D, device=gpu, generator=g).bfloat16() for _ in range(3)]
    xs = [t.requires_grad_(True) for t in
          (*xs, torch.randn(1, 1, 2, N, N, device=gpu, generator=g).bfloat16())]
    mask = torch.zeros(1, 5, 1, 1, N, device=gpu)
    dout = torch.randn(1, 5, N, 2, D, device=gpu, generator=g).bfloat16()

    def run(d):
        return torch.autograd.grad(attn(*xs[:3], mask, xs[3]), xs, d)

    ref = run(dout)
    for got in (run(_misaligned(dout)), python_path(lambda: run(_misaligned(dout)))):
        assert all(torch.equal(a, b) for a, b in zip(got, ref))


@pytest.mark.gpu
@pytest.mark.parametrize("N,C", [(17, 64), (24, 128)])
def test_trimul_misaligned_pair_and_gradient(gpu, python_path, N, C):
    """As above for TriMul's upstream gradient and for its pair input."""
    from openfold3_triangle_kernel_amd import turbo_trimul

    print(f"[misaligned trimul] N={N} C={C}", flush=True)
    g = torch.Generator(device=gpu).manual_seed(N)
    z, dout = (torch.randn(1, N, N, C, device=gpu, generator=g).bfloat16() for _ in range(2))
    w = [torch.randn(s, device=gpu, generator=g) / C ** 0.5
         for s in ((C,), (C,), (2 * C, C), (2 * C, C), (C,), (C,), (C, C), (C, C))]

    def run(z, d):
        xs = [z.detach().requires_grad_(True), *(t.detach().requires_grad_(True) for t in w)]
        return torch.autograd.grad(turbo_trimul(xs[0], "incoming", None, *xs[1:]), xs, d)

    ref = run(z, dout)
    bad = _misaligned(z), _misaligned(dout)
    for got in (run(z, bad[1]), run(*bad), python_path(lambda: run(*bad))):
        assert all(torch.equal(a, b) for a, b in zip(got, ref))


@pytest.mark.gpu
def test_host_path_threads_streams_and_environment(gpu):
    """Two threads, each on a stream of its own, run both operators forward
    and backward while a third assigns environment variables (the policy
    variables are read under the GIL, as those assignments are made): the bits
    of one thread on the default stream."""
    import os
    import threading

    from openfold3_triangle_kernel_amd import turbo_trimul
    from openfold3_triangle_kernel_amd import turbopairformer_triangle_attention as attn

    g = torch.Generator(device=gpu).manual_seed(3)
    q, k, v = (torch.randn(1, 9, 2, 70, 32, device=gpu, generator=g).bfloat16() for _ in range(3))
    bias = torch.randn(1, 1, 2, 70, 70, device=gpu, generator=g).bfloat16()
    mask, z = torch.zeros(1, 9, 1, 1, 70, device=gpu), torch.randn(
        1, 33, 33, 64, device=gpu, generator=g).bfloat16()
    w = [torch.randn(s, device=gpu, generator=g) / 8
         for s in ((64,), (64,), (128, 64), (128, 64), (64,), (64,), (64, 64), (64, 64))]

    def both():
        xs = [t.detach().requires_grad_(True) for t in (q, k, v, bias, z, *w)]
        a = attn(*xs[:3], mask, xs[3])
        t = turbo_trimul(xs[4], "outgoing", None, *xs[5:])
        return [a, t, *torch.autograd.grad((a, t), xs, (a.detach(), t.detach()))]

    ref = [t.clone() for t in both()]
    torch.cuda.synchronize()
    failed, done = [], threading.Event()

    def work():
        try:
            with torch.cuda.stream(torch.cuda.Stream(gpu)):
                for _ in range(20):
                    got = both()
                torch.cuda.current_stream().synchronize()
                if not all(torch.equal(a, b) for a, b in zip(got, ref)):
                    failed.append("outputs differ")
        except Exception as e:  # reported by the main thread
            failed.append(repr(e))

    def assign():
        i = 0
        while not done.is_set() and i < 100_000:
            os.environ[f"TPF_TEST_{i % 300}"] = "x" * (i % 50)
            i += 1

    workers = [threading.Thread(target=work) for _ in range(2)]
    writer = threading.Thread(target=assign)
    try:
        for t in (writer, *workers):
            t.start()
        for t in workers:
            t.join()
    finally:
        done.set()
        writer.join()
        for i in range(300):
            os.environ.pop(f"TPF_TEST_{i}", None)
    assert not failed, failed


@pytest.mark.gpu
def test_host_path_leaves_torch_function_modes_to_python(gpu):
    """An active TorchFunctionMode sees the torch calls of both operators; a
    default device (a mode of torch's own, for tensor factories) keeps the
    host path."""
    from openfold3_triangle_kernel_amd import _native, turbo_trimul
    from openfold3_triangle_kernel_amd import turbopairformer_triangle_attention as attn

    class Seen(torch.overrides.TorchFunctionMode):
        def __init__(self):
            super().__init__()
            self.names = []

        def __torch_function__(self, func, types, args=(), kwargs=None):
            self.names.append(getattr(func, "__name__", str(func)))
            return func(*args, **(kwargs or {}))

    q = torch.randn(1, 2, 1, 16, 8, device=gpu).bfloat16()
    mask, bias = torch.zeros(1, 2, 1, 1, 16, device=gpu), torch.zeros(1, 1, 1, 16, 16, device=gpu)
    z, w = torch.randn(1, 8, 8, 32, device=gpu).bfloat16(), torch.randn(64, 32, device=gpu)
    ln = torch.ones(32, device=gpu)

    def trimul():
        return turbo_trimul(z, "outgoing", None, ln, ln, w, w, ln, ln, w[:32], w[:32])

    ref = attn(q, q, q, mask, bias), trimul()
    for call, want in zip((lambda: attn(q, q, q, mask, bias), trimul), ref):
        with Seen() as mode:
            assert torch.equal(call(), want)
        assert mode.names
        with torch.device(gpu):
            assert _native.host_eligible(q)
            assert torch.equal(call(), want)


@pytest.mark.parametrize("version,loads", [(None, True), ("1.13.0", False), ("{0}1", False),
                                           ("{0}+other", True)])
def test_host_extension_declines_another_torch(version, loads):
    """Beside another torch than it was built for the extension is reported
    and left out, and the Python path serves the operators; the budget call
    that forwards to it works either way."""
    import subprocess
    import sys

    code = f"""
import warnings, torch
version = {version!r}
if version:
    torch.__version__ = version.format(torch.__version__.split('+')[0])
warnings.simplefilter("always")
with warnings.catch_warnings(record=True) as seen:
    from openfold3_triangle_kernel_amd import _native, attention
    hosts = [_native.host(), _native.host()]
    attention.set_sr_workspace_budget(1 << 30)
msgs = [w for w in seen if "host extension" in str(w.message)]
assert [h is not None for h in hosts] == [{loads}] * 2 and len(msgs) == {int(not loads)}, (hosts, msgs)
assert _native.query("tpf_abi_version") > 0
"""
    r = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-2000:]
