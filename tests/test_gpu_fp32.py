"""GPU parity of the inference-only FP32 paths against the numpy FP64 oracle.

Tolerance (north star, fp32 mode): every output at max-rel <= 1e-4,
max-rel = max|got - ref| / max|ref|, oracle in float64 on the same f32
inputs (full f32 values, not bf16-rounded).
"""

import numpy as np
import pytest
import torch

from oracle.attention import attention_forward
from tests._util import max_rel

TOL = 1e-4


def _f32_case(B, O, H, N, D, *, mask_tail=0, full_planes=0, bias_batch=1, seed=0):
    g = torch.Generator().manual_seed(seed)
    q, k, v = (torch.randn(B, O, H, N, D, generator=g) for _ in range(3))
    bias = torch.randn(bias_batch, 1, H, N, N, generator=g) * 2
    mask = torch.zeros(B, O, 1, 1, N)
    if mask_tail:
        tails = torch.randint(0, mask_tail + 1, (B, O), generator=g)
        for b in range(B):
            for o in range(O):
                if int(tails[b, o]):
                    mask[b, o, ..., N - int(tails[b, o]):] = float("-inf")
    if full_planes:
        mask[:, :full_planes] = float("-inf")
    return q, k, v, mask, bias


ATTN_CASES = [
    # B, O, H, N, D, mask_tail, full_planes, bias_batch
    (1, 8, 4, 128, 32, 13, 0, 1),
    (1, 16, 4, 384, 32, 32, 0, 1),
    (1, 6, 4, 100, 12, 7, 1, 1),
    (2, 4, 4, 200, 20, 5, 0, 2),
    (1, 6, 4, 256, 64, 0, 2, 1),
    (1, 2, 8, 96, 48, 9, 0, 1),
    (1, 3, 1, 33, 3, 0, 0, 1),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", ATTN_CASES, ids=lambda c: "B{}O{}H{}N{}D{}".format(*c[:5]))
def test_attention_fp32(gpu, case):
    from openfold3_triangle_kernel_amd import turbopairformer_attention_fp32

    B, O, H, N, D, tail, full, bb = case
    q, k, v, mask, bias = _f32_case(B, O, H, N, D, mask_tail=tail, full_planes=full, bias_batch=bb)
    print(f"fp32 attention case={case}", flush=True)
    with torch.no_grad():
        out = turbopairformer_attention_fp32(*(t.to(gpu) for t in (q, k, v, mask, bias)))
    torch.cuda.synchronize()
    assert out.dtype == torch.float32 and out.shape == (B, O, N, H, D)
    ref, _, _ = attention_forward(q.numpy(), k.numpy(), v.numpy(), mask.numpy(), bias.numpy())
    got = out.cpu().numpy()
    if full:
        assert np.all(got[:, :full] == 0)
    err = max_rel(got, ref)
    assert err <= TOL, err


@pytest.mark.gpu
def test_attention_fp32_sequence_major(gpu):
    """The transposed-projection view (sequence-major storage) is read in place."""
    from openfold3_triangle_kernel_amd import turbopairformer_attention_fp32

    q, k, v, mask, bias = _f32_case(1, 4, 4, 128, 32, mask_tail=9)
    qs, ks, vs = (t.transpose(2, 3).contiguous().to(gpu).transpose(2, 3) for t in (q, k, v))
    with torch.no_grad():
        out = turbopairformer_attention_fp32(qs, ks, vs, mask.to(gpu), bias.to(gpu))
    ref, _, _ = attention_forward(q.numpy(), k.numpy(), v.numpy(), mask.numpy(), bias.numpy())
    assert max_rel(out.cpu().numpy(), ref) <= TOL


def _trimul_module(C, H, outgoing, *, biases=False, fused=False, affine=True, seed=0):
    """An object with the official TriMul module's attribute names, FP32 on CPU."""
    from types import SimpleNamespace

    torch.manual_seed(seed)

    def lin(i, o):
        layer = torch.nn.Linear(i, o, bias=biases)
        with torch.no_grad():
            layer.weight.normal_(0, i ** -0.5)
            if biases:
                layer.bias.normal_(0, 0.2)
        return layer

    m = SimpleNamespace(c_z=C, c_hidden=H, _outgoing=outgoing)
    if fused:
        m.linear_ab_p, m.linear_ab_g = lin(C, 2 * H), lin(C, 2 * H)
    else:
        m.linear_a_p, m.linear_a_g, m.linear_b_p, m.linear_b_g = (lin(C, H) for _ in range(4))
    m.linear_g, m.linear_z = lin(C, C), lin(H, C)
    m.layer_norm_in = torch.nn.LayerNorm(C, eps=1e-5, elementwise_affine=affine)
    m.layer_norm_out = torch.nn.LayerNorm(H, eps=1e-5, elementwise_affine=affine)
    if affine:
        with torch.no_grad():
            for ln in (m.layer_norm_in, m.layer_norm_out):
                ln.weight.normal_(1, 0.1)
                ln.bias.normal_(0, 0.1)
    return m


def _oracle_weights(m, C, H):
    def wb(layer, lo=None):
        w = layer.weight.detach().cpu().double().numpy()
        b = None if layer.bias is None else layer.bias.detach().cpu().double().numpy()
        if lo is not None:
            w = w[:H] if lo else w[H:]
            b = None if b is None else (b[:H] if lo else b[H:])
        return w, b

    if hasattr(m, "linear_ab_p"):
        parts = {"ap": wb(m.linear_ab_p, True), "ag": wb(m.linear_ab_g, True),
                 "bp": wb(m.linear_ab_p, False), "bg": wb(m.linear_ab_g, False)}
    else:
        parts = {"ap": wb(m.linear_a_p), "ag": wb(m.linear_a_g), "bp": wb(m.linear_b_p),
                 "bg": wb(m.linear_b_g)}
    parts["g"], parts["z"] = wb(m.linear_g), wb(m.linear_z)
    w = {}
    for n, (wt, b) in parts.items():
        w["w_" + n] = wt
        if b is not None:
            w["bias_" + n] = b

    def aff(ln, n):
        if ln.weight is None:
            return np.ones(n), np.zeros(n)
        return ln.weight.detach().cpu().double().numpy(), ln.bias.detach().cpu().double().numpy()

    w["g_in"], w["b_in"] = aff(m.layer_norm_in, C)
    w["g_out"], w["b_out"] = aff(m.layer_norm_out, H)
    return w


def _to(m, dev):
    from types import SimpleNamespace

    out = SimpleNamespace(**vars(m))
    for name, v in vars(m).items():
        if isinstance(v, torch.nn.Module):
            setattr(out, name, v.to(dev))
    return out


TRIMUL_CASES = [
    # B, N, C, H, outgoing, biases, fused, affine, mask_kind
    (1, 64, 128, 128, True, False, False, True, "float"),
    (1, 64, 128, 128, False, False, False, True, "float"),
    (1, 33, 64, 64, True, True, False, True, "bool"),
    (2, 40, 48, 40, False, True, True, True, "float"),
    (1, 17, 30, 22, True, False, False, False, "none"),
    (1, 96, 128, 96, False, True, False, True, "bool"),
    (1, 36, 64, 150, True, False, False, True, "float"),   # 16 channels per thread, H4 pad
    (1, 32, 48, 30, False, True, False, True, "float"),    # 8 channels per thread, H4 pad
    (2, 35, 128, 200, False, False, False, True, "float"),  # 1 pad position, 16 channels per thread
    (1, 129, 32, 32, True, False, False, True, "float"),    # 3 pad positions, tiles end past N
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", TRIMUL_CASES,
                         ids=lambda c: "B{}N{}C{}H{}{}{}{}".format(
                             c[0], c[1], c[2], c[3], "out" if c[4] else "in",
                             "_bias" if c[5] else "", "_fused" if c[6] else ""))
def test_trimul_fp32(gpu, case):
    from oracle.trimul import trimul_forward
    from openfold3_triangle_kernel_amd.trimul_fp32 import run_trimul_fp32

    B, N, C, H, outgoing, biases, fused, affine, mk = case
    m = _trimul_module(C, H, outgoing, biases=biases, fused=fused, affine=affine)
    g = torch.Generator().manual_seed(1)
    z = torch.randn(B, N, N, C, generator=g)
    if mk == "none":
        mask, mask_np = None, np.ones((B, N, N))
    else:
        mb = torch.rand(B, N, N, generator=g) > 0.2
        mask = mb if mk == "bool" else mb.float()
        mask_np = mb.double().numpy()
    print(f"fp32 trimul case={case}", flush=True)
    with torch.no_grad():
        out = run_trimul_fp32(_to(m, gpu), z.to(gpu), None if mask is None else mask.to(gpu))
    torch.cuda.synchronize()
    assert out.dtype == torch.float32 and out.shape == z.shape
    ref, _ = trimul_forward(z.double().numpy(), mask_np, _oracle_weights(m, C, H), outgoing)
    err = max_rel(out.cpu().numpy(), ref)
    assert err <= TOL, err


@pytest.mark.gpu
@pytest.mark.parametrize("seq_major", [False, True])
@pytest.mark.parametrize("B,O,H,N,D", [(1, 2, 1, 1, 4), (1, 3, 2, 31, 32), (2, 2, 2, 33, 20),
                                       (1, 2, 2, 63, 64), (1, 4, 2, 95, 44), (1, 3, 1, 130, 32)])
def test_attention_fp32_any_sequence_length(gpu, B, O, H, N, D, seq_major):
    """N that is not a multiple of 64 is bitwise the caller-padded problem and
    reads nothing past its tensors (NaN there); <= 1e-4 against the oracle."""
    from openfold3_triangle_kernel_amd import turbopairformer_attention_fp32

    print(f"[fp32 attn any N] {B, O, H, N, D} seq={seq_major}", flush=True)
    q, k, v, mask, bias = _f32_case(B, O, H, N, D, mask_tail=max(0, min(7, N - 1)), seed=N)

    def poisoned(t):
        flat = torch.full((t.numel() + 64 * 64 * 8,), float("nan"), device=gpu)
        flat[: t.numel()] = t.reshape(-1)
        return flat[: t.numel()].view(t.shape)

    def run(q, k, v, mask, bias):
        if seq_major:
            q, k, v = (poisoned(t.transpose(-2, -3).contiguous()).transpose(-2, -3)
                       for t in (q, k, v))
        else:
            q, k, v = (poisoned(t) for t in (q, k, v))
        with torch.no_grad():
            return turbopairformer_attention_fp32(q, k, v, poisoned(mask), poisoned(bias))

    out = run(*(t.to(gpu) for t in (q, k, v, mask, bias)))
    p, pad = (-N) % 64, torch.nn.functional.pad
    ref = run(*(pad(t, (0, 0, 0, p)).to(gpu) for t in (q, k, v)),
              pad(mask, (0, p), value=float("-inf")).to(gpu), pad(bias, (0, p, 0, p)).to(gpu))
    assert torch.equal(out, ref[:, :, :N])
    want, _, _ = attention_forward(q.numpy(), k.numpy(), v.numpy(), mask.numpy(), bias.numpy())
    assert max_rel(out.cpu().numpy(), want) <= TOL


@pytest.mark.gpu
@pytest.mark.parametrize("scale", [1.0, 2.0 ** -60, 2.0 ** 50])
@pytest.mark.parametrize("M,N,K", [(1, 1, 4), (130, 65, 36), (257, 128, 100)])
def test_gemm_f32_products_are_fp32(gpu, M, N, K, scale):
    """tpf_gemm_f32 forms its products from three-way bf16 splits: rel-L2
    against FP64 within 2 K^0.5 eps (K additions of random sign; a dropped
    split term of 2^-16 would exceed it), for operands of ordinary and of
    extreme magnitude, and exact on values of one split part."""
    from openfold3_triangle_kernel_amd import _native

    g = torch.Generator().manual_seed(M + K)
    Np = (N + 3) // 4 * 4
    a, b = torch.randn(M, K, generator=g) * scale, torch.randn(Np, K, generator=g) * scale

    def run(a, b):
        a, b = a.to(gpu), b.to(gpu)
        c = torch.empty(M, Np, device=gpu)
        _native.call("tpf_gemm_f32", a.data_ptr(), 1, K, 0, b.data_ptr(), 1, K, 0, c.data_ptr(), Np,
                     0, M, Np, K, 1, 1.0, None, torch.cuda.current_stream().cuda_stream)
        return c.cpu().double()

    ref = a.double() @ b.double().t()
    err = ((run(a, b) - ref).norm() / ref.norm()).item()
    print(f"gemm f32 M={M} N={N} K={K} scale={scale:.1e} rel {err:.2e}", flush=True)
    assert err <= 2 * K ** 0.5 * 2.0 ** -24
    ai, bi = torch.randint(-9, 10, (M, K), generator=g).float(), torch.randint(-9, 10, (Np, K), generator=g).float()
    assert torch.equal(run(ai, bi), ai.double() @ bi.double().t())


def _gemm_f32(a, b, dev):
    """a [M, K] @ b [N, K]^T on tpf_gemm_f32 (K and N multiples of 4), as FP64."""
    from openfold3_triangle_kernel_amd import _native

    (M, K), N = a.shape, b.shape[0]
    a, b, c = a.to(dev), b.to(dev), torch.empty(M, N, device=dev)
    _native.call("tpf_gemm_f32", a.data_ptr(), 1, K, 0, b.data_ptr(), 1, K, 0, c.data_ptr(), N, 0,
                 M, N, K, 1, 1.0, None, torch.cuda.current_stream().cuda_stream)
    return c.cpu().double()


@pytest.mark.gpu
def test_gemm_f32_single_products(gpu):
    """One product per output, over random significands and those whose split
    parts are largest: the dropped terms are below 2^-24 of it and the last sum
    rounds within one unit in the last place, 2^-23 of it (the sums before are
    below 2^-7 of it, hence the factor)."""
    g = torch.Generator().manual_seed(0)
    bits = torch.randint(1 << 23, (256,), generator=g)
    bits[:8] = torch.tensor([0x00FFFF, 0x7FFFFF, 0x008080, 0x008000, 0x007FFF, 0x7F7FFF, 0x018181,
                             0x000001])
    x = ((bits + 0x3F800000).to(torch.int32)).view(torch.float32)
    a = torch.zeros(256, 4)
    a[:, 0] = x
    ref = a.double() @ a.double().t()
    err = ((_gemm_f32(a, a, gpu) - ref).abs() / ref).max().item()
    print(f"single products: largest error {err * 2 ** 24:.3f} * 2^-24", flush=True)
    assert err <= 3 * 2.0 ** -24 * (1 + 2.0 ** -7)


@pytest.mark.gpu
def test_gemm_f32_same_sign_sums_are_unbiased(gpu):
    """Operands of one sign just below 1 + 2^-7 (K = 16, one MFMA step): every
    sum within its 16 roundings and the dropped terms, and no error of one
    sign: the mean over 2^16 sums stays below a quarter of one rounding."""
    g = torch.Generator().manual_seed(1)
    a, b = (1 + 2.0 ** -7 * (1 - 0.1 * torch.rand(256, 16, generator=g)) for _ in range(2))
    ref = a.double() @ b.double().t()
    err = (_gemm_f32(a, b, gpu) - ref) / ref
    print(f"same-sign sums: mean {err.mean() * 2 ** 24:.3f}, largest "
          f"{err.abs().max() * 2 ** 24:.3f} (* 2^-24)", flush=True)
    assert err.abs().max() <= 17 * 2.0 ** -24
    assert err.mean().abs() <= 2.0 ** -26


@pytest.mark.gpu
@pytest.mark.parametrize("special", [float("inf"), float("-inf"), float("nan"), 3.4e38, -3.4e38])
def test_gemm_f32_infinities_and_largest_values(gpu, special):
    """Operands that are infinite, NaN or round to infinity in bf16 act as in
    f32 arithmetic, beside ordinary outputs that keep their values."""
    g = torch.Generator().manual_seed(2)
    a, b = torch.randn(130, 36, generator=g), torch.randn(68, 36, generator=g)
    b[:, 5] = torch.tensor([1.0, -1.0, 0.5, 2.0 ** -20]).repeat(17)  # one split part: m = l = 0
    b[7, 5] = 0.0
    clean = _gemm_f32(a, b, gpu)
    a[3, 5] = special
    a[70, 5] = -special
    got, ref = _gemm_f32(a, b, gpu), a.double() @ b.double().t()
    rows = torch.tensor([r not in (3, 70) for r in range(130)])
    assert torch.equal(got[rows], clean[rows])
    ref = ref.float().double()  # overflow where f32 overflows
    assert torch.equal(got.isnan(), ref.isnan()) and torch.equal(got.isinf(), ref.isinf())
    fin = ref.isfinite()
    assert torch.equal(got[ref.isinf()], ref[ref.isinf()])
    assert ((got - ref).abs()[fin] <= 37 * 2.0 ** -24 * (a.double().abs() @ b.double().abs().t())[fin]).all()


@pytest.mark.gpu
@pytest.mark.parametrize("N,D", [(64, 32), (70, 64)])
def test_attention_fp32_infinities(gpu, N, D):
    """FP32 attention with an infinite value at an unmasked key, a key whose
    score is -inf (weight 0) and a value near the largest float, against the
    same in FP64."""
    from openfold3_triangle_kernel_amd import turbopairformer_attention_fp32

    q, k, v, mask, bias = _f32_case(1, 3, 2, N, D, seed=N)
    q[..., 0] = q[..., 0].abs() + 0.1
    k[0, 0, 0, 5, 0] = float("-inf")
    v[0, 1, 1, 9, 3] = float("inf")
    v[0, 1, 1, 11, 4] = float("-inf")
    v[0, 2, 0, 40, 7] = 3.4e38
    bias[..., 40] -= 30  # (its weight well below 1: the sums are unnormalised)
    with torch.no_grad():
        out = turbopairformer_attention_fp32(*(t.to(gpu) for t in (q, k, v, mask, bias))).cpu()
    s = (q.double() @ k.double().transpose(-1, -2)) / D ** 0.5 + mask.double() + bias.double()
    ref = (torch.softmax(s, -1) @ v.double()).transpose(-2, -3)
    assert torch.equal(out.isnan(), ref.isnan()) and torch.equal(out.isinf(), ref.isinf())
    assert torch.equal(out[ref.isinf()].double(), ref[ref.isinf()]) and ref.isinf().any()
    assert not ref.isnan().any()
    fin = ref.isfinite()
    rel = (out.double() - ref).abs()[fin] / ref.abs()[fin].clamp(min=1e-2)
    assert rel.max() <= TOL
