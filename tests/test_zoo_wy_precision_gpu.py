"""GPU test of the precision of the delta family's WY transform (zoo_wy_ns.hip: no or scalar decay; zoo_diag_prep.h: per-channel decay)
against float64: T = (I + G)^-1 holds 24 bits per entry whatever its size beside the others of its row; W and U of the first are no
further from the float64 transform than those of the same transform in plain fp32 (torch on the CPU, no kernel of this library), those of
the second no further than the measured ones of the stand-alone kernel that it replaced."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _transform(k, v, beta, gc, sigma, dtype=torch.float64):
    """W, U in ``dtype``, from the half-precision operands (64-token chunks): T by forward substitution into the identity, then T.X.
    gc: cumulative decay (B, T, H), or (B, T, H, K) per channel."""
    B, T, H, _ = k.shape
    chunks = lambda t: t.to(dtype).reshape(B, T // 64, 64, H, -1).permute(0, 1, 3, 2, 4).contiguous()  # noqa: E731
    kd, vd, b = chunks(k), chunks(v), chunks(beta)
    bs, bh = b ** sigma, b ** (1 - sigma)
    X, Y = kd * bs, kd * bh
    if gc is None or gc.dim() == 3:
        G = X @ Y.transpose(-1, -2).contiguous()
    else:
        G = torch.empty(*X.shape[:-1], 64, dtype=dtype, device=k.device)
        g = chunks(gc)
        for i in range(64):  # (row by row: the decays of all pairs at once would be 64 times k)
            G[..., i, :] = ((X[..., i:i + 1, :] * Y) * torch.exp((g[..., i:i + 1, :] - g).clamp(max=0))).sum(-1)
        X = X * torch.exp(g)
    if gc is not None and gc.dim() == 3:
        g = chunks(gc)
        G, X = G * torch.exp(g - g.transpose(-1, -2)), X * torch.exp(g)
    eye = torch.eye(64, dtype=dtype, device=k.device)
    Tm = torch.linalg.solve_triangular(torch.tril(G, -1) + eye, eye.expand(G.shape), upper=False, unitriangular=True)
    back = lambda t: t.permute(0, 1, 3, 2, 4).reshape(B, T, H, -1)  # noqa: E731
    return [back(Tm @ t) for t in (X, bs * vd)]


@pytest.mark.parametrize("K,V", [(64, 64), (128, 128)])
def test_strongly_decayed_entries_of_T_keep_their_bits(cuda, K, V):
    """Orthogonal keys behind a first one that meets them all, a large value at the head of the chunk and zeros behind it: U_i is
    the one entry -G_i0 of T, down to 2^-28 of its row's largest, times that value.  Bound: half a unit of fp16 (2^-11), and 2^-17
    for the handful of fp32 roundings in front of it, of which the exponential's argument (up to 24 times 2^-24) is the largest."""
    from linquant_amd.kernels.zoo import _common as C

    B, T, H = 2, 128, 3
    gen = torch.Generator(device="cuda").manual_seed(K)
    k = torch.zeros(64, K, device="cuda")
    k[torch.arange(1, 64), torch.arange(1, 64)] = 1.0
    k[0, 1:64] = 63 ** -0.5
    k = k.half().repeat(T // 64, 1).view(1, T, 1, K).expand(B, T, H, K).contiguous()
    v = torch.zeros(B, T, H, V, device="cuda")
    v[:, ::64] = torch.randint(20000, 60000, (B, T // 64, H, V), generator=gen, device="cuda").float()
    v = v.half()
    beta = torch.rand(B, T, H, generator=gen, device="cuda") * 0.5 + 0.5
    gc = (-0.26 * torch.arange(1, 65, device="cuda").float()).repeat(T // 64).view(1, T, 1).expand(B, T, H).contiguous()
    _, W, U, _, _ = C.run_wy_prep(k, v, beta, gc, 0.5, 1.0, (B, T, H, K, V), C.DECAY_SCALAR)
    ref = _transform(k, v, beta, gc, 0.5)[1]
    normal = ref.abs() > 2.0 ** -14
    assert (normal & (ref.abs() < 2.0 ** -9)).float().mean().item() > 0.1  # the decayed end of the chunk is in the comparison
    err = ((U.double() - ref).abs() / ref.abs())[normal].max().item()
    assert err <= 2.0 ** -11 + 2.0 ** -17, err * 2.0 ** 11


def _misrounded(decay, dtype, K, V, sigma, norm):
    """Shares of the W and U entries on the other side of a rounding boundary than the float64 transform, over 2 M entries or more:
    [(kernel, plain fp32 or None)]."""
    from linquant_amd.kernels.zoo import _common as C

    B, T, H = 4, 1024, 8
    gen = torch.Generator(device="cuda").manual_seed(7)
    rn = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    k = (torch.nn.functional.normalize(rn(B, T, H, K), dim=-1) * norm).to(dtype)
    v, beta = rn(B, T, H, V).to(dtype), torch.sigmoid(rn(B, T, H) - (2.0 if norm > 1 else 0.0))
    gc = None
    if decay != "none":
        g = torch.nn.functional.logsigmoid(rn(B, T, H) + 2.0 if decay == "scalar" else rn(B, T, H, K) + 1.0)
        gc = g.reshape(B, T // 64, 64, H, -1).double().cumsum(2).float().reshape(g.shape).contiguous()
    code = {"none": C.DECAY_NONE, "scalar": C.DECAY_SCALAR, "diagonal": C.DECAY_DIAGONAL}[decay]
    _, W, U, _, _ = C.run_wy_prep(k, v, beta, gc, sigma, 1.0, (B, T, H, K, V), code)
    ref = [t.to(dtype) for t in _transform(k, v, beta, gc, sigma)]
    share = lambda t, r: (t.to(r) != r).double().mean().item()  # noqa: E731
    if decay == "diagonal":
        return [(share(t, r), None) for t, r in zip((W, U), ref)]
    plain = _transform(*(None if t is None else t.cpu() for t in (k, v, beta, gc)), sigma, torch.float32)
    return [(share(t, r), share(p, r)) for t, p, r in zip((W, U), plain, ref)]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("decay", ["none", "scalar"])
@pytest.mark.parametrize("K,V,sigma,norm", [(128, 128, 1.0, 1.0), (64, 64, 0.5, 1.0), (128, 64, 0.5, 3.0)])
def test_W_and_U_are_no_further_from_float64_than_in_plain_fp32(cuda, dtype, decay, K, V, sigma, norm):
    """Measured: 0.52 to 0.84 of the plain form's misrounded entries."""
    for name, (off, off0) in zip("WU", _misrounded(decay, dtype, K, V, sigma, norm)):
        assert off <= off0 < 0.01, f"{name}: {off:.2e} of the entries, plain fp32 {off0:.2e}"


# W and U of the kernel that made the transform alone (Gram product anchored at the chunk's middle row, the same three bf16 pieces in
# T.X), measured on these inputs
@pytest.mark.parametrize("dtype,K,V,sigma,norm,before", [
    (torch.float16, 128, 128, 1.0, 1.0, (9.73e-5, 1.74e-4)), (torch.bfloat16, 128, 128, 1.0, 1.0, (3.73e-4, 2.48e-5)),
    (torch.float16, 64, 64, 0.5, 1.0, (1.67e-4, 2.26e-4)), (torch.bfloat16, 64, 64, 0.5, 1.0, (4.06e-4, 4.29e-5)),
    (torch.float16, 128, 64, 0.5, 3.0, (3.11e-4, 4.82e-4)), (torch.bfloat16, 128, 64, 0.5, 3.0, (5.76e-4, 6.91e-5))])
def test_W_and_U_under_per_channel_decay_are_no_further_from_float64_than_before(cuda, dtype, K, V, sigma, norm, before):
    """Decay of its own on every channel.  Measured: 0.45 to 0.85 of the former kernel's misrounded entries."""
    for name, (off, _), off0 in zip("WU", _misrounded("diagonal", dtype, K, V, sigma, norm), before):
        assert off <= off0, f"{name}: {off:.2e} of the entries, before {off0:.2e}"
