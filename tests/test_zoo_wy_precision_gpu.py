"""GPU test of the precision of the delta family's WY transform without or with scalar decay (zoo_wy_ns.hip) against float64:
T = (I + G)^-1 holds 24 bits per entry whatever its size beside the others of its row, and W and U are no further from the float64
transform than those of the fp32 form (the per-channel-decay kernel given the same decay on every channel)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


def _transform(k, v, beta, gc, sigma):
    """W, U in float64 on the GPU, from the half-precision operands (64-token chunks)."""
    B, T, H, _ = k.shape
    chunks = lambda t: t.double().reshape(B, T // 64, 64, H, -1).permute(0, 1, 3, 2, 4).contiguous()  # noqa: E731
    kd, vd, b = chunks(k), chunks(v), chunks(beta)
    bs, bh = b ** sigma, b ** (1 - sigma)
    G, X = (kd * bs) @ (kd * bh).transpose(-1, -2).contiguous(), kd * bs
    if gc is not None:
        g = chunks(gc)
        G, X = G * torch.exp(g - g.transpose(-1, -2)), X * torch.exp(g)
    A = torch.tril(G, -1) + torch.eye(64, dtype=torch.float64, device=k.device)
    back = lambda t: t.permute(0, 1, 3, 2, 4).reshape(B, T, H, -1)  # noqa: E731
    return [back(torch.linalg.solve_triangular(A, t, upper=False, unitriangular=True)) for t in (X, bs * vd)]


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


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("scalar", [False, True])
@pytest.mark.parametrize("K,V,sigma,norm", [(128, 128, 1.0, 1.0), (64, 64, 0.5, 1.0), (128, 64, 0.5, 3.0)])
def test_W_and_U_are_no_further_from_float64_than_the_fp32_form(cuda, dtype, scalar, K, V, sigma, norm):
    """Share of W and U entries on the other side of a rounding boundary than the float64 transform, over 2 M entries or more: no
    larger than in the fp32 form (measured: 0.4 to 0.8 of it)."""
    from linquant_amd.kernels.zoo import _common as C

    B, T, H = 4, 1024, 8
    gen = torch.Generator(device="cuda").manual_seed(7)
    rn = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    k = (torch.nn.functional.normalize(rn(B, T, H, K), dim=-1) * norm).to(dtype)
    v, beta = rn(B, T, H, V).to(dtype), torch.sigmoid(rn(B, T, H) - (2.0 if norm > 1 else 0.0))
    gc = None
    if scalar:
        g = torch.nn.functional.logsigmoid(rn(B, T, H) + 2.0)
        gc = g.reshape(B, T // 64, 64, H).double().cumsum(2).float().reshape(B, T, H).contiguous()
    dims = (B, T, H, K, V)
    _, W, U, _, _ = C.run_wy_prep(k, v, beta, gc, sigma, 1.0, dims, C.DECAY_SCALAR if scalar else C.DECAY_NONE)
    per_channel = (torch.zeros(B, T, H, device="cuda") if gc is None else gc)[..., None].expand(B, T, H, K).contiguous()
    _, W0, U0, _, _ = C.run_wy_prep(k, v, beta, per_channel, sigma, 1.0, dims, C.DECAY_DIAGONAL)
    for name, got, other, ref in zip("WU", (W, U), (W0, U0), _transform(k, v, beta, gc, sigma)):
        off, off0 = [(t != ref.to(dtype)).double().mean().item() for t in (got, other)]
        assert off <= off0 < 0.01, f"{name}: {off:.2e} of the entries, the fp32 form {off0:.2e}"
