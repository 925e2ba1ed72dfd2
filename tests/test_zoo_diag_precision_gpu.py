"""GPU test of the precision of the intra-chunk product under per-channel decay (zoo_diag_prep.h) against float64."""

import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

BC = 16


def _chunks(t, H):
    B, T = t.shape[:2]
    return t.reshape(B, T // 64, 64, H, -1).permute(0, 1, 3, 2, 4)


def _off_diagonal(q, k, g, rot, sq, sk, scale, dtype):
    """The blocks of A below the diagonal ones in ``dtype``, every product and exponential rounded on its own (e^x as 2^(x log2 e), one
    for each element and anchor); the rotation's operands in fp16.  q, k, g [B, NT, H, 64, K]."""
    q, k, g, sq, sk = (t.to(dtype) for t in (q, k, g, sq, sk))
    ex = lambda x: torch.exp2(x * 1.4426950408889634) if dtype == torch.float32 else torch.exp(x)  # noqa: E731
    code = lambda x, s: torch.trunc(x * (1 / s) + torch.copysign(torch.full_like(x, 0.5), x)).clamp(-127, 127)  # noqa: E731
    A = q.new_zeros(*q.shape[:-1], 64)
    for i in range(BC, 64, BC):
        a = g[..., i:i + 1, :]
        x, y = q[..., i:i + BC, :] * ex(g[..., i:i + BC, :] - a) * scale, k[..., :i, :] * ex(a - g[..., :i, :])
        if rot is not None:
            x, y = (t.half().to(dtype) @ rot.to(dtype) for t in (x, y))
        A[..., i:i + BC, :i] = (code(x, sq) @ code(y, sk).transpose(-1, -2).contiguous()) * (sq * sk)
    return A


@pytest.mark.parametrize("K,dtype,rotate", [(128, torch.float16, True), (128, torch.bfloat16, True), (64, torch.float16, True),
                                            (128, torch.float16, False)])
@pytest.mark.parametrize("gscale", [0.3, 1.0, 3.0])
def test_off_diagonal_blocks_are_no_further_from_float64_than_their_fp32_form(cuda, K, dtype, rotate, gscale):
    """Entries of A that are not the float64 value's fp16: at most those of the fp32 form, a quarter more for the hardware's exp2 (one
    unit in the last place) and the order of the rotation's sums, and 64 for a code on the other side of a tie, which moves up to 16
    entries of its row or column: four of them at once."""
    from linquant_amd.kernels.zoo import _common as C

    B, T, H = 2, 4096, 16
    gen = torch.Generator(device="cuda").manual_seed(K)
    rn = lambda *s: torch.randn(*s, generator=gen, device="cuda")  # noqa: E731
    q, k = rn(B, T, H, K).to(dtype), torch.nn.functional.normalize(rn(B, T, H, K), dim=-1).to(dtype)
    g = torch.nn.functional.logsigmoid(rn(B, T, H, K) + 1.0) * gscale
    gc = g.reshape(B, T // 64, 64, H, K).double().cumsum(2).float().reshape(B, T, H, K).contiguous()
    scale = K ** -0.5
    sq, sk = ((t.float().abs().amax(dim=(0, 1, 3)) / 127).contiguous() for t in (q, k))
    sq = sq * scale
    rot = None
    if rotate:
        R = torch.ones(1, 1, device="cuda")
        while R.shape[0] < K:
            R = torch.cat([torch.cat([R, R], 1), torch.cat([R, -R], 1)], 0)
        rot = (R / math.sqrt(K) * (torch.randint(0, 2, (K,), generator=gen, device="cuda") * 2 - 1)).half().contiguous()
    A, _ = C.run_gla_A(q, k, gc, sq, sk, scale, 127, (B, T, H, K, K), rot=rot)
    got = _chunks(A, H)
    scales = [t.view(1, 1, H, 1, 1) for t in (sq, sk)]
    ref, plain = [_off_diagonal(_chunks(q, H), _chunks(k, H), _chunks(gc, H), rot, *scales, scale, d).half() for d in (torch.float64, torch.float32)]
    below = torch.arange(64, device="cuda")[:, None] // BC > torch.arange(64, device="cuda")[None, :] // BC
    off, off32 = [int((t != ref)[..., below].sum()) for t in (got, plain)]
    print(f"K {K} {dtype} rotate {rotate} gscale {gscale}: {off} entries, fp32 form {off32}")
    assert float(ref[..., below].float().abs().max()) > 0
    assert off <= 1.25 * off32 + 64, (off, off32)


@pytest.mark.parametrize("K", [64, 128])
def test_entries_of_A_are_rounded_once(cuda, K):
    """Without decay every entry is a whole number times the fp32 product of the two scales: it is stored as the fp16 nearest to that
    exact product, not to its fp32 rounding."""
    from linquant_amd.kernels.zoo import _common as C

    B, T, H = 2, 1024, 8
    gen = torch.Generator().manual_seed(K)
    cq, ck = (torch.randint(-127, 128, (B, T, H, K), generator=gen) for _ in range(2))
    sq, sk = (torch.rand(H, generator=gen) * 0.01 + 0.005 for _ in range(2))
    q, k = ((c * s[None, None, :, None]).half() for c, s in ((cq, sq), (ck, sk)))  # (fp16: within 0.07 of the code's middle)
    A, _ = C.run_gla_A(q.cuda(), k.cuda(), torch.zeros(B, T, H, K, device="cuda"), sq.cuda(), sk.cuda(), 1.0, 127, (B, T, H, K, K))
    dots = (_chunks(cq.double(), H) @ _chunks(ck.double(), H).transpose(-1, -2)).tril().numpy()
    sqk = (sq * sk).view(1, 1, H, 1, 1).numpy()
    once = (dots * sqk.astype(np.float64)).astype(np.float16)  # (the product is exact in 53 bits)
    twice = (dots.astype(np.float32) * sqk).astype(np.float16)
    assert (once != twice).sum() > 8
    assert np.array_equal(_chunks(A.cpu(), H).numpy(), once)
