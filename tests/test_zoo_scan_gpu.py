"""GPU test of the launch that runs the chunk recurrence and the output together (zoo_scan.hip) at the edges of its loops and
grids, against the stage-by-stage kernels, which the float64 oracle pins in test_zoo_gpu.py: every value is the same arithmetic
in the same order, so outputs and final states are equal bit for bit."""

import pytest
import torch

from linquant_amd import _lib
from tests import zoo_cases as zc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cell", list(zc.CELLS))
# chunks: fewer than the operand sets in rotation (3 and 2), exactly as many, remainders of one and of all but one; grids that
# do and do not divide over the 8 XCDs; one and several V tiles per head, a V the operand prologue is not built for (192)
@pytest.mark.parametrize("NT,B,H,K,V,dtype,out_dtype", [
    (1, 1, 1, 128, 64, torch.float16, None), (2, 1, 8, 64, 128, torch.bfloat16, None), (3, 2, 3, 128, 192, torch.float16, None),
    (5, 1, 5, 64, 64, torch.float16, torch.float32), (6, 3, 2, 128, 128, torch.bfloat16, torch.float32),
    (11, 2, 4, 128, 128, torch.float16, None),
    # more than 128 workgroups of 32 value columns: the 32-column kernel, over the same edges of loops, grids, widths and types, with
    # more workgroups than fit the chip at once in the last two
    (1, 5, 14, 64, 64, torch.float16, None), (2, 3, 23, 128, 64, torch.bfloat16, None), (3, 1, 36, 64, 128, torch.float16, torch.float32),
    (4, 2, 17, 128, 128, torch.bfloat16, None), (5, 5, 13, 64, 64, torch.bfloat16, torch.float32), (6, 3, 11, 128, 128, torch.float16, None),
    (7, 1, 24, 128, 192, torch.bfloat16, None), (8, 9, 8, 128, 128, torch.float16, torch.float32), (3, 5, 27, 64, 128, torch.bfloat16, None),
    # more than 128 steps of few chains: the linear family's stages one after the other behind the same call, the delta family's one launch
    (130, 1, 2, 128, 64, torch.bfloat16, None)])
def test_recurrence_and_output_in_one_launch_equal_the_staged_kernels(cuda, cell, NT, B, H, K, V, dtype, out_dtype):
    from linquant_amd.kernels import zoo
    from oracle.zoo_reference import signed_hadamard

    q, k, v, g, beta = [t.to(cuda) if t is not None else None for t in zc.inputs(cell, B=B, T=64 * NT, H=H, K=K, V=V, seed=NT, dtype=dtype)]
    gen = torch.Generator().manual_seed(NT)
    r = lambda *shape, lo, hi: (torch.rand(*shape, generator=gen) * (hi - lo) + lo).to(cuda)  # noqa: E731
    sc = {"q": r(H, lo=0.001, hi=0.003), "k": r(H, lo=0.005, hi=0.01), "w": r(H, lo=0.02, hi=0.04), "kw": r(H, K, lo=0.005, hi=0.015),
          "vw": r(H, V, lo=0.02, hi=0.04), "vl": r(H, V, lo=0.02, hi=0.04), "el": r(H, V, lo=0.04, hi=0.06),
          "ew": r(H, V, lo=0.04, hi=0.06), "state": r(H, V, lo=0.02, hi=0.07)}
    fam, dec = zc.CELLS[cell]
    kw = dict(eta=0.25, output_final_state=True, out_dtype=out_dtype)
    if dec == "diagonal":
        kw["rot"] = signed_hadamard(K, 2).float().to(cuda)
    if fam == "delta":
        kw.update(sigma=0.5, tau=0.5)
        fn = zoo.chunk_kda_int8 if dec == "diagonal" else zoo.chunk_delta_int8
        args = (q, k, v, g, beta, sc)
    else:
        fn = zoo.chunk_gla_int8 if dec == "diagonal" else zoo.chunk_simple_gla_int8
        args = (q, k, v, g, sc)
    o1, h1 = fn(*args, **kw)
    o0, h0 = fn(*args, _debug={}, **kw)
    torch.cuda.synchronize()
    assert o1.dtype == (out_dtype or dtype) and float(o1.float().abs().max()) > 0
    assert torch.equal(o0, o1) and torch.equal(h0, h1)


# row widths that share the workgroup's waves differently, the scalar decay's fp64 running sum, every part of the prologue
@pytest.mark.parametrize("cell,NT,B,H,K,V,dtype,parts", [
    ("linear_none", 2, 1, 3, 128, 128, torch.float16, ("signs_qk", "signs_v", "dqk")), ("mamba2", 3, 2, 4, 64, 128, torch.bfloat16, ("signs_v",)),
    ("mamba2", 1, 1, 1, 128, 64, torch.float16, ("signs_qk", "dqk")), ("linear_none", 4, 2, 2, 64, 64, torch.bfloat16, ("dqk",)),
    # 40 chunks: one launch for few chains and for many
    ("mamba2", 40, 1, 2, 128, 64, torch.float16, ("signs_qk", "signs_v")), ("linear_none", 40, 4, 8, 128, 128, torch.bfloat16, ("signs_qk", "dqk")),
    # the stages one after the other behind the same call: few chains of more than 128 steps; K = V = 64 and more than 2048 chunks
    ("mamba2", 130, 1, 2, 128, 64, torch.float16, ("signs_qk", "signs_v")), ("linear_none", 40, 2, 32, 64, 64, torch.bfloat16, ("signs_qk", "dqk")),
    # 32 value columns per workgroup
    ("mamba2", 3, 5, 8, 128, 128, torch.bfloat16, ("signs_qk",)), ("mamba2", 2, 3, 23, 64, 64, torch.float16, ("signs_v", "dqk"))])
def test_operand_prologue_in_the_one_call_forward_equals_the_staged_kernels(cuda, cell, NT, B, H, K, V, dtype, parts):
    from linquant_amd.kernels import zoo

    q, k, v, g, _ = [t.to(cuda) if t is not None else None for t in zc.inputs(cell, B=B, T=64 * NT, H=H, K=K, V=V, seed=NT, dtype=dtype)]
    gen = torch.Generator().manual_seed(NT)
    r = lambda *shape, lo, hi: (torch.rand(*shape, generator=gen) * (hi - lo) + lo).to(cuda)  # noqa: E731
    sc = {"q": r(H, lo=0.001, hi=0.003), "k": r(H, lo=0.005, hi=0.03), "kw": r(H, K, lo=0.005, hi=0.03), "vw": r(H, V, lo=0.02, hi=0.04),
          "vl": r(H, V, lo=0.02, hi=0.04), "state": r(H, V, lo=0.02, hi=0.07)}
    every = {"signs_qk": (r(K, lo=-1, hi=1)).sign(), "signs_v": (r(V, lo=-1, hi=1)).sign(), "dqk": r(H, K, lo=0.5, hi=2.0)}
    kw = dict(eta=0.75, output_final_state=True, prologue={n: every[n] for n in parts})
    o1, h1 = zoo.chunk_simple_gla_int8(q, k, v, g, sc, **kw)
    o0, h0 = zoo.chunk_simple_gla_int8(q, k, v, g, sc, _staged=True, **kw)
    torch.cuda.synchronize()
    assert float(o1.float().abs().max()) > 0
    assert torch.equal(o0, o1) and torch.equal(h0, h1)


# chains in segments: cuts at multiples of four (three: K = 128, 32 value columns), as many as the chain has room for (16 segments of
# at least one cut step, fewer), one that starts in the last chunk; the lines between 16 and 32 columns (12, 32 and 256 steps; 42 and 64
# tiles of 32), the last grid with two segments and the first with one
@pytest.mark.parametrize("cell", ["linear_none", "mamba2", "gla"])
@pytest.mark.parametrize("NT,B,H,K,V,dtype,out_dtype", [
    (4, 1, 1, 64, 64, torch.float16, None), (5, 1, 1, 128, 64, torch.bfloat16, None), (13, 1, 2, 64, 64, torch.float16, torch.float32),
    (64, 1, 1, 64, 64, torch.bfloat16, None), (65, 2, 1, 128, 128, torch.float16, None), (30, 3, 1, 128, 192, torch.float16, None),
    (33, 1, 11, 128, 128, torch.bfloat16, None), (34, 2, 11, 64, 64, torch.float16, torch.float32), (32, 1, 16, 128, 128, torch.float16, None),
    (12, 1, 17, 128, 128, torch.float16, None), (13, 1, 17, 128, 128, torch.float16, None), (14, 1, 32, 64, 128, torch.bfloat16, None),
    (13, 3, 11, 128, 128, torch.float16, torch.float32), (257, 1, 9, 64, 128, torch.float16, None), (258, 1, 17, 128, 64, torch.bfloat16, None)])
def test_a_chain_in_segments_equals_the_staged_kernels(cuda, cell, NT, B, H, K, V, dtype, out_dtype):
    test_recurrence_and_output_in_one_launch_equal_the_staged_kernels(cuda, cell, NT, B, H, K, V, dtype, out_dtype)


# the same with the operand prologue, whose route differs: chains of more than 128 steps in segments, and on the other side of its line
# (K = V = 64, more than 80 tiles, more than 64 steps) the stages behind the same call
@pytest.mark.parametrize("cell", ["linear_none", "mamba2"])
@pytest.mark.parametrize("NT,B,H,K,V,dtype,parts", [
    (257, 1, 9, 64, 128, torch.float16, ("signs_qk",)), (258, 1, 17, 128, 64, torch.bfloat16, ("signs_qk", "signs_v")),
    (131, 1, 3, 128, 128, torch.float16, ("dqk",)), (64, 1, 41, 64, 64, torch.float16, ("signs_qk",)), (65, 1, 41, 64, 64, torch.float16, ("signs_qk",))])
def test_a_chain_in_segments_behind_the_prologue_equals_the_staged_kernels(cuda, cell, NT, B, H, K, V, dtype, parts):
    test_operand_prologue_in_the_one_call_forward_equals_the_staged_kernels(cuda, cell, NT, B, H, K, V, dtype, parts)


# the running sum of a 64-token chunk by its thread-wide form (lq_zoo_cumsum) against fp64: the orders differ by fp64 roundings only, which
# move an fp32 result by one unit in the last place at most; one token that forgets everything, in each 16 of the chunk
@pytest.mark.parametrize("at", [None, 0, 15, 16, 40, 63])
def test_cumulative_scalar_decay_of_64_tokens(cuda, at):
    from linquant_amd.kernels.zoo import _common as C

    B, NT, H = 3, 5, 7
    g = -torch.rand(B, 64 * NT, H, generator=torch.Generator().manual_seed(3)) ** 4 * 8
    if at is not None:
        g[1, 128 + at, 2] = float("-inf")
    out = C.cumsum(g.to(cuda), B, 64 * NT, H, 0)[0].cpu().view(B, NT, 64, H)
    ref = g.double().view(B, NT, 64, H).cumsum(2)
    assert torch.equal(torch.isinf(out), torch.isinf(ref))
    fin = torch.isfinite(ref)
    assert ((out[fin].double() - ref[fin]).abs() <= ref[fin].abs() * 2.0 ** -23).all()


# its order, to the bit: inside each 16 tokens by sums over the last 1, 2, 4, 8 values, then the totals of the 16s before; columns that fill
# a workgroup's 64 and that do not, also where the result takes the place of the input
@pytest.mark.parametrize("B,NT,H", [(1, 1, 1), (1, 3, 21), (2, 2, 16), (5, 13, 1), (3, 17, 5), (1, 5, 130)])
@pytest.mark.parametrize("in_place", [False, True])
def test_cumulative_scalar_decay_takes_the_order_of_the_waves(cuda, B, NT, H, in_place):
    g = -torch.rand(B, 64 * NT, H, generator=torch.Generator().manual_seed(H)) ** 4 * 8
    x = g.double().view(B, NT, 4, 16, H)
    for s in (1, 2, 4, 8):
        x = torch.cat([x[..., :s, :], x[..., s:, :] + x[..., :-s, :]], 3)
    t0, t1, t2 = x[:, :, :3, -1:].clone().unbind(2)
    x[:, :, 1] += t0
    x[:, :, 3] += t2
    x[:, :, 2:] += (t1 + t0)[:, :, None]
    gin = g.to(cuda)
    out = gin if in_place else torch.empty_like(gin)
    _lib.call("lq_zoo_cumsum", gin.device, g=gin.data_ptr(), gc=out.data_ptr(), batch=B, seqlen=64 * NT, nheads=H, kdim=0, chunk_size=64)
    assert torch.equal(out.cpu(), x.float().view(g.shape))


# the same sum across the lanes of a wave, in the launches that make it themselves: what a decay of minus infinity cuts off is cut off
@pytest.mark.parametrize("cell", ["mamba2", "gated_deltanet"])
@pytest.mark.parametrize("at", [0, 15, 16, 40, 63])
def test_a_scalar_decay_that_forgets_everything_equals_the_staged_kernels(cuda, cell, at):
    from linquant_amd.kernels import zoo

    B, T, H, K, V = 1, 192, 3, 64, 64
    q, k, v, g, beta = [t.to(cuda) if t is not None else None for t in zc.inputs(cell, B=B, T=T, H=H, K=K, V=V, seed=at, dtype=torch.float16)]
    g[0, 64 + at, 1] = -200.0
    sc = {n: torch.full((H,), x, device=cuda) for n, x in (("q", 0.002), ("k", 0.008), ("w", 0.03))}
    sc.update(kw=torch.full((H, K), 0.01, device=cuda), **{n: torch.full((H, V), 0.03, device=cuda) for n in ("vw", "vl", "el", "ew", "state")})
    fn, args = (zoo.chunk_simple_gla_int8, (q, k, v, g, sc)) if cell == "mamba2" else (zoo.chunk_delta_int8, (q, k, v, g, beta, sc))
    o1, h1 = fn(*args, eta=0.25, output_final_state=True)
    o0, h0 = fn(*args, eta=0.25, output_final_state=True, _staged=True)
    assert float(o1.float().abs().max()) > 0 and torch.isfinite(o1).all()
    assert torch.equal(o0, o1) and torch.equal(h0, h1)
