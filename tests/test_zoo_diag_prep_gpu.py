"""GPU test of the launch in front of the recurrence under per-channel decay (zoo_diag_prep.h) at the edges of its branches: sub-blocks
whose decay is factorized and sub-blocks that take one exponential per product in one chunk, grids that do and do not divide over the
8 XCDs, both key widths, value widths of one pass, several and a partial last one, with and without rotation and D_QK.  Its fused forms
run the code of the stage entry points, so outputs and final states are equal bit for bit: that comparison pins the forms to each other,
the last test here and test_zoo_gpu.py pin them to the float64 oracle."""

import pytest
import torch

from tests import zoo_cases as zc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cell", ["gla", "kda"])
@pytest.mark.parametrize("B,NT,H,K,V,dtype,rot,dqk,sigma", [
    (1, 1, 1, 64, 64, torch.float16, False, False, 1.0), (2, 4, 3, 128, 128, torch.bfloat16, True, True, 0.5),
    (1, 3, 5, 128, 64, torch.float16, True, False, 1.0), (2, 2, 4, 64, 192, torch.bfloat16, True, True, 0.0),
    (3, 8, 2, 128, 192, torch.float16, False, True, 0.5), (1, 2, 3, 64, 128, torch.float16, True, False, 0.5),
    (1, 5, 1, 128, 320, torch.bfloat16, False, False, 1.0), (1, 130, 1, 64, 64, torch.float16, True, False, 1.0)])
def test_one_launch_equals_the_stages_in_every_branch(cuda, cell, B, NT, H, K, V, dtype, rot, dqk, sigma):
    from linquant_amd.kernels import zoo
    from oracle.zoo_reference import signed_hadamard

    T = 64 * NT
    q, k, v, g, beta = zc.inputs(cell, B=B, T=T, H=H, K=K, V=V, seed=NT, dtype=dtype)
    gen = torch.Generator().manual_seed(H)
    # sub-blocks of 16 tokens: a third as drawn, a third near the factorization's limit, a third far beyond it in some channels
    kind = torch.randint(0, 3, (B, T // 16, H, 1), generator=gen).repeat_interleave(16, dim=1)
    far = torch.where(torch.rand(B, T, H, K, generator=gen) < 0.1, 60.0, 1.0)
    g = (g * torch.where(kind == 0, torch.ones(()), torch.where(kind == 1, torch.tensor(4.0), far))).contiguous()
    q, k, v, g = q.to(cuda), k.to(cuda), v.to(cuda), g.to(cuda)
    r = lambda *shape, lo, hi: (torch.rand(*shape, generator=gen) * (hi - lo) + lo).to(cuda)  # noqa: E731
    sc = {"q": r(H, lo=0.001, hi=0.003), "k": r(H, lo=0.005, hi=0.01), "w": r(H, lo=0.02, hi=0.04), "kw": r(H, K, lo=0.005, hi=0.015),
          "vw": r(H, V, lo=0.02, hi=0.04), "vl": r(H, V, lo=0.02, hi=0.04), "el": r(H, V, lo=0.04, hi=0.06),
          "ew": r(H, V, lo=0.04, hi=0.06), "state": r(H, V, lo=0.02, hi=0.07)}
    kw = dict(eta=0.25, output_final_state=True, rot=signed_hadamard(K, 2).float().to(cuda) if rot else None)
    if cell == "kda":
        kw.update(sigma=sigma, tau=0.5, dqk=r(H, K, lo=0.25, hi=1.75) if dqk else None)
        call = lambda **x: zoo.chunk_kda_int8(q, k, v, g, beta.to(cuda), sc, **kw, **x)  # noqa: E731
    else:
        call = lambda **x: zoo.chunk_gla_int8(q, k, v, g, sc, **kw, **x)  # noqa: E731
    o1, h1 = call()
    o0, h0 = call(_debug={})
    torch.cuda.synchronize()
    assert torch.isfinite(o1.float()).all() and float(o1.float().abs().max()) > 0
    assert torch.equal(o0, o1) and torch.equal(h0, h1)


@pytest.mark.parametrize("cell", ["gla", "kda"])
@pytest.mark.parametrize("K,rot", [(64, False), (128, False), (128, True)])
@pytest.mark.parametrize("staged", [False, True])
def test_halves_of_a_sub_block_that_decide_apart_match_the_oracle(cuda, cell, K, rot, staged):
    """The two waves of a 16-token sub-block, half of the channels each, decide for themselves whether its decay is factorized: here the
    lower, the upper, both or neither half of the channels decays by far more than e^40 in it, every order of the four in a chunk."""
    from oracle.zoo_reference import signed_hadamard

    B, T, H, V = 1, 64 * 6, 4, 64
    q, k, v, g, beta = zc.inputs(cell, B=B, T=T, H=H, K=K, V=V, seed=K)
    gen = torch.Generator().manual_seed(3)
    order = torch.stack([torch.randperm(4, generator=gen) for _ in range(T // 64 * H)]).view(T // 64, H, 4).permute(0, 2, 1)
    kind = order.reshape(T // 16, H).repeat_interleave(16, dim=0)  # bit 0: the lower half of the channels, bit 1: the upper
    far = torch.stack([kind & 1, kind >> 1], dim=-1).repeat_interleave(K // 2, dim=-1).bool()
    some = torch.rand(T, H, K, generator=gen) < 0.2  # (in one channel of five, so that the others still carry the output)
    g = torch.where(far & some, g * 60.0, g).contiguous()
    rise = g.view(B, T // 16, 16, H, 2, K // 2)[:, :, 1:].sum(2).amin(-1)  # spread of each half over its sub-block
    wide = (rise < -40.0).view(B, T // 16, H, 2)
    assert ((wide[..., 0] == far.view(1, T // 16, 16, H, K)[:, :, 0, :, 0]) & (wide[..., 1] == far.view(1, T // 16, 16, H, K)[:, :, 0, :, -1])).float().mean() > 0.9
    tensors = (q, k, v, g, beta)
    R = signed_hadamard(K, 3) if rot else None
    qz, run = zc.calibrated(cell, tensors, eta=0.0, rot_qk=R)
    scales = qz.kernel_scales(0, H, K, V, delta=cell == "kda")
    out = zc.run_kernel(cell, tensors, scales, eta=0.0, rot=R, debug={} if staged else None)[0]
    zc.check(out, run, qz, f"{cell} K={K} rot={rot} staged={staged}")


# every way in which R_QK comes to the launch, below and from fp32's line (1024 chunks and heads) on: fp32 as it is, fp32 that is not on a
# 16-byte boundary, fp32 whose rows are not contiguous, fp16, fp64; a matrix without symmetry, so that a transposed operand shows
@pytest.mark.parametrize("cell", ["gla", "kda"])
@pytest.mark.parametrize("NT,H,K", [(31, 33, 64), (32, 32, 64), (33, 31, 128), (16, 64, 128)])
@pytest.mark.parametrize("form", ["fp32", "unaligned", "transposed", "fp16", "fp64"])
def test_every_form_of_the_local_rotation_equals_the_stages(cuda, cell, NT, H, K, form):
    from linquant_amd.kernels import zoo

    q, k, v, g, beta = [t if t is None else t.to(cuda) for t in zc.inputs(cell, B=1, T=64 * NT, H=H, K=K, V=64, seed=NT, dtype=torch.float16)]
    R = torch.linalg.qr(torch.randn(K, K, generator=torch.Generator().manual_seed(K), dtype=torch.float64))[0].contiguous().to(cuda)
    R = {"fp32": R.float(), "transposed": R.float().T, "fp16": R.half(), "fp64": R,
         "unaligned": torch.cat([torch.zeros(1, device=cuda), R.float().flatten()])[1:].view(K, K)}[form]
    assert R.is_contiguous() == (form != "transposed") and (form != "unaligned" or R.data_ptr() % 16 == 4)
    full = lambda x, *shape: torch.full(shape, x, device=cuda)  # noqa: E731
    sc = {"q": full(0.002, H), "k": full(0.008, H), "w": full(0.03, H), "kw": full(0.01, H, K)}
    sc.update({n: full(0.03, H, 64) for n in ("vw", "vl", "el", "ew", "state")})
    kw = dict(eta=0.25, output_final_state=True, rot=R)
    call = lambda **x: zoo.chunk_kda_int8(q, k, v, g, beta, sc, dqk=full(0.75, H, K), **kw, **x) if cell == "kda" else zoo.chunk_gla_int8(q, k, v, g, sc, **kw, **x)  # noqa: E731
    (o1, h1), (o0, h0) = call(), call(_staged=True)
    assert float(o1.float().abs().max()) > 0
    assert torch.equal(o0, o1) and torch.equal(h0, h1)


# what only callers of the C entry choose, below and from the lines of R_QK's operand launch (1024 chunks and heads fp32, 4096 fp16) on: fp16
# or fp32 R_QK, without room for its operands too, and KDA's D_QK with reciprocals of the caller's or without
@pytest.mark.parametrize("cell,tables", [("gla", None), ("kda", "dqk"), ("kda", "dq")])
@pytest.mark.parametrize("NT,H,K", [(31, 33, 64), (32, 32, 128), (63, 65, 64), (64, 64, 64)])
@pytest.mark.parametrize("rot", ["rot", "rot_f32"])
@pytest.mark.parametrize("room", [False, True])
def test_tables_of_the_c_entry_equal_the_wrapper(cuda, cell, tables, NT, H, K, rot, room):
    import ctypes

    from linquant_amd import _lib
    from linquant_amd.kernels import zoo

    T, V = 64 * NT, 64
    q, k, v, g, beta = [t if t is None else t.to(cuda) for t in zc.inputs(cell, B=1, T=T, H=H, K=K, V=V, seed=NT, dtype=torch.float16)]
    gen = torch.Generator().manual_seed(K)
    r = lambda *shape, lo, hi: (torch.rand(*shape, generator=gen) * (hi - lo) + lo).to(cuda)  # noqa: E731
    R = torch.linalg.qr(torch.randn(K, K, generator=gen))[0].contiguous().to(cuda)
    D = r(H, K, lo=0.25, hi=1.75)
    sc = {"q": r(H, lo=0.001, hi=0.003), "k": r(H, lo=0.005, hi=0.01), "w": r(H, lo=0.02, hi=0.04), "kw": r(H, K, lo=0.005, hi=0.015)}
    sc.update({n: r(H, V, lo=0.02, hi=0.05) for n in ("vw", "vl", "el", "ew", "state")})
    kda = cell == "kda"
    fn = (lambda **x: zoo.chunk_kda_int8(q, k, v, g, beta, sc, dqk=D, **x)) if kda else (lambda **x: zoo.chunk_gla_int8(q, k, v, g, sc, **x))
    o1, h1 = fn(eta=0.25, output_final_state=True, rot=R)

    dims = dict(family=int(kda), decay=2, batch=1, seqlen=T, nheads=H, kdim=K, vdim=V, chunk_size=64)
    n = ctypes.c_int64(0)
    st = _lib.fill("lq_zoo_chunk_forward_args", **dims)
    assert _lib.load().lq_zoo_chunk_forward_workspace_bytes(ctypes.byref(st), ctypes.byref(n)) == 0
    ws, ops = torch.empty(n.value, dtype=torch.uint8, device=cuda), torch.empty(2 * K * K, dtype=torch.uint8, device=cuda)
    o0, h0 = torch.zeros_like(v), torch.zeros(1, H, K, V, device=cuda)
    Rt, rcp = R if rot == "rot_f32" else R.half(), 1.0 / D
    extra = {rot: Rt.data_ptr()}
    if room:
        extra["rot_ws"] = ops.data_ptr()
    if kda:
        extra.update(beta=beta.data_ptr(), sw=sc["w"].data_ptr())
        extra.update({"dqk": D.data_ptr()} if tables == "dqk" else {"dq": D.data_ptr(), "dq_rcp": rcp.data_ptr()})
    p = lambda name: sc[name].data_ptr()  # noqa: E731
    _lib.call("lq_zoo_chunk_forward", q.device, q=q.data_ptr(), k=k.data_ptr(), v=v.data_ptr(), g=g.data_ptr(), o=o0.data_ptr(), ht=h0.data_ptr(),
              sq=p("q"), sk=p("k"), skw=p("kw"), svw=p("ew" if kda else "vw"), svl=p("el" if kda else "vl"), ss=p("state"), sigma=1.0, tau=1.0,
              eta=0.25, scale=K ** -0.5, qmax=127, act_dtype=_lib.LQ_DT_F16, workspace=ws.data_ptr(), workspace_bytes=n.value, **dims, **extra)
    assert float(o1.float().abs().max()) > 0
    assert torch.equal(o0, o1) and torch.equal(h0, h1)
