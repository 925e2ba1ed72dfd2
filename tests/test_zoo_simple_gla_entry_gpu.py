"""GPU test of lq_zoo_simple_gla's contract through the C entry: which calls with an operand prologue are accepted does not depend on
the route that their size takes (one launch for recurrence and output, or one after the other)."""

import ctypes

import pytest
import torch

from linquant_amd import _lib
from tests import zoo_cases as zc

pytestmark = pytest.mark.gpu


def _call(q, k, v, g, sc, ht, unaligned=(), **prologue):
    """(return code, o) of the C entry; the tables named in ``unaligned`` start 4 bytes behind a 16-byte boundary."""
    B, T, H, K = q.shape
    V = v.shape[-1]
    keep = []

    def ptr(name, t):
        if t is None:
            return None
        if name in unaligned:
            room = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
            room[1:] = t.reshape(-1)
            t = room[1:]
            assert t.data_ptr() % 16 == 4
        keep.append(t)
        return t.data_ptr()

    o = torch.zeros_like(v)
    st = _lib.fill("lq_zoo_simple_gla_args", q=q.data_ptr(), k=k.data_ptr(), v=v.data_ptr(), g=ptr("g", g), o=o.data_ptr(),
                   ht=ht.data_ptr(), sq=ptr("sq", sc["q"]), sk=ptr("sk", sc["k"]), skw=ptr("skw", sc["kw"]), svw=ptr("svw", sc["vw"]),
                   svl=ptr("svl", sc["vl"]), ss=ptr("ss", sc["state"]), eta=0.75, scale=K ** -0.5, qmax=127, batch=B, seqlen=T,
                   nheads=H, kdim=K, vdim=V, chunk_size=64, act_dtype=_lib.LQ_DT_F16, **{n: ptr(n, t) for n, t in prologue.items()})
    n = ctypes.c_int64(0)
    lib = _lib.load()
    assert lib.lq_zoo_simple_gla_workspace_bytes(ctypes.byref(st), ctypes.byref(n)) == 0
    ws = torch.empty(n.value, dtype=torch.uint8, device=q.device)
    st.workspace, st.workspace_bytes = ws.data_ptr(), n.value
    rc = lib.lq_zoo_simple_gla(ctypes.byref(st), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return rc, o


@pytest.mark.parametrize("cell", ["linear_none", "mamba2"])
# a short chain, and a few long ones
@pytest.mark.parametrize("NT", [2, 136])
@pytest.mark.parametrize("K,V,parts,unaligned", [(64, 192, ("signs_qk",), ()), (128, 64, ("signs_qk", "dqk"), ("dq", "dq_rcp")),
                                                 (64, 64, ("signs_v",), ("skw", "svw"))])
def test_a_prologue_is_accepted_on_either_route(cuda, cell, NT, K, V, parts, unaligned):
    from linquant_amd.kernels import zoo

    B, H = 1, 2
    q, k, v, g, _ = [t.to(cuda) if t is not None else None for t in zc.inputs(cell, B=B, T=64 * NT, H=H, K=K, V=V, seed=NT)]
    gen = torch.Generator().manual_seed(NT)
    r = lambda *shape, lo, hi: (torch.rand(*shape, generator=gen) * (hi - lo) + lo).to(cuda)  # noqa: E731
    sc = {"q": r(H, lo=0.001, hi=0.003), "k": r(H, lo=0.005, hi=0.03), "kw": r(H, K, lo=0.005, hi=0.03), "vw": r(H, V, lo=0.02, hi=0.04),
          "vl": r(H, V, lo=0.02, hi=0.04), "state": r(H, V, lo=0.02, hi=0.07)}
    every = {"signs_qk": r(K, lo=-1, hi=1).sign(), "signs_v": r(V, lo=-1, hi=1).sign(), "dqk": r(H, K, lo=0.5, hi=2.0)}
    ref, href = zoo.chunk_simple_gla_int8(q, k, v, g, sc, eta=0.75, output_final_state=True, prologue={n: every[n] for n in parts}, _staged=True)
    fields = {n: every[n] for n in parts if n != "dqk"}
    if "dqk" in parts:
        fields.update(dq=every["dqk"], dq_rcp=1.0 / every["dqk"])
    ht = torch.zeros(B, H, K, V, device=cuda)
    rc, o = _call(q, k, v, g, sc, ht, unaligned, **fields)
    assert rc == 0
    assert torch.equal(o, ref) and torch.equal(ht, href) and float(o.float().abs().max()) > 0
    # signs_v needs V in {64, 128}, on either route
    if V == 192:
        rc, o = _call(q, k, v, g, sc, ht, signs_v=every["signs_v"])
        assert rc == -22 and float(o.abs().max()) == 0
