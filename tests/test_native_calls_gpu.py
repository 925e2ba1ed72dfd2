"""The wrappers' native short calls (csrc/binding.cpp) against their general path: the same bits for every form of a call that they
take, and the general path for every form that they do not."""

import pytest
import torch

from linquant_amd import _lib
from linquant_amd.calibration import Mamba2Shape
from linquant_amd.kernels import zoo
from linquant_amd.kernels.mamba2 import ssd_combined
from linquant_amd.kernels.mamba2.fused_split_rotate_xBC import fused_split_rotate_quant_xBC
from tests import zoo_cases as zc
from tests.mamba2_cases import build_case

pytestmark = pytest.mark.gpu


def _flat(out):
    for t in out if isinstance(out, (tuple, list)) else [out]:
        if isinstance(t, (tuple, list)):
            yield from _flat(t)
        else:
            yield t


def _both(monkeypatch, name, call, native=True):
    """The call as it is and without its native form; whether that served it."""
    served, fn = [], getattr(_lib.native(), name)
    monkeypatch.setattr(_lib.native(), name, lambda *a: served.append(fn(*a)) or served[-1])
    here = list(_flat(call()))
    monkeypatch.setattr(_lib.native(), name, lambda *a: None)
    there = list(_flat(call()))
    assert [r is not None for r in served] in ([[True]] if native else [[False], []])  # ([]: not offered at all)
    assert len(here) == len(there)
    for a, b in zip(here, there):
        assert (a is None) == (b is None)
        if a is not None:
            assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride() and a.device == b.device and torch.equal(a, b)


def _unaligned(t):
    return torch.cat([torch.zeros(1, dtype=t.dtype, device=t.device), t.flatten()])[1:].view(t.shape)


def _zoo(cuda, cell, dtype, B=2, T=128, H=3, K=64, V=128):
    q, k, v, g, beta = [t if t is None else t.to(cuda) for t in zc.inputs(cell, B=B, T=T, H=H, K=K, V=V, seed=1, dtype=dtype)]
    gen = torch.Generator().manual_seed(2)
    r = lambda *shape: (torch.rand(*shape, generator=gen) * 0.02 + 0.01).to(cuda)  # noqa: E731
    sc = {"q": r(H) / 8, "k": r(H) / 2, "w": r(H) * 2, "kw": r(H, K), **{n: r(H, V) for n in ("vw", "vl", "el", "ew", "state")}}
    return q, k, v, g, beta, sc


# what changes in the arguments -> whether the native form serves it
FORMS = {"plain": True, "final": True, "fp32 out": True, "numbers": True, "no bits": True, "q strided": False, "scales fp16": False,
         "scale unaligned": False, "scale tensor": False, "short chunk": False, "ragged width": False, "dispatch mode": False}


@pytest.mark.parametrize("cell", list(zc.CELLS))
@pytest.mark.parametrize("form", list(FORMS))
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_zoo_calls(cuda, monkeypatch, cell, form, dtype):
    fam, dec = zc.CELLS[cell]
    q, k, v, g, beta, sc = _zoo(cuda, cell, dtype, V=96 if form == "ragged width" else 128)
    kw = {"final": dict(output_final_state=True), "fp32 out": dict(out_dtype=torch.float32, output_final_state=True),
          "numbers": dict(eta=1, scale=0.07), "no bits": dict(bits=6), "scale tensor": dict(scale=torch.tensor(0.07)),
          "short chunk": dict(chunk_size=32)}.get(form, {})
    if form == "q strided":
        q = torch.cat([q, q], -1)[..., :64]
    if form == "scales fp16":
        sc["q"] = sc["q"].half()
    if form == "scale unaligned":
        sc["state"] = _unaligned(sc["state"])
    if dec == "diagonal":
        kw["rot"] = torch.linalg.qr(torch.randn(64, 64, generator=torch.Generator().manual_seed(3)))[0].contiguous().to(cuda)
    if cell == "kda":
        kw["dqk"] = sc["kw"] * 40
    if fam == "delta":
        kw.update(sigma=0.5, tau=0.25)
    if cell in ("linear_none", "mamba2"):
        name, call = "simple_gla", lambda: zoo.chunk_simple_gla_int8(q, k, v, g, sc, **kw)  # noqa: E731
    else:
        fn = {"gla": zoo.chunk_gla_int8, "kda": zoo.chunk_kda_int8}.get(cell, zoo.chunk_delta_int8)
        name, call = "chunk_forward", lambda: fn(q, k, v, g, *((beta,) if fam == "delta" else ()), sc, **kw)  # noqa: E731
    if form == "dispatch mode":
        from torch.utils._python_dispatch import TorchDispatchMode

        class Watch(TorchDispatchMode):
            def __torch_dispatch__(self, func, types, args=(), kwargs=None):
                return func(*args, **(kwargs or {}))

        inner = call

        def call():
            with Watch():
                return inner()
    _both(monkeypatch, name, call, FORMS[form])


@pytest.mark.parametrize("parts,native", [(("signs_qk",), True), (("signs_qk", "signs_v"), True), (("dqk",), False), ((), True), (("none",), True)])
def test_linear_prologue(cuda, monkeypatch, parts, native):
    q, k, v, g, _, sc = _zoo(cuda, "mamba2", torch.float16)
    signs = lambda n: torch.randint(0, 2, (n,), generator=torch.Generator().manual_seed(n)).float().to(cuda) * 2 - 1  # noqa: E731
    every = {"signs_qk": signs(64), "signs_v": signs(128), "dqk": sc["kw"] * 40, "none": None}
    pro = {"signs_qk" if n == "none" else n: every[n] for n in parts}
    _both(monkeypatch, "simple_gla", lambda: zoo.chunk_simple_gla_int8(q, k, v, g, sc, prologue=pro), native)


@pytest.mark.parametrize("form,native", [("qk", True), ("v", True), ("all", True), ("dqk", False), ("unaligned", False), ("out", None)])
def test_rotate_qkv(cuda, monkeypatch, form, native):
    q, k, v, *_ , sc = _zoo(cuda, "linear_none", torch.bfloat16)
    s = torch.ones(64, device=cuda)
    s[::3] = -1
    sv = torch.cat([s, -s])
    kw = dict(qk=dict(q=q, k=k, signs_qk=s), v=dict(v=v, signs_v=sv), all=dict(q=q, k=k, v=v, signs_qk=s, signs_v=sv),
              dqk=dict(q=q, k=k, signs_qk=s, dqk=sc["kw"] * 40), unaligned=dict(q=q, k=k, signs_qk=_unaligned(s)),
              out=dict(q=q, signs_qk=s, out=(torch.empty_like(q), None, None)))[form]
    if native is None or form == "dqk":  # never offered
        ref = zoo.rotate_qkv(**kw)
        monkeypatch.setattr(_lib.native(), "rotate_qkv", lambda *a: pytest.fail("offered"))
        assert all(a is b or torch.equal(a, b) for a, b in zip(ref, zoo.rotate_qkv(**kw)))
    else:
        _both(monkeypatch, "rotate_qkv", lambda: zoo.rotate_qkv(**kw), native)


@pytest.mark.parametrize("keyside", [True, False])
@pytest.mark.parametrize("form,native", [("plain", True), ("no bias", True), ("dt fp32", True), ("no D", True), ("D per channel", True),
                                         ("dt scale a number", False), ("scales fp16", False), ("x a view", True), ("ragged", True)])
def test_ssd_layer(cuda, monkeypatch, keyside, form, native):
    s = Mamba2Shape(batch=2, seqlen=256, nheads=4, headdim=64, dstate=128, ngroups=2, chunk=128)
    case = build_case(s)
    p, sc = ({n: t.to(cuda) for n, t in case[x].items()} for x in ("params", "scales"))
    xBC, dt = case["xBC"].to(cuda), case["dt_raw"].to(cuda)
    if form == "ragged":
        xBC, dt = xBC[:, :200], dt[:, :200]
    if form == "x a view":
        xBC = torch.cat([xBC, xBC], -1)[..., :xBC.shape[-1]]
    args = (xBC, p["r_signs"], s.nheads, s.ngroups, s.dstate, s.headdim, sc["B_inv_scale"], sc["C_inv_scale"])
    kw = dict(return_b_fp=True, return_b_rowmax=True) if keyside else {}
    _both(monkeypatch, "split_rotate", lambda: fused_split_rotate_quant_xBC(*args, **kw))
    x, qB, qC, *rest = fused_split_rotate_quant_xBC(*args, **kw)
    kw = dict(keyside=True, x_scale_hp=sc["x_scale_hp"], b_fp=rest[0], b_gate_scale=sc["b_gate_scale"], b_rowmax=rest[1]) if keyside else {}
    D, bias = p["D"], p["dt_bias"]
    if form == "no D":
        D = None
    if form == "D per channel":
        D = D[:, None].repeat(1, 64)
    if form == "dt fp32":
        dt = dt.float()
    a = [x, dt, 1.0 if form == "dt scale a number" else p["dt_scale"], p["A_log"], p["A_log_scale"], qB, sc["B_scale"], qC,
         sc["C_scale"].half() if form == "scales fp16" else sc["C_scale"], s.chunk, D, p["D_scale"]]
    call = lambda: ssd_combined._quant_mamba_chunk_scan_combined_fwd(  # noqa: E731
        *a, dt_bias=None if form == "no bias" else bias, dt_softplus=True, static_state_scale=sc["static_state_scale"],
        static_cb_scale=sc["static_cb_scale"], alpha_hp=sc["alpha_hp"], bscale_g=sc["bscale_g"], **kw)
    _both(monkeypatch, "ssd", call, native)


def test_a_failed_call_raises(cuda):
    q, k, v, g, _, sc = _zoo(cuda, "mamba2", torch.float16)
    q = _unaligned(q)  # dense, but not on a 16-byte boundary: refused by the library
    with pytest.raises(_lib.LinQuantHipError, match="lq_zoo_simple_gla failed with code -22"):
        zoo.chunk_simple_gla_int8(q, k, v, g, sc)
