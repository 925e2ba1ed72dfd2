"""The work that a user of this package has it do, as cases that can be timed and compared.

Three paths, all prefill (there is no decode and no backward pass here), each through the calls a user's program makes:
  zoo     one layer of a zoo cell: the operand rotation where the cell rotates q and k up front, then the chunk forward
          (``linquant_amd.kernels.zoo``)
  ssd     one Mamba-2 SSD layer: split / rotate / quantize of B and C, then the combined INT8 forward
          (``linquant_amd.kernels.mamba2``)
  mixer   the native stages of a whole Mamba-2 mixer around the user's own two projections: activation quantizer,
          conv1d + SiLU, the SSD as above, gated norm + Hadamard + INT8

Sizes are the repository's benchmark and test configurations, the batch and length grids its reference is timed on
(batch 1 to 32, length 256 to 8192 and above) and odd neighbours of both.  Activations are drawn as the benchmark draws
them (``linquant_amd.calibration``), on the GPU; static scales come from a separate calibration batch, as a user's do.
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as Fn

from linquant_amd import hadamard_utils
from linquant_amd.calibration import Mamba2Shape, calibrate_mamba2, dqk_from_absmax
from linquant_amd.kernels import zoo
from linquant_amd.kernels.mamba2.causal_conv1d import causal_conv1d_fn
from linquant_amd.kernels.mamba2.fused_split_rotate_xBC import fused_split_rotate_quant_xBC
from linquant_amd.kernels.mamba2.ssd_combined import _quant_mamba_chunk_scan_combined_fwd
from linquant_amd.norm import rmsnorm_gated_qhad
from linquant_amd.w4a8_linear import _fused_fp16_to_int8

CELLS = {"linear": ("linear", "none"), "mamba2": ("linear", "scalar"), "gla": ("linear", "diagonal"),
         "deltanet": ("delta", "none"), "gdn": ("delta", "scalar"), "kda": ("delta", "diagonal")}
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def _zoo(cell, B, T, H, K, V, *, dtype="fp16", rotate=True, final=False, sigma=1.0, dqk=False, name=None):
    c = dict(path="zoo", cell=cell, B=B, T=T, H=H, K=K, V=V, dtype=dtype, rotate=rotate, final=final, sigma=sigma, dqk=dqk)
    return c if name is None else dict(c, name=name)


def _ssd(B, L, H, *, G=1, N=128, Q=256, keyside=True, decay="strong", path="ssd", name=None):
    c = dict(path=path, B=B, L=L, H=H, P=64, G=G, N=N, Q=Q, keyside=keyside, decay=decay)
    return c if name is None else dict(c, name=name)


def listed():
    return [
        # the smallest calls: one short sequence, where launches, host work and the chain of chunk steps count
        _zoo("mamba2", 1, 2048, 8, 64, 64, rotate=False, name="mamba2_cell_b1"),
        _ssd(1, 512, 80, name="ssd_b1_l512"),                       # a short prompt through a 2.7B-shape layer
        _zoo("kda", 1, 2048, 8, 128, 128, dtype="bf16", final=True, name="kda_b1"),  # one prompt, state kept for decoding
        # ordinary prefills of every recurrence
        _zoo("linear", 4, 4096, 16, 128, 128, name="linear_attention_b4"),
        _zoo("gla", 4, 4096, 16, 128, 128, name="gla_b4"),
        _zoo("deltanet", 8, 2048, 8, 128, 128, dtype="bf16", rotate=False, name="deltanet_b8"),
        _zoo("gdn", 4, 4096, 16, 128, 128, sigma=0.5, final=True, name="gdn_b4"),
        _ssd(8, 2048, 64, keyside=False, name="ssd_value_side_b8"),  # 1.3B-shape layer, value-side scale absorption
        _ssd(3, 5000, 80, decay="weak", name="ssd_weak_ragged_b3"),  # slowly forgetting layer, length off the chunk grid
        _ssd(4, 2048, 80, decay="weak", path="mixer", name="mixer_b4"),  # everything between the two projections
        # the largest: long context
        _zoo("kda", 2, 8192, 32, 128, 128, dqk=True, name="kda_b2_t8192"),
        _ssd(4, 8192, 80, name="ssd_b4_l8192"),                     # the shape the metric is quoted on
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """Another case of the same ranges: any cell, batch, length (in whole chunks for the zoo), head count, width, dtype."""
    path = rng.choice(["zoo", "zoo", "zoo", "ssd", "ssd", "mixer"])
    if path == "zoo":
        cell = rng.choice(list(CELLS))
        H = rng.choice([4, 5, 8, 12, 16, 24, 32])
        most = 2 * 8192 * 32 // H if cell == "kda" else 4 * 8192 * 16 // H
        tokens = _log(rng, 2048, most)
        B = rng.choice([b for b in (1, 2, 3, 4, 8) if b * 1024 <= tokens])
        T = 64 * max(1, round(tokens / B / 64))
        K = V = 128
        if rng.random() < 0.25:
            K, V = rng.choice([(64, 64), (64, 128), (128, 64)])
        return _zoo(cell, B, T, H, K, V, dtype=rng.choice(["fp16", "bf16"]), rotate=rng.random() < 0.6, final=rng.random() < 0.5,
                    sigma=rng.choice([0.5, 1.0]), dqk=cell == "kda" and rng.random() < 0.5)
    H = rng.choice([24, 48, 64, 80])
    tokens = _log(rng, 256, 4 * 8192 if path == "ssd" else 4 * 2048)
    B = rng.choice([b for b in (1, 2, 3, 4, 8, 16) if b * 256 <= tokens])
    L = max(256, int(tokens / B))
    if rng.random() < 0.5:
        L -= L % 256
    return _ssd(B, L, H, G=rng.choice([1, 1, 1, 8]), N=rng.choice([128, 128, 64]), Q=rng.choice([256, 256, 128]),
                keyside=rng.random() < 0.7, decay=rng.choice(["strong", "weak"]), path=path)


# ------------------------------------------------------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed % (1 << 62))


def _signs(n, seed):
    g = _generator(seed)
    return torch.randint(0, 2, (n,), generator=g, device="cuda").float() * 2 - 1


def _hadamard(n, signs):
    H = torch.ones(1, 1, device="cuda")
    while H.shape[0] < n:
        H = torch.cat([torch.cat([H, H], 1), torch.cat([H, -H], 1)], 0)
    return H / math.sqrt(n) * signs


def _zoo_inputs(c, B, seed):
    """q, k, v, g, beta of ``linquant_amd.calibration.zoo_synthetic``'s distributions, drawn on the GPU."""
    fam, dec = CELLS[c["cell"]]
    T, H, K, V, dt = c["T"], c["H"], c["K"], c["V"], DTYPES[c["dtype"]]
    gen = _generator(seed)
    rn = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")  # noqa: E731
    q, k = rn(B, T, H, K).to(dt), rn(B, T, H, K)
    k = (Fn.normalize(k, dim=-1) if fam == "delta" else k).to(dt)
    v = rn(B, T, H, V).to(dt)
    beta = torch.sigmoid(rn(B, T, H)) if fam == "delta" else None
    g = None
    if c["cell"] == "gla":
        g = Fn.logsigmoid(rn(B, T, H, K)) / 16
    elif c["cell"] == "kda":
        g = Fn.logsigmoid(rn(B, T, H, K) + 1.0)
    elif c["cell"] == "gdn":
        g = Fn.logsigmoid(rn(B, T, H) + 2.0)
    elif c["cell"] == "mamba2":
        g = -Fn.softplus(rn(B, T, H) * 0.5 - 2.0) * torch.exp(torch.rand(H, generator=gen, device="cuda") * 2.77)
    return q, k, v, g, beta


def _prepare_zoo(c, seed):
    fam, dec = CELLS[c["cell"]]
    H, K, V = c["H"], c["K"], c["V"]
    q, k, v, g, beta = _zoo_inputs(c, c["B"], seed)
    s = dict(cell=c["cell"], q=q, k=k, v=v, g=g, beta=beta, sigma=c["sigma"], final=c["final"], eta=0.0 if dec == "diagonal" else 1.0,
             scale=K ** -0.5, signs=None, rot=None, dqk=None)
    if c["rotate"]:  # local R_QK inside the kernels under per-channel decay, persistent R_QK up front otherwise
        signs = _signs(K, 17)
        s["rot" if dec == "diagonal" else "signs"] = _hadamard(K, signs) if dec == "diagonal" else signs
    # static scales: absmax of a calibration batch, the recurrence's own roles from a pilot run over it
    cal = dict(s)
    cal.update(zip(("q", "k", "v", "g", "beta"), _zoo_inputs(c, 1, 1234567)))
    if c["dqk"]:
        s["dqk"] = cal["dqk"] = dqk_from_absmax(cal["q"].float(), cal["k"].float(), 0.5)
    cq, ck, _ = zoo.rotate_qkv(cal["q"], cal["k"], None, signs_qk=s["signs"], dqk=s["dqk"])
    ph = lambda t: (t.float().abs().amax(dim=(0, 1, 3)) / 127).clamp_min(1e-6)  # noqa: E731
    pc = lambda t: (t.float().abs().amax(dim=(0, 1)) / 127).clamp_min(1e-6)  # noqa: E731
    vs = pc(cal["v"])
    sc = {"q": ph(cq) * s["scale"], "k": ph(ck), "w": ph(ck) * 2, "kw": pc(ck), "vw": vs, "vl": vs.clone(), "el": vs * 2, "ew": vs * 2,
          "state": torch.ones(H, V, device="cuda")}
    seen = {}
    cal.update(scales=sc, final=True)
    _, ht = _run_zoo(cal, _debug=seen)
    sc["state"] = (ht.abs().amax(dim=(0, 2)) / 127 * 1.5).clamp_min(1e-6)
    if fam == "delta":
        sc["el"] = pc(seen["e_out"])
        sc["ew"], sc["w"] = sc["el"].clone(), ph(seen["W"])
    s["scales"] = {n: t.contiguous() for n, t in sc.items()}
    return s


def _mamba2_inputs(c, B, L, seed):
    gen = _generator(seed)
    rn = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")  # noqa: E731
    xBC = rn(B, L, c["H"] * c["P"] + 2 * c["G"] * c["N"]).half()
    dt = (rn(B, L, c["H"]) * 0.5 + (-2.0 if c["decay"] == "strong" else -4.5)).half()
    return xBC, dt


def _prepare_ssd(c, seed):
    H, G, N, Q = c["H"], c["G"], c["N"], c["Q"]
    gen = _generator(42)
    rand = lambda *shape: torch.rand(*shape, generator=gen, device="cuda")  # noqa: E731
    a_log = rand(H) * math.log(16.0 if c["decay"] == "strong" else 1.3)
    D = torch.randn(H, generator=gen, device="cuda")
    a_scale, d_scale = (a_log.abs().amax() / 127.0).clamp_min(1e-8), (D.abs().amax() / 127.0).clamp_min(1e-8)
    p = dict(A_log=torch.round(a_log / a_scale).clamp(-127, 127).to(torch.int8), A_log_scale=a_scale,
             D=torch.round(D / d_scale).clamp(-127, 127).to(torch.int8), D_scale=d_scale,
             dt_bias=torch.zeros(H, device="cuda"), dt_scale=torch.ones((), device="cuda"), r_signs=_signs(G * N, 43).view(G, N))
    cal = Mamba2Shape(batch=1, seqlen=2048, nheads=H, headdim=c["P"], dstate=N, ngroups=G, chunk=Q)
    s = dict(c, p=p)
    if c["path"] == "ssd":
        s["xBC"], s["dt"] = _mamba2_inputs(c, c["B"], c["L"], seed)
        cx, cdt = _mamba2_inputs(c, 1, 2048, 7654321)
        s["sc"] = calibrate_mamba2(cal, cx, cdt, p)
        return s
    # the mixer: hidden states, the output of the user's in_proj ([z | xBC | dt]), conv and norm weights
    d_ssm, gn = H * c["P"], G * N
    conv_dim = d_ssm + 2 * gn
    gen = _generator(seed)
    rn = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")  # noqa: E731
    s["hidden"] = rn(c["B"], c["L"], d_ssm // 2).half()
    s["proj"] = rn(c["B"], c["L"], d_ssm + conv_dim + H).half()
    s["proj"][..., -H:] = s["proj"][..., -H:] * 0.5 + (-2.0 if c["decay"] == "strong" else -4.5)
    gen = _generator(44)
    s["conv_w"], s["conv_b"] = (rn(conv_dim, 4) * 0.5).half(), (rn(conv_dim) * 0.1).half()
    s["norm_w"] = (1 + 0.1 * rn(d_ssm)).half()
    s["in_scale"], s["out_scale"] = torch.tensor(4.0 / 127, device="cuda"), 4.0 / 127
    small = hadamard_utils.small_order(d_ssm)
    if small != 1 and small not in hadamard_utils._SMALL:
        hadamard_utils.register_hadamard(small, hadamard_utils.hadamard_matrix(small))
    cx = causal_conv1d_fn(rn(1, 2048, conv_dim).half().transpose(1, 2), s["conv_w"], s["conv_b"], activation="silu").transpose(1, 2)
    s["sc"] = calibrate_mamba2(cal, cx, _mamba2_inputs(c, 1, 2048, 7654321)[1], p)
    return s


def prepare(case, seed):
    return _prepare_zoo(case, seed) if case["path"] == "zoo" else _prepare_ssd(case, seed)


# -------------------------------------------------------------------------------------------------------------- calls
def _run_zoo(s, **kw):
    cell, q, k, v, g, sc = s["cell"], s["q"], s["k"], s["v"], s["g"], s["scales"]
    kw.update(eta=s["eta"], scale=s["scale"], output_final_state=s["final"])
    if cell in ("linear", "mamba2"):
        return zoo.chunk_simple_gla_int8(q, k, v, g, sc, prologue=None if s["signs"] is None else dict(signs_qk=s["signs"]), **kw)
    if cell == "gla":
        return zoo.chunk_gla_int8(q, k, v, g, sc, rot=s["rot"], **kw)
    if cell == "kda":
        return zoo.chunk_kda_int8(q, k, v, g, s["beta"], sc, sigma=s["sigma"], rot=s["rot"], dqk=s["dqk"], **kw)
    if s["signs"] is not None:
        q, k, _ = zoo.rotate_qkv(q, k, None, signs_qk=s["signs"])
    return zoo.chunk_delta_int8(q, k, v, g, s["beta"], sc, sigma=s["sigma"], **kw)


def _run_ssd(s, xBC, dt):
    p, sc, kw = s["p"], s["sc"], {}
    args = (xBC, p["r_signs"], s["H"], s["G"], s["N"], s["P"], sc["B_inv_scale"], sc["C_inv_scale"])
    if s["keyside"]:
        x, qB, qC, b_fp, b_rowmax = fused_split_rotate_quant_xBC(*args, return_b_fp=True, return_b_rowmax=True)
        kw = dict(keyside=True, x_scale_hp=sc["x_scale_hp"], b_fp=b_fp, b_gate_scale=sc["b_gate_scale"], b_rowmax=b_rowmax)
    else:
        x, qB, qC = fused_split_rotate_quant_xBC(*args)
    return _quant_mamba_chunk_scan_combined_fwd(
        x, dt, p["dt_scale"], p["A_log"], p["A_log_scale"], qB, sc["B_scale"], qC, sc["C_scale"], s["Q"], p["D"], p["D_scale"],
        dt_bias=p["dt_bias"], dt_softplus=True, static_state_scale=sc["static_state_scale"], static_cb_scale=sc["static_cb_scale"],
        alpha_hp=sc["alpha_hp"], bscale_g=sc["bscale_g"], **kw)[0]


def _run_mixer(s):
    hidden, d_ssm = s["hidden"], s["H"] * s["P"]
    h_i8 = _fused_fp16_to_int8(hidden.view(-1, hidden.shape[-1]), s["in_scale"], clamp_min=-128.0, reciprocal=False)
    z, xBC, dt = s["proj"].split([d_ssm, d_ssm + 2 * s["G"] * s["N"], s["H"]], dim=-1)
    xBC = causal_conv1d_fn(xBC.transpose(1, 2), s["conv_w"], s["conv_b"], activation="silu").transpose(1, 2)
    y = _run_ssd(s, xBC, dt)
    y = y.view(y.shape[0], y.shape[1], d_ssm)
    y_i8, _ = rmsnorm_gated_qhad(y, z, s["norm_w"], s["out_scale"], 1e-5, d_ssm // s["G"])
    return {"h_i8": h_i8, "y": y, "y_i8": y_i8}


def run(state):
    """ONE layer's forward over inputs resident in HBM."""
    if "cell" in state:
        return [t for t in _run_zoo(state) if t is not None]
    return _run_mixer(state) if state["path"] == "mixer" else _run_ssd(state, state["xBC"], state["dt"])


# --------------------------------------------------------------------------------------------------------------- work
def work(case):
    """Every input read once, every output written once; the chunked recurrence's multiply-adds (two operations each):
    per token and head the chunk-local products (half of the C x C squares) and the state write and read."""
    if case["path"] == "zoo":
        fam, dec = CELLS[case["cell"]]
        B, T, H, K, V, C = case["B"], case["T"], case["H"], case["K"], case["V"], 64
        n = B * T * H
        nbytes = n * 2 * (2 * K + 2 * V) + (n * 4 if fam == "delta" else 0)
        nbytes += {"none": 0, "scalar": n * 4, "diagonal": n * K * 4}[dec] + (B * H * K * V * 4 if case["final"] else 0)
        macs = n * (C / 2 * (K + V) + 2 * K * V)
        if fam == "delta":  # the Gram matrix, T.k and T.v, the state read of W
            macs += n * (C / 2 * (2 * K + V) + K * V)
        return {"bytes": nbytes, "flops": 2 * macs}
    B, L, H, P, G, N, Q = (case[k] for k in ("B", "L", "H", "P", "G", "N", "Q"))
    n = B * L
    x, bc = n * H * P, n * G * N
    flops = 2 * (Q / 2 * (bc + x) + 2 * x * N)
    if case["path"] == "ssd":
        return {"bytes": 2 * (x + 2 * bc) + 2 * n * H + 2 * x, "flops": flops}
    # hidden (d_ssm / 2) in and its codes out, z, xBC, dt in, y and its INT8 codes out; the Hadamard factors are adds
    return {"bytes": 3 * x // 2 + 2 * (2 * x + 2 * bc + n * H) + 3 * x, "flops": flops + 2 * 4 * (x + 2 * bc)}


def tolerance(case):
    """Four times what the kernels measure against the float64 oracle of the same quantized recurrence.  Operands and states are
    INT8 codes: where a 32-bit sum lies within its own noise of a rounding boundary two correct implementations pick
    neighbouring codes, so single outputs differ by a code step (``max``) while the norm of the difference stays small.
    Without decay the delta rule never forgets such a step (measured 3e-3 in fp16, 9e-3 in bf16 over 4096 tokens); the other
    cells measure up to 1.2e-4 in fp16 and 9e-4 in bf16, the SSD 2.2e-4 in fp16 with 1.9e-3 of the mixer's INT8 outputs on
    the other side of a tie."""
    if case["path"] == "zoo":
        bf16 = case["dtype"] == "bf16"
        if case["cell"] == "deltanet":
            return {"rel": 0.03 if bf16 else 0.014, "max": 0.4}
        return {"rel": 4e-3 if bf16 else 5e-4, "max": 0.12}
    return {"rel": 9e-4, "max": 0.012, "differ": 0.008}
