"""GPU test of the launch that runs the cumulative sum and C.B^T side by side (mamba2_cumsum_bmm.hip): the one-call forward equals the
stages one after the other bit for bit at the edges of its dispatch: every chunk size that the other stages take, units that
do and do not divide over the 8 XCDs, either with one tile to a workgroup and with several and a partial last workgroup, a ragged last
chunk, heads off the 16-head tile, groups, and a d_state it leaves to two launches."""

import pytest
import torch

from linquant_amd.calibration import Mamba2Shape
from tests.mamba2_cases import build_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("keyside", [True, False])
@pytest.mark.parametrize("B,L,H,G,N,Q", [
    (1, 64, 1, 1, 64, 64), (2, 1000, 6, 2, 128, 128), (8, 256, 16, 1, 128, 256), (3, 700, 17, 1, 64, 256), (2, 1024, 4, 1, 128, 512),
    (4, 2560, 32, 4, 64, 256), (8, 4096, 80, 1, 128, 256), (3, 5000, 80, 1, 128, 256), (1, 6300, 80, 2, 64, 256), (1, 300, 4, 1, 256, 256)])
def test_one_call_equals_the_stages(cuda, B, L, H, G, N, Q, keyside):
    from linquant_amd.kernels.hadamard import kronecker_hadamard_fwd
    from linquant_amd.kernels.mamba2 import ssd_combined as M

    s = Mamba2Shape(batch=B, seqlen=-(-L // Q) * Q, nheads=H, headdim=64, dstate=N, ngroups=G, chunk=Q)
    case = build_case(s, device=cuda)
    p, sc, gn = case["params"], case["scales"], G * N
    xBC, dt = case["xBC"][:, :L].contiguous(), case["dt_raw"][:, :L].contiguous()
    x = xBC[..., :s.d_ssm].view(B, L, H, 64)
    gen = torch.Generator(device="cuda").manual_seed(L)
    qB, qC = (torch.randint(-127, 128, (B, L, G, N), generator=gen, device="cuda", dtype=torch.int8) for _ in range(2))
    b_fp = kronecker_hadamard_fwd(xBC[..., s.d_ssm:s.d_ssm + gn].view(B, L, G, N), p["r_signs"], G)

    def run():
        return M._quant_mamba_chunk_scan_combined_fwd(
            x, dt, p["dt_scale"], p["A_log"], p["A_log_scale"], qB, sc["B_scale"], qC, sc["C_scale"], Q, p["D"],
            p["D_scale"], dt_bias=p["dt_bias"], dt_softplus=True, static_state_scale=sc["static_state_scale"],
            static_cb_scale=sc["static_cb_scale"], alpha_hp=sc["alpha_hp"], bscale_g=sc["bscale_g"], keyside=keyside,
            x_scale_hp=sc["x_scale_hp"], b_fp=b_fp, b_gate_scale=sc["b_gate_scale"])[0]

    one = run()
    orig = M._quant_bmm_chunk_fwd
    M._quant_bmm_chunk_fwd = lambda *a, **k: orig(*a, **k)  # a re-bound stage: the stages one after the other
    try:
        staged = run()
    finally:
        M._quant_bmm_chunk_fwd = orig
    torch.cuda.synchronize()
    assert torch.equal(one, staged) and float(one.float().abs().max()) > 0
