"""GPU test of the order in which the launches in front of the recurrence take a call's (batch, chunk)s: wherever eight of them come
together (chunks of one sequence, of several, one of each of eight) or do not, a batched call gives each sequence what a call of its own
gives it, bit for bit; and no chunk is lost where the grid's last dimension does not hold them all."""

import pytest
import torch

from tests import zoo_cases as zc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cell", ["linear_none", "mamba2", "gla", "deltanet", "gated_deltanet", "kda"])
@pytest.mark.parametrize("B,NT,H", [(3, 8, 2), (2, 4, 3), (4, 6, 1), (8, 1, 3), (3, 3, 2), (2, 12, 2), (16, 3, 1)])
def test_a_batch_equals_its_sequences(cuda, cell, B, NT, H):
    from linquant_amd.kernels import zoo

    K = V = 64
    q, k, v, g, beta = (None if t is None else t.to(cuda) for t in zc.inputs(cell, B=B, T=64 * NT, H=H, K=K, V=V, seed=B, dtype=torch.float16))
    gen = torch.Generator().manual_seed(NT)
    r = lambda *shape, lo, hi: (torch.rand(*shape, generator=gen) * (hi - lo) + lo).to(cuda)  # noqa: E731
    sc = {"q": r(H, lo=0.001, hi=0.003), "k": r(H, lo=0.005, hi=0.01), "w": r(H, lo=0.02, hi=0.04), "kw": r(H, K, lo=0.005, hi=0.015),
          "vw": r(H, V, lo=0.02, hi=0.04), "vl": r(H, V, lo=0.02, hi=0.04), "el": r(H, V, lo=0.04, hi=0.06),
          "ew": r(H, V, lo=0.04, hi=0.06), "state": r(H, V, lo=0.02, hi=0.07)}

    def call(s):
        c = [None if t is None else t[s].contiguous() for t in (q, k, v, g, beta)]
        if cell in ("linear_none", "mamba2"):
            return zoo.chunk_simple_gla_int8(*c[:4], sc, output_final_state=True)
        if cell == "gla":
            return zoo.chunk_gla_int8(*c[:4], sc, output_final_state=True)
        return (zoo.chunk_kda_int8 if cell == "kda" else zoo.chunk_delta_int8)(*c, sc, output_final_state=True)

    o, ht = call(slice(None))
    for b in range(B):
        o1, h1 = call(slice(b, b + 1))
        assert torch.equal(o[b:b + 1], o1) and torch.equal(ht[b:b + 1], h1), b
    assert float(o.float().abs().amax(dim=(1, 2, 3)).min()) > 0


def test_more_chunks_than_the_grid_holds_in_one_dimension(cuda):
    from linquant_amd.kernels.zoo import _common

    H, K, NT = 2, 64, 32771  # (two folds of 32768 chunks, the second nearly empty)
    T = 64 * NT
    gen = torch.Generator(device=cuda).manual_seed(1)
    k = torch.nn.functional.normalize(torch.randn(1, T, H, K, generator=gen, device=cuda), dim=-1).half()
    v = torch.randn(1, T, H, K, generator=gen, device=cuda).half()
    beta = torch.rand(1, T, H, generator=gen, device=cuda)

    def prep(s):
        n = len(range(*s.indices(T)))
        return _common.run_wy_prep(k[:, s].contiguous(), v[:, s].contiguous(), beta[:, s].contiguous(), None, 0.5, 0.5,
                                   (1, n, H, K, K), _common.DECAY_NONE)

    whole = prep(slice(0, T))
    for s in (slice(0, 64 * 5), slice(64 * 32764, T)):
        for name, a, b in zip(("Hw", "W", "U", "fw"), whole, prep(s)):
            assert torch.equal(a[:, s], b), (name, s)


@pytest.mark.parametrize("cell", ["linear_none", "mamba2"])
@pytest.mark.parametrize("H,NT,prologue", [(31, 129, False), (32, 129, False), (9, 129, True), (10, 129, True), (10, 256, True), (10, 257, True),
                                           (10, 385, True), (13, 513, True), (14, 385, True), (16, 513, True), (22, 513, True)])
def test_long_chains_on_either_side_of_the_rule(cuda, cell, H, NT, prologue):
    """More than 128 chunk steps, K = V = 128: one launch or two by the numbers of workgroups and steps and the decay, the same bits as the stages."""
    from linquant_amd.kernels import zoo
    from linquant_amd.kernels.zoo.prologue import rotation_signs
    from oracle.zoo_reference import signed_hadamard

    K = V = 128
    q, k, v, g, _ = (None if t is None else t.to(cuda) for t in zc.inputs(cell, B=1, T=64 * NT, H=H, K=K, V=V, seed=H, dtype=torch.float16))
    gen = torch.Generator().manual_seed(H)
    r = lambda *shape, lo, hi: (torch.rand(*shape, generator=gen) * (hi - lo) + lo).to(cuda)  # noqa: E731
    sc = {"q": r(H, lo=0.001, hi=0.003), "k": r(H, lo=0.005, hi=0.01), "kw": r(H, K, lo=0.005, hi=0.015), "vw": r(H, V, lo=0.02, hi=0.04),
          "vl": r(H, V, lo=0.02, hi=0.04), "state": r(H, V, lo=0.02, hi=0.07)}
    kw = dict(output_final_state=True)
    if prologue:
        kw["prologue"] = dict(signs_qk=rotation_signs(signed_hadamard(K, 2)).to(cuda))
    o1, h1 = zoo.chunk_simple_gla_int8(q, k, v, g, sc, **kw)
    o0, h0 = zoo.chunk_simple_gla_int8(q, k, v, g, sc, _debug={}, **kw)
    assert torch.equal(o0, o1) and torch.equal(h0, h1) and float(o1.float().abs().max()) > 0
