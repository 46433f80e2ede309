"""The fp32 attention kernels at the edges of their tiles (32 queries, 32 keys, 32 dims) and
on both sides of the rule that picks four or eight waves a workgroup, against a 64-bit
torch reference.

The tolerance: a score is a sum of D fp32 products, off by about sqrt(D) 2^-24 of
sum |q k| scale (below 8 for these inputs, so 5e-6); the output moves by that times the
spread of V (about 1) and adds its own sum over the keys, weighted by probabilities: 2e-5
bounds both.
"""
import numpy as np
import pytest
import torch

from conftest import announce
from oracle import delta_oracle as O
from oracle import select_oracle_c as OC

pytestmark = pytest.mark.gpu

TOL = 2e-5


def _dense64(q, k, v, causal):
    g = q.shape[1] // k.shape[1]
    k, v = k.double().repeat_interleave(g, 1), v.double().repeat_interleave(g, 1)
    out = torch.empty(q.shape, dtype=torch.float64)
    for b in range(q.shape[0]):
        for h in range(q.shape[1]):
            s = q[b, h].double() @ k[b, h].t() * q.shape[-1] ** -0.5
            if causal:
                s = s.masked_fill(torch.ones_like(s, dtype=torch.bool).triu(1), -float("inf"))
            out[b, h] = torch.softmax(s, -1) @ v[b, h]
    return out


@pytest.mark.parametrize("B,Hq,Hkv,N,D,causal", [
    (1, 2, 1, 1, 64, True), (1, 2, 2, 31, 8, True), (2, 3, 1, 33, 32, True), (1, 4, 4, 257, 40, True),
    (1, 6, 3, 130, 96, False), (1, 2, 1, 200, 104, True), (1, 8, 2, 300, 128, False), (2, 40, 8, 225, 128, True),
    (1, 64, 64, 289, 64, True), (1, 72, 8, 250, 24, False)])
def test_dense_fp32_edges(gpu, B, Hq, Hkv, N, D, causal):
    from deltaattention_amd import ops
    gen = torch.Generator().manual_seed(N * D)
    q, k, v = (torch.randn((B, h, N, D), generator=gen) for h in (Hq, Hkv, Hkv))
    announce(f"fp32 dense B={B} Hq={Hq} N={N} D={D} causal={causal}")
    out = ops.dense_prefill(q.to(gpu), k.to(gpu), v.to(gpu), causal=causal).cpu()
    err = (out.double() - _dense64(q, k, v, causal)).abs().max()
    assert err <= TOL, err


@pytest.mark.parametrize("variant", ["hybrid", "sanity", "pure_phase1"])
@pytest.mark.parametrize("Hq,Hkv,N,D", [(2, 2, 97, 64), (4, 2, 515, 40), (3, 1, 700, 96), (40, 8, 641, 128)])
def test_delta_fp32_edges(gpu, variant, Hq, Hkv, N, D):
    from deltaattention_amd import ops, synth
    q, k, v = synth.make_layer_inputs(1, Hq, Hkv, N, D, seed=N, rope_base=10000.0, dtype=torch.float32)
    tau = 9.0 * (D / 128) ** 0.5
    announce(f"fp32 {variant} Hq={Hq} N={N} D={D}")
    out = ops.delta_prefill(q.to(gpu), k.to(gpu), v.to(gpu), tau, 128, window=64, variant=variant).cpu().numpy()
    qn, kn, vn = q.numpy(), k.numpy(), v.numpy()
    keep, _ = OC.select_delta(kn, tau, 128, arith="fp32")
    p = O.pack(kn, vn, keep)
    want = O.hybrid_attention(qn, kn, vn, p["k_packed"], p["v_packed"], p["timestamps"], p["counts"], 64,
                              variant=variant)
    assert np.abs(out - want).max() <= TOL, np.abs(out - want).max()
