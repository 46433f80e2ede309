"""The fp32 attention kernel at the edges of its tiles (32 queries, 32 keys, 32 dims) and in
both orders of its workgroups: long and short row blocks paired on a grid of at most two
workgroups a CU, the longest first on larger ones (each case asserts its side), against a 64-bit
torch reference.

The tolerance: a score is a sum of D fp32 products, off by about sqrt(D) 2^-24 of
sum |q k| scale (below 8 for these inputs, so 5e-6 at worst, a tenth of it in the mean); the
output moves by that times the spread of V (about 1) and adds its own sum over the keys,
weighted by probabilities: 1e-5 at worst and 1e-6 in the mean bound both.
"""
import numpy as np
import pytest
import torch

from conftest import announce
from oracle import delta_oracle as O
from oracle import select_oracle_c as OC

pytestmark = pytest.mark.gpu

MAX_TOL, MEAN_TOL = 1e-5, 1e-6


def _close(err):
    assert err.max() <= MAX_TOL and err.mean() <= MEAN_TOL, (float(err.max()), float(err.mean()))


def _paired(gpu, B, Hq, N):
    """The launch's rule: at most two workgroups (32 rows of one head) a CU."""
    return B * Hq * -(-N // 32) <= 2 * torch.cuda.get_device_properties(gpu).multi_processor_count


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


@pytest.mark.parametrize("B,Hq,Hkv,N,D,causal,paired", [
    (1, 2, 1, 1, 64, True, True), (1, 2, 2, 31, 8, True, True), (2, 3, 1, 33, 32, True, True),
    (1, 4, 4, 257, 40, True, True), (1, 6, 3, 130, 96, False, True), (1, 2, 1, 200, 104, True, True),
    (1, 8, 2, 300, 128, False, True), (2, 40, 8, 225, 128, True, False), (1, 64, 64, 289, 64, True, False),
    (1, 72, 8, 250, 24, False, False)])
def test_dense_fp32_edges(gpu, B, Hq, Hkv, N, D, causal, paired):
    from deltaattention_amd import ops
    assert _paired(gpu, B, Hq, N) == paired
    gen = torch.Generator().manual_seed(N * D)
    q, k, v = (torch.randn((B, h, N, D), generator=gen) for h in (Hq, Hkv, Hkv))
    announce(f"fp32 dense B={B} Hq={Hq} N={N} D={D} causal={causal}")
    out = ops.dense_prefill(q.to(gpu), k.to(gpu), v.to(gpu), causal=causal).cpu()
    _close((out.double() - _dense64(q, k, v, causal)).abs())


@pytest.mark.parametrize("variant", ["hybrid", "sanity", "pure_phase1"])
@pytest.mark.parametrize("Hq,Hkv,N,D,paired", [(2, 2, 97, 64, True), (4, 2, 515, 40, True), (3, 1, 700, 96, True),
                                               (40, 8, 641, 128, False)])
def test_delta_fp32_edges(gpu, variant, Hq, Hkv, N, D, paired):
    from deltaattention_amd import ops, synth
    assert _paired(gpu, 1, Hq, N) == paired
    q, k, v = synth.make_layer_inputs(1, Hq, Hkv, N, D, seed=N, rope_base=10000.0, dtype=torch.float32)
    tau = 9.0 * (D / 128) ** 0.5
    announce(f"fp32 {variant} Hq={Hq} N={N} D={D}")
    out = ops.delta_prefill(q.to(gpu), k.to(gpu), v.to(gpu), tau, 128, window=64, variant=variant).cpu().numpy()
    qn, kn, vn = q.numpy(), k.numpy(), v.numpy()
    keep, _ = OC.select_delta(kn, tau, 128, arith="fp32")
    p = O.pack(kn, vn, keep)
    want = O.hybrid_attention(qn, kn, vn, p["k_packed"], p["v_packed"], p["timestamps"], p["counts"], 64,
                              variant=variant)
    _close(np.abs(out - want))
