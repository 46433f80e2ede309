"""The 16-bit attention kernel at the edges of its items (64, 128 and 256 rows), tiles and
grids, for every kind of GQA group, against the oracle (fp32 on the same 16-bit inputs).

Tolerance: the bars every bf16 / fp16 attention output of this build is held to (max-abs
2e-2, mean-abs 1e-3): P is rounded to the 16-bit type before P.V and the output is stored in
it, 2^-9 of values below 4 each.
"""
import numpy as np
import pytest
import torch

from conftest import announce, oracle_arith
from oracle import delta_oracle as O
from oracle import select_oracle_c as OC

pytestmark = pytest.mark.gpu


def _close(out, want):
    err = np.abs(out.float().cpu().numpy() - want)
    assert err.max() <= 2e-2 and err.mean() <= 1e-3, (err.max(), err.mean())


@pytest.mark.parametrize("variant", ["hybrid", "sanity", "pure_phase1"])
@pytest.mark.parametrize("B,Hq,Hkv,N,D,W,chunk", [
    (1, 3, 3, 255, 64, 0, 64), (1, 2, 2, 257, 128, 64, 64), (1, 2, 1, 385, 128, 128, 100),
    (2, 6, 2, 640, 72, 0, 32), (1, 8, 1, 65, 128, 64, 512), (1, 12, 3, 193, 128, 0, 64),
    (1, 4, 4, 1400, 128, 128, 128), (1, 5, 1, 900, 8, 64, 128)])
def test_groups_and_row_edges(gpu, variant, B, Hq, Hkv, N, D, W, chunk):
    """One head over two logical blocks (their schedules differ), two heads over one, four
    over half of one; the last item partly or wholly past the rows."""
    from deltaattention_amd import ops, synth
    q, k, v = synth.make_layer_inputs(B, Hq, Hkv, N, D, seed=N + D)
    tau = 9.0 * (D / 128) ** 0.5
    announce(f"attn edges {variant} B={B} Hq={Hq} Hkv={Hkv} N={N} D={D} W={W}")
    out = ops.delta_prefill(q.to(gpu), k.to(gpu), v.to(gpu), tau, chunk, window=W, variant=variant)
    kf, vf = k.float().numpy(), v.float().numpy()
    keep, _ = OC.select_delta(kf, tau, chunk, arith=oracle_arith(k))
    p = O.pack(kf, vf, keep)
    _close(out, O.hybrid_attention(q.float().numpy(), kf, vf, p["k_packed"], p["v_packed"], p["timestamps"],
                                   p["counts"], W, variant=variant))


@pytest.mark.parametrize("Hq,Hkv,N,causal", [
    (1, 1, 1, True), (7, 7, 63, True), (2, 2, 256, False), (6, 3, 129, True), (32, 8, 1056, True),
    (16, 16, 513, True), (40, 8, 300, False), (64, 16, 600, True), (32, 8, 2048, False), (32, 8, 2080, False),
    (300, 300, 100, False)])
def test_dense_small_grids(gpu, Hq, Hkv, N, causal):
    """Grids of less than one, between one and two, and more workgroups than run at once; unmasked
    ones on both sides of one 64-row item a CU and with half an item past the rows."""
    from deltaattention_amd import ops, synth
    q, k, v = synth.make_layer_inputs(1, Hq, Hkv, N, 128, seed=N)
    announce(f"dense Hq={Hq} Hkv={Hkv} N={N} causal={causal}")
    out = ops.dense_prefill(q.to(gpu), k.to(gpu), v.to(gpu), causal=causal)
    _close(out, O.dense_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(), causal))


def test_pure_phase1_unsorted_timestamps(gpu):
    """Pure Phase 1 ends a row group's keys at the last packed block that holds a timestamp it
    sees: with the packed rows in a random order, and some of weight 0, that is the bound the
    suffix minima give, and the result the oracle's."""
    from deltaattention_amd import ops, synth
    N, P = 1000, 300
    q, k, v = synth.make_layer_inputs(1, 4, 2, N, 128, seed=3)
    rng = np.random.default_rng(0)
    ts = np.stack([1 + rng.permutation(N - 1)[:P] for _ in range(2)])[None].astype(np.int32)
    cnt = rng.integers(0, 4, size=ts.shape).astype(np.int32)
    ts[..., 5], cnt[..., 5] = 0, 2  # every row sees a key in the first block
    kp = torch.stack([k[0, h, torch.from_numpy(ts[0, h]).long()] for h in range(2)])[None].contiguous()
    vp = torch.stack([v[0, h, torch.from_numpy(ts[0, h]).long()] for h in range(2)])[None].contiguous()
    announce("pure phase 1, unsorted timestamps")
    out = ops.hybrid_prefill(q.to(gpu), k.to(gpu), v.to(gpu), kp.to(gpu), vp.to(gpu), torch.from_numpy(ts).to(gpu),
                             torch.from_numpy(cnt).to(gpu), window=64, variant="pure_phase1")
    _close(out, O.hybrid_attention(q.float().numpy(), k.float().numpy(), v.float().numpy(), kp.float().numpy(),
                                   vp.float().numpy(), ts, cnt, 64, variant="pure_phase1"))


@pytest.mark.parametrize("variant", ["hybrid", "sanity", "pure_phase1", "dense"])
@pytest.mark.parametrize("Hq,Hkv,N,D,W,dtype", [
    (3, 3, 255, 64, 0, torch.bfloat16), (2, 2, 385, 128, 64, torch.float16), (5, 1, 900, 8, 128, torch.bfloat16),
    (6, 3, 129, 128, 0, torch.bfloat16), (8, 1, 65, 128, 64, torch.float16), (12, 3, 193, 72, 64, torch.bfloat16),
    (8, 2, 1400, 128, 128, torch.bfloat16)])
def test_32_row_waves_match_64_row_ones(gpu, variant, Hq, Hkv, N, D, W, dtype):
    """A grid of at most two 64-row items a CU takes 32 rows a wave instead of 64.  Every row's
    sums are the same: a batch of copies beyond that line repeats the one sequence's output bit
    for bit."""
    from deltaattention_amd import ops, synth
    q, k, v = synth.make_layer_inputs(1, Hq, Hkv, N, D, seed=N, dtype=dtype, device=str(gpu))
    G = Hq // Hkv
    hpw = 4 if G % 4 == 0 else 2 if G % 2 == 0 else 1   # query heads a workgroup takes
    items = Hkv * (G // hpw) * -(-N // (256 // hpw))    # of one sequence, 64 rows a wave
    line = 2 * torch.cuda.get_device_properties(gpu).multi_processor_count
    copies = 1 + line // items
    assert items <= line < copies * items
    qb, kb, vb = (x.repeat(copies, 1, 1, 1) for x in (q, k, v))
    announce(f"32- and 64-row waves {variant} Hq={Hq} Hkv={Hkv} N={N} D={D} W={W} {dtype}")
    if variant == "dense":
        one, many = ops.dense_prefill(q, k, v), ops.dense_prefill(qb, kb, vb)
    else:
        tau = 9.0 * (D / 128) ** 0.5
        one, many = (ops.delta_prefill(x, y, z, tau, 100, window=W, variant=variant)
                     for x, y, z in ((q, k, v), (qb, kb, vb)))
    assert torch.equal(one.expand_as(many), many)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16], ids=["fp32", "bf16", "fp16"])
@pytest.mark.parametrize("variant", ["hybrid", "sanity", "pure_phase1"])
@pytest.mark.parametrize("Hq,Hkv,Nq,Nk,P,W", [(4, 2, 1024, 256, 70, 64), (8, 2, 900, 130, 33, 0), (3, 3, 700, 100, 1, 64)])
def test_more_queries_than_keys(gpu, variant, Hq, Hkv, Nq, Nk, P, W, dtype):
    """Query blocks with start_m - W > Nk + 1 take the partly filled last packed block: its
    rows past P weigh nothing and are not read (here they are NaN, in views of wider buffers).
    The oracle has them as zero rows of count 0 and timestamp Nk + 1, which is what the
    reference's masked loads give (deltaFlashAttention.py:70, 84-90)."""
    from deltaattention_amd import ops, synth
    D, room = 128, 256
    q = synth.make_layer_inputs(1, Hq, Hkv, Nq, D, seed=Nq, dtype=dtype)[0]
    _, k, v = synth.make_layer_inputs(1, Hq, Hkv, Nk, D, seed=Nk, dtype=dtype)
    at = torch.linspace(0, Nk - 1, P).long()
    ts = at.to(torch.int32).expand(1, Hkv, P)
    cnt = torch.randint(1, 5, (1, Hkv, P), generator=torch.Generator().manual_seed(P), dtype=torch.int32)

    def wide(x, fill):
        buf = torch.full((*x.shape[:2], room, *x.shape[3:]), fill, dtype=x.dtype, device=gpu)
        buf[:, :, :P] = x.to(gpu)
        return buf[:, :, :P]
    announce(f"more queries than keys {variant} Nq={Nq} Nk={Nk} P={P} W={W} {dtype}")
    out = ops.hybrid_prefill(q.to(gpu), k.to(gpu), v.to(gpu), wide(k[:, :, at], float("nan")),
                             wide(v[:, :, at], float("nan")), wide(ts, -1), wide(cnt, 1 << 20), window=W,
                             variant=variant).float().cpu().numpy()
    n = -(-P // 128) * 128 - P
    pad = lambda x, fill: np.pad(x, [(0, 0), (0, 0), (0, n)] + [(0, 0)] * (x.ndim - 3), constant_values=fill)
    kf, vf = k.float().numpy(), v.float().numpy()
    want = O.hybrid_attention(q.float().numpy(), kf, vf, pad(kf[:, :, at.numpy()], 0), pad(vf[:, :, at.numpy()], 0),
                              pad(ts.numpy(), Nk + 1), pad(cnt.numpy(), 0), W, variant=variant)
    # a block past every key of both phases has no weight at all: 0 / 0 in the reference
    some = np.isfinite(want)
    assert np.isfinite(out)[some].all()
    err = np.abs(out - want)[some]
    bars = (1e-5, 1e-6) if dtype == torch.float32 else (2e-2, 1e-3)
    assert err.max() <= bars[0] and err.mean() <= bars[1], (err.max(), err.mean())
