"""GPU parity of vq_moe_rows (vq2_moe_rows: the pairs of one expert grouped
for the matrix cores) against fp64, and of the modules' choice between it and
the one-pair kernels: tiles of 32 and 64 pairs and their remainders, experts
with no, one and many pairs, a token that names an expert twice, short k tiles
and column blocks, both codebook types, ids outside the pool, a captured call.

Tolerance: the chain of a pair is ~40 fp32 roundings (two transforms of at most
11 stages, scales, silu, the weighted sum) around exact 24-bit products, each
at most 2^-24 of the values there: 5e-6 of max |out| bounds it (3e-7 to 4e-7
observed).  In the 2-norm it may not exceed the one-pair kernels' error by more
than the scatter of their difference."""
import numpy as np
import pytest
import torch

from compressai_amd import kernels as K, synth
from compressai_amd.moe import MoELayer, ResidentMoEExperts
from oracle import vq2_oracle as O

pytestmark = pytest.mark.gpu

TOL = 5e-6


def _pools(seed, E, H, I):
    gu = synth.indices16(seed, (E, 2 * I, H // 8))
    dn = synth.indices16(seed + 1, (E, H, I // 8))
    return gu, synth.scales(seed + 2, (E, 2 * I)), dn, synth.scales(seed + 3, (E, H))


def _tables(n, hb, seed, dev):
    perm, sign = synth.permutation(seed, n), synth.signs(seed + 1, n)
    return (perm.to(dev), sign.to(dev), hb, hb ** -0.5), perm.numpy(), sign.numpy()


def _reference(h, ids, w, gu, gus, dn, dns, cb, th, ti, hb_h, hb_i):
    h, w, ids = h.double().numpy(), w.double().numpy(), ids.numpy()
    I = dn.shape[2] * 8
    xr = np.stack([O.np_rht64(v, th[1], th[2], hb=hb_h)[0] for v in h])
    out = np.zeros((h.shape[0], dn.shape[1]))
    for e in range(gu.shape[0]):
        t, k = np.nonzero(ids == e)
        if not t.size:
            continue
        g = xr[t] @ O.np_dequant64(gu[e], None, cb, None, gus[e]).T
        act = g[:, :I] / (1.0 + np.exp(-g[:, :I])) * g[:, I:]
        ar = np.stack([O.np_rht64(v, ti[1], ti[2], hb=hb_i)[0] for v in act])
        y = ar @ O.np_dequant64(dn[e], None, cb, None, dns[e]).T
        np.add.at(out, t, w[t, k][:, None] * y)
    return out


# (T, P, E): pairs 96 of 3 experts (tiles of 64), 33 on one expert (32 + 1)
@pytest.mark.parametrize("T,P,E,H,I,hb_h,hb_i,h_dtype,cb_dtype,ids_dtype,out_dtype", [
    (1, 1, 1, 64, 64, 64, 64, torch.float32, torch.float16, torch.int32, torch.float32),
    (33, 1, 9, 320, 192, 64, 64, torch.float16, torch.bfloat16, torch.int64, torch.float32),
    (32, 3, 3, 2048, 512, 2048, 512, torch.bfloat16, torch.float16, torch.int32, torch.float32),
    (29, 9, 24, 2048, 512, 2048, 512, torch.float16, torch.bfloat16, torch.int64, torch.bfloat16),
    (5, 2, 300, 512, 1088, 256, 64, torch.float32, torch.float16, torch.int32, torch.float32),
])
def test_moe_rows_vs_fp64(dev, T, P, E, H, I, hb_h, hb_i, h_dtype, cb_dtype, ids_dtype, out_dtype):
    seed = 9800 + T
    gu, gus, dn, dns = _pools(seed, E, H, I)
    cb = synth.codebook(seed + 5, dtype=cb_dtype)
    # scales that keep the activation near 1
    gus, dns = (gus.float() * H ** -0.5).half(), (dns.float() * I ** -0.5).to(torch.bfloat16)
    th, ti = _tables(H, hb_h, seed + 6, dev), _tables(I, hb_i, seed + 8, dev)
    h = synth.activations(seed + 10, (T, H), dtype=h_dtype)
    g = synth.gen(seed + 11)
    ids = torch.randint(0, E, (T, P), generator=g).to(ids_dtype)
    if T == 33:
        ids[:] = 4  # one expert holds every pair
    w = torch.rand(T, P, generator=g)
    out = K.vq_moe_rows(h.to(dev), ids.to(dev), w.to(dev), gu.to(dev), gus.to(dev), dn.to(dev), dns.to(dev), cb.to(dev),
                        th[0], ti[0], out_dtype=out_dtype)
    ref = _reference(h, ids, w, gu, gus, dn, dns, cb, th, ti, hb_h, hb_i)
    eps = 2.0 ** -8 if out_dtype == torch.bfloat16 else 0.0
    err = np.abs(out.float().cpu().numpy() - ref)
    assert np.all(err <= TOL * np.abs(ref).max() + eps * np.abs(ref)), err.max() / np.abs(ref).max()


def test_ids_outside_the_pool_poison_their_token_alone(dev):
    E, T, P = 5, 40, 2
    gu, gus, dn, dns = _pools(9850, E, 512, 64)
    cb = synth.codebook(9855).to(dev)
    th, ti = _tables(512, 512, 9856, dev), _tables(64, 64, 9858, dev)
    args = [t.to(dev) for t in (gu, gus, dn, dns)]
    h = synth.activations(9860, (T, 512)).to(dev)
    ids = torch.randint(0, E, (T, P), generator=synth.gen(9861)).to(dev)
    w = torch.rand(T, P, generator=synth.gen(9862)).to(dev)
    call = lambda i: K.vq_moe_rows(h, i, w, *args[:2], *args[2:], cb, th[0], ti[0])
    good = call(ids)
    bad = ids.clone()
    bad[3, 1], bad[7, 0], bad[39, 1] = E, -1, 1 << 40
    out = call(bad)
    rows = torch.tensor([3, 7, 39], device=dev)
    assert bool(torch.isnan(out[rows]).all())
    keep = [t for t in range(T) if t not in (3, 7, 39)]
    assert torch.equal(out[keep], good[keep])


def test_more_pairs_than_the_sorting_workgroup_holds_in_registers(dev):
    """Above 5120 pairs (256 threads, 20 ids each) the pairs are sorted in
    several batches, their ids read again in the second pass: every token's
    result is the one that a call of few tokens gives, bit for bit (it depends
    on the token's own pairs alone), tokens with ids outside the pool NaN."""
    E, T, P, H, I = 9, 1811, 3, 512, 64  # 5433 pairs
    gu, gus, dn, dns = _pools(9910, E, H, I)
    args = [t.to(dev) for t in (gu, gus, dn, dns)]
    cb = synth.codebook(9915).to(dev)
    th, ti = _tables(H, H, 9916, dev), _tables(I, I, 9918, dev)
    h = synth.activations(9920, (T, H)).to(dev)
    ids = torch.randint(0, E, (T, P), generator=synth.gen(9921))
    ids[5, 1], ids[1700, 0], ids[1810, 2] = E, -1, E + 7
    ids, w = ids.to(dev), torch.rand(T, P, generator=synth.gen(9922)).to(dev)
    call = lambda t0, t1: K.vq_moe_rows(h[t0:t1], ids[t0:t1], w[t0:t1], *args, cb, th[0], ti[0])
    out = call(0, T)
    parts = torch.cat([call(t, min(T, t + 600)) for t in range(0, T, 600)])
    bad = torch.zeros(T, dtype=torch.bool, device=dev)
    bad[[5, 1700, 1810]] = True
    assert bool(torch.isnan(out[bad]).all()) and torch.equal(out[~bad], parts[~bad])


@pytest.mark.parametrize("cb_dtype", [torch.float16, torch.bfloat16])
def test_layer_takes_the_grouped_path_and_keeps_its_precision(dev, cb_dtype):
    """A layer with enough tokens: its result against 64 bits is no further
    off than the one-pair kernels' (2-norm, 2 % of scatter allowed), repeats
    and graph replays with new inputs are bit-identical, and without the
    reference pools the layer stays on the one-pair kernels."""
    E, k, T = 8, 4, 60
    gu, gus, dn, dns = _pools(9870, E + 1, 2048, 512)
    gus, dns = (gus.float() * 2048 ** -0.5).half(), (dns.float() * 512 ** -0.5).half()
    cb = synth.codebook(9875, dtype=cb_dtype)
    gate = synth.activations(9876, 2048) * 0.02
    layer = MoELayer(gu.to(dev), gus.to(dev), dn.to(dev), dns.to(dev), cb.to(dev), gate.to(dev), top_k=k)
    m = layer.experts_mod
    assert K.moe_rows_faster(T * (k + 1), E + 1, 2048, 512) and not K.moe_rows_faster(2 * (k + 1), E + 1, 2048, 512)
    h = synth.activations(9877, (T, 2048)).to(dev)
    lg = synth.activations(9878, (T, E), dtype=torch.float32).to(dev)
    out = layer(h, lg)
    ids, w = layer.route(h, lg)
    assert torch.equal(out, m._rows(h, ids, w)) and torch.equal(out, m.experts(h, ids, w))
    assert torch.equal(out, layer(h, lg))
    th, ti = ((None, r.perm.cpu().numpy(), r.sign.float().cpu().numpy()) for r in (m.rot_h, m.rot_i))
    ref = _reference(h.cpu(), ids.cpu(), w.cpu(), gu, gus, dn, dns, cb, th, ti, 2048, 512)
    static_h, static_l = h.clone(), lg.clone()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        gout = layer(static_h, static_l)
    for i in range(4):
        static_h.copy_(h if i % 2 else h.flip(0))
        static_l.copy_(lg if i % 2 else lg.flip(0))
        g.replay()
        eager = layer(static_h, static_l)
        torch.cuda.synchronize()
        assert torch.equal(gout, eager), i
    m.release_reference_pools()
    one = layer(h, lg)
    norm = lambda a: np.linalg.norm(a.double().cpu().numpy() - ref) / np.linalg.norm(ref)
    assert norm(out) <= 1.02 * norm(one), (norm(out), norm(one))


def test_layer_with_a_top_k_above_the_router_entrys_runs_for_any_token_count(dev):
    """Forty experts a token: more than vq_router_topk selects, so a chunk
    that would be grouped stays on the one-pair kernels and its router, and
    gives each token what a call of few tokens gives it."""
    E, k, T = 64, 40, 40
    gu, gus, dn, dns = _pools(9890, E + 1, 512, 64)
    layer = MoELayer(gu.to(dev), (gus.float() * 512 ** -0.5).half().to(dev), dn.to(dev),
                     (dns.float() * 64 ** -0.5).half().to(dev), synth.codebook(9895).to(dev),
                     synth.activations(9896, 512).to(dev) * 0.02, top_k=k)
    assert K.moe_rows_faster(T * (k + 1), E + 1, 512, 64)
    h = synth.activations(9897, (T, 512)).to(dev)
    lg = synth.activations(9898, (T, E), dtype=torch.float32).to(dev)
    out = layer(h, lg)
    few = torch.cat([layer(h[t:t + 4], lg[t:t + 4]) for t in range(0, T, 4)])
    assert float((out - few).abs().max()) <= TOL * float(few.abs().max())


@pytest.mark.parametrize("sign", [1, -1])
def test_a_product_past_fp32_is_infinite_as_in_the_one_pair_kernels(dev, sign):
    """Every centroid value 1e15 (bf16 codebooks reach that far): the gate_up
    sums are 1e13, their activation rotates to one value of ~8e26 and zeros,
    and the down product leaves fp32.  The result is infinite, not NaN."""
    E, H, I, P = 3, 64, 64, 2
    T = 20
    gu, dn = synth.indices16(9901, (E, 2 * I, H // 8)), synth.indices16(9902, (E, H, I // 8))
    gus, dns = torch.full((E, 2 * I), 1e-2 / 8), torch.ones(E, H)
    cb = torch.full((65536, 8), 1e15, dtype=torch.bfloat16)
    mod = ResidentMoEExperts.from_pools(gu.to(dev), gus.to(dev), dn.to(dev), dns.to(dev), cb.to(dev), sorted_layout=True)
    rot = (None, None, 64, 0.125)
    h = torch.ones(T, H, device=dev)
    ids = torch.randint(0, E, (T, P), generator=synth.gen(9903)).to(dev)
    w = torch.full((T, P), 0.5 * sign, device=dev)
    one = K.vq_sorted_moe(h, mod.sorted_gu, mod.gate_up_scale, mod.sorted_dn, mod.down_scale, mod.cb16, rot, rot,
                          ids=ids, w=w)
    assert bool((one == sign * float("inf")).all())
    out = K.vq_moe_rows(h, ids, w, mod.gate_up_idx, mod.gate_up_scale, mod.down_idx, mod.down_scale, mod.cb16, rot, rot)
    assert torch.equal(out, one)
