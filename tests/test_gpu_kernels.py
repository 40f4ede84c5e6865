"""GPU parity tests: every kernel through the C ABI against the CPU oracle on the same seeded inputs.

Bars: bit-exact for packing, router indices, histogram / permutation (and for the RoPE / KV writes,
whose rounding is per element); bf16 outputs within max-abs-rel 2e-2 and cosine >= 0.999."""
import numpy as np
import pytest
import torch

from flyai_amd import kvlayout

from oracle import attention as oattn
from oracle import experts as oexperts
from oracle import layer as olayer
from oracle import packing as opack
from oracle import routing as oroute
from oracle.numerics import bf16

pytestmark = pytest.mark.gpu

MAR, COS = 2e-2, 0.999
DEV = "cuda"


def _metrics(a, b):
    from gpu_harness import metrics
    return metrics(a, b)


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


# ---- a1 ----------------------------------------------------------------------------------------

@pytest.mark.parametrize("q_lens,starts", [([1, 1, 3, 7], [0, 5, 9, 100]),
                                           ([1] * 24 + [4] * 8, list(range(512, 512 + 32 * 200, 200))),
                                           ([2048] + [1] * 48, [4096] + list(range(600, 648)))])
def test_pack_ragged_bit_exact(q_lens, starts):
    from flyai_amd import ops
    S = len(q_lens)
    base = [s * 1000 * 64 for s in range(S)]
    cap = [8192] * S
    t = lambda v, dt: torch.tensor(v, dtype=dt, device=DEV)
    out = ops.pack_ragged(t(q_lens, torch.int32), t(starts, torch.int32), t(base, torch.int64),
                          t(cap, torch.int32), 64, 4096)
    ref = opack.pack_ragged(q_lens, starts, kv_base=base, kv_cap=cap, head_dim=64)
    T = sum(q_lens)
    assert out["status"].item() == 0
    assert out["cu_seqlens"].cpu().numpy().tolist() == ref["cu_seqlens"].tolist()
    assert out["positions"][:T].cpu().numpy().tolist() == ref["positions"].tolist()
    assert out["seq_id"][:T].cpu().numpy().tolist() == ref["seq_id"].tolist()
    assert out["kv_slot"][:T].cpu().numpy().tolist() == ref["kv_slot"].tolist()
    assert out["kv_len"].cpu().numpy().tolist() == ref["kv_len"].tolist()


def test_pack_ragged_overflow_status():
    from flyai_amd import ops
    t = lambda v, dt: torch.tensor(v, dtype=dt, device=DEV)
    out = ops.pack_ragged(t([8, 8], torch.int32), t([92, 93], torch.int32), t([0, 0], torch.int64),
                          t([100, 100], torch.int32), 64, 64)
    assert out["status"].item() & 1
    slots = out["kv_slot"][:16].cpu().numpy()
    assert (slots[:8] >= 0).all() and slots[15] == -1      # only the out-of-capacity token is blanked


# ---- a2 / a3 / a4 ------------------------------------------------------------------------------

def _rms_input(T, H, seed):
    x = torch.randn(T, H, device=DEV, generator=_gen(seed))
    x = x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-5)
    return x.to(torch.bfloat16)


# (300, *, *, *) and (2096, ...) take the prefill-sized logits kernel, whose 1-D grid runs a token group's
# expert groups back to back on one XCD and exits the token groups past T (300 = 37.5 groups of 8)
@pytest.mark.parametrize("T,E,k,H", [(56, 128, 4, 2880), (12, 128, 4, 2880), (300, 32, 4, 256), (5, 8, 2, 128),
                                     (300, 128, 4, 2880), (2096, 128, 4, 2880)])
def test_router_indices_bit_exact(T, E, k, H):
    from flyai_amd import ops
    x = _rms_input(T, H, 1)
    w = (torch.randn(E, H, device=DEV, generator=_gen(2)) * 0.02).to(torch.bfloat16)
    b = (torch.randn(E, device=DEV, generator=_gen(3)) * 0.02).to(torch.bfloat16)
    ids, wts, logits = ops.router_topk_softmax(x, w, b, k, want_logits=True)
    rids, rw, rlog = oroute.gptoss_route(x.float().cpu(), w.float().cpu(), b.float().cpu(), k)
    assert torch.equal(logits.cpu(), rlog), "router logits differ from the fixed-order oracle"
    assert np.array_equal(ids.cpu().numpy(), rids)
    np.testing.assert_allclose(wts.cpu().numpy(), rw, rtol=2e-6, atol=1e-7)


def test_router_exact_ties_go_to_lower_id():
    from flyai_amd import ops
    T, E, H = 16, 64, 128
    x = _rms_input(T, H, 4)
    base = (torch.randn(8, H, device=DEV, generator=_gen(5)) * 0.05).to(torch.bfloat16)
    w = base.repeat(8, 1).contiguous()                      # experts e and e+8 are identical rows
    b = torch.zeros(E, dtype=torch.bfloat16, device=DEV)
    ids, _ = ops.router_topk_softmax(x, w, b, 4)
    rids, _, _ = oroute.gptoss_route(x.float().cpu(), w.float().cpu(), b.float().cpu(), 4)
    assert np.array_equal(ids.cpu().numpy(), rids)
    # the winning row has 8 identical copies (r, r+8, ..., r+56): top-4 must be its 4 lowest ids
    got = ids.cpu().numpy()
    r = got[:, :1] % 8
    assert (got == r + np.arange(4)[None, :] * 8).all()


@pytest.mark.parametrize("T,E,H", [(56, 128, 2880), (12, 128, 2880), (1024, 128, 2880), (1025, 128, 2880),
                                   (33, 256, 7168)])
def test_fused_route_permute_bit_exact(T, E, H):
    """The stage's fused path (one-workgroup top-k + permute for T*k <= 4096, split above)."""
    from flyai_amd import ops
    k = 4 if E == 128 else 8
    x = _rms_input(T, H, 12)
    w = (torch.randn(E, H, device=DEV, generator=_gen(13)) * 0.02).to(torch.bfloat16)
    b = (torch.randn(E, device=DEV, generator=_gen(14)) * 0.02).to(torch.bfloat16)
    ids, wts, hist, off, perm, inv = ops.moe_route_permute(x, w, b, k)
    rids, rw, _ = oroute.gptoss_route(x.float().cpu(), w.float().cpu(), b.float().cpu(), k)
    rh, ro, rp, ri = oroute.permute(rids, E)
    assert np.array_equal(ids.cpu().numpy(), rids)
    np.testing.assert_allclose(wts.cpu().numpy(), rw, rtol=2e-6, atol=1e-7)
    for got, ref in ((hist, rh), (off, ro), (perm, rp), (inv, ri)):
        assert np.array_equal(got.cpu().numpy(), ref)


@pytest.mark.parametrize("T,E,k", [(20, 128, 4), (56, 128, 8), (7, 64, 2)])
def test_fused_route_permute_ties_go_to_lower_id(T, E, k):
    """Zero router weights leave logits = bias; a bias with many equal values makes ties inside a
    lane's quarter and across the four lanes that share a token.  Bit-exact ids and weights."""
    from flyai_amd import ops
    x = _rms_input(T, 2880, 15)
    w = torch.zeros(E, 2880, device=DEV, dtype=torch.bfloat16)
    b = torch.tensor([((e * 7) % 5) * 0.125 for e in range(E)], device=DEV).to(torch.bfloat16)
    ids, wts, hist, off, perm, inv = ops.moe_route_permute(x, w, b, k)
    rids, rw, _ = oroute.gptoss_route(x.float().cpu(), w.float().cpu(), b.float().cpu(), k)
    assert np.array_equal(ids.cpu().numpy(), rids)
    np.testing.assert_allclose(wts.cpu().numpy(), rw, rtol=2e-6, atol=1e-7)
    rh, ro, rp, ri = oroute.permute(rids, E)
    for got, ref in ((hist, rh), (off, ro), (perm, rp), (inv, ri)):
        assert np.array_equal(got.cpu().numpy(), ref)


@pytest.mark.parametrize("T,k,E,mode", [(1, 4, 128, "rand"), (56, 4, 128, "rand"), (2096, 4, 128, "rand"),
                                        (4096, 4, 256, "skew"), (64, 4, 8, "one"), (16384, 4, 128, "rand")])
def test_permute_bit_exact(T, k, E, mode):
    from flyai_amd import ops
    rng = np.random.default_rng(T + E)
    if mode == "one":
        ids = np.tile(np.arange(k), (T, 1))
    elif mode == "skew":
        hot = rng.choice(E, E // 10, replace=False)
        ids = np.stack([np.sort(rng.choice(hot, k, replace=False)) if rng.random() < 0.5
                        else np.sort(rng.choice(E, k, replace=False)) for _ in range(T)])
    else:
        ids = np.sort(np.stack([rng.choice(E, k, replace=False) for _ in range(T)]), axis=1)
    ids_d = torch.tensor(ids, dtype=torch.int32, device=DEV)
    hist, off, perm, inv = ops.moe_permute(ids_d, E)
    rh, ro, rp, ri = oroute.permute(ids, E)
    assert np.array_equal(hist.cpu().numpy(), rh)
    assert np.array_equal(off.cpu().numpy(), ro)
    assert np.array_equal(perm.cpu().numpy(), rp)
    assert np.array_equal(inv.cpu().numpy(), ri)


@pytest.mark.parametrize("P,E", [(1, 1), (63, 3), (1023, 128), (1024, 256), (1025, 255), (4097, 64), (8384, 7),
                                 (65536, 256)])
def test_permute_blocks_bit_exact(P, E):
    """The permute's blocks of 1,024 assignments: one short, full, one over, many; ids outside [0, E) count as
    expert 0 in the counts of a block and in the counts before it."""
    from flyai_amd import ops
    rng = np.random.default_rng(P + E)
    ids = rng.integers(-1, E + 1, size=(P, 1)).astype(np.int32)
    got = ops.moe_permute(torch.tensor(ids, device=DEV), E)
    ref = oroute.permute(np.where((ids >= 0) & (ids < E), ids, 0), E)
    for g, r in zip(got, ref):
        assert np.array_equal(g.cpu().numpy(), r)


@pytest.mark.parametrize("P,first", [(1024, 1024), (2048, 1024), (3000, 1), (5000, 0), (5000, 4999)])
def test_permute_counts_before_and_after_a_block_bit_exact(P, first):
    """Long runs of one expert: a block's counts of the ids before it and of the rest are kept apart and added."""
    from flyai_amd import ops
    ids = np.where(np.arange(P) < first, 200, 7).astype(np.int32)[:, None]
    got = ops.moe_permute(torch.tensor(ids, device=DEV), 256)
    for g, r in zip(got, oroute.permute(ids, 256)):
        assert np.array_equal(g.cpu().numpy(), r)


# the last batch of the one-workgroup kernel and the first of the two launches, per E and selection kernel
@pytest.mark.parametrize("T,E,k", [(62, 128, 4), (63, 128, 4), (31, 256, 8), (32, 256, 8), (64, 4, 2), (65, 4, 4),
                                   (64, 120, 4), (70, 120, 8), (64, 16, 8), (300, 112, 2)])
def test_route_selection_order_bit_exact(T, E, k):
    """Logits of every kind the selection's integer order has to rank: both signs, zeros, ties, subnormals, the
    largest magnitudes and -infinity (zero weights: the bias is the logit)."""
    from flyai_amd import ops
    x = _rms_input(T, 256, 16)
    w = torch.zeros(E, 256, device=DEV, dtype=torch.bfloat16)
    kinds = torch.tensor([-1.5, 0.0, 2.0**-130, -2.0**-130, 0.75, -3.38e38, float("-inf"), 0.75, -0.25, 1e-3, 1.0])
    b = kinds[torch.randperm(E, generator=torch.Generator().manual_seed(E)) % len(kinds)].to(torch.bfloat16)
    w[:, 0] = torch.linspace(-2, 2, E).to(torch.bfloat16).to(DEV) * (torch.arange(E, device=DEV) % 3 == 0)
    ids, wts, *perm = ops.moe_route_permute(x, w, b.to(DEV), k)
    rids, rw, _ = oroute.gptoss_route(x.float().cpu(), w.float().cpu(), b.float(), k)
    assert np.array_equal(ids.cpu().numpy(), rids)
    np.testing.assert_allclose(wts.cpu().numpy(), rw, rtol=2e-6, atol=1e-7)
    for g, r in zip(perm, oroute.permute(rids, E)):
        assert np.array_equal(g.cpu().numpy(), r)


def test_nan_router_rows_route_consistently():
    """A router row of NaN (a NaN hidden state) must not break the routing's index invariants: the
    expert and combine kernels index with perm, inv and offsets.  The top-k gives such a row
    in-range ids, and the permute counts any id outside [0, E) as expert 0, so the histogram sums to
    T*k and perm / inv stay a permutation and its inverse."""
    from flyai_amd import ops
    T, H, E, k = 40, 2880, 128, 4
    g = _gen(140)
    x = torch.randn(T, H, device=DEV, generator=g).to(torch.bfloat16)
    x[3] = float("nan")
    x[17, 5] = float("nan")
    rw = (0.02 * torch.randn(E, H, device=DEV, generator=g)).to(torch.bfloat16)
    rb = torch.zeros(E, device=DEV, dtype=torch.bfloat16)
    ids, wts = ops.router_topk_softmax(x, rw, rb, k)
    ids_h = ids.cpu().numpy()
    assert ((ids_h >= 0) & (ids_h < E)).all(), "router ids out of range on a NaN row"
    # ids outside [0, E) straight into the permute: counted as expert 0
    bad = ids_h.copy()
    bad[0] = [-1, E, 2**31 - 1, 7]
    hist, off, perm, inv = ops.moe_permute(torch.tensor(bad, dtype=torch.int32, device=DEV), E)
    want = np.where((bad >= 0) & (bad < E), bad, 0)
    rh, ro, rp, ri = oroute.permute(want, E)
    assert np.array_equal(hist.cpu().numpy(), rh) and np.array_equal(off.cpu().numpy(), ro)
    assert np.array_equal(perm.cpu().numpy(), rp) and np.array_equal(inv.cpu().numpy(), ri)


def test_combine_matches_oracle():
    from flyai_amd import ops
    T, k, H = 56, 4, 2880
    rng = np.random.default_rng(9)
    y = torch.randn(T * k, H, device=DEV, generator=_gen(9)) * 5
    inv = torch.tensor(rng.permutation(T * k), dtype=torch.int32, device=DEV)
    w = torch.softmax(torch.randn(T, k, device=DEV, generator=_gen(10)), -1)
    res = torch.randn(T, H, device=DEV, generator=_gen(11)).to(torch.bfloat16)
    out = ops.moe_combine(y, inv, w, residual=res.clone())
    ref = oroute.combine(y.cpu(), inv.cpu().numpy(), w.cpu(), residual=res.float().cpu())
    mar, cos = _metrics(out.float().cpu().numpy(), ref.numpy())
    assert mar < 1e-2 and cos > 0.99999


# ---- a5 / a6 -----------------------------------------------------------------------------------

@pytest.mark.parametrize("T,E,hot", [(12, 128, None), (128, 8, None), (3, 4, None), (320, 4, None), (600, 16, 5)])
def test_moe_experts_vs_oracle(T, E, hot):
    """gate_up (+SwiGLU) and down through the packed MXFP4 layout.  (12, 128) and (3, 4) are
    decode-sized (row-pass kernel); (128, 8) averages 64 rows per expert (dense kernel, one pass);
    (320, 4) puts all 320 tokens on every expert (dense kernel, four passes of up to 96 rows, each its
    own work unit); (600, 16, hot 5) biases the router to one expert, which then holds nearly every
    token (seven passes) beside groups of about 120 rows."""
    from flyai_amd import ops
    from flyai_amd.weights import GptOssShape, synthetic_moe
    shape = GptOssShape(n_experts=E)
    m = synthetic_moe(shape, _gen(20 + E), DEV)
    w13 = ops.mxfp4_repack(m["w13_blocks"], m["w13_scales"])
    w2 = ops.mxfp4_repack(m["w2_blocks"], m["w2_scales"])
    x = _rms_input(T, shape.hidden, 21)
    rw = (torch.randn(E, shape.hidden, device=DEV, generator=_gen(22)) * 0.02).to(torch.bfloat16)
    rb = torch.zeros(E, dtype=torch.bfloat16, device=DEV)
    if hot is not None:
        rb[hot] = 4.0
    ids, wts = ops.router_topk_softmax(x, rw, rb, 4)
    hist, off, perm, inv = ops.moe_permute(ids, E)
    if hot is not None:
        hc = hist.cpu().numpy()
        assert hc[hot] > 5 * 96, hc
    h = ops.moe_gate_up(x, perm, off, 4, w13, m["b13"], E, shape.intermediate)
    y = ops.moe_down(h, off, w2, m["b2"], E, shape.hidden)
    torch.cuda.synchronize()
    wts_o = oexperts.MxExpertWeights(*(m[n].cpu().numpy() for n in
                                       ("w13_blocks", "w13_scales", "b13", "w2_blocks", "w2_scales", "b2")))
    ry, rh = oexperts.experts_mxfp4(x.float().cpu(), perm.cpu().numpy(), off.cpu().numpy(), 4, wts_o,
                                    return_h=True)
    mar, cos = _metrics(h.float().cpu().numpy(), rh.numpy())
    assert mar <= MAR and cos >= COS, f"gate_up+swiglu: {mar:.3g} {cos:.6f}"
    mar, cos = _metrics(y.cpu().numpy(), ry.numpy())
    assert mar <= MAR and cos >= COS, f"down: {mar:.3g} {cos:.6f}"


# ---- a9 ----------------------------------------------------------------------------------------

def test_rmsnorm_and_linear_vs_oracle():
    from flyai_amd import ops
    T, H, N = 56, 2880, 5120
    x = torch.randn(T, H, device=DEV, generator=_gen(30)).to(torch.bfloat16) * 3
    w = (1 + 0.1 * torch.randn(H, device=DEV, generator=_gen(31))).float()
    y = ops.rmsnorm(x, w)
    ref = olayer.rmsnorm(x.float().cpu(), w.cpu())
    mar, cos = _metrics(y.float().cpu().numpy(), ref.numpy())
    assert mar < 1e-2 and cos > 0.9999
    W = (torch.randn(N, H, device=DEV, generator=_gen(32)) * 0.02).to(torch.bfloat16)
    b = (torch.randn(N, device=DEV, generator=_gen(33)) * 0.02).to(torch.bfloat16)
    out = ops.linear(y, W, b)
    ref = olayer.linear(y.float().cpu(), W.float().cpu(), b.float().cpu())
    mar, cos = _metrics(out.float().cpu().numpy(), ref.numpy())
    assert mar < 1e-2 and cos > 0.9999
    Wo = (torch.randn(H, 4096, device=DEV, generator=_gen(34)) * 0.02).to(torch.bfloat16)
    a = torch.randn(T, 4096, device=DEV, generator=_gen(35)).to(torch.bfloat16)
    res = x.clone()
    ops.linear(a, Wo, None, residual=res)
    ref = bf16(x.float().cpu() + olayer.linear(a.float().cpu(), Wo.float().cpu()))
    mar, cos = _metrics(res.float().cpu().numpy(), ref.numpy())
    assert mar < 1e-2 and cos > 0.9999


@pytest.mark.parametrize("M", [2, 16, 17, 48, 64, 65, 80, 128, 129, 255, 256])
@pytest.mark.parametrize("N,K,off", [(16, 32, 0), (144, 544, 1), (272, 2880, 0), (64, 8192, 3)])
def test_linear_rows_do_not_depend_on_the_batch(M, N, K, off):
    """Row tiles and passes of the projections: every row of a batch equals that row alone bit for bit, with
    and without bias and residual, for N past the last whole workgroup, K of partial groups and slices, tensors
    that start `off` elements past a 16-byte boundary, and an infinity and a NaN in the first and last rows."""
    from flyai_amd import ops

    def at(t):
        buf = torch.empty(t.numel() + off, dtype=t.dtype, device=DEV)
        buf[off:] = t.reshape(-1)
        return buf[off:].view(t.shape)

    x = torch.randn(M, K, device=DEV, generator=_gen(71)).to(torch.bfloat16)
    x[0, K - 1], x[M - 1, 0] = float("inf"), float("nan")
    w = at((torch.randn(N, K, device=DEV, generator=_gen(72)) * 0.02).to(torch.bfloat16))
    b = at(torch.randn(N, device=DEV, generator=_gen(73)).to(torch.bfloat16))
    res = torch.randn(M, N, device=DEV, generator=_gen(74)).to(torch.bfloat16)
    x, res0 = at(x), at(res)
    y = ops.linear(x, w, b)
    y0 = ops.linear(x, w)
    yr = ops.linear(x, w, b, residual=res0)
    for r in sorted({0, 1, 15, 16, M // 2, 63, 64, M - 2, M - 1}):
        if r >= M:
            continue
        one = at(x[r:r + 1])
        assert torch.equal(ops.linear(one, w, b).view(torch.int16), y[r:r + 1].view(torch.int16)), r
        assert torch.equal(ops.linear(one, w).view(torch.int16), y0[r:r + 1].view(torch.int16)), r
        assert torch.equal(ops.linear(one, w, b, residual=at(res[r:r + 1])).view(torch.int16), yr[r:r + 1].view(torch.int16)), r
    # fp32 sums of K exact products: K 2^-24 of the sum of magnitudes; then bf16 roundings (2^-8 each) of y
    ref = x[1:M - 1].double() @ w.double().T + b.double()
    mag = x[1:M - 1].double().abs() @ w.double().abs().T
    assert bool(((y[1:M - 1].double() - ref).abs() <= K * 2.0**-24 * mag + 2.0**-8 * ref.abs() + 1e-30).all())


# grids of eight waves a workgroup (the first), and of four on both sides of them
@pytest.mark.parametrize("M", [65, 128, 137, 255])
@pytest.mark.parametrize("N,K,off", [(2896, 2880, 1), (1040, 2880, 0), (5136, 4608, 0), (272, 512, 3)])
def test_linear_passes_of_64_rows_bit_exact(M, N, K, off):
    """Batches of several passes by workgroups of four and of eight waves: every tile's first and last row equals
    that row alone bit for bit (a last workgroup with tiles past N, a last slice of fewer groups than the others)."""
    from flyai_amd import ops

    def at(t):
        buf = torch.empty(t.numel() + off, dtype=t.dtype, device=DEV)
        buf[off:] = t.reshape(-1)
        return buf[off:].view(t.shape)

    x = torch.randn(M, K, device=DEV, generator=_gen(75)).to(torch.bfloat16)
    x[M - 1, 0] = float("nan")
    w = at((torch.randn(N, K, device=DEV, generator=_gen(76)) * 0.02).to(torch.bfloat16))
    b = at(torch.randn(N, device=DEV, generator=_gen(77)).to(torch.bfloat16))
    y = ops.linear(at(x), w, b)
    for r in sorted({r for m in range(0, M, 16) for r in (m, min(m + 15, M - 1))}):
        assert torch.equal(ops.linear(at(x[r:r + 1]), w, b).view(torch.int16), y[r:r + 1].view(torch.int16)), r


@pytest.mark.parametrize("N,K", [(5120, 2880), (2880, 4096), (2000, 2880), (1008, 2080), (512, 7168)])
def test_linear_tiled_equals_split_k_bit_exact(N, K):
    """Prefill-sized batches (>= 256 rows) take a tiled GEMM, decode-sized ones the split-K GEMM;
    a row's projection must come out the same bits either way (batch invariance), and within the bar
    of the oracle.  K % 64 == 0 takes the direct-to-LDS tiled kernel (2880: 5 slices and a partial
    one; 4096 and 7168: whole slices only), K = 2080 the register-staged one."""
    from flyai_amd import ops
    M = 300
    x = torch.randn(M, K, device=DEV, generator=_gen(110)).to(torch.bfloat16)
    w = (0.02 * torch.randn(N, K, device=DEV, generator=_gen(111))).to(torch.bfloat16)
    b = (0.1 * torch.randn(N, device=DEV, generator=_gen(112))).to(torch.bfloat16)
    big = ops.linear(x, w, b)                       # tiled path
    parts = [ops.linear(x[r0:r0 + 60].contiguous(), w, b) for r0 in range(0, M, 60)]  # split-K path
    torch.cuda.synchronize()
    assert torch.equal(big, torch.cat(parts)), "tiled and split-K projections differ"
    ref = olayer.linear(x.float().cpu(), w.float().cpu(), b.float().cpu())
    mar, cos = _metrics(big.float().cpu().numpy(), ref.numpy())
    assert mar < 1e-2 and cos > 0.99999


def test_rope_kv_append_bit_exact():
    from flyai_amd import ops
    from flyai_amd.rope import YarnRotary
    q_lens, starts = [1, 4, 3], [100, 7, 4090]
    T, Hq, Hkv, D, cap = sum(q_lens), 64, 8, 64, 4160
    rot = YarnRotary(cap, device=DEV)
    pk = opack.pack_ragged(q_lens, starts)
    qkv = torch.randn(T, (Hq + 2 * Hkv) * D, device=DEV, generator=_gen(40)).to(torch.bfloat16)
    slab = Hkv * cap * D
    kp = torch.zeros(3 * slab, dtype=torch.bfloat16, device=DEV)
    vp = torch.zeros(3 * slab, dtype=torch.bfloat16, device=DEV)
    base = torch.tensor([0, slab, 2 * slab], dtype=torch.int64, device=DEV)
    capt = torch.tensor([cap] * 3, dtype=torch.int32, device=DEV)
    pos = torch.tensor(pk["positions"], device=DEV)
    sid = torch.tensor(pk["seq_id"], device=DEV)
    q = ops.rope_kv_append(qkv, pos, sid, rot.cos, rot.sin, Hq, Hkv, D, base, capt, kp, vp)
    cos, sin = olayer.rope_table(cap)
    p = torch.from_numpy(pk["positions"].astype(np.int64))
    qc = qkv.float().cpu()
    rq = olayer.apply_rope(qc[:, :Hq * D].view(T, Hq, D), cos[p], sin[p])
    rk = olayer.apply_rope(qc[:, Hq * D:(Hq + Hkv) * D].view(T, Hkv, D), cos[p], sin[p])
    assert torch.equal(q.float().cpu(), rq)
    kcpu = [kvlayout.gather(kp[b * slab:(b + 1) * slab], Hkv, cap, "k").float().cpu() for b in range(3)]
    vcpu = [kvlayout.gather(vp[b * slab:(b + 1) * slab], Hkv, cap, "v").float().cpu() for b in range(3)]
    written = set()
    for t in range(T):
        b, ps = int(pk["seq_id"][t]), int(pk["positions"][t])
        written.add((b, ps))
        assert torch.equal(kcpu[b][:, ps, :], rk[t])
        assert torch.equal(vcpu[b][:, ps, :], qc[t, (Hq + Hkv) * D:].view(Hkv, D))
    # nothing else in the slabs was touched (the tiled offsets of distinct positions never overlap)
    for b in range(3):
        others = [p_ for p_ in range(cap) if (b, p_) not in written]
        assert not kcpu[b][:, others].any() and not vcpu[b][:, others].any()


# ---- a8 ----------------------------------------------------------------------------------------

@pytest.mark.parametrize("window", [0, 128])
@pytest.mark.parametrize("q_lens,starts", [([1] * 6 + [4] * 2, [700, 5, 64, 129, 1000, 2047, 300, 0]),
                                           ([130, 1, 9], [0, 3000, 511]),
                                           ([1, 8, 3], [0, 1, 4093])])
def test_attention_vs_oracle(window, q_lens, starts):
    from flyai_amd import ops
    Hq, Hkv, D, cap = 64, 8, 64, 4160
    S, T = len(q_lens), sum(q_lens)
    slab = Hkv * cap * D
    kp = torch.randn(S * slab, device=DEV, generator=_gen(50)).to(torch.bfloat16)
    vp = torch.randn(S * slab, device=DEV, generator=_gen(51)).to(torch.bfloat16)
    q = torch.randn(T, Hq, D, device=DEV, generator=_gen(52)).to(torch.bfloat16)
    sinks = torch.randn(Hq, device=DEV, generator=_gen(53)).to(torch.bfloat16).float()
    base = torch.tensor([b * slab for b in range(S)], dtype=torch.int64, device=DEV)
    capt = torch.tensor([cap] * S, dtype=torch.int32, device=DEV)
    items, groups, n_small = ops.attn_plan(q_lens, starts, Hkv, window, 512)
    out = ops.attn_ragged(q, kp, vp, base, capt, sinks, window, items, groups, n_small, Hkv)
    ks = [kvlayout.gather(kp[b * slab:(b + 1) * slab], Hkv, cap, "k").float().cpu() for b in range(S)]
    vs = [kvlayout.gather(vp[b * slab:(b + 1) * slab], Hkv, cap, "v").float().cpu() for b in range(S)]
    ref = oattn.ragged_attention(q.float().cpu(), ks, vs, q_lens, starts, sinks.cpu(), window)
    mar, cos = _metrics(out.float().cpu().numpy(), ref.numpy())
    assert mar <= MAR and cos >= COS, f"attention: {mar:.3g} {cos:.6f}"


@pytest.mark.parametrize("window", [0, 128])
def test_attention_many_splits_vs_oracle(window):
    """128-key splits: up to 32 splits per (token, head), so the merge reads its split maxima and
    records over several batches, including a partial last batch."""
    from flyai_amd import ops
    Hq, Hkv, D, cap = 64, 8, 64, 4160
    q_lens, starts = [1, 4, 2], [4093, 2301, 17]
    S, T = len(q_lens), sum(q_lens)
    slab = Hkv * cap * D
    kp = torch.randn(S * slab, device=DEV, generator=_gen(60)).to(torch.bfloat16)
    vp = torch.randn(S * slab, device=DEV, generator=_gen(61)).to(torch.bfloat16)
    q = torch.randn(T, Hq, D, device=DEV, generator=_gen(62)).to(torch.bfloat16)
    sinks = torch.randn(Hq, device=DEV, generator=_gen(63)).to(torch.bfloat16).float()
    base = torch.tensor([b * slab for b in range(S)], dtype=torch.int64, device=DEV)
    capt = torch.tensor([cap] * S, dtype=torch.int32, device=DEV)
    items, groups, n_small = ops.attn_plan(q_lens, starts, Hkv, window, 128)
    if window == 0:
        assert max(int(g[1]) for g in groups.cpu().view(-1, 8).tolist()) >= 32
    out = ops.attn_ragged(q, kp, vp, base, capt, sinks, window, items, groups, n_small, Hkv)
    ks = [kvlayout.gather(kp[b * slab:(b + 1) * slab], Hkv, cap, "k").float().cpu() for b in range(S)]
    vs = [kvlayout.gather(vp[b * slab:(b + 1) * slab], Hkv, cap, "v").float().cpu() for b in range(S)]
    ref = oattn.ragged_attention(q.float().cpu(), ks, vs, q_lens, starts, sinks.cpu(), window)
    mar, cos = _metrics(out.float().cpu().numpy(), ref.numpy())
    assert mar <= MAR and cos >= COS, f"attention: {mar:.3g} {cos:.6f}"


@pytest.mark.parametrize("window", [0, 128])
def test_attention_prefill_items_vs_oracle(window):
    """Chunked-prefill rows (q_len >= 32) on the prefill kernel, mixed with decode and verify rows on
    the split kernel, into one output; against the oracle.  The unwritten slots past each sequence
    hold NaN, which neither kernel may read into a result."""
    from flyai_amd import ops
    Hq, Hkv, D, cap = 64, 8, 64, 1600
    q_lens, starts = [300, 1, 4, 45, 33], [700, 1000, 64, 0, 1200]
    S, T = len(q_lens), sum(q_lens)
    slab = Hkv * cap * D
    kp = torch.full((S * slab,), float("nan"), device=DEV).to(torch.bfloat16)
    vp = torch.full((S * slab,), float("nan"), device=DEV).to(torch.bfloat16)
    for b, (ql, st) in enumerate(zip(q_lens, starts)):
        pos = torch.arange(st + ql, device=DEV)
        kvlayout.scatter(kp[b * slab:(b + 1) * slab], Hkv, cap, "k",
                         torch.randn(Hkv, st + ql, D, device=DEV, generator=_gen(90 + b)), pos)
        kvlayout.scatter(vp[b * slab:(b + 1) * slab], Hkv, cap, "v",
                         torch.randn(Hkv, st + ql, D, device=DEV, generator=_gen(95 + b)), pos)
    q = torch.randn(T, Hq, D, device=DEV, generator=_gen(52)).to(torch.bfloat16)
    sinks = torch.randn(Hq, device=DEV, generator=_gen(53)).to(torch.bfloat16).float()
    base = torch.tensor([b * slab for b in range(S)], dtype=torch.int64, device=DEV)
    capt = torch.tensor([cap] * S, dtype=torch.int32, device=DEV)
    items, groups, n_small, pitems = ops.attn_plan_prefill(q_lens, starts, Hkv, window, 512, 32)
    assert pitems.shape[0] == (19 + 3 + 3) * Hkv
    out = ops.attn_ragged(q, kp, vp, base, capt, sinks, window, items, groups, n_small, Hkv)
    ops.attn_prefill(q, kp, vp, base, capt, sinks, window, pitems, Hkv, out)
    torch.cuda.synchronize()
    ks = [kvlayout.gather(kp[b * slab:(b + 1) * slab], Hkv, cap, "k").float().cpu() for b in range(S)]
    vs = [kvlayout.gather(vp[b * slab:(b + 1) * slab], Hkv, cap, "v").float().cpu() for b in range(S)]
    ref = oattn.ragged_attention(q.float().cpu(), ks, vs, q_lens, starts, sinks.cpu(), window)
    got = out.float().cpu().numpy()
    assert np.isfinite(got).all()
    mar, cos = _metrics(got, ref.numpy())
    assert mar <= MAR and cos >= COS, f"prefill attention: {mar:.3g} {cos:.6f}"
    # the prefill path against the split path on the same rows: same math, different blocking
    items0, groups0, ns0 = ops.attn_plan(q_lens, starts, Hkv, window, 512)
    out0 = ops.attn_ragged(q, kp, vp, base, capt, sinks, window, items0, groups0, ns0, Hkv)
    torch.cuda.synchronize()
    mar0, cos0 = _metrics(got, out0.float().cpu().numpy())
    assert mar0 < 1e-2 and cos0 > 0.99999


@pytest.mark.parametrize("window,split", [(0, 1024), (0, 192), (128, 1024)])
def test_attention_few_items_equal_many_items_bit_exact(window, split):
    """A launch of few items gives each one four waves, a launch of many one wave each: every sequence
    alone (few items) equals the same sequence among the others (many items), bit for bit.  Lengths at the
    edges of blocks, of a super-block (256 and 512 keys) and of a split; 1 to 8 query tokens; logits large
    enough to move the running max often; NaN in the unwritten slots."""
    from flyai_amd import ops
    Hq, Hkv, D = 64, 8, 64
    ends = [1, 2, 63, 64, 65, 129, 255, 256, 257, 512, 513, 1000, 1023, 1024, 1025, 2047, 2300]
    seqs = [(q, max(0, e - q)) for e in ends for q in (1, 2, 3, 8)]
    q_lens, starts = [q for q, _ in seqs], [s for _, s in seqs]
    cap = 2432
    S, T, slab = len(seqs), sum(q_lens), Hkv * cap * D
    kp = torch.full((S * slab,), float("nan"), device=DEV, dtype=torch.bfloat16)
    vp = torch.full((S * slab,), float("nan"), device=DEV, dtype=torch.bfloat16)
    for b, (ql, st) in enumerate(seqs):
        pos = torch.arange(st + ql, device=DEV)
        kvlayout.scatter(kp[b * slab:(b + 1) * slab], Hkv, cap, "k",
                         4 * torch.randn(Hkv, st + ql, D, device=DEV, generator=_gen(300 + b)), pos)
        kvlayout.scatter(vp[b * slab:(b + 1) * slab], Hkv, cap, "v",
                         torch.randn(Hkv, st + ql, D, device=DEV, generator=_gen(500 + b)), pos)
    q = (4 * torch.randn(T, Hq, D, device=DEV, generator=_gen(54))).to(torch.bfloat16)
    sinks = torch.randn(Hq, device=DEV, generator=_gen(55)).to(torch.bfloat16).float()

    def run(sel, rows):
        base = torch.tensor([b * slab for b in sel], dtype=torch.int64, device=DEV)
        capt = torch.tensor([cap] * len(sel), dtype=torch.int32, device=DEV)
        items, groups, n_small = ops.attn_plan([q_lens[b] for b in sel], [starts[b] for b in sel], Hkv, window, split)
        return ops.attn_ragged(rows.contiguous(), kp, vp, base, capt, sinks, window, items, groups, n_small, Hkv), len(items)

    many, n = run(range(S), q)
    assert n > 640
    t = 0
    for b, ql in enumerate(q_lens):
        few, n = run([b], q[t:t + ql])
        assert n <= 512
        assert torch.equal(few.view(torch.int16), many[t:t + ql].view(torch.int16)), (q_lens[b], starts[b])
        t += ql
    assert torch.isfinite(many.float()).all()


def _attention_item_count_rules(q_len, window, S, few_counts):
    from flyai_amd import ops
    Hq, Hkv, D, cap = 64, 8, 64, 640
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    starts = [(64 * (1 + b % 9) + (b % 5) - 2) - q_len for b in range(S)]
    slab = Hkv * cap * D
    kp = torch.full((S * slab,), float("nan"), device=DEV, dtype=torch.bfloat16)
    vp = torch.full((S * slab,), float("nan"), device=DEV, dtype=torch.bfloat16)
    for b, st in enumerate(starts):
        pos = torch.arange(st + q_len, device=DEV)
        kvlayout.scatter(kp[b * slab:(b + 1) * slab], Hkv, cap, "k",
                         4 * torch.randn(Hkv, st + q_len, D, device=DEV, generator=_gen(700 + b)), pos)
        kvlayout.scatter(vp[b * slab:(b + 1) * slab], Hkv, cap, "v",
                         torch.randn(Hkv, st + q_len, D, device=DEV, generator=_gen(800 + b)), pos)
    q = (4 * torch.randn(S * q_len, Hq, D, device=DEV, generator=_gen(56))).to(torch.bfloat16)
    sinks = torch.randn(Hq, device=DEV, generator=_gen(57)).to(torch.bfloat16).float()

    def run(n):
        base = torch.arange(n, dtype=torch.int64, device=DEV) * slab
        capt = torch.full((n,), cap, dtype=torch.int32, device=DEV)
        items, groups, n_small = ops.attn_plan([q_len] * n, starts[:n], Hkv, window, 1024)
        out = ops.attn_ragged(q[:n * q_len].contiguous(), kp, vp, base, capt, sinks, window, items, groups, n_small, Hkv)
        return out.view(torch.int16), len(items)

    many, n_many = run(S)
    assert n_many > 2 * cus and n_many == 8 * S and torch.isfinite(many.view(torch.bfloat16).float()).all()
    for n in few_counts(cus):
        few, n_items = run(n)
        assert n_items == 8 * n
        assert torch.equal(few, many[:n * q_len]), n


@pytest.mark.parametrize("window", [0, 128])
@pytest.mark.parametrize("q_len", [1, 2, 4])
def test_attention_item_count_rules_bit_exact(q_len, window):
    """The launch's item count decides how many waves take an item and up to how many blocks one wave takes it
    alone (one workgroup a CU, two a CU, more): the same sequences in launches on both sides of every line, with
    key counts at both sides of every block line, give the same bits."""
    _attention_item_count_rules(q_len, window, 72, lambda cus: (1, cus // 8, cus // 8 + 1, cus // 4, cus // 4 + 1))


@pytest.mark.parametrize("q_len", [1, 2, 4])
@pytest.mark.parametrize("window", [0, 128, 129])
def test_attention_full_and_sliding_lines_bit_exact(window, q_len):
    """The lines that depend on the layer: a full layer's items stay with four waves up to two and a half workgroups a
    CU; a sliding layer's go to one wave where its window holds every item in the blocks one wave takes."""
    _attention_item_count_rules(q_len, window, 100, lambda cus: (2, cus // 4, 5 * cus // 16, 5 * cus // 16 + 1))


def test_attention_ignores_unwritten_nan_slots():
    """Keys/values past each sequence's length (and before its window) are never read into the
    result even when they hold NaN: the kernel masks scores and zeroes out-of-range values."""
    from flyai_amd import ops
    Hq, Hkv, D, cap = 64, 8, 64, 1024
    q_lens, starts = [1, 3], [200, 517]
    S, T = 2, 4
    slab = Hkv * cap * D
    kp = torch.full((S * slab,), float("nan"), device=DEV).to(torch.bfloat16)
    vp = torch.full((S * slab,), float("nan"), device=DEV).to(torch.bfloat16)
    for b, (ql, st) in enumerate(zip(q_lens, starts)):
        pos = torch.arange(st + ql, device=DEV)
        kvlayout.scatter(kp[b * slab:(b + 1) * slab], Hkv, cap, "k",
                         torch.randn(Hkv, st + ql, D, device=DEV, generator=_gen(60 + b)), pos)
        kvlayout.scatter(vp[b * slab:(b + 1) * slab], Hkv, cap, "v",
                         torch.randn(Hkv, st + ql, D, device=DEV, generator=_gen(70 + b)), pos)
    q = torch.randn(T, Hq, D, device=DEV, generator=_gen(80)).to(torch.bfloat16)
    sinks = torch.zeros(Hq, device=DEV)
    base = torch.tensor([0, slab], dtype=torch.int64, device=DEV)
    capt = torch.tensor([cap, cap], dtype=torch.int32, device=DEV)
    for window in (0, 128):
        items, groups, n_small = ops.attn_plan(q_lens, starts, Hkv, window, 128)
        out = ops.attn_ragged(q, kp, vp, base, capt, sinks, window, items, groups, n_small, Hkv)
        assert torch.isfinite(out.float()).all()


# ---- a10: the stage step ------------------------------------------------------------------------

def test_stage_step_per_layer_vs_oracle():
    from gpu_harness import run_stage_vs_oracle, small_stage_case
    case = small_stage_case(n_layers=2, n_experts=8, seed=1)
    outs, refs = run_stage_vs_oracle(case, per_layer=True)
    for l, (o, r) in enumerate(zip(outs, refs)):
        mar, cos = _metrics(o, r)
        assert mar <= MAR and cos >= COS, f"layer {l}: max-abs-rel {mar:.3g} cos {cos:.6f}"


def test_stage_step_hidden_3584_per_layer_vs_oracle():
    """Hidden 3584 (> 3072): the router-logits finalizer's wide variant, which keeps one split-K
    slice in registers and adds the other 7 of the 4096-wide o-proj in its tail loop."""
    from gpu_harness import oracle_layer_params, oracle_kv, fill_kv_random, metrics
    from flyai_amd.rope import YarnRotary
    from flyai_amd.runtime import KVWorkspace, RaggedStage
    from flyai_amd.weights import GptOssShape, synthetic_layer
    shape = GptOssShape(hidden=3584, n_experts=8)
    lw = synthetic_layer(shape, 77, DEV, sliding=False, keep_hf=True)
    rot = YarnRotary(2048, device=DEV)
    q_lens, starts = [1, 4, 1], [300, 17, 1500]
    kv = KVWorkspace(1, 3, 2048, shape.n_kv_heads, shape.head_dim, DEV)
    fill_kv_random(kv, 78)
    T = sum(q_lens)
    h = torch.randn(T, shape.hidden, device=DEV, generator=_gen(79)).to(torch.bfloat16)
    okv = oracle_kv(kv, 0, [0, 1, 2])
    st = RaggedStage(shape, [lw], rot, kv, max_tokens=64, max_seqs=3)
    out = st.forward(h.clone(), q_lens, starts, [0, 1, 2])
    torch.cuda.synchronize()
    cos, sin = olayer.rope_table(2048)
    ref = olayer.decoder_layer(h.float().cpu(), oracle_layer_params(lw, False), okv, q_lens, starts, cos, sin)
    mar, cs = metrics(out.float().cpu().numpy(), ref.numpy())
    assert mar <= MAR and cs >= COS, f"hidden 3584 layer: {mar:.3g} {cs:.6f}"


def test_c0_moe_block_vs_oracle():
    """Workload C0: one GPT-OSS MoE block (H=I=2880, 128 experts, top-4) on 4 sequences of lengths
    {1,1,3,7}, E2M1 codes uniform, E8M0 scales 2^-8..2^-4, bf16 N(0,1) activations RMSNorm'd."""
    from flyai_amd import ops
    from flyai_amd.weights import GptOssShape, synthetic_moe
    shape = GptOssShape()
    m = synthetic_moe(shape, _gen(0), DEV)
    w13 = ops.mxfp4_repack(m["w13_blocks"], m["w13_scales"])
    w2 = ops.mxfp4_repack(m["w2_blocks"], m["w2_scales"])
    T = 12
    x = torch.randn(T, shape.hidden, device=DEV, generator=_gen(1)).to(torch.bfloat16)
    lnw = torch.ones(shape.hidden, device=DEV)
    rw = (torch.randn(128, shape.hidden, device=DEV, generator=_gen(2)) * 0.02).to(torch.bfloat16)
    rb = (torch.randn(128, device=DEV, generator=_gen(3)) * 0.02).to(torch.bfloat16)
    xn = ops.rmsnorm(x, lnw)
    ids, wts = ops.router_topk_softmax(xn, rw, rb, 4)
    hist, off, perm, inv = ops.moe_permute(ids, 128)
    h = ops.moe_gate_up(xn, perm, off, 4, w13, m["b13"], 128, shape.intermediate)
    y = ops.moe_down(h, off, w2, m["b2"], 128, shape.hidden)
    out = ops.moe_combine(y, inv, wts, residual=x.clone())
    torch.cuda.synchronize()
    xn_ref = olayer.rmsnorm(x.float().cpu(), lnw.cpu())
    rids, rwts, _ = oroute.gptoss_route(xn.float().cpu(), rw.float().cpu(), rb.float().cpu(), 4)
    assert np.array_equal(ids.cpu().numpy(), rids)
    _, roff, rperm, rinv = oroute.permute(rids, 128)
    assert np.array_equal(perm.cpu().numpy(), rperm)
    wo = oexperts.MxExpertWeights(*(m[n].cpu().numpy() for n in
                                    ("w13_blocks", "w13_scales", "b13", "w2_blocks", "w2_scales", "b2")))
    ry = oexperts.experts_mxfp4(xn.float().cpu(), rperm, roff, 4, wo)
    ref = oroute.combine(ry, rinv, rwts, residual=x.float().cpu())
    mar, cos = _metrics(out.float().cpu().numpy(), ref.numpy())
    assert mar <= MAR and cos >= COS, f"C0 MoE block: {mar:.3g} {cos:.6f}"
    mar, cos = _metrics(xn.float().cpu().numpy(), xn_ref.numpy())
    assert mar < 1e-2 and cos > 0.9999


def test_stage_step_with_prefill_chunk_per_layer_vs_oracle():
    """A chunked-prefill row (q_len 96, prefill attention items) packed with decode and verify rows,
    layer by layer from the GPU's own input: the attention output within a tight bar, and the layer
    output on every token routed alike (a token may route differently only on a near-tie of the
    oracle's logits, which the bf16 rounding of its input can flip)."""
    import gpu_harness as gh
    from flyai_amd.runtime import RaggedStage
    q_lens, starts = [96, 1, 4, 1], [300, 40, 1000, 0]
    case = gh.small_stage_case(n_layers=2, n_experts=32, seed=4, q_lens=q_lens, starts=starts)
    shape, kv, T = case["shape"], case["kv"], case["T"]
    cos, sin = olayer.rope_table(case["maxlen"])
    h = case["hidden"].clone()
    for l, lw in enumerate(case["layers"]):
        okv = gh.oracle_kv(kv, l, case["slots"])
        st = RaggedStage(shape, [lw], case["rot"], gh._SingleLayerKV(kv, l), max_tokens=128, max_seqs=4)
        hin = gh.cpu_f32(h)
        h = st.forward(h.clone(), q_lens, starts, case["slots"])
        torch.cuda.synchronize()
        tr = {}
        ids = st.debug_buffer(4, torch.int32, (T, shape.top_k)).cpu().numpy()
        ref = olayer.decoder_layer(hin, gh.oracle_layer_params(lw, lw.sliding), okv, q_lens, starts, cos, sin,
                                   trace=tr, force_ids=ids)
        attn = gh.cpu_f32(st.debug_buffer(3, torch.bfloat16, (T, shape.n_q_heads * shape.head_dim))).numpy()
        mar_a, cos_a = _metrics(attn, tr["attn"].reshape(T, -1).numpy())
        assert mar_a <= 1e-2 and cos_a >= 0.9999, (l, mar_a, cos_a)
        gh.tokens_with_same_routing(ids, tr["ids"], tr["logits"], shape.top_k)
        mar, cos_ = _metrics(gh.cpu_f32(h).numpy(), ref.numpy())
        assert mar <= MAR and cos_ >= COS, f"layer {l}: max-abs-rel {mar:.3g} cos {cos_:.6f}"
        del st


def test_batched_equals_solo_bit_exact():
    """Size-independent property on a C1-shaped batch: a stream's output inside a ragged batch equals
    running that stream alone (per-row fixed reduction orders everywhere), bit for bit."""
    from gpu_harness import small_stage_case
    from flyai_amd.runtime import KVWorkspace, RaggedStage
    q_lens = [1] * 6 + [4] * 2
    starts = [600, 513, 4000, 800, 1, 2500, 1500, 7000]
    case = small_stage_case(n_layers=2, n_experts=16, seed=3, q_lens=q_lens, starts=starts, maxlen=8192)
    kv0 = [(k.clone(), v.clone()) for k, v in zip(case["kv"].k, case["kv"].v)]
    st = RaggedStage(case["shape"], case["layers"], case["rot"], case["kv"], 64, 8)
    batched = st.forward(case["hidden"].clone(), q_lens, starts, list(range(8)))
    torch.cuda.synchronize()
    cu = np.concatenate([[0], np.cumsum(q_lens)])
    for b in (0, 6, 7):
        for l, (k, v) in enumerate(kv0):
            case["kv"].k[l].copy_(k)
            case["kv"].v[l].copy_(v)
        solo = st.forward(case["hidden"][cu[b]:cu[b + 1]].clone(), [q_lens[b]], [starts[b]], [b])
        torch.cuda.synchronize()
        assert torch.equal(solo, batched[cu[b]:cu[b + 1]]), f"stream {b} differs solo vs batched"


def test_prefill_batch_decode_rows_equal_solo_bit_exact():
    """A 300-token prefill chunk makes the batch prefill-sized: the qkv projection then runs the tiled
    GEMM with the finalize, RoPE and KV append in its epilogue, the o-projection the tiled GEMM and the
    router the unfused path.  The decode rows beside it must come out as they do alone (split-K
    projections, the separate qkv finalize kernel, the fused router finalizer), bit for bit."""
    from gpu_harness import small_stage_case
    from flyai_amd.runtime import RaggedStage
    q_lens = [300, 1, 1, 4]
    starts = [0, 700, 2100, 1500]
    case = small_stage_case(n_layers=2, n_experts=16, seed=5, q_lens=q_lens, starts=starts, maxlen=4096)
    kv0 = [(k.clone(), v.clone()) for k, v in zip(case["kv"].k, case["kv"].v)]
    st = RaggedStage(case["shape"], case["layers"], case["rot"], case["kv"], 320, 4)
    batched = st.forward(case["hidden"].clone(), q_lens, starts, list(range(4)))
    torch.cuda.synchronize()
    assert torch.isfinite(batched.float()).all()
    cu = np.concatenate([[0], np.cumsum(q_lens)])
    for b in (1, 2, 3):
        for l, (k, v) in enumerate(kv0):
            case["kv"].k[l].copy_(k)
            case["kv"].v[l].copy_(v)
        solo = st.forward(case["hidden"][cu[b]:cu[b + 1]].clone(), [q_lens[b]], [starts[b]], [b])
        torch.cuda.synchronize()
        assert torch.equal(solo, batched[cu[b]:cu[b + 1]]), f"stream {b} differs solo vs beside a prefill chunk"


def test_dense_and_row_pass_experts_bit_identical():
    """The same rows through the row-pass expert kernel (a batch below the dense cutoff of 8 rows per
    expert on average) and through the dense tiled GEMM (a batch above it) give bit-identical h and y:
    both feed the MFMA the same K-to-lane mapping, accumulate the 128-K groups in the same order from
    zero and share the epilogue arithmetic.  So a row's tokens do not depend on whether its batch
    mates push the batch across the cutoff (the reference's Triton path measured the opposite,
    docs/receipts/batched-verify-20260623.json:27-30).  Dense groups of 100 rows take a 96-row pass
    and a 32-row pass; H = I = 2880 leaves a partial last 128-K group."""
    from flyai_amd import ops
    from flyai_amd.weights import GptOssShape, synthetic_moe
    E, k = 4, 4
    shape = GptOssShape(n_experts=E)
    m = synthetic_moe(shape, _gen(31), DEV)
    w13 = ops.mxfp4_repack(m["w13_blocks"], m["w13_scales"])
    w2 = ops.mxfp4_repack(m["w2_blocks"], m["w2_scales"])
    T = 100
    x = _rms_input(T, shape.hidden, 32)
    ids = torch.arange(E, dtype=torch.int32, device=DEV).repeat(T, 1).contiguous()  # every token on every expert
    _, off_a, perm_a, _ = ops.moe_permute(ids, E)
    h_a = ops.moe_gate_up(x, perm_a, off_a, k, w13, m["b13"], E, shape.intermediate)   # 400 rows: dense
    y_a = ops.moe_down(h_a, off_a, w2, m["b2"], E, shape.hidden)
    for sel in ([0, 1, 2, 3, 4, 5, 6], [99, 17, 50], [64, 95, 96, 97]):   # 4 * len(sel) < 32: row-pass
        sel_t = torch.tensor(sel, device=DEV)
        ids_b = ids[:len(sel)].contiguous()
        _, off_b, perm_b, _ = ops.moe_permute(ids_b, E)
        xb = x[sel_t].contiguous()
        h_b = ops.moe_gate_up(xb, perm_b, off_b, k, w13, m["b13"], E, shape.intermediate)
        y_b = ops.moe_down(h_b, off_b, w2, m["b2"], E, shape.hidden)
        torch.cuda.synchronize()
        oa, ob = off_a.cpu().tolist(), off_b.cpu().tolist()
        for e in range(E):
            ra = torch.tensor([oa[e] + t for t in sel], device=DEV)   # expert e's rows are its tokens in order
            rb = torch.arange(ob[e], ob[e] + len(sel), device=DEV)
            assert torch.equal(h_a[ra], h_b[rb]), f"expert {e}, tokens {sel}: gate_up differs"
            assert torch.equal(y_a[ra], y_b[rb]), f"expert {e}, tokens {sel}: down differs"


@pytest.mark.parametrize("E,groups", [(130, {0: 2, 63: 1, 64: 9, 127: 1, 128: 3, 129: 1}), (130, {129: 1}), (4, {2: 5}),
                                      (64, {63: 17}), (200, {e: 1 for e in range(3, 200, 2)})])
def test_few_groups_experts_bit_identical(E, groups):
    """The row-pass kernel's workgroups are counted over the groups that have rows (128 experts counted at a
    time): each group's h and y equal that expert's alone in a one-expert call, bit for bit."""
    from flyai_amd import ops
    from flyai_amd.weights import GptOssShape, synthetic_moe
    H, I = 160, 96
    m = synthetic_moe(GptOssShape(hidden=H, intermediate=I, n_experts=E), _gen(63), DEV)
    w13 = ops.mxfp4_repack(m["w13_blocks"], m["w13_scales"])
    w2 = ops.mxfp4_repack(m["w2_blocks"], m["w2_scales"])
    ids = torch.tensor([e for e, n in groups.items() for _ in range(n)], dtype=torch.int32, device=DEV)[:, None]
    x = _rms_input(len(ids), H, 64)
    _, off, perm, _ = ops.moe_permute(ids, E)
    h = ops.moe_gate_up(x, perm, off, 1, w13, m["b13"], E, I)
    y = ops.moe_down(h, off, w2, m["b2"], E, H)
    lo = 0
    for e, n in groups.items():
        one = [ops.mxfp4_repack(m[f"{w}_blocks"][e:e + 1].contiguous(), m[f"{w}_scales"][e:e + 1].contiguous())
               for w in ("w13", "w2")]
        for r in range(lo, lo + n, 5):  # at most 5 rows: the row-pass kernel
            rows = x[r:min(r + 5, lo + n)].contiguous()
            _, off1, perm1, _ = ops.moe_permute(torch.zeros(len(rows), 1, dtype=torch.int32, device=DEV), 1)
            h1 = ops.moe_gate_up(rows, perm1, off1, 1, one[0], m["b13"][e:e + 1].contiguous(), 1, I)
            y1 = ops.moe_down(h1, off1, one[1], m["b2"][e:e + 1].contiguous(), 1, H)
            assert torch.equal(h1.view(torch.int16), h[r:r + len(rows)].view(torch.int16)), f"gate_up of expert {e}"
            assert torch.equal(y1.view(torch.int32), y[r:r + len(rows)].view(torch.int32)), f"down of expert {e}"
        lo += n


@pytest.mark.parametrize("H,I", [(2880, 2880), (128, 160), (544, 2048)])
def test_medium_group_experts_bit_identical(H, I):
    """A batch of 6 to 18 rows per expert on average runs the medium-group kernel; the same rows in batches
    of at most 5 per expert run the row-pass kernel: h and y equal bit for bit.  Groups of 0 rows, of one
    row tile and its neighbours, of two and their neighbours, and of more than a pass; K of whole and partial
    128-K groups; one weight block a unit; rows holding an infinity (first and last group) and a NaN."""
    from flyai_amd import ops
    from flyai_amd.weights import GptOssShape, synthetic_moe
    sizes = [1, 15, 0, 16, 17, 32, 33, 14]
    E, T = len(sizes), sum(sizes)
    assert 6 * E <= T < 18 * E
    m = synthetic_moe(GptOssShape(hidden=H, intermediate=I, n_experts=E), _gen(61), DEV)
    w13 = ops.mxfp4_repack(m["w13_blocks"], m["w13_scales"])
    w2 = ops.mxfp4_repack(m["w2_blocks"], m["w2_scales"])
    x = _rms_input(T, H, 62)
    x[3, 5], x[40, H - 1], x[70, 1] = float("inf"), float("-inf"), float("nan")
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(sizes)])[torch.randperm(T, generator=torch.Generator().manual_seed(3))]
    ids = ids.to(torch.int32).to(DEV)[:, None].contiguous()

    def run(rows):
        _, off, perm, inv = ops.moe_permute(ids[rows].contiguous(), E)
        h = ops.moe_gate_up(x[rows].contiguous(), perm, off, 1, w13, m["b13"], E, I)
        return h[inv.long()], ops.moe_down(h, off, w2, m["b2"], E, H)[inv.long()]

    h_all, y_all = run(torch.arange(T, device=DEV))
    for t0 in range(0, T, 5 * E):
        rows = torch.arange(t0, min(T, t0 + 5 * E), device=DEV)
        h, y = run(rows)
        assert torch.equal(h.view(torch.int16), h_all[rows].view(torch.int16)), "gate_up differs"
        assert torch.equal(y.view(torch.int32), y_all[rows].view(torch.int32)), "down differs"

@pytest.mark.parametrize("K", [32, 160, 2880])
def test_mxfp4_repack_leaves_padding_scales_zero(K):
    """The tiled expert kernels multiply the padding of K with zero activations and rely on its scale bytes for finite
    weights: the re-pack writes zeros there, whatever the real scales are and whatever the buffer held."""
    from flyai_amd import ops
    E, N, G = 2, 48, K // 32
    blocks = torch.full((E, N, G, 16), 0xff, dtype=torch.uint8, device=DEV)
    del_me = torch.full((ops.mxfp4_packed_bytes(E, N, K),), 0xff, dtype=torch.uint8, device=DEV)
    del del_me  # the allocator hands the re-pack this memory
    packed = ops.mxfp4_repack(blocks, torch.full((E, N, G), 0xff, dtype=torch.uint8, device=DEV)).cpu().numpy()
    KG4 = (G + 15) // 16  # scale words of 4 groups of 4 blocks
    words = packed[E * N * G * 16:].reshape(E * N // 16, KG4, 4, 16, 4)  # [tile][word][block of a group][row][group]
    for kg in range(4 * KG4):
        for g in range(4):
            want = 0xff if 4 * kg + g < G else 0
            assert (words[:, kg // 4, g, :, kg % 4] == want).all(), (kg, g)


def _expert_batches_equal_parts(ids, H, I, E, part, seed):
    """gate_up and down of a batch of `ids` [T, k] against the same tokens in batches of `part`, bit for bit."""
    from flyai_amd import ops
    from flyai_amd.weights import GptOssShape, synthetic_moe
    m = synthetic_moe(GptOssShape(hidden=H, intermediate=I, n_experts=E), _gen(seed), DEV)
    w13 = ops.mxfp4_repack(m["w13_blocks"], m["w13_scales"])
    w2 = ops.mxfp4_repack(m["w2_blocks"], m["w2_scales"])
    T, k = ids.shape
    x = _rms_input(T, H, seed + 1)
    x[T // 2, 1], x[T - 1, H - 1] = float("inf"), float("nan")

    def run(rows):
        _, off, perm, inv = ops.moe_permute(ids[rows].contiguous(), E)
        h = ops.moe_gate_up(x[rows].contiguous(), perm, off, k, w13, m["b13"], E, I)
        return (h[inv.long()].view(len(rows), k, I).view(torch.int16),
                ops.moe_down(h, off, w2, m["b2"], E, H)[inv.long()].view(len(rows), k, H).view(torch.int32))

    h_all, y_all = run(torch.arange(T, device=DEV))
    for t0 in range(0, T, part):
        rows = torch.arange(t0, min(T, t0 + part), device=DEV)
        h, y = run(rows)
        assert torch.equal(h, h_all[rows]), "gate_up differs"
        assert torch.equal(y, y_all[rows]), "down differs"


@pytest.mark.parametrize("skewed", [False, True])
def test_medium_group_experts_full_size_bit_identical(skewed):
    """The medium-group kernel with three weight blocks a unit (128 experts, H = I = 2880: a chunk's later blocks, the
    ring running over them, their bias, a last chunk of two blocks): 333 tokens against batches of the row-pass
    kernel, with even routing and with half of the rows on a tenth of the experts (groups of two and more passes)."""
    E, k, T = 128, 4, 333
    g = torch.Generator().manual_seed(7)
    p = torch.ones(E)
    if skewed:
        p[torch.randperm(E, generator=g)[:E // 10]] = 9.0
    ids = (-torch.rand(T, E, generator=g).log() / p).topk(k, 1, largest=False)[1].sort(1)[0].to(torch.int32)
    most = int(torch.bincount(ids.flatten(), minlength=E).max())
    assert 6 * E <= T * k < 18 * E and (most > 32) == skewed
    _expert_batches_equal_parts(ids.to(DEV), 2880, 2880, E, 150, 73)


@pytest.mark.parametrize("sizes", [(6, 6, 6, 6), (7, 9, 8, 7), (8, 8, 9, 8), (1, 17, 0, 6, 33, 8, 2, 1)])
def test_few_experts_medium_rule_bit_identical(sizes):
    """Where the medium-group kernel's units leave most of the chip idle it starts at 8 rows per expert: batches on
    both sides of that line and on it, against batches of the row-pass kernel."""
    T = sum(sizes)
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(sizes)])[torch.randperm(T, generator=torch.Generator().manual_seed(5))]
    _expert_batches_equal_parts(ids.to(torch.int32).to(DEV)[:, None], 544, 1024, len(sizes), 5 * len(sizes), 71)


@pytest.mark.parametrize("H", [32, 128, 160, 288, 2880])
@pytest.mark.parametrize("n,V", [(1, 16), (16, 144), (17, 272), (48, 128), (64, 1040)])
def test_lm_head_rows_do_not_depend_on_the_batch(n, V, H):
    """K shorter than the weight ring and of partial chunks, vocabularies past the last whole workgroup, 1 to 4
    row tiles, rows picked in any order, an infinite hidden value: every row's logits equal that row's alone bit
    for bit and the token is their first maximum; finite rows against float64."""
    from flyai_amd import ops
    x = torch.randn(n + 3, H, device=DEV, generator=_gen(91)).to(torch.bfloat16)
    w = (torch.randn(V, H, device=DEV, generator=_gen(92)) * 0.05).to(torch.bfloat16)
    rows = torch.randperm(n + 3, generator=torch.Generator().manual_seed(n))[:n].to(torch.int32).to(DEV)
    x[int(rows[0]), H - 1] = float("inf")
    wp = ops.bf16_tile_repack(w)
    ids, logits = ops.lm_head_argmax(x, wp, V, rows=rows, want_logits=True)
    for i in sorted({0, 1, 15, 16, n - 1}):
        if i < n:
            i1, l1 = ops.lm_head_argmax(x, wp, V, rows=rows[i:i + 1].contiguous(), want_logits=True)
            assert torch.equal(l1.view(torch.int16), logits[i:i + 1].view(torch.int16)) and int(i1[0]) == int(ids[i])
    best = logits.float().amax(1, keepdim=True)
    first = (logits.float() == best).int().argmax(1)
    assert torch.equal(first[1:].cpu().int(), ids[1:].cpu().int())
    # fp32 sums of H exact products: H 2^-24 of the sum of magnitudes; then one bf16 rounding (2^-8)
    xs = x[rows.long()][1:].double()
    ref, mag = xs @ w.double().T, xs.abs() @ w.double().abs().T
    assert bool(((logits[1:].double() - ref).abs() <= H * 2.0**-24 * mag + 2.0**-8 * ref.abs() + 1e-30).all())
