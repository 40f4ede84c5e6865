"""flyai_sample_rows / flyai_sample_probs and the kernel-backed Sampler against the sampler oracle,
bit for bit: integer weights make the kernel's sums independent of its reduction order, so the fp32
probabilities, the drafted-token probabilities and every draw for given uniforms must be identical.
Vocabulary of GPT-OSS (201088) and small odd sizes; rows with heavy bf16 ties so that the top-k and
top-p boundaries fall inside runs of equal logits."""
import numpy as np
import pytest
import torch

from oracle import sampling as S

pytestmark = pytest.mark.gpu

DEV = "cuda"
V_GPTOSS = 201088


def _logits(R, V, seed, ties=False, scale=3.0):
    g = torch.Generator(device="cpu")
    g.manual_seed(seed)
    x = torch.randn(R, V, generator=g) * scale
    if ties:
        x = torch.round(x * 2) / 2
    return x.to(torch.bfloat16)


CASES = [  # (V, temp, top_k, top_p, ties)
    (V_GPTOSS, 0.7, 0, 0.9, False),
    (V_GPTOSS, 1.0, 50, 1.0, False),
    (V_GPTOSS, 1.3, 1000, 0.95, True),
    (V_GPTOSS, 1e-3, 0, 0.9, False),
    (V_GPTOSS, 0.8, 0, 1e-6, False),
    (V_GPTOSS, 2.0, 0, 0.5, True),
    (1, 1.0, 0, 0.9, False),
    (1000, 0.9, 999, 0.99, True),
    (3001, 1.0, 0, 1.0, True),
]


@pytest.mark.parametrize("V,temp,top_k,top_p,ties", CASES)
def test_sample_rows_bit_exact(V, temp, top_k, top_p, ties):
    from flyai_amd import ops
    R = 4
    x = _logits(R, V, seed=V + top_k, ties=ties)
    xf = x.float().numpy()
    rng = np.random.default_rng(V)
    w = [S.weights(xf[r], temp, top_k, top_p) for r in range(R)]
    # drafts: the most likely token, a kept mid token, a dropped token (if any), none
    draft = []
    for r in range(R):
        kept = np.flatnonzero(w[r])
        dead = np.flatnonzero(w[r] == 0)
        choice = [int(np.argmax(w[r])), int(kept[len(kept) // 2]), int(dead[0]) if dead.size else 0, -1][r]
        draft.append(choice)
    u = rng.random(R)
    u[0] = 0.0
    xd = x.to(DEV)
    out = ops.sample_rows(xd, temp, top_k, top_p, draft=torch.tensor(draft, dtype=torch.int32, device=DEV),
                          u=torch.tensor(u, dtype=torch.float64, device=DEV),
                          want_p_draft=True, want_draw=True, want_probs=True)
    torch.cuda.synchronize()
    probs = out["probs"].cpu().numpy()
    for r in range(R):
        assert np.array_equal(probs[r], S.probs(w[r])), f"row {r}: probabilities differ"
        want_p = float(S.p_of(w[r], draft[r])) if draft[r] >= 0 else 0.0
        assert out["p_draft"][r].item() == want_p, f"row {r}: p_draft"
        assert out["draw"][r].item() == S.draw(w[r], u[r], exclude=draft[r]), f"row {r}: draw"


def test_sample_rows_greedy():
    from flyai_amd import ops
    x = _logits(6, V_GPTOSS, seed=3, ties=True)
    x[2, 7] = x[2].max() + 1
    x[2, 9] = x[2, 7]                       # a tie for the maximum: the first id
    xd = x.to(DEV)
    d = torch.tensor([0, 1, 7, 9, -1, 5], dtype=torch.int32, device=DEV)
    out = ops.sample_rows(xd, 0.0, draft=d, want_p_draft=True, want_draw=True, want_probs=True)
    torch.cuda.synchronize()
    want = [S.greedy(r) for r in x.float().numpy()]
    assert out["draw"].tolist() == want and want[2] == 7
    assert out["p_draft"].tolist() == [1.0 if a == b else 0.0 for a, b in zip(d.tolist(), want)]
    p = out["probs"].cpu()
    assert torch.equal(p.argmax(-1), torch.tensor(want)) and (p.sum(-1) == 1).all()


def test_sample_probs_bit_exact():
    from flyai_amd import ops
    x = _logits(1, V_GPTOSS, seed=9)[0].float().numpy()
    p = S.probs(S.weights(x, 0.9, 0, 0.97))
    pd = torch.from_numpy(p).to(DEV)
    for u in (0.0, 0.123456789, 0.5, 0.999999):
        assert ops.sample_probs(pd, u).item() == S.draw_probs(p, u)
    assert ops.sample_probs(torch.zeros(17, device=DEV), 0.4).item() == 0


@pytest.mark.parametrize("temp,top_k,top_p", [(0.8, 0, 0.95), (1.0, 20, 1.0), (0.0, 0, 1.0)])
def test_sampler_accept_matches_oracle(temp, top_k, top_p):
    """The kernel-backed Sampler and the oracle's accept, fed the same uniforms, return the same doctored
    list; drafts mix likely, unlikely and filtered-out tokens so both accept and reject paths run."""
    from flyai_amd.sampling import Sampler
    K = 4
    for trial in range(6):
        x = _logits(K + 1, V_GPTOSS, seed=100 + trial, ties=trial % 2 == 1)
        xf = x.float().numpy()
        w = [S.weights(xf[j], max(temp, 1e-6), top_k, top_p) for j in range(K)]
        draft = [int(np.argmax(w[j])) if (trial + j) % 3 else int(np.argsort(xf[j])[trial]) for j in range(K)]
        seed = 1000 + trial
        sm = Sampler(temp=temp, top_p=top_p, top_k=top_k, seed=seed, device=DEV)
        got = sm.accept(x.to(DEV), draft)
        uni = np.random.Generator(np.random.PCG64(seed))
        want = S.accept(list(xf), draft, temp, top_k, top_p, iter(lambda: float(uni.random()), None))
        assert got == want, f"trial {trial}: {got} vs {want}"


def test_sampler_api():
    from flyai_amd.sampling import Sampler
    x = _logits(1, 5000, seed=4)[0]
    sm = Sampler(temp=0.0, device=DEV)
    assert sm.greedy and sm.sample_logits(x.to(DEV)) == S.greedy(x.float().numpy())
    sm = Sampler(temp=0.9, top_p=0.9, seed=5, device=DEV)
    p = sm.dist(x.to(DEV))
    assert p.dtype == torch.float32 and p.shape == (5000,)
    assert np.array_equal(p.cpu().numpy(), S.probs(S.weights(x.float().numpy(), 0.9, 0, 0.9)))
    u = np.random.Generator(np.random.PCG64(5))
    assert sm.sample_logits(x.to(DEV)) == S.draw(S.weights(x.float().numpy(), 0.9, 0, 0.9), float(u.random()))
    assert sm.sample(p) == S.draw_probs(p.cpu().numpy(), float(u.random()))
    with pytest.raises(ValueError):
        sm.accept(_logits(2, 5000, seed=1).to(DEV), [1, 2])           # K=2 needs 3 rows
    with pytest.raises(TypeError):
        sm.dist(x.float().to(DEV))


def test_tail_tokens_over_the_lm_head():
    """tail_tokens on the stage parts (final norm + lm_head over the 201088-token vocabulary): greedy
    replies are bit-identical to the fused lm_head argmax; sampled replies (prefill, per-row, accept over
    K+1 rows) equal the oracle's for the same uniforms over the same bf16 logits."""
    from flyai_amd.sampling import Sampler, tail_tokens
    from flyai_amd.stage_parts import FinalNorm, LmHead
    H = 2880
    g = torch.Generator(device="cpu")
    g.manual_seed(21)
    parts = {"norm": FinalNorm((1 + 0.1 * torch.randn(H, generator=g)).to(DEV)),
             "lm_head": LmHead((torch.randn(V_GPTOSS, H, generator=g) * 0.03).to(torch.bfloat16).to(DEV))}
    h = (torch.randn(1, 5, H, generator=g) * 2).to(torch.bfloat16).to(DEV)
    logits = parts["lm_head"](parts["norm"](h))[0].float().cpu().numpy()
    greedy = Sampler(device=DEV)
    want = [S.greedy(r) for r in logits]
    assert tail_tokens(parts, h, greedy) == want
    assert tail_tokens(parts, h, greedy, draft=[want[0], 3, want[2], 4]) == want
    assert tail_tokens(parts, h, greedy, prefill=True) == [want[-1]]
    temp, top_k, top_p, seed = 0.9, 0, 0.95, 77
    ws = [S.weights(r, temp, top_k, top_p) for r in logits]

    def uni():
        u = np.random.Generator(np.random.PCG64(seed))
        return iter(lambda: float(u.random()), None)
    sm = lambda: Sampler(temp=temp, top_p=top_p, top_k=top_k, seed=seed, device=DEV)  # noqa: E731
    u = uni()
    assert tail_tokens(parts, h, sm(), prefill=True) == [S.draw(ws[-1], next(u))]
    u = uni()
    assert tail_tokens(parts, h, sm()) == [S.draw(w, next(u)) for w in ws]
    draft = [int(np.argmax(ws[0])), int(np.argmax(ws[1])), 5, 6]
    assert tail_tokens(parts, h, sm(), draft=draft) == S.accept(list(logits), draft, temp, top_k, top_p, uni())


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_sample_rows_non_finite_logits_and_out_of_range_uniforms(bad):
    """A row with a NaN or infinite logit: the kernel's weights and draw equal the oracle's (every weight
    0 for NaN/+inf, so the draw is id 0, inside the vocabulary); uniforms outside [0, 1) are held to its
    ends, so they draw what 0 and the largest double below 1 draw."""
    from flyai_amd import ops
    V = 3001
    x = _logits(4, V, seed=5)
    x[0, 17] = bad
    x[1, 0] = bad
    x[1, V - 1] = bad
    xf = x.float().numpy()
    u = np.array([0.3, 0.6, -0.25, 1.5])
    u_eff = np.array([0.3, 0.6, 0.0, np.nextafter(1.0, 0.0)])
    out = ops.sample_rows(x.to(DEV), 0.9, 0, 1.0, draft=torch.tensor([17, -1, 5, 9], dtype=torch.int32, device=DEV),
                          u=torch.tensor(u, dtype=torch.float64, device=DEV), want_draw=True, want_probs=True)
    draw = out["draw"].cpu().numpy()
    probs = out["probs"].cpu().numpy()
    for r, d in enumerate([17, -1, 5, 9]):
        w = S.weights(xf[r], 0.9)
        want = S.draw(w, float(u_eff[r]), exclude=d)
        assert 0 <= draw[r] < V and draw[r] == want, (r, draw[r], want)
        if w.sum(dtype=np.uint64) > 0:
            assert np.array_equal(probs[r], S.probs(w)), r
        else:
            assert not probs[r].any(), r


CHUNKED = [  # (rows, V, temp, top_k, top_p): ids per chunk 4096 up to 262,144 ids, then a multiple of 2048
    (3, 4096, 0.8, 0, 0.9), (3, 4097, 1.0, 40, 1.0), (2, 8191, 1.1, 40, 0.9), (2, 16392, 0.7, 3, 0.5),
    (5, V_GPTOSS, 1.2, 0, 0.95), (2, V_GPTOSS, 0.9, 200, 0.9), (2, 262153, 0.9, 0, 0.97), (300, 4104, 0.9, 5, 0.9),
]


@pytest.mark.parametrize("R,V,temp,top_k,top_p", CHUNKED)
def test_split_rows_equal_one_workgroup_rows(R, V, temp, top_k, top_p):
    """The rows split over workgroups (a workspace) against one workgroup a row (no workspace), bit for bit:
    ragged last chunks, odd row lengths (no vector loads), ties across chunks at the top-k and top-p
    boundaries, drafted tokens inside the ties, -inf masks, and rows for the general path (NaN, +inf,
    quotients near the denormals, an overflowing temperature)."""
    import ctypes as C
    from flyai_amd import _lib, ops
    x = _logits(R, V, seed=V + R, ties=True)
    if R >= 2:
        x[1, :V // 2] = float("-inf")                 # masked vocabulary
        x[1, V // 3] = 1e-36                           # a quotient near the denormals
    if R >= 3:
        x[2] = 1.25                                    # one tie over the whole row
    if R >= 5:
        x[3, 11], x[4, 7], x[4, 8] = float("nan"), 3e38, float("-inf")
    g = torch.Generator().manual_seed(V)
    d = torch.randint(-1, V, (R,), generator=g, dtype=torch.int32)
    d[0] = int(x[0].float().argmax())
    u = torch.rand(R, generator=g, dtype=torch.float64)
    xd, dd, ud = x.to(DEV), d.to(DEV), u.to(DEV)
    for t in (temp, 1e-30, 0.0):
        got = ops.sample_rows(xd, t, top_k, top_p, draft=dd, u=ud, want_p_draft=True, want_draw=True, want_probs=True)
        want = {n: torch.empty_like(v) for n, v in got.items()}
        p = lambda v: C.c_void_p(v.data_ptr())  # noqa: E731
        _lib.check(_lib.lib().flyai_sample_rows(p(xd), R, V, t, top_k, top_p, p(dd), p(ud), p(want["p_draft"]),
                                                p(want["draw"]), p(want["probs"]),
                                                C.c_void_p(torch.cuda.current_stream().cuda_stream)))
        torch.cuda.synchronize()
        for n in got:
            assert torch.equal(got[n], want[n]), (t, n, (got[n] != want[n]).nonzero()[:4].tolist())


@pytest.mark.parametrize("R", [1, 255, 256, 257])
@pytest.mark.parametrize("V", [1, 12288, 12289, 16384, 16385])
def test_greedy_rows_on_both_sides_of_the_split(R, V):
    """Greedy rows of few ids are one workgroup each, longer ones are split; 256 rows move the line."""
    from flyai_amd import ops
    x = _logits(R, V, seed=V + R, ties=True)
    want = x.float().numpy().argmax(-1)
    d = torch.from_numpy(np.where(np.arange(R) % 2 == 0, want, V - 1).astype(np.int32))
    out = ops.sample_rows(x.to(DEV), 0.0, draft=d.to(DEV), want_p_draft=True, want_draw=True, want_probs=True)
    assert np.array_equal(out["draw"].cpu().numpy(), want)
    assert np.array_equal(out["p_draft"].cpu().numpy(), (d.numpy() == want).astype(np.float32))
    p = out["probs"].cpu().numpy()
    assert (p[np.arange(R), want] == 1).all() and (p.sum(-1) == 1).all()
