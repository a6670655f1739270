"""Selection stage on the GPU vs the CPU oracle, given identical scores.

Top-k indices and values, block masks and CSR lists must be bit-exact; tau
must be bit-exact too (same fp32 recurrence, same rounding conventions).
Reference: adasplashattention.cu:35-242.
"""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from tests._util import causal_idx

pytestmark = pytest.mark.gpu


def _run(dev, S, vis_qidx, vis_kidx, k, alpha, B, H, with_topk=True):
    import splash_attention as sa

    BH, NQ, NK = S.shape
    st = sa.ops.select_from_scores(torch.from_numpy(S).to(dev), vis_qidx.to(dev),
                                   vis_kidx.to(dev), alpha, k, batch=B, heads=H,
                                   with_topk=with_topk)
    torch.cuda.synchronize()
    return st


def _oracle(S, qidx, kidx, k, alpha):
    qi = qidx.numpy()
    ki = kidx.numpy()
    vis = (ki[:, None, :] <= qi[:, :, None]).astype(np.uint8)
    Sc = np.clip(S, -10, 10).astype(np.float32)
    sel = orc.select(Sc, vis, k, alpha)
    c = orc.csr(sel.mask)
    return sel, c


def _compare(st, sel, c):
    if st.topk_idx is not None:
        np.testing.assert_array_equal(st.topk_idx.cpu().numpy(), sel.topk_idx)
        np.testing.assert_array_equal(st.topk_val.cpu().numpy(), sel.topk_val)
    np.testing.assert_array_equal(st.mask.cpu().numpy(), sel.mask)
    np.testing.assert_array_equal(st.q_ptr.cpu().numpy(), c.q_ptr)
    np.testing.assert_array_equal(st.q_list.cpu().numpy(), c.q_list)
    np.testing.assert_array_equal(st.k_ptr.cpu().numpy(), c.k_ptr)
    np.testing.assert_array_equal(st.k_list.cpu().numpy(), c.k_list)
    taus = st.taus.cpu().numpy()
    np.testing.assert_array_equal(taus.view(np.uint32), sel.taus.astype(np.float32).view(np.uint32))


CASES = [
    # (name, B, H, NQ, NK, k, alpha, kind)
    ("causal_c1", 1, 2, 256, 256, 8, 1.5, "normal"),
    ("causal_k32", 1, 2, 320, 320, 32, 1.5, "normal"),
    ("sparsemax_k64", 1, 1, 256, 256, 64, 2.0, "normal"),
    ("alpha125_k128", 1, 1, 192, 192, 128, 1.25, "normal"),
    ("ties_quantised", 2, 1, 200, 200, 16, 1.5, "ties"),
    ("clamp_saturated", 1, 1, 128, 256, 8, 2.0, "saturated"),
    ("ragged_nq_ne_nk", 1, 3, 100, 333, 8, 1.5, "normal"),
    ("alpha_general", 1, 1, 130, 130, 8, 1.7, "normal"),
]


# with_topk=False is the path asa_forward takes: values sorted alone, the
# mask from the candidates scoring above the k-th value plus the
# lowest-index ties (the "ties" and "saturated" cases split tie runs at the
# k-th value)
@pytest.mark.parametrize("with_topk", [True, False], ids=["topk", "values"])
@pytest.mark.parametrize("name,B,H,NQ,NK,k,alpha,kind", CASES, ids=[c[0] for c in CASES])
def test_select_bit_exact(dev, name, B, H, NQ, NK, k, alpha, kind, with_topk):
    print(f"[select] {name} B={B} H={H} NQ={NQ} NK={NK} k={k} alpha={alpha} "
          f"topk={with_topk}", flush=True)
    rng = np.random.default_rng(hash(name) % 2**32)
    BH = B * H
    if kind == "normal":
        S = rng.normal(size=(BH, NQ, NK)).astype(np.float32)
    elif kind == "ties":
        S = (np.round(rng.normal(size=(BH, NQ, NK)) * 2) / 2).astype(np.float32)
    else:
        S = (rng.normal(size=(BH, NQ, NK)) * 30).astype(np.float32)
    qidx = causal_idx(BH, NQ) + (NK - NQ if NK > NQ else 0)
    kidx = causal_idx(BH, NK)
    st = _run(dev, S, qidx, kidx, k, alpha, B, H, with_topk)
    sel, c = _oracle(S, qidx, kidx, k, alpha)
    _compare(st, sel, c)


def test_select_noncausal_and_scattered_positions(dev):
    """Arbitrary (non-monotone) positions: visibility is K_idx <= Q_idx."""
    rng = np.random.default_rng(7)
    BH, NQ, NK, k = 2, 150, 260, 12
    S = rng.normal(size=(BH, NQ, NK)).astype(np.float32)
    qidx = torch.from_numpy(rng.integers(0, 300, size=(BH, NQ)).astype(np.int32))
    kidx = torch.from_numpy(rng.integers(0, 300, size=(BH, NK)).astype(np.int32))
    print("[select] scattered positions", flush=True)
    st = _run(dev, S, qidx, kidx, k, 1.5, 1, 2)
    sel, c = _oracle(S, qidx, kidx, k, 1.5)
    _compare(st, sel, c)



def _rising_scores(N, k):
    """Scores that make the score pass run many overflow rounds: in every
    64-key tile the keys at offsets below (k - 1) // R (R = 2 class maxima
    per tile offset for k <= 32, else 4: the tile ordinal mod R) score
    2 + 1e-4 j, rising with the key index j, and all other keys
    -1 - 1e-4 j.  Those offsets make fewer than k of the 64 R classes, so
    the floor falls among the low keys and every high key is a candidate;
    they arrive in ascending tile order, worst first, so each round's
    stored candidates give a threshold that only cap - k of them fail."""
    R = 2 if k <= 32 else 4
    nh = (k - 1) // R
    j = np.arange(N)
    row = np.where(j % 64 < nh, 2 + 1e-4 * j, -1 - 1e-4 * j).astype(np.float32)
    return np.broadcast_to(row, (1, N, N)).copy()


@pytest.mark.parametrize("with_topk", [True, False], ids=["topk", "values"])
@pytest.mark.parametrize("k,min_rounds", [(8, 2), (32, 4), (64, 4)])
def test_select_overflow_rounds_bit_exact(dev, k, min_rounds, with_topk):
    """Rows with many more candidates than the per-row capacity (k + 32)
    run several overflow rounds; the result must still be the oracle's,
    bit for bit, and the status word must report the rounds (without the
    round-bound flag)."""
    import splash_attention as sa

    N = 2048
    S = _rising_scores(N, k)
    idx = causal_idx(1, N)
    print(f"[select] overflow rounds N={N} k={k} topk={with_topk}", flush=True)
    st = _run(dev, S, idx, idx, k, 1.5, 1, 1, with_topk)
    rounds = st.overflow_rounds()
    print(f"[select] overflow rounds N={N} k={k}: {rounds} rounds", flush=True)
    assert not st.status_word() & sa._lib.STATUS_SELECT_ROUNDS
    assert rounds >= min_rounds, rounds
    sel, c = _oracle(S, idx, idx, k, 1.5)
    _compare(st, sel, c)


@pytest.mark.parametrize("with_topk", [True, False], ids=["topk", "values"])
@pytest.mark.parametrize("k", [1, 8, 64, 100, 128])
def test_select_ties_beyond_the_list_bit_exact(dev, k, with_topk):
    """Rows whose candidates tie at the score clamp in numbers around and far
    beyond the list's capacity (a row is then done without another sweep
    when every left-out tie comes after the kept ones), and, in the last
    third of the rows, tied candidates below better ones that arrive late
    (another sweep must follow).  One oracle, bit for bit."""
    N = 1100
    rng = np.random.default_rng(k)
    S = rng.normal(size=(1, N, N)).astype(np.float32)
    cap = k + max(32, k * 3 // 4)
    for i in range(N):
        m = rng.integers(max(1, cap - 8), cap + 9) if i % 2 else N // 2
        at = rng.choice(N, size=min(N, m), replace=False)
        if i < 2 * N // 3:
            S[0, i, at] = 12.0 + rng.random(at.size)    # clamped to 10
        else:
            S[0, i, at] = 5.0
            S[0, i, -min(N, 2 * k):] = 6.0 + 0.25 * rng.integers(0, 3, size=min(N, 2 * k))
    qidx = torch.full((1, N), N - 1, dtype=torch.int32)
    kidx = causal_idx(1, N)
    print(f"[select] ties beyond the list k={k} topk={with_topk}", flush=True)
    st = _run(dev, S, qidx, kidx, k, 1.5, 1, 1, with_topk)
    sel, c = _oracle(S, qidx, kidx, k, 1.5)
    _compare(st, sel, c)


@pytest.mark.parametrize("layout", ["dense", "rows"])
@pytest.mark.parametrize("k", [1, 8, 9, 16, 17, 32, 42, 43, 64, 65, 128])
@pytest.mark.parametrize("d,dtype", [(64, torch.bfloat16), (128, torch.bfloat16), (128, torch.float16),
                                     (96, torch.bfloat16), (64, torch.float32), (128, torch.float32)])
def test_score_pass_variants(dev, d, dtype, k, layout):
    """Every variant of the score pass (4 or 8 waves per block, LDS rings or
    register loads, contiguous or strided K) on visible lists of more than
    128 tiles (two refills of the per-lane list window, an odd number of
    tiles, a ragged last one) and on short ones: top-k, mask and tau against
    the oracle, on scores that are exact in fp32."""
    import splash_attention as sa

    B, H, NQ, NK, scale = 1, 2, 75, 64 * 130 + 5, 0.125
    print(f"[select] variants d={d} {dtype} k={k} {layout}", flush=True)
    g = torch.Generator().manual_seed(100 * d + k)
    Q, K = ((torch.round(torch.randn(B, H, n, d, generator=g) * 16) / 16).clamp(-4, 4)
            for n in (NQ, NK))
    K[:, :, 3000:3300] = K[:, :, 5000:5300]  # ties across tiles
    kidx = causal_idx(B * H, NK)
    qidx = torch.randint(40, NK, (B * H, NQ), generator=g).to(torch.int32)
    qidx[:, :64] = qidx[:, :64].clamp(min=64 * 129)  # the first block sees every tile
    q, kk = Q.to(dtype).to(dev), K.to(dtype).to(dev)
    if layout == "rows":
        kk = torch.cat((kk, kk), -1)[..., :d]  # rows 2 d elements apart
    got = [sa.ops.splash_forward(q, kk, kk, qidx.to(dev), kidx.to(dev), 1.5, k, scale,
                                 with_topk=t, with_support=False)[1] for t in (True, False)]
    torch.cuda.synchronize()
    S, vis = orc.scores(Q.reshape(B * H, NQ, d).numpy(), K.reshape(B * H, NK, d).numpy(),
                        qidx.numpy(), kidx.numpy(), scale)
    sel = orc.select(S, vis, k, 1.5)
    np.testing.assert_array_equal(got[0].topk_idx.cpu().numpy(), sel.topk_idx)
    np.testing.assert_array_equal(got[0].topk_val.cpu().numpy(), sel.topk_val)
    for st in got:
        np.testing.assert_array_equal(st.mask.cpu().numpy(), sel.mask)
        np.testing.assert_array_equal(st.taus.cpu().numpy(), sel.taus)


@pytest.mark.parametrize("d,dtype,k", [(128, torch.bfloat16, 32), (128, torch.float16, 64),
                                       (64, torch.bfloat16, 128), (64, torch.float32, 8)])
def test_captured_variants(dev, d, dtype, k):
    """The variants with more than 64 KiB of LDS (and the two-group fp32
    forward) captured in a graph: every replay on new inputs, with eager work
    between, bit-equal to the eager call."""
    import splash_attention as sa

    B, H, N = 1, 2, 700
    print(f"[select] captured d={d} {dtype} k={k}", flush=True)
    idx = causal_idx(B * H, N).to(dev)
    g = torch.Generator(device=dev).manual_seed(d + k)
    new = lambda: torch.randn(B, H, N, d, generator=g, device=dev).to(dtype)
    bufs = [new() for _ in range(3)]
    call = lambda q, kk, v: sa.splash_attention(q, kk, v, idx, idx, 1.5, k)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        call(*bufs)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = call(*bufs)
    for _ in range(3):
        fresh = [new() for _ in range(3)]
        want = call(*fresh)
        for b, f in zip(bufs, fresh):
            b.copy_(f)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


@pytest.mark.parametrize("heads", [128, 129])
@pytest.mark.parametrize("NK", [64 * 9 + 5, 64 * 130 + 5])
@pytest.mark.parametrize("d,dtype,k", [(64, torch.bfloat16, 8), (64, torch.float16, 64),
                                       (128, torch.bfloat16, 32), (96, torch.bfloat16, 16),
                                       (64, torch.float32, 1), (64, torch.float32, 64)])
def test_score_pass_by_block_count(dev, d, dtype, k, NK, heads):
    """The score pass's waves per block change where the blocks exceed the
    compute units (two blocks per head here, 256 units): both sides on short
    and long lists against the oracle, on scores that are exact in fp32.
    Q and K are one head's, repeated, with other positions per head."""
    import splash_attention as sa

    NQ, scale = 75, 0.125
    print(f"[select] blocks d={d} {dtype} k={k} NK={NK} heads={heads}", flush=True)
    g = torch.Generator().manual_seed(1000 * d + k)
    Q, K = ((torch.round(torch.randn(1, 1, n, d, generator=g) * 16) / 16).clamp(-4, 4)
            for n in (NQ, NK))
    kidx = causal_idx(heads, NK)
    qidx = torch.randint(40, NK, (1, NQ), generator=g).to(torch.int32).repeat(heads, 1)
    qidx[1::2] = NK - 1  # odd heads see every key
    q, kk = (x.to(dtype).to(dev).expand(1, heads, -1, -1) for x in (Q, K))
    got = [sa.ops.splash_forward(q, kk, kk, qidx.to(dev), kidx.to(dev), 1.5, k, scale,
                                 with_topk=t, with_support=False)[1] for t in (True, False)]
    torch.cuda.synchronize()
    S, vis = orc.scores(Q.repeat(1, 2, 1, 1)[0].numpy(), K.repeat(1, 2, 1, 1)[0].numpy(),
                        qidx[:2].numpy(), kidx[:2].numpy(), scale)
    sel = orc.select(S, vis, k, 1.5)
    for name, sts in (("topk_idx", got[:1]), ("topk_val", got[:1]), ("mask", got), ("taus", got)):
        for st in sts:
            x, want = getattr(st, name).cpu().numpy(), getattr(sel, name)
            for h in range(heads):
                np.testing.assert_array_equal(x[h], want[h % 2])


@pytest.mark.parametrize("d,dtype,k,heads", [
    (64, torch.bfloat16, 32, 3), (64, torch.bfloat16, 32, 257), (64, torch.float16, 128, 3),
    (128, torch.bfloat16, 64, 3), (128, torch.float16, 32, 257), (80, torch.bfloat16, 64, 257),
    (64, torch.float32, 64, 3), (64, torch.float32, 8, 257)])
def test_operand_overflow_rounds(dev, d, dtype, k, heads):
    """Overflow rounds with the scores formed from Q and K (rings or register
    loads, four or eight waves per block, 3 or 257 blocks): head 0 has
    _rising_scores' pattern, head 1 half of its keys tied at the score clamp
    and the others just below, head 2 both.  Against the oracle, on scores
    that are exact in fp32."""
    import splash_attention as sa

    NQ, NK, scale = 64, 2048 + 37, 0.125
    print(f"[select] operand overflow d={d} {dtype} k={k} heads={heads}", flush=True)
    j = np.arange(NK)
    high = j % 64 < (k - 1) // (2 if k <= 64 else 4)
    rng = np.random.default_rng(d + k)
    raw = [np.where(high, 16 + j / 128, -8 - j / 128),       # 2 .. 4.1 after scaling
           np.where(rng.random(NK) < 0.5, 96, 64 + j / 128),  # 10 (clamped) or 8 ..
           np.where(high, 48 + j / 64, np.where(rng.random(NK) < 0.5, 40, -8))]
    # raw = its floor + a multiple of 1/128, each exact in 16 bits
    K = np.zeros((1, 3, NK, d), np.float32)
    for h in range(3):
        K[0, h, :, 0], K[0, h, :, d - 1] = np.floor(raw[h]), raw[h] - np.floor(raw[h])
    Q = np.zeros((1, 3, NQ, d), np.float32)
    Q[..., 0] = Q[..., d - 1] = 1.0
    kidx = causal_idx(heads, NK)
    qidx = (NK - 1 - 3 * torch.arange(NQ, dtype=torch.int32)).expand(heads, NQ).contiguous()
    rep = torch.arange(heads) % 3
    q, kk = (torch.from_numpy(x)[:, rep].contiguous().to(dtype).to(dev) for x in (Q, K))
    got = [sa.ops.splash_forward(q, kk, kk, qidx.to(dev), kidx.to(dev), 1.5, k, scale,
                                 with_topk=t, with_support=False)[1] for t in (True, False)]
    rounds = [st.overflow_rounds() for st in got]
    print(f"[select] operand overflow: {rounds} rounds", flush=True)
    S, vis = orc.scores(Q[0], K[0], qidx[:3].numpy(), kidx[:3].numpy(), scale)
    sel = orc.select(S, vis, k, 1.5)
    for st, n in zip(got, rounds):
        assert n >= 1 and not st.status_word() & sa._lib.STATUS_SELECT_ROUNDS
        for name in ("mask", "taus") + (("topk_idx", "topk_val") if st.topk_idx is not None else ()):
            x, want = getattr(st, name).cpu().numpy(), getattr(sel, name)
            for h in range(heads):
                np.testing.assert_array_equal(x[h], want[h % 3])
