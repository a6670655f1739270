"""fp32 at d <= 64: the forward's score and P V products are split bf16 products.
Against the oracle at the GPU's tau (1e-5, the fp32 tolerance of the other
parity tests), with operands whose split matters: wide magnitudes, values
past bf16's largest; and values below 2^-109, infinities and NaN (fp32
products from there on, or for that tile).  One and two wave groups per
block, few and many blocks, ragged lengths, a head dimension that is not a
whole split step.  Rows whose best scores tie at tau."""
import numpy as np
import pytest
import torch

import splash_attention as sa
from oracle import oracle as orc
from tests._util import assert_close, causal_idx, make_inputs, np32, oracle_at_gpu_tau

pytestmark = pytest.mark.gpu

CASES = [
    ("one_row", 1, 1, 1, 65, 64, 64),
    ("two_groups_odd", 1, 2, 70, 64 * 5 + 3, 64, 64),
    ("d40", 1, 2, 129, 130, 40, 64),
    ("d36_m32", 1, 2, 129, 200, 36, 32),
    ("one_group", 3, 16, 400, 400, 64, 64),
]


@pytest.mark.parametrize("alpha", [1.5, 1.25, 1.7, 2.0])
@pytest.mark.parametrize("kind", ["normal", "wide", "huge", "tiny", "nonfinite", "low_tile", "low_row"])
@pytest.mark.parametrize("name,B,H,NQ,NK,d,bm", CASES, ids=[c[0] for c in CASES])
def test_split_forward(dev, name, B, H, NQ, NK, d, bm, kind, alpha):
    print(f"[split] {name} {kind} B{B} H{H} NQ{NQ} NK{NK} d{d} block_m {bm} alpha {alpha}", flush=True)
    BH, k = B * H, 8
    Q, K, V, dO = make_inputs(B, H, NQ, NK, d, seed=NQ + d)
    if kind == "wide":  # rows over 2^-40 .. 2^40, scores of order one
        s = torch.exp2(torch.randint(-40, 41, (d,), generator=torch.Generator().manual_seed(1)).float())
        Q, K = Q * s, K / s
        V = V * torch.exp2(torch.randint(-30, 31, (d,), generator=torch.Generator().manual_seed(2)).float())
    elif kind == "huge":
        K[:, :, NK // 2, 0] = 3.4e38   # past bf16's largest value
        Q[..., 0] *= 1e-38             # and values below the split's range
    elif kind == "tiny":
        V *= 1e-37
    elif kind == "low_tile":  # one value below 2^-109 late in the lists: split products until there
        K[:, ::2, NK // 2, 5] = 1e-35
        V[:, 1::2, 2 * NK // 3, 7] = -1e-38
    elif kind == "low_row":   # and in one row of Q
        Q[:, :, NQ // 2, 9] = 1e-36
    elif kind == "nonfinite":
        K[:, :, NK // 2, 0] = float("inf")
        K[:, :, NK // 3, 1] = float("nan")
        Q[:, :, NQ // 2, 2] = float("-inf")
    qidx, kidx = causal_idx(BH, NQ) + (NK - NQ), causal_idx(BH, NK)
    args = [t.to(dev) for t in (Q, K, V)]
    q, kk, v, qi, ki = sa.ops.check_inputs(*args, qidx.to(dev), kidx.to(dev))
    out, st = sa.ops.splash_forward(q, kk, v, qi, ki, alpha, k, d ** -0.5, block_m=bm)
    torch.cuda.synchronize()
    heads = slice(0, min(BH, 3))
    f = lambda t: np32(t)[heads]
    own, fw, _ = oracle_at_gpu_tau(f(Q), f(K), f(V), f(dO), qidx[heads].numpy(), kidx[heads].numpy(),
                                   alpha, d ** -0.5, k, st.taus.cpu().numpy()[heads], 0, block_m=bm)
    np.testing.assert_array_equal(st.mask.cpu().numpy()[heads], own.mask)
    got = np32(out)[heads]
    # Relative to the column's largest |V|: an output is a convex combination
    # of V's column, so rounding of scores, weights and sums moves it by at
    # most that bound times a few 1e-7, however much the column cancels; and
    # (kind "tiny") each of the row's products rounds to a multiple of 2^-149
    # before the division by the row sum.
    scale = np.abs(f(V)).max(axis=(0, 1)).astype(np.float64)
    tol = 1e-5 + NK * 2.0 ** -150 / (fw.norms[..., None] + 1e-8) / scale
    assert (np.abs(got / scale - fw.out / scale) <= tol).all()
    assert_close("norms", st.norms.cpu().numpy()[heads], fw.norms, 1e-5)


@pytest.mark.parametrize("alpha", [1.25, 1.5, 2.0])
@pytest.mark.parametrize("N", [1024, 4096])
def test_split_error_no_larger_than_fp32_products(dev, N, alpha):
    """2-norm error of the output against float64, split and with the fp32
    products of the same call with four zero columns appended (above d = 64
    nothing is split), both at the threshold that the score pass found."""
    B, H, d, k = 1, 4, 64, 8
    Q, K, V, dO = make_inputs(B, H, N, N, d, seed=5)
    idx = causal_idx(B * H, N)
    q, kk, v, i = (t.to(dev) for t in (Q, K, V, idx))
    outs = []
    for pad in (0, 4):
        p = [torch.nn.functional.pad(t, (0, pad)) for t in (q, kk, v)]
        o, st = sa.ops.splash_forward(*p, i, i, alpha, k, 0.125)
        outs.append(np32(o[..., :d]))
    f = lambda t: t.reshape(H, N, -1).numpy()
    ref = orc.forward(f(Q), f(K), f(V), idx.numpy(), idx.numpy(), alpha, 0.125, k, precision="f64",
                      taus_in=st.taus.cpu().numpy().reshape(H, N)).out
    e, e32 = (np.linalg.norm(o - ref) / np.linalg.norm(ref) for o in outs)
    print(f"[split] error against float64 N={N} alpha={alpha}: {e:.2e}, fp32 products {e32:.2e}", flush=True)
    assert e <= 1.02 * e32


@pytest.mark.parametrize("heads", [2, 129])
@pytest.mark.parametrize("alpha", [1.25, 1.5, 1.7, 2.0, 2.5, 3.0])
@pytest.mark.parametrize("k,bm", [(1, 64), (2, 64), (8, 64), (8, 32), (128, 64)])
def test_rows_whose_best_keys_tie(dev, k, bm, alpha, heads):
    """Keys repeated more than k times, so that a row's k best scores are equal
    (below the clamp, inexact in fp32) and tau can end within a rounding of
    them: the forward has to see the very scores that tau came from.  Against
    the same call with four zero columns appended (above d = 64 nothing is
    split, and zeros change no sum): rows without weight are the same ones,
    support masks bit-equal.  One and two wave groups per block (heads 129
    and 2).  Each row's p, as both backward passes form it, sums to
    norm / (norm + 1e-8)."""
    N, d, scale = 64 * 3 + 6, 64, 0.125
    print(f"[split] ties k={k} bm={bm} alpha={alpha} heads={heads}", flush=True)
    g = torch.Generator().manual_seed(int(100 * alpha) + k)
    Q, V = (torch.randn(1, heads, N, d, generator=g) for _ in range(2))
    # one key vector in a third of the heads, two or three in the others
    which = torch.randint(0, 3, (1, heads, N), generator=g) % (torch.arange(heads)[None, :, None] % 3 + 1)
    K = torch.gather(torch.randn(1, heads, 3, d, generator=g), 2, which[..., None].expand(-1, -1, -1, d))
    qidx = torch.full((heads, N), N - 1, dtype=torch.int32, device=dev)
    kidx = causal_idx(heads, N).to(dev)
    q, kk, v = (t.to(dev) for t in (Q, K, V))
    got = []
    for pad in (0, 4):
        p = [torch.nn.functional.pad(t, (0, pad)) for t in (q, kk, v)]
        got.append(sa.ops.splash_forward(*p, qidx, kidx, alpha, k, scale, block_m=bm))
    (out, st), (want, ref) = got
    assert torch.equal(st.taus, ref.taus)
    if bm == 64:  # the lists that index the masks are the state's
        for h in range(heads):
            n = int(st.q_ptr[h, -1])
            masks = [x.sup_mask.view(torch.uint8).reshape(heads, -1, 512)[h, :n] for x in (st, ref)]
            assert torch.equal(*masks)
    assert bool((ref.norms < 1e-3).any())  # the draw has such rows
    assert torch.equal(st.norms == 0, ref.norms == 0)
    # Rows of split scores have u > 1/16, and u >= k^-1/2 at alpha = 1.5
    # (k = 128: 0.09): u's rounding moves a weight by at most a / u = 23 times
    # that, and (alpha - 1) times a sum of 64 products rounds by 1e-6 at most
    # in these draws.
    tol = 2.4e-5
    torch.testing.assert_close(st.norms, ref.norms, rtol=tol, atol=0)
    torch.testing.assert_close(out, want[..., :d], rtol=0, atol=tol * float(v.abs().max()))
    # Sums of p: dO with row i of a 64-row block marking column i.  The support
    # passes gather their own dot products: there rows with weights of a
    # score's rounding are left out, and the others' k equal weights, with
    # u = k^-(alpha - 1), move by a / u times that rounding.
    wide = max(tol, 1e-6 * k ** (alpha - 1) / (alpha - 1))
    eye = torch.eye(d, device=dev).repeat(4, 1)[:N].expand(1, heads, N, d)
    norms = st.norms.view(heads, N)
    for passes in ("support", "tiles"):
        if passes == "tiles":
            st.sup_mask = None
        for b in range(4):
            rows = slice(64 * b, min(64 * b + 64, N))
            dO = torch.zeros_like(eye)
            dO[:, :, rows] = eye[:, :, rows]
            _, _, dV = sa.ops.splash_backward(q, kk, v, qidx, kidx, out, dO, st, alpha, k, scale)
            sums, n = dV.sum(2)[0, :, :rows.stop - rows.start], norms[:, rows]
            on, at = ((n == 0) | (n > 0.5), wide) if passes == "support" else (n >= 0, tol)
            torch.testing.assert_close(sums[on], (n / (n + 1e-8))[on], rtol=0, atol=at)
