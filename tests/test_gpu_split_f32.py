"""fp32 at d <= 64: the forward's score and P V products are split bf16 products.
Against the oracle at the GPU's tau (1e-5, the fp32 tolerance of the other
parity tests), with operands whose split matters: wide magnitudes, values
past bf16's largest; and values below 2^-109, infinities and NaN (the tiles
that hold those run again with fp32 products).  One and two wave groups per block, few and many
blocks, ragged lengths, a head dimension that is not a whole split step."""
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


@pytest.mark.parametrize("kind", ["normal", "wide", "huge", "tiny", "nonfinite"])
@pytest.mark.parametrize("name,B,H,NQ,NK,d,bm", CASES, ids=[c[0] for c in CASES])
def test_split_forward(dev, name, B, H, NQ, NK, d, bm, kind):
    print(f"[split] {name} {kind} B{B} H{H} NQ{NQ} NK{NK} d{d} block_m {bm}", flush=True)
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
    elif kind == "nonfinite":
        K[:, :, NK // 2, 0] = float("inf")
        K[:, :, NK // 3, 1] = float("nan")
        Q[:, :, NQ // 2, 2] = float("-inf")
    qidx, kidx = causal_idx(BH, NQ) + (NK - NQ), causal_idx(BH, NK)
    args = [t.to(dev) for t in (Q, K, V)]
    q, kk, v, qi, ki = sa.ops.check_inputs(*args, qidx.to(dev), kidx.to(dev))
    out, st = sa.ops.splash_forward(q, kk, v, qi, ki, 1.5, k, d ** -0.5, block_m=bm)
    torch.cuda.synchronize()
    heads = slice(0, min(BH, 3))
    f = lambda t: np32(t)[heads]
    own, fw, _ = oracle_at_gpu_tau(f(Q), f(K), f(V), f(dO), qidx[heads].numpy(), kidx[heads].numpy(),
                                   1.5, d ** -0.5, k, st.taus.cpu().numpy()[heads], 0, block_m=bm)
    np.testing.assert_array_equal(st.mask.cpu().numpy()[heads], own.mask)
    got = np32(out)[heads]
    # Relative to the column's largest |V|: an output is a convex combination
    # of V's column, so rounding of scores, weights and sums moves it by at
    # most that bound times a few 1e-7, however much the column cancels.
    scale = np.abs(f(V)).max(axis=(0, 1))
    np.testing.assert_allclose(got / scale, fw.out / scale, rtol=0, atol=1e-5)
    assert_close("norms", st.norms.cpu().numpy()[heads], fw.norms, 1e-5)


def test_split_error_no_larger_than_fp32_products(dev):
    """2-norm error of the output against float64: below 1.5e-6 (fp32 matrix
    products measured 0.7 to 1.2e-6 on the same inputs)."""
    B, H, N, d = 1, 4, 1024, 64
    print("[split] error against float64", flush=True)
    Q, K, V, _ = make_inputs(B, H, N, N, d, seed=5)
    idx = causal_idx(B * H, N)
    out = sa.splash_attention(*(t.to(dev) for t in (Q, K, V)), idx.to(dev), idx.to(dev), 1.5, 8, 0.125)
    q, k, v = (t.reshape(H, N, d).numpy() for t in (Q, K, V))
    ref = orc.forward(q, k, v, idx.numpy(), idx.numpy(), 1.5, 0.125, 8, precision="f64").out
    e = np.linalg.norm(np32(out) - ref) / np.linalg.norm(ref)
    print(f"[split] {e:.2e}", flush=True)
    assert e < 1.5e-6
