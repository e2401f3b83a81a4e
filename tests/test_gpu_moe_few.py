"""The expert FFN for few tokens per expert (dq_moe_few.hip) against the oracle's expert FFN: both form the same
integer sums, so gate, up and down differ by float summation order only (about 1e-6 relative). silu(gate) * up is
quantized per 256 in between; where that order moves a value across a rounding tie, one of the n_ff inputs of the down
projection changes by a step, 1/127 of its block's maximum (about 0.03 of the rms): 0.03 / sqrt(n_ff) of a token's
output, 2e-3 for one step at n_ff = 256 and less above."""
import numpy as np
import pytest
import torch

from desireeia_amd import ops, synth

pytestmark = pytest.mark.gpu
Q4K = synth.Q4_K
TOL = 2e-3


def build(gpu, n_exp, E, F, seed):
    ws = [synth.gen_weights(Q4K, n_exp * r, c, seed + i) for i, (r, c) in enumerate(((F, E), (F, E), (E, F)))]
    return ws, [ops.QuantMatrix.from_gguf(Q4K, w, n_exp * r, c, device=gpu) for w, (r, c) in
                zip(ws, ((F, E), (F, E), (E, F)))]


@pytest.mark.parametrize("n_tok,n_exp,k,E,F,one", [
    (1, 8, 2, 256, 256, False),     # one super-block: one wave, two 16-row tiles past a 128-row tile's start
    (3, 4, 1, 512, 1280, False),    # two and five super-blocks; experts without a token
    (16, 8, 1, 256, 512, True),     # one expert gets a whole 16-row tile
    (17, 8, 1, 768, 512, True),     # ... and one entry more: a second pass
    (40, 8, 2, 256, 768, True),     # three passes
    (2, 2, 2, 8192, 256, False),    # eight waves over 32 super-blocks
    (1, 3, 3, 256, 8448, False),    # 33 super-blocks over eight waves
    (48, 8, 2, 256, 256, False),    # 12 entries per expert: the last of the few-token form
    (49, 8, 2, 256, 256, False),    # the first of the other (fp16 operands: 4e-3)
])
def test_few(gpu, orc, n_tok, n_exp, k, E, F, one):
    print(f"moe few n_tok={n_tok} experts={n_exp} k={k} E={E} F={F} one={one}", flush=True)
    ws, mats = build(gpu, n_exp, E, F, seed=E + F + n_tok)
    x = synth.gen_act((n_tok, E), seed=n_tok)
    x[0] *= 1e4
    lg = synth.gen_act((n_tok, n_exp), seed=n_tok + 1)
    if one:
        lg[:, 2] += 20.0
    want = np.asarray(orc.moe_ffn(Q4K, *ws, n_exp, E, F, x, lg, n_tok, k), np.float64).reshape(n_tok, E)
    xd, ld = torch.from_numpy(x).to(gpu), torch.from_numpy(lg).to(gpu)
    tiled = ops.MoeLayer(*mats, n_exp, k)(xd, ld)
    rows = ops.MoeLayer(*mats, n_exp, k, tiled=False)(xd, ld)
    assert torch.equal(tiled, rows)
    got = tiled.cpu().numpy().astype(np.float64)
    tol = TOL if n_tok * k <= 12 * n_exp else 1e-2
    for t in range(n_tok):
        assert np.linalg.norm(got[t] - want[t]) <= tol * np.linalg.norm(want[t]), t
