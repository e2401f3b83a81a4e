"""The few-token prefill GEMM (dq_gemm_direct.hip, behind dq_gemm up to 128 tokens) against the 128-token-tile kernel
of the two-call form (dq_quantize_act_f16 + dq_gemm_f16act): the same fp16 operands, so only the order of the fp32
sums differs. Each of the n products of a sum is rounded once more at most in either order, and their errors are
independent: the two results differ by at most a few 2^-24 sqrt(n) of the root of the summed squares, 1e-5 over
14336 columns."""
import ctypes

import pytest
import torch

from desireeia_amd import _lib, ops, synth

pytestmark = pytest.mark.gpu
TOL = 1e-5


def two_calls(mat, x):
    lib = _lib.load()
    n = ctypes.c_size_t(0)
    fmt = mat.fmt & ~ops.GEMM_TILES
    _lib.check(lib.dq_gemm_workspace_bytes(fmt, mat.rows, mat.cols, x.shape[0], ctypes.byref(n)), "workspace")
    work = torch.empty(n.value, dtype=torch.uint8, device=x.device)
    y = torch.empty(x.shape[0], mat.rows, device=x.device)
    _lib.check(lib.dq_quantize_act_f16(fmt, ops._ptr(x), mat.cols, x.shape[0], ops._ptr(work), ops._stream()), "quantize")
    _lib.check(lib.dq_gemm_f16act(mat.fmt, ops._ptr(mat.buf), mat.rows, mat.cols, ops._ptr(work), x.shape[0],
                                  ops._ptr(y), ops._stream()), "gemm")
    return y


@pytest.mark.parametrize("qtype", [synth.Q4_K, synth.Q6_K, synth.Q8_0, synth.Q4_0])
@pytest.mark.parametrize("rows,cols,n_tok", [
    (1, 256, 1),        # one row, one super-block, one token: one wave
    (17, 768, 16),      # a row past a tile; three waves; a whole token tile
    (33, 1024, 17),     # a token past a tile; four waves
    (300, 2304, 33),    # nine super-blocks over four waves; rows past a 256-row weight tile
    (16, 8192, 64),     # eight waves; a whole 64-token block
    (130, 8448, 65),    # 33 super-blocks over eight waves; a token past a block
    (4096, 512, 128),   # two row tiles per wave; the largest token count
])
def test_direct_matches_tiles(gpu, qtype, rows, cols, n_tok):
    print(f"direct gemm type={qtype} rows={rows} cols={cols} n_tok={n_tok}", flush=True)
    m = ops.QuantMatrix.from_gguf(qtype, synth.gen_weights(qtype, rows, cols, seed=rows + cols), rows, cols)
    x = torch.from_numpy(synth.gen_act((n_tok, cols), seed=n_tok)).to(gpu)
    x[0] *= 3000.0  # another range scale
    if n_tok > 2:
        x[1] = 0.0
    got, want = ops.gemm(m, x).double(), two_calls(m, x).double()
    for t in range(n_tok):
        assert (got[t] - want[t]).norm() <= TOL * want[t].norm()
    assert torch.equal(ops.gemm(ops.GemmTiles(m), x).double(), got)
    # a token's sum does not depend on the tokens beside it
    k = max(1, n_tok // 3)
    parts = torch.cat([ops.gemm(m, x[:k].contiguous()), ops.gemm(m, x[k:].contiguous())]) if n_tok > 1 else got
    assert torch.equal(parts.double(), got)


def test_direct_keeps_padding_out(gpu):
    """Tokens past n_tok of a 16-token tile are read from unwritten workspace: NaN there reaches no output."""
    m = ops.QuantMatrix.from_gguf(synth.Q4_K, synth.gen_weights(synth.Q4_K, 64, 512, seed=1), 64, 512)
    x = torch.from_numpy(synth.gen_act((5, 512), seed=2)).to(gpu)
    work = ops.gemm_workspace(m, 5)
    work.fill_(0xFF)
    y = torch.full((6, 64), 7.0, device=gpu)
    ops.gemm(m, x, out=y[:5], work=work)
    assert torch.isfinite(y).all() and (y[5] == 7.0).all()
    assert torch.equal(y[:5], ops.gemm(m, x))
