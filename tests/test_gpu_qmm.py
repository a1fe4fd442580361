"""Dense quantized matmul (QmmCall, metal/lib.rs:357-380, 684-734) on the
GPU vs the oracle's sequential-FMA matvec per token row. Bar: max|d| /
max|ref| <= 1e-3 per token."""
import numpy as np
import pytest

from helpers import gen_quant_matrix, rel_err
from test_gpu_decode import dev, host, oracle_matvec, qweights

pytestmark = pytest.mark.gpu

TOL = 1e-3


@pytest.mark.parametrize("out_dim,in_dim,group,bits,n", [
    (512, 2048, 64, 4, 1),     # shared-expert gate/up shape, one token
    (2048, 512, 64, 4, 7),     # shared-expert down shape, ragged block
    (4096, 2048, 32, 4, 33),   # two 32-token blocks
    (1024, 1024, 128, 3, 64),  # packed 3-bit
    (256, 256, 64, 4, 100),    # four blocks, last ragged
    # Without bf16 GEMM tiles (the limb GEMM): Flash-Next's 640 and 2560, a
    # 7168-wide projection, a 96-input matrix.
    (640, 2560, 64, 4, 9), (2560, 640, 32, 3, 5), (300, 7168, 64, 4, 3), (64, 96, 32, 4, 17),
])
def test_qmm_matches_oracle(kernels, out_dim, in_dim, group, bits, n):
    import torch

    rng = np.random.default_rng(out_dim + 3 * in_dim + 7 * n + bits)
    codes, s, b = gen_quant_matrix(rng, out_dim, in_dim, group, bits)
    x = rng.standard_normal((n, in_dim)).astype(np.float32)
    w = qweights(codes, s, b, group, bits)
    y = torch.empty((n, out_dim), dtype=torch.float32, device="cuda")
    ws = torch.empty(kernels.qmm_workspace_size(in_dim, group, n), dtype=torch.uint8, device="cuda")
    assert kernels.qmm(w, dev(x), y, out_dim, in_dim, n, ws) == 0
    got = host(y)
    worst = 0.0
    for t in range(n):
        want, _ = oracle_matvec(codes, s, b, in_dim, out_dim, group, bits, x[t])
        worst = max(worst, rel_err(got[t], want))
    print(f"qmm {n}x{in_dim} -> {out_dim} g{group} {bits}-bit: worst rel_err {worst:.3e}")
    assert worst <= TOL


def test_qmm_argument_errors(kernels):
    import torch

    from streamoe_amd import _abi

    c = _abi.CODES
    rng = np.random.default_rng(5)
    codes, s, b = gen_quant_matrix(rng, 512, 2048, 64, 4)
    w = qweights(codes, s, b, 64, 4)
    x = torch.zeros((4, 2048), dtype=torch.float32, device="cuda")
    y = torch.zeros((4, 512), dtype=torch.float32, device="cuda")
    need = kernels.qmm_workspace_size(2048, 64, 4)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    small = torch.empty(need // 2, dtype=torch.uint8, device="cuda")
    assert kernels.qmm(w, x, y, 512, 2048, 4, small) == c["SMOE_ERR_WORKSPACE_TOO_SMALL"]
    assert kernels.qmm(w, x, y, 500, 2048, 4, ws) == 0  # out_dim % 256: the limb GEMM
    assert kernels.qmm(w, x, y, 512, 2048, 0, ws) == c["SMOE_ERR_INVALID_ARG"]
    assert kernels.qmm(w, x[:, 1:], y, 512, 2044, 4, ws) == c["SMOE_ERR_IN_DIM_NOT_MULTIPLE"]


@pytest.mark.parametrize("out_dim,in_dim,group,bits,n", [
    (16896, 2048, 32, 4, 82),    # one unit per block, 792 limb blocks
    (15104, 4096, 32, 4, 103),
    (4096, 2048, 32, 4, 256),    # a whole round of limb blocks, group 32
    (4096, 1024, 64, 4, 256),    # 1024 inputs
    (1024, 4096, 32, 4, 1000),
    (5376, 256, 64, 4, 96),      # 252 blocks, 256 inputs
])
def test_qmm_stays_on_the_tiles_where_they_are_faster(kernels, out_dim, in_dim, group, bits, n):
    """Rows of a call that the bf16 tiles take have the same bits within a call
    of 1024 rows, which they take at any of these shapes."""
    import torch

    rng = np.random.default_rng(out_dim + n)
    w = qweights(*gen_quant_matrix(rng, out_dim, in_dim, group, bits), group, bits)
    x = dev(rng.standard_normal((1024, in_dim)).astype(np.float32))

    def run(rows):
        y = torch.empty((rows, out_dim), dtype=torch.float32, device="cuda")
        ws = torch.empty(kernels.qmm_workspace_size(in_dim, group, rows), dtype=torch.uint8, device="cuda")
        assert kernels.qmm(w, x, y, out_dim, in_dim, rows, ws) == 0
        return y

    few, many = run(n), run(1024)
    torch.cuda.synchronize()
    assert torch.equal(few, many[:n])


@pytest.mark.parametrize("out_dim,in_dim,group,bits,n,room", [
    (300, 7168, 32, 4, 2, "all"),      # two rows that are faster one after the other
    (640, 1152, 64, 3, 2, "all"),
    (17000, 1536, 32, 4, 2, "all"),
    (300, 704, 64, 4, 5, "one byte"),  # a workspace too small for the limb GEMM
    (300, 704, 64, 3, 5, "unaligned"),
])
def test_qmm_row_by_row_is_qmv(kernels, out_dim, in_dim, group, bits, n, room):
    import torch

    rng = np.random.default_rng(out_dim + in_dim + n)
    w = qweights(*gen_quant_matrix(rng, out_dim, in_dim, group, bits), group, bits)
    x = dev(rng.standard_normal((n, in_dim)).astype(np.float32))
    y, rows = (torch.zeros((n, out_dim), dtype=torch.float32, device="cuda") for _ in range(2))
    ws = torch.empty(kernels.qmm_workspace_size(in_dim, group, n) + 16, dtype=torch.uint8, device="cuda")
    ws = {"all": ws, "one byte": ws[:1], "unaligned": ws[16:]}[room]
    assert kernels.qmm(w, x, y, out_dim, in_dim, n, ws) == 0
    for t in range(n):
        assert kernels.qmv(w, x[t], rows[t], out_dim, in_dim) == 0
    torch.cuda.synchronize()
    assert torch.equal(y, rows)


@pytest.mark.parametrize("out_dim,in_dim,group,bits,n", [
    (4096, 2048, 32, 4, 257),   # one row past eight blocks of 32
    (4096, 2048, 32, 3, 300),
    (4096, 2048, 64, 3, 515),   # 17 blocks, the last of three rows
    (4096, 2048, 64, 4, 515),
    (4096, 2048, 128, 4, 300),
    (4096, 2048, 128, 3, 257),
    (256, 8448, 128, 4, 40),    # past the limb GEMM's 8192 inputs
    (512, 16384, 128, 3, 70),   # the most
])
def test_qmm_bf16_tiles_match_oracle(kernels, out_dim, in_dim, group, bits, n):
    """Calls that the bf16 tiles take. Bar 1e-4: x as bf16 pairs is off by 2^-17
    per value, whose sum over 2048 inputs and more stays below 2e-5 of the
    largest output."""
    import torch

    rng = np.random.default_rng(in_dim + 7 * n + group + bits)
    codes, s, b = gen_quant_matrix(rng, out_dim, in_dim, group, bits)
    x = rng.standard_normal((n, in_dim)).astype(np.float32)
    y = torch.full((n, out_dim), 7.0, dtype=torch.float32, device="cuda")
    ws = torch.empty(kernels.qmm_workspace_size(in_dim, group, n), dtype=torch.uint8, device="cuda")
    assert kernels.qmm(qweights(codes, s, b, group, bits), dev(x), y, out_dim, in_dim, n, ws) == 0
    got = host(y)
    assert np.all(np.isfinite(got))
    for t in sorted({0, 31, 32, n // 2, n - 1, min(n - 1, 255), min(n - 1, 256)}):
        assert rel_err(got[t], oracle_matvec(codes, s, b, in_dim, out_dim, group, bits, x[t])[0]) <= 1e-4
