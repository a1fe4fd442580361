"""The int8-limb GEMMs (csrc/limb.hip) at the edges of their tiles, against the
oracle's f32 path. Bar: max|d| / max|ref| <= 1e-5. Both sides round their
sums to f32: a sequential sum of K terms is off by about sqrt(K) 2^-24 of its
size (5.4e-6 at 8192), the gate, up and down sums add in quadrature, and the
limb side adds less than that."""
import numpy as np
import pytest

import oracle
from helpers import dequant_f64, gen_quant_matrix, rel_err
from test_gpu_decode import dev, oracle_matvec, qweights
from test_gpu_prefill import _case, _torch, host

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.mark.parametrize("name,n,H,I,E,k,bits,group,x_bf16,routing", [
    ("one-chunk", 3, 32, 32, 4, 2, 4, 32, True, "zipf"),             # a quarter step, a quarter column block
    ("g32-tail", 17, 96, 160, 6, 3, 3, 32, False, "hot"),            # 17 entries: an item of one row
    ("g64-half-step", 33, 320, 192, 5, 2, 4, 64, True, "hot"),       # K = 2.5 steps, odd group counts
    ("g128-odd", 40, 1152, 384, 9, 4, 4, 128, False, "zipf"),        # K split, 9 groups per row
    ("g64-3bit", 48, 704, 832, 12, 6, 3, 64, True, "zipf"),          # columns not a multiple of 128
    ("wide-g32", 7, 8160, 96, 3, 2, 3, 32, False, "zipf"),           # largest scale area
    ("inter-2048", 5, 2080, 2016, 4, 3, 4, 32, True, "zipf"),
    ("e1500", 20, 256, 64, 1500, 16, 4, 64, True, "zipf"),           # more experts than entries
    ("max-entries", 1024, 64, 64, 40, 16, 4, 64, True, "zipf"),      # 16384 entries
])
def test_limb_prefill_matches_oracle(kernels, name, n, H, I, E, k, bits, group, x_bf16, routing):
    got, want, _ = _case(kernels, n, H, I, E, k, bits, group, x_bf16, seed=sum(map(ord, name)), routing=routing)
    err = rel_err(got, want)
    print(f"limb prefill {name}: rel_err={err:.3e}")
    assert np.all(np.isfinite(got))
    assert err <= TOL


def test_limb_prefill_workspace_alignment_and_nonfinite_rows(kernels):
    """3-bit blobs at a base that is only 4-byte aligned; a workspace just
    below the grouped call's runs token by token to the same result; a row
    with a NaN or an infinity turns its own token's outputs into NaN and no
    other's."""
    import streamoe_amd as sa

    torch = _torch()
    lay = sa.ExpertLayout(320, 192, 3, 64)
    E, n, k = 6, 19, 3
    stride = (lay.expert_size + 15) // 16 * 16
    buf = torch.empty(E * stride + 16, dtype=torch.uint8, device="cuda")
    arena = buf[4:4 + E * stride]
    assert kernels.synth_experts(arena, E, stride, lay, 77) == 0
    idx, w = sa.zipf_routing(n, E, k, 1.1, seed=3)
    x = torch.empty((n, 320), dtype=torch.float32, device="cuda")
    assert kernels.synth_normal_f32(x, 78, 1.0) == 0
    idx_d, w_d = torch.from_numpy(idx).cuda(), torch.from_numpy(w).cuda()
    need = kernels.moe_prefill_workspace_size(lay, n, E, k)

    def run(ws_bytes, rows):
        out = torch.full((n, 320), 7.0, dtype=torch.float32, device="cuda")
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device="cuda")
        assert kernels.moe_prefill(lay, arena, stride, E, idx_d, w_d, rows, False, n, k, out, ws) == 0
        kernels.sync()
        return host(out)

    got = run(need, x)
    want = oracle.moe_permute_fuse(host(arena), stride, 3, 320, 192, 64, host(x),
                                   oracle.build_expert_buckets(idx, w, n, k, E), n)
    assert rel_err(got, want) <= TOL
    assert rel_err(run(need - 256, x), want) <= TOL
    bad = x.clone()
    bad[4, 100] = float("nan")
    bad[9, 319] = float("-inf")
    out = run(need, bad)
    rest = [t for t in range(n) if t not in (4, 9)]
    assert np.all(np.isnan(out[[4, 9]]))
    assert np.array_equal(out[rest], got[rest])


@pytest.mark.parametrize("out_dim,in_dim,group,bits,n", [
    (31, 32, 32, 4, 2),       # fewer columns than a tile, one chunk
    (33, 96, 32, 3, 16),      # one column past two tiles, a full row tile
    (640, 2560, 64, 4, 17),   # 2 tiles per wave, one row past a row tile
    (1000, 704, 64, 3, 50),   # half a step at the end of K
    (8200, 1152, 128, 4, 33), # 4 tiles per wave, 9 groups
    (16500, 320, 64, 4, 40),  # 8 tiles, K split, 2.5 steps over four waves
    (32900, 640, 32, 3, 30),  # more blocks than fit at once: columns split
    (16640, 8192, 32, 4, 20), # largest scale area
    (512, 2048, 64, 4, 100),  # a shape with bf16 tiles
    (4096, 2048, 64, 4, 257), # one row block past the rule: the bf16 tiles
])
def test_limb_qmm_matches_oracle(kernels, out_dim, in_dim, group, bits, n):
    torch = _torch()
    rng = np.random.default_rng(out_dim + 3 * in_dim + 7 * n + bits)
    codes, s, b = gen_quant_matrix(rng, out_dim, in_dim, group, bits)
    x = rng.standard_normal((n, in_dim)).astype(np.float32)
    x[0, 5] = 1000.0  # an outlier channel: one exponent per row
    w = qweights(codes, s, b, group, bits)
    y = torch.full((n, out_dim), 7.0, dtype=torch.float32, device="cuda")
    ws = torch.empty(kernels.qmm_workspace_size(in_dim, group, n), dtype=torch.uint8, device="cuda")
    assert kernels.qmm(w, dev(x), y, out_dim, in_dim, n, ws) == 0
    got = host(y)
    rows = sorted({0, n // 2, n - 1})
    worst = max(rel_err(got[t], oracle_matvec(codes, s, b, in_dim, out_dim, group, bits, x[t])[0]) for t in rows)
    print(f"limb qmm {n}x{in_dim} -> {out_dim} g{group} {bits}-bit: worst rel_err {worst:.3e}")
    assert np.all(np.isfinite(got))
    # The bf16 tiles split x into bf16 pairs: 2^-17 per value.
    assert worst <= (1e-4 if n == 257 else TOL)


@pytest.mark.parametrize("out_dim,in_dim,bits,n", [
    (48, 64, 3, 5),       # two of a step's four groups
    (100, 160, 4, 9),     # five groups: the second step's first alone
    (272, 2144, 4, 40),   # 67: 17 steps over four waves, the last of three groups
    (8300, 224, 3, 33),   # 4 tiles per wave
    (33000, 480, 4, 18),  # columns split, an odd step
])
def test_limb_groups_of_32(kernels, out_dim, in_dim, bits, n):
    """Outputs that see one group each (all other scales and biases zero): a code
    or an input in another group's operand shows at full size."""
    torch = _torch()
    rng = np.random.default_rng(out_dim + in_dim)
    codes, s, b = gen_quant_matrix(rng, out_dim, in_dim, 32, bits)
    keep = np.arange(in_dim // 32) == (np.arange(out_dim) % (in_dim // 32))[:, None]
    s, b = np.where(keep, s, 0).astype(np.uint16), np.where(keep, b, 0).astype(np.uint16)
    x = rng.standard_normal((n, in_dim)).astype(np.float32)
    y = torch.full((n, out_dim), 7.0, dtype=torch.float32, device="cuda")
    ws = torch.empty(kernels.qmm_workspace_size(in_dim, 32, n), dtype=torch.uint8, device="cuda")
    assert kernels.qmm(qweights(codes, s, b, 32, bits), dev(x), y, out_dim, in_dim, n, ws) == 0
    got = host(y)
    for t in sorted({0, n // 2, n - 1}):
        assert rel_err(got[t], oracle_matvec(codes, s, b, in_dim, out_dim, 32, bits, x[t])[0]) <= TOL


def test_limb_outlier_bound(kernels):
    """One exponent per row: a large input moves the others by up to 2^-30 of it
    each, which shows where its own weight is zero (even outputs here, their
    group's bias and its code zero). Bound, output by output: that times the sum
    of s q + |b|, and 64 roundings of f32 partial sums (11 groups in two sums of
    two roundings each, the bias chain, four K shares). The other rows keep
    theirs."""
    torch = _torch()
    out_dim, in_dim, n, at, big = 300, 704, 5, 5, 1e6
    rng = np.random.default_rng(21)
    codes, s, b = gen_quant_matrix(rng, out_dim, in_dim, 64, 4)
    codes[::2, at // 2] &= 0x0F  # input 5: the high nibble of byte 2
    b[::2, 0] = 0
    x = rng.standard_normal((n, in_dim)).astype(np.float32)
    x[2, at] = big
    y = torch.empty((n, out_dim), dtype=torch.float32, device="cuda")
    ws = torch.empty(kernels.qmm_workspace_size(in_dim, 64, n), dtype=torch.uint8, device="cuda")
    assert kernels.qmm(qweights(codes, s, b, 64, 4), dev(x), y, out_dim, in_dim, n, ws) == 0
    got = host(y).astype(np.float64)
    words = np.ascontiguousarray(codes).view(np.uint32)
    w = dequant_f64(words, s, b, in_dim, out_dim, 64)
    parts = dequant_f64(words, s & 0x7FFF, b & 0x7FFF, in_dim, out_dim, 64)  # s q + |b|
    want = x.astype(np.float64) @ w.T
    assert np.all(w[::2, at] == 0)
    parts[::2, at] = 0
    size = parts @ np.abs(x[2].astype(np.float64))
    bound = 2.0 ** -30 * big * parts.sum(axis=1) + 64 * 2.0 ** -24 * size
    err = np.abs(got[2] - want[2])
    print(f"outlier {big:g}: zero-weight outputs off by {(err / bound)[::2].max():.2f} of the bound, "
          f"{(err / np.abs(want[2]).max())[::2].max():.1e} of the largest output")
    assert np.all(err[::2] <= bound[::2])
    assert rel_err(got[2][1::2], want[2][1::2]) <= TOL
    for t in (0, 1, 3, 4):
        assert rel_err(got[t], want[t]) <= TOL
