"""The one-token expert kernels with limbs in LDS (csrc/phase.hip) at the edges
of their tiles and of the rules that choose between kernels, against the
oracle. Bar: max|d| / max|ref| <= 1e-5 of the output and of the MoE part: the
oracle's sequential f32 sums of K <= 8128 terms are off by about sqrt(K) 2^-24,
5.4e-6, the device's by less."""
import numpy as np
import pytest

import oracle
from helpers import gen_expert_blob, rel_err
from test_gpu_decode import _chain, _experts_case, _layer_case, _torch, dev, host
from test_gpu_softmax import _same_bits as same_bits, ulp_cases

pytestmark = pytest.mark.gpu

TOL = 1e-5


@pytest.mark.parametrize("H,I,k,bits,shared", [
    (64, 64, 1, 4, False),      # two chunks: a sixteenth of a row's lanes
    (576, 192, 3, 3, True),     # 18 chunks: one round of four, two of them used
    (2048, 448, 9, 4, False),   # 4032 rows: 4 per wave
    (2048, 576, 8, 4, True),    # 4608 rows: 8 per wave
    (2624, 704, 7, 3, True),    # 82 chunks: two rounds of four; three waves of 8 down rows
    (2560, 1600, 10, 4, True),  # 8 down waves
    (2560, 1664, 10, 4, True),  # 9: half the rows per block
    (8128, 128, 2, 4, False),   # 254 chunks
    (4096, 320, 4, 3, True),    # hidden 4096: whole-wave gate/up rows
    (128, 1984, 16, 4, True),   # 992 chunks, the most that fit
    (128, 2048, 16, 3, True),   # 1024: a wave per row
])
def test_phase_experts_match_oracle(kernels, H, I, k, bits, shared):
    _check_experts(kernels, H, I, k, bits, shared)


def _check_experts(kernels, H, I, k, bits, shared):
    if H > 4096:
        kernels.reserve(H, 2048, 1024)
    got, want, h_mid = _experts_case(kernels, H, I, k, bits, shared, seed=H + I + k + bits)
    err, moe = rel_err(got, want), rel_err(got - h_mid, want - h_mid)
    print(f"experts H={H} I={I} k={k} {bits}-bit rel_err={err:.3e} MoE part {moe:.3e}")
    assert err <= TOL and moe <= TOL


@pytest.mark.parametrize("name,H,I,E,k,bits,shared", [
    ("small-3bit", 320, 192, 20, 5, 3, True),   # 3-bit routed slots beside the 4-bit shared wave
    ("ungated", 2560, 640, 40, 10, 4, "ungated"),
    ("most-chunks", 256, 1856, 18, 16, 4, True),   # 17 slots, 986 chunks
    ("wave-per-row", 256, 1920, 18, 16, 3, True),  # 1020
])
def test_phase_layers_match_oracle(kernels, name, H, I, E, k, bits, shared):
    kernels.set_decode_path(1)
    try:
        got, gi, gw, want, wi, ww, _ = _layer_case(kernels, H, I, E, k, bits, True, shared, seed=sum(map(ord, name)))
    finally:
        kernels.set_decode_path(0)
    kernels.sync()
    err = rel_err(got, want)
    print(f"layer {name}: rel_err={err:.3e}")
    assert np.array_equal(gi, wi)
    assert err <= TOL


def test_phase_nonfinite_input(kernels):
    """A NaN in the hidden vector reaches every output; the next call is clean."""
    import streamoe_amd as sa

    torch = _torch()
    lay = sa.ExpertLayout(576, 192, 4, 64)
    arena = torch.empty(2 * lay.expert_size, dtype=torch.uint8, device="cuda")
    assert kernels.synth_experts(arena, 2, lay.expert_size, lay, 3) == 0
    x = torch.ones(576, device="cuda")
    out, h = torch.empty(576, device="cuda"), torch.zeros(576, device="cuda")
    bind = [(arena, 0), (arena, lay.expert_size)]
    x[100] = float("nan")
    assert kernels.experts_decode(lay, bind, [0.5, 0.5], x, h, None, 0.0, out) == 0
    kernels.sync()
    assert bool(torch.isnan(out).all())
    x[100] = 1.0
    assert kernels.experts_decode(lay, bind, [0.5, 0.5], x, h, None, 0.0, out) == 0
    kernels.sync()
    assert bool(torch.isfinite(out).all())


@pytest.mark.parametrize("scale", [1.0, 2e-19, 1e-19])
def test_phase_range_ends(kernels, scale):
    """SwiGLU outputs near the smallest normal float keep their precision, and
    an infinity in the hidden vector reaches every output, zero biases
    included. Bar 1e-5 as above, and 1152 steps of the smallest subnormal: both
    sides round 192 SwiGLU outputs (times a weight <= 1.1), 192 products and
    192 sums by at most one each."""
    import streamoe_amd as sa

    H, I = 576, 192
    rng = np.random.default_rng(11)
    blob = gen_expert_blob(rng, H, I, 64, 4)
    blob.reshape(3, -1)[:, H * I // 2 + H * I // 32:] = 0
    lay = sa.ExpertLayout(H, I, 4, 64)
    arena = dev(blob)
    x = (rng.standard_normal(H) * scale).astype(np.float32)
    zero, out = dev(np.zeros(H, np.float32)), dev(np.zeros(H, np.float32))

    def run():
        assert kernels.experts_decode(lay, [(arena, 0)], [1.0], dev(x), zero, None, 0.0, out) == 0
        kernels.sync()
        return host(out)

    want = oracle.expert_swiglu(blob, 4, H, I, 64, x)
    top = float(np.abs(want).max())
    got = run()
    err = float(np.abs(got.astype(np.float64) - want).max()) / top
    print(f"scale {scale}: largest output {top:.3e}, rel_err={err:.3e}")
    assert err <= TOL + 1152 * 2.0 ** -149 / top
    x[100] = np.inf
    assert not np.isfinite(run()).any()


@pytest.mark.parametrize("T,H,I,E,k,bits,norm", [
    (4, 2560, 640, 64, 10, 4, 0.1),
    (2, 2048, 640, 41, 3, 3, 0.0),     # odd logit rows
    (3, 320, 192, 300, 16, 4, 0.1),    # eight logits per lane, most slots
    (4, 7168, 1920, 18, 8, 4, 0.1),    # two rounds of chunks, down blocks of four rows
    (4, 3072, 512, 20, 4, 4, 0.1),     # a wave per gate/up row, 2048 rows of a token
    (3, 7168, 192, 300, 3, 3, 0.0),    # the same, four chunks per lane
    (4, 1024, 576, 20, 3, 4, 0.1),     # 4 rows per wave alone, 8 together; down 4 and 8 rows
])
def test_phase_tokens_match_single_token(kernels, T, H, I, E, k, bits, norm):
    """Several tokens through the per-phase kernels at once: outputs, indices
    and weights bit for bit those of each token alone."""
    torch = _torch()
    kernels.reserve(max(H, 4096), 2048, 1024)
    c = _chain(kernels, 2, E, k, bits, seed=H + E + T, norm_sigma=norm, I=I, H=H)
    xs = dev(np.random.default_rng(T).standard_normal((T, H)).astype(np.float32))
    xs[:, 0] *= 50

    def run(rows):
        r, n = rows.clone(), rows.shape[0]
        idx = torch.empty((n, k), dtype=torch.int32, device="cuda")
        w = torch.empty((n, k), dtype=torch.float32, device="cuda")
        assert kernels.moe_decode_tokens(c["layers"], c["norms"], 1e-6, n, rows, r, torch.empty_like(rows), idx, w) == 0
        kernels.sync()
        return host(r).view(np.uint32), host(idx), host(w).view(np.uint32)

    kernels.set_decode_path(1)
    try:
        got = run(xs)
        one = [run(xs[t:t + 1].contiguous()) for t in range(T)]
    finally:
        kernels.set_decode_path(0)
    for a, b in zip(got, zip(*one)):
        assert np.array_equal(a, np.concatenate(b))


@pytest.mark.parametrize("E,k", [(256, 8), (257, 16), (300, 4), (512, 10)])
def test_phase_routing_boundary(kernels, E, k):
    """Four tokens at once whose k-th and (k+1)-th logits are 0, 1 and 2 ulps
    apart (every gate/up wave then runs the reference's softmax and scan) beside
    one with a clear margin: indices and weights bit for bit the oracle's,
    together and one at a time."""
    import streamoe_amd as sa

    torch = _torch()
    H, I, T = 320, 192, 4
    rng = np.random.default_rng(E + k)
    cols = ulp_cases(E, k, 3, 60 + E + k) + [rng.standard_normal(E).astype(np.float32)]
    router = np.zeros((E, H), np.float32)
    router[:, :T] = np.stack(cols, axis=1)
    lay = sa.ExpertLayout(H, I, 4, 64)
    arena = torch.empty(E * lay.expert_size, dtype=torch.uint8, device="cuda")
    assert kernels.synth_experts(arena, E, lay.expert_size, lay, E) == 0
    shared = dev(gen_expert_blob(rng, H, I, 64, 4))
    gate = rng.standard_normal(H).astype(np.float32)
    router_d, gate_d = dev(router), dev(gate)  # the layer holds their addresses
    layer = kernels.layer(lay, arena, lay.expert_size, E, k, True, router_d, shared, gate_d)
    x = np.eye(T, H, dtype=np.float32)
    want = [oracle.moe_decode_layer(host(arena), lay.expert_size, H, I, E, k, 64, 4, True, router, x[t], x[t],
                                    host(shared), gate) for t in range(T)]
    for t in range(T):
        assert same_bits(want[t][3], cols[t])  # one-hot rows: the logits are the columns

    def run(rows):
        r, n = dev(rows), len(rows)
        idx = torch.empty((n, k), dtype=torch.int32, device="cuda")
        w = torch.empty((n, k), dtype=torch.float32, device="cuda")
        assert kernels.moe_decode_tokens([layer], None, 1e-6, n, dev(rows), r, torch.empty_like(r), idx, w) == 0
        kernels.sync()
        return host(r), host(idx), host(w)

    got = run(x)
    for t in range(T):
        out, idx, w = run(x[t:t + 1])
        assert np.array_equal(got[1][t], want[t][1]) and np.array_equal(idx[0], want[t][1])
        assert same_bits(got[2][t], want[t][2]) and same_bits(w[0], want[t][2])
        assert rel_err(got[0][t], want[t][0]) <= TOL and same_bits(out[0], got[0][t])


@pytest.mark.parametrize("H,I,k,bits,shared", [
    # The row's limbs in one to four rounds of a block's threads.
    (2112, 64, 4, 4, False),    # 66 chunks: two rounds, the second of two
    (6208, 320, 7, 3, True),    # 194: four
    (8192, 192, 11, 4, False),  # 256: four whole ones
])
def test_phase_long_rows_match_oracle(kernels, H, I, k, bits, shared):
    _check_experts(kernels, H, I, k, bits, shared)


@pytest.mark.parametrize("H,I,k,bits,shared", [
    (576, 64, 1, 4, False),  # 18 chunks: two per lane, most of the second's past the row
    (1024, 576, 8, 4, True),      # 32: two, 8 rows per wave
    (1088, 192, 3, 3, False),     # 34: three
    (1536, 320, 14, 3, True),     # 48: three, 8 rows per wave
])
def test_phase_short_rows_match_oracle(kernels, H, I, k, bits, shared):
    _check_experts(kernels, H, I, k, bits, shared)


@pytest.mark.parametrize("H,I,k,bits,shared", [
    (1024, 1536, 8, 3, True),    # down blocks of four rows in six waves
    (1984, 512, 5, 4, False),    # 248 blocks of eight would be fewer than CUs
    (2048, 512, 5, 4, False),    # 256 are not
    (64, 2048, 15, 4, False),    # 16 blocks, 15 waves
])
def test_phase_down_rows_match_oracle(kernels, H, I, k, bits, shared):
    _check_experts(kernels, H, I, k, bits, shared)


@pytest.mark.parametrize("H,I,k,bits,shared", [
    (2624, 128, 16, 4, False),  # 2048 rows of 82 chunks: the most that take a wave per row
    (2624, 192, 11, 4, False),  # 2112: 16 lanes
    (3648, 64, 1, 3, False),    # 114 chunks
    (4160, 64, 2, 4, True),     # 130: four per lane, half of the third's past the row
    (8192, 128, 15, 3, True),   # 256
])
def test_phase_wave_per_row_match_oracle(kernels, H, I, k, bits, shared):
    _check_experts(kernels, H, I, k, bits, shared)
