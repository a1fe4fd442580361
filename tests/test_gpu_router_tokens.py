"""smoe_router over many tokens (k_router_mm) at the edges of its tiles: the
logits against float64, the routing against smoe_softmax_topk of the returned
logits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,E,H", [
    (129, 127, 96),     # one logit short of the rule: a block per row
    (129, 128, 96),     # three pieces over eight waves, one token past a tile
    (33, 500, 32),      # one piece, experts not a multiple of a tile
    (17, 1000, 2560),   # one token past a tile
    (1024, 16, 2080),   # half an expert tile, 65 pieces
    (500, 256, 2048),
    (70, 256, 100),     # not whole pieces: a block per row
])
def test_router_many_tokens(kernels, n, E, H):
    import torch

    rng = np.random.default_rng(n + E + H)
    W = (rng.standard_normal((E, H)) * 0.02).astype(np.float32)
    x = rng.standard_normal((n, H)).astype(np.float32)
    x[n // 2, 3] = 1e4
    k = min(8, E)
    wd, xd = torch.from_numpy(W).cuda(), torch.from_numpy(x).cuda()
    new = lambda dt, *s: torch.zeros(s, dtype=dt, device="cuda")
    idx, w, lg = new(torch.int32, n, k), new(torch.float32, n, k), new(torch.float32, n, E)
    assert kernels.router(wd, xd, n, E, H, k, True, idx, w, lg) == 0
    idx2, w2 = new(torch.int32, n, k), new(torch.float32, n, k)
    assert kernels.softmax_topk(lg, n, E, k, True, idx2, w2) == 0
    kernels.sync()
    assert torch.equal(idx, idx2) and torch.equal(w, w2)
    want = x.astype(np.float64) @ W.astype(np.float64).T
    # Rounding of chains of 4 products per 1024 inputs (12 at most here) and 8
    # pairwise levels, 2^-24 of the partial sums each, which sum |w x| bounds.
    bound = 21 * 2.0 ** -24 * (np.abs(x).astype(np.float64) @ np.abs(W).astype(np.float64).T)
    assert np.all(np.abs(lg.cpu().numpy() - want) <= bound)


@pytest.mark.parametrize("few,n,E,H", [
    (1, 129, 128, 2048),
    (63, 64, 256, 2048),
    (5, 40, 500, 32),      # one piece
    (3, 130, 128, 96),     # three pieces
    (7, 70, 256, 1376),    # 43: some leaves of two turns
    (15, 20, 1000, 2560),
    (900, 1024, 16, 2080),
    (4, 32, 512, 7168),    # seven turns
    (2, 17, 1000, 8224),   # a ninth turn of one piece
    (2, 70, 256, 100),     # not whole pieces
])
def test_router_token_bits_do_not_depend_on_the_call(kernels, few, n, E, H):
    import torch

    g = torch.Generator(device="cuda").manual_seed(n + E + H)
    W = torch.randn((E, H), generator=g, device="cuda") * 0.02
    x = torch.randn((n, H), generator=g, device="cuda")
    x[0, 3] = 1e4
    W[E - 1] = 0
    k = min(8, E)

    def run(m):
        idx = torch.zeros((m, k), dtype=torch.int32, device="cuda")
        w, lg = torch.zeros((m, k), device="cuda"), torch.zeros((m, E), device="cuda")
        assert kernels.router(W, x, m, E, H, k, True, idx, w, lg) == 0
        return idx, w.view(torch.int32), lg.view(torch.int32)

    assert few * E < 2 ** 14 <= n * E
    a, b = run(few), run(n)
    torch.cuda.synchronize()
    for p, q in zip(a, b):
        assert torch.equal(p, q[:few])
