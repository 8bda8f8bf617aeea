"""Forward of layers with several positions per sample by the kernel that has the positions on its lanes: rows and channels that do not
fill a wavefront or a workgroup, inputs that are no multiple of 4 or 8, wavefronts that reach into several samples, slices,
groups, ties and undefined inputs.  Maxima and positions bit for bit against the oracle; powers against 64-bit sums: a term's
rounding (at most 24 halves of an ulp) and that of N additions (a random walk, four times its spread) are divided by p in the root,
which adds 2 ulp of its own."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _data(B, N, M, G, HW, kind):
    g = torch.Generator().manual_seed(B + N + HW)
    x, w = torch.randn(B, G * N, HW, generator=g), torch.randn(G * M, N, generator=g)
    if kind == "ties":
        x, w = x.round(), w.round()
    if kind == "odd":
        x[0, 1, 3], w[2, min(5, N - 1)], x[-1, :, -1] = float("nan"), float("inf"), float("nan")
    return x, w


# at least 16 positions and 2^22 terms with positions, 25 and 2^26 without
@pytest.mark.parametrize("B,N,M,G,HW,kind", [
    (9, 33, 901, 1, 16, "ties"), (3, 27, 61, 1, 1024, ""), (70, 75, 33, 1, 49, "odd"), (5, 2701, 20, 1, 17, ""), (40, 32, 24, 4, 65, "ties"),
    (1, 4, 1100, 1, 1000, ""), (2, 700, 96, 2, 25, ""), (64, 290, 65, 1, 64, "odd"), (33, 145, 224, 1, 63, "ties")])
def test_maxima_and_positions(oracle, B, N, M, G, HW, kind):
    from sortnet_amd import _lib, ext
    x, w = _data(B, N, M, G, HW, kind)
    ry, rp = oracle.inf_dist_forward(x.numpy(), w.numpy(), G)
    y, pos = torch.full((B, G * M, HW), 7.0, device="cuda"), torch.full((B, G * M, HW), 7, device="cuda", dtype=torch.int32)
    ext.inf_dist_forward(x.cuda(), w.cuda(), y, pos, G)
    assert _lib.last_forward_kernel().startswith("fwd_cols_kernel")
    np.testing.assert_array_equal(y.cpu().numpy(), ry)
    np.testing.assert_array_equal(pos.cpu().numpy(), np.asarray(rp).astype(np.int32))
    y.fill_(7.0)
    ext.inf_dist_forward_nograd(x.cuda(), w.cuda(), y, G)
    assert _lib.last_forward_kernel().startswith("fwd_cols_kernel") == (HW >= 25 and B * N * M * G * HW >= 1 << 26)
    np.testing.assert_array_equal(y.cpu().numpy(), ry)


@pytest.mark.parametrize("p", [1.0, 2.0, 3.0, 4.0, 5.0, 6.0, 7.0, 8.0])
@pytest.mark.parametrize("B,N,M,G,HW", [(150, 75, 501, 1, 49), (4, 2701, 33, 1, 784), (60, 34, 65, 2, 1030)])
def test_powers(p, B, N, M, G, HW):
    from sortnet_amd import _lib, ext
    x, w = (t.cuda() for t in _data(B, N, M, G, HW, ""))
    y = torch.full((B, G * M, HW), 7.0, device="cuda")
    ext.norm_dist_forward(x, w, y, G, p)
    assert _lib.last_forward_kernel().startswith("fwd_cols_kernel")
    rtol = (4 * N ** 0.5 + 24) * 2 ** -24 / p + 2 ** -22
    for b in {0, B - 1}:
        for m in range(0, G * M, 16):
            g = m // M
            d = (x[b, None, g * N:(g + 1) * N].double() - w[m:min(m + 16, (g + 1) * M), :, None].double()).abs()
            ref = d.pow(p).sum(1).pow(1 / p)
            torch.testing.assert_close(y[b, m:m + ref.shape[0]].double(), ref, rtol=rtol, atol=0)


@pytest.mark.parametrize("p", [2.0, 8.0])
@pytest.mark.parametrize("B,N,M,HW,slices", [(24, 800, 512, 256, 4), (12, 4000, 256, 256, 8), (64, 400, 256, 256, 2)])
def test_sums_are_no_longer_than_slices(p, B, N, M, HW, slices):
    """Long rows of many outputs, where a wavefront sums a whole row or half of it: the spread of the error is not above (by more than its
    sampling, a tenth) that of 32-bit sums over `slices` parts of the row, as many as tiles of 32 x 128 outputs are cut in."""
    from sortnet_amd import _lib, ext
    x, w = (t.cuda() for t in _data(B, N, M, 1, HW, ""))
    y = torch.full((B, M, HW), 7.0, device="cuda")
    ext.norm_dist_forward(x, w, y, 1, p)
    assert _lib.last_forward_kernel().startswith("fwd_cols_kernel")
    rows, cols, chunks = x[:: B // 6], w[:: M // 32], -(-N // 32)
    exact = torch.zeros(rows.shape[0], cols.shape[0], HW, device="cuda", dtype=torch.float64)
    parts = []
    for k in range(slices):
        s = torch.zeros_like(exact, dtype=torch.float32)
        for n in range(k * chunks // slices * 32, min((k + 1) * chunks // slices * 32, N)):
            t = (rows[:, None, n] - cols[None, :, n, None]).abs()
            exact += (rows[:, None, n].double() - cols[None, :, n, None].double()).abs() ** p
            if p == 8.0:
                t = t * t
                t = t * t
            s = (s.double() + t.double() * t.double()).float()   # one fused multiply-add
        parts.append(s)
    spread = lambda got: float(((got.double() - exact ** (1 / p)) / exact ** (1 / p)).pow(2).mean().sqrt())   # noqa: E731
    assert spread(y[:: B // 6][:, :: M // 32]) <= 1.1 * spread(sum(parts) ** (1 / p))
