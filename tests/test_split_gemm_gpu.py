"""GEMM of 32-bit operands in three bf16 parts: values of many magnitudes, values without parts, routed rows."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def K():
    from nats_llm_studio_amd.ops import stack
    stack.lib()
    return stack


def st():
    return torch.cuda.current_stream().cuda_stream


def launch(K, x, w, cfg, ks=1):
    M, Kd = x.shape
    N = w.shape[0]
    xa = torch.zeros(M, K.act_ld(Kd), device="cuda")
    xa[:, :Kd] = x
    y = torch.full((ks * M + 1, N), 9.0, device="cuda")
    p = K.PackedLinear(w, True, "cuda")
    a = K.LinLaunch([K.Seg(p, xa, y, slabs=ks, slab_rows=M)]).a
    a.s[0].M, a.s[0].ks = M, ks
    K._check(K.lib().nls_lin_gemm(ctypes.byref(a), 1, cfg, st()), "gemm")
    assert (y[-1] == 9).all()
    return y[:-1].view(ks, M, N).sum(0).cpu()


@pytest.mark.parametrize("cfg", [0, 1, 2])
@pytest.mark.parametrize("M,N,Kd,ks", [(1, 16, 64, 1), (63, 130, 97, 1), (64, 128, 320, 2), (65, 200, 33, 1), (129, 300, 515, 3)])
def test_values_of_many_magnitudes(K, cfg, M, N, Kd, ks):
    """Parts leave out less than 2^-24 of a product (three at 2^-9 2^-18 and below), and 32 products are added at a time in 32 bits, six times:
    |error| <= 2^-24 (K + 8) sum |x| |w|."""
    g = torch.Generator().manual_seed(M + Kd)
    x, w = (torch.randn(n, Kd, generator=g) * torch.exp2(torch.randint(-30, 31, (n, Kd), generator=g).float()) for n in (M, N))
    got = launch(K, x.cuda(), w.cuda(), cfg, ks).double()
    want, mag = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    assert ((got - want).abs() <= 2.0 ** -24 * (Kd + 8) * mag).all()


@pytest.mark.parametrize("cfg", [0, 1, 2])
def test_values_without_parts(K, cfg):
    """An infinite operand gives what 32-bit products give, as do the largest numbers, which a bf16 does not reach; other rows do not change."""
    g = torch.Generator().manual_seed(1)
    x, w = torch.randn(140, 160, generator=g), torch.randn(140, 160, generator=g)
    w[:, :2] = 2.0 ** -20                     # (row 139's sums stay inside the range)
    plain = launch(K, x.cuda(), w.cuda(), cfg)
    x[3, 7], x[70, 9], x[139, 0], x[139, 1], w[20, 5] = float("inf"), float("nan"), 3.4e38, -3.4e38, float("-inf")
    got, want = launch(K, x.cuda(), w.cuda(), cfg).double(), x.double() @ w.double().T
    assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.isinf(), want.isinf())
    assert torch.equal(got[got.isinf()], want[want.isinf()])
    rows, cols = [r for r in range(140) if r not in (3, 70, 139)], [c for c in range(140) if c != 20]
    kept = plain[rows][:, cols].double()
    assert (got[rows][:, cols] - kept).abs().max() <= 2.0 ** -23 * 168 * (x[rows].abs() @ w[cols].abs().T).max()
    assert (got[139, cols] - want[139, cols]).abs().max() <= 2.0 ** -24 * 168 * (x[139].double().abs() @ w[cols].double().abs().T).max()


@pytest.mark.parametrize("T", [40, 130, 700])
def test_routed_rows(K, T):
    """Experts' lists in tiles of 64 and of 128 rows, 32-bit operands."""
    g = torch.Generator().manual_seed(T)
    d, n, E = 330, 200, 4
    x, z, w = torch.randn(T, d, generator=g), torch.randn(T, E, generator=g), torch.randn(E, n, d, generator=g) * d ** -0.5
    plan = K.MoePlan(T, E, 2, 1, 1, 1.0, "cuda")
    assert plan.bm(T) == (128 if T == 700 else 64)
    plan.run(z.cuda(), T, st())
    xa = torch.zeros(T, K.act_ld(d), device="cuda")
    xa[:, :d] = x
    y = torch.zeros(2 * T, n, device="cuda")
    K.LinLaunch([K.Seg(K.PackedLinear(w, True, "cuda"), xa, y, routed=(plan.rows, 2))], plan).run(T, st())
    sel = plan.sel.cpu().long()
    want = torch.stack([w[e].double() @ x[i // 2].double() for i, e in enumerate(sel.tolist())])
    assert ((y.cpu().double() - want).norm() / want.norm()).item() < 2e-6


def test_lists_of_256_rows(K):
    """Tiles of a list that are taller than any 32-bit one are refused, by the launch's own choice and as a config."""
    T, d, n, E = 700, 320, 200, 4
    plan = K.MoePlan(T, E, 2, 1, 1, 1.0, "cuda", tall=True)
    assert plan.bm(T) == 256
    plan.run(torch.randn(T, E, device="cuda"), T, st())
    y = torch.full((2 * T, n), 7.0, device="cuda")
    L = K.LinLaunch([K.Seg(K.PackedLinear(torch.randn(E, n, d), True, "cuda"), torch.zeros(T, K.act_ld(d), device="cuda"), y, routed=(plan.rows, 2))], plan)
    for cfg in (None, 4):
        if cfg is not None:
            L._cfg[T] = (True, cfg), 1
        with pytest.raises(RuntimeError):
            L.run(T, st())
    assert (y == 7).all()


@pytest.mark.parametrize("cfg", [0, 1, 2])
def test_rows_beside_values_without_parts(K, cfg):
    """Sums of finite rows and columns have the same bits whatever the others of their tile hold."""
    g = torch.Generator().manual_seed(2)
    x, w = torch.randn(140, 160, generator=g), torch.randn(140, 160, generator=g)
    plain = launch(K, x.cuda(), w.cuda(), cfg)
    x[3, 7], x[70, 9], w[20, 5], w[100, 2] = float("inf"), float("nan"), float("-inf"), 3.4e38
    got = launch(K, x.cuda(), w.cuda(), cfg)
    rows, cols = [r for r in range(140) if r not in (3, 70)], [c for c in range(140) if c not in (20, 100)]
    assert torch.equal(got[rows][:, cols], plain[rows][:, cols]) and not got[3, cols].isfinite().any()


@pytest.mark.parametrize("cfg", [0, 1, 2])
@pytest.mark.parametrize("ex,ew", [(-100, 0), (-111, 0), (-118, 5), (-123, 0), (0, -119), (-60, -55)])
def test_small_values(K, cfg, ex, ew):
    """Operands, themselves normal numbers, whose parts or whose parts' products would lie below those: the bound of 32-bit products. Few
    inputs of one sign, so that an operand's missing digits show and no sum passes below the normal numbers itself."""
    g = torch.Generator().manual_seed(-ex)
    x, w = ((torch.rand(70, 4, generator=g) + 1) * 2.0 ** e for e in (ex, ew))
    x[1] = 0
    got = launch(K, x.cuda(), w.cuda(), cfg).double()
    want, mag = x.double() @ w.double().T, x.double().abs() @ w.double().abs().T
    assert ((got - want).abs() <= 2.0 ** -24 * 12 * mag).all() and not got[1].any()


@pytest.mark.parametrize("cfg", [0, 1, 5])
def test_routed_rows_on_each_tile(K, cfg):
    """Lists in tiles of 64 rows on every 32-bit tile that takes them: lists of one tile, of two and of few rows."""
    T, d, n, E = 130, 330, 200, 4
    g = torch.Generator().manual_seed(3)
    x, z, w = torch.randn(T, d, generator=g), torch.randn(T, E, generator=g), torch.randn(E, n, d, generator=g) * d ** -0.5
    z[:, 1] += 2.0
    plan = K.MoePlan(T, E, 2, 1, 1, 1.0, "cuda")
    assert plan.bm(T) == 64
    plan.run(z.cuda(), T, st())
    xa = torch.zeros(T, K.act_ld(d), device="cuda")
    xa[:, :d] = x
    y = torch.full((2 * T + 1, n), 7.0, device="cuda")
    L = K.LinLaunch([K.Seg(K.PackedLinear(w, True, "cuda"), xa, y, routed=(plan.rows, 2))], plan)
    L._cfg[T] = (True, cfg), 1
    L.run(T, st())
    sel = plan.sel.cpu().long()
    assert sel.bincount(minlength=E).max() > 64
    want = torch.stack([w[e].double() @ x[i // 2].double() for i, e in enumerate(sel.tolist())])
    assert ((y[:-1].cpu().double() - want).norm() / want.norm()).item() < 2e-6 and (y[-1] == 7).all()
