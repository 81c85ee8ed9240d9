"""Launch forms of the stack kernels at the sizes where their tiles, splits and groups end."""
import math

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


def rnd(*shape, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed), dtype=torch.float64)


def relerr(got, want):
    want = want.double()
    return float((got.double().cpu() - want).norm() / want.norm())


def act(x, ld):
    out = torch.zeros(x.shape[0], ld, dtype=torch.bfloat16)
    out[:, :x.shape[1]] = x.to(torch.bfloat16)
    return out.cuda()


@pytest.mark.parametrize("M", [1, 255, 256, 257, 513, 1300])
@pytest.mark.parametrize("Kd", [150, 192, 530])
def test_phased_gemm(K, M, Kd):
    """256 x 256 tiles: rows and columns around a tile's edge, three to nine steps of K, more tiles than a pass of an XCD takes, every
    kind of epilogue, whole and ragged columns, outputs of both types, segments beside each other."""
    bf = torch.bfloat16
    x = rnd(M, Kd, seed=1).to(bf)
    xd, X = x.double(), act(x, K.act_ld(Kd))
    ws = {n: (rnd(N, Kd, seed=10 + i) * Kd ** -0.5).to(bf) for i, (n, N) in enumerate(
        [("none", 515), ("silu", 260), ("tanh", 64), ("geglu", 512), ("f32", 2304), ("rope", 96)])}
    z = {n: xd @ w.double().T for n, w in ws.items()}
    y = {n: torch.full((M + 1, {"geglu": 256, "rope": 200}.get(n, w.shape[0])), 7.0, dtype=torch.float32 if n in ("f32", "none") else bf,
                       device="cuda") for n, w in ws.items()}
    P = {n: K.PackedLinear(w, False, "cuda") for n, w in ws.items()}
    pos = torch.arange(M, dtype=torch.int32).flip(0) % 50
    ang = rnd(50, 10, seed=5)
    cs = torch.stack([torch.cos(ang), torch.sin(ang)], -1).float()
    turn = dict(block=(32, 64), rope=(cs.cuda(), pos.cuda(), 10))          # 20 of a block's 32 columns turn
    L = K.LinLaunch([K.Seg(P[n], X, y[n][:M], "none" if n == "f32" else n, **(turn if n == "rope" else {})) for n in ws])
    L._cfg[M] = (True, 7), 1
    L.run(M, st())
    gelu = torch.nn.functional.gelu
    want = {"none": z["none"], "silu": z["silu"] * torch.sigmoid(z["silu"]), "tanh": torch.tanh(z["tanh"]),
            "geglu": gelu(z["geglu"][:, 0::2], approximate="tanh") * z["geglu"][:, 1::2], "f32": z["f32"]}
    for n, w in want.items():
        # f32 sums of Kd products; bf16 outputs round to 2^-9
        assert relerr(y[n][:M], w) < (2e-6 if y[n].dtype == torch.float32 else 3e-3), n
    o = y["rope"][:M].cpu()
    u = z["rope"].view(M, 3, 16, 2)
    c, s = (torch.cat([v[pos.long()].double()[:, None], torch.full((M, 1, 6), one, dtype=torch.float64)], 2)
            for v, one in ((cs[..., 0], 1.0), (cs[..., 1], 0.0)))
    w = torch.stack([u[..., 0] * c - u[..., 1] * s, u[..., 1] * c + u[..., 0] * s], -1).view(M, 96)
    assert relerr(torch.cat([o[:, 64 * i:64 * i + 32] for i in range(3)], 1), w) < 3e-3
    assert (o[:, 32:64] == 7).all() and all((t[M] == 7).all() for t in y.values())


@pytest.mark.parametrize("M,N,Kd,ks", [(1, 256, 400, 2), (300, 515, 700, 2), (257, 512, 700, 3), (600, 1028, 1100, 5), (1300, 4096, 700, 3),
                                        (513, 2304, 1300, 6)])
def test_phased_splits(K, M, N, Kd, ks):
    """Split products: 3 to 6 steps, not the same to every split, whole and ragged columns, up to 288 tiles, so that a workgroup walks from
    a split's tile to another split's; each slab holds its own steps' sums."""
    bf, steps = torch.bfloat16, K.act_ld(Kd) // 64
    x, w = rnd(M, Kd, seed=1).to(bf), (rnd(N, Kd, seed=2) * Kd ** -0.5).to(bf)
    y = torch.full((ks * M + 1, N), 7.0, device="cuda")
    L = K.LinLaunch([K.Seg(K.PackedLinear(w, False, "cuda"), act(x, K.act_ld(Kd)), y, slabs=ks, slab_rows=M)])
    L._cfg[M] = (True, 7), ks
    assert L.run(M, st()) == ks and L.slab_rows == M
    for i in range(ks):
        k0, k1 = (min(Kd, 64 * (steps * j // ks)) for j in (i, i + 1))
        assert relerr(y[i * M:(i + 1) * M], x[:, k0:k1].double() @ w[:, k0:k1].double().T) < 2e-6
    assert (y[ks * M] == 7).all()


@pytest.mark.parametrize("M", [200, 600])
@pytest.mark.parametrize("N", [256, 516, 518])
def test_phased_gates_and_groups(K, M, N):
    """256 x 256 tiles: the gated and the weighted epilogues, whole 4-column groups and not, and a batch of groups with columns of their
    own in x and y."""
    bf, Kd, G = torch.bfloat16, 250, 3
    ld = K.act_ld(Kd)
    x = rnd(M, G * Kd, seed=1).to(bf)
    X = torch.cat([act(x[:, g * Kd:(g + 1) * Kd], ld) for g in range(G)], 1).contiguous()
    w = {n: (rnd(N, Kd, seed=10 + i) * Kd ** -0.5).to(bf) for i, n in enumerate(("swiglu", "siluglu", "sigmoid"))}
    wg = (rnd(G, N, Kd, seed=20) * Kd ** -0.5).to(bf)
    y = {n: torch.full((M + 1, N if n == "sigmoid" else N // 2), 7.0, dtype=bf, device="cuda") for n in w}
    yg = torch.full((M + 1, G * (N + 8)), 7.0, device="cuda")
    segs = [K.Seg(K.PackedLinear(v, False, "cuda"), X, y[n][:M], n, alpha={"swiglu": 0.9, "sigmoid": 1.5}.get(n, 1.0)) for n, v in w.items()]
    L = K.LinLaunch(segs + [K.Seg(K.PackedLinear(wg, False, "cuda"), X, yg[:M], xgs=ld, ygs=N + 8)])
    L._cfg[M] = (True, 7), 1
    L.run(M, st())
    z = {n: x[:, :Kd].double() @ v.double().T for n, v in w.items()}
    g, u = z["swiglu"][:, 0::2].clamp(max=0.9), z["swiglu"][:, 1::2].clamp(-0.9, 0.9)
    silu = torch.nn.functional.silu
    want = {"swiglu": g * torch.sigmoid(1.702 * g) * (u + 1), "siluglu": silu(z["siluglu"][:, 0::2]) * z["siluglu"][:, 1::2],
            "sigmoid": 1.5 * torch.sigmoid(z["sigmoid"])}
    for n, v in want.items():                        # bf16 outputs round to 2^-9
        assert relerr(y[n][:M], v) < 3e-3 and (y[n][M] == 7).all(), n
    o = yg.view(M + 1, G, N + 8)
    for i in range(G):
        assert relerr(o[:M, i, :N], x[:, i * Kd:(i + 1) * Kd].double() @ wg[i].double().T) < 2e-6
    assert (o[:, :, N:] == 7).all() and (o[M] == 7).all()


@pytest.mark.parametrize("cfg", [8, 9, 10, 11])
@pytest.mark.parametrize("M,N,Kd", [(17, 96, 70), (64, 160, 192), (65, 161, 256), (129, 500, 330), (40, 1000, 1000)])
def test_balanced_tiles(K, cfg, M, N, Kd):
    """Tiles of 96, 128 and 160 weight rows: row and column edges, one to sixteen steps of K (fewer than the stages)."""
    bf = torch.bfloat16
    x, w = rnd(M, Kd, seed=1).to(bf), (rnd(N, Kd, seed=2) * Kd ** -0.5).to(bf)
    y = torch.full((M + 1, N), 7.0, device="cuda")
    L = K.LinLaunch([K.Seg(K.PackedLinear(w, False, "cuda"), act(x, K.act_ld(Kd)), y[:M])])
    L._cfg[M] = (True, cfg), 1
    L.run(M, st())
    assert relerr(y[:M], x.double() @ w.double().T) < 2e-6 and (y[M] == 7).all()


@pytest.mark.parametrize("nt,mt", [(4, 4), (4, 5), (5, 4), (6, 4), (6, 5), (8, 4), (8, 5)])
def test_paired_wave_groups(K, nt, mt):
    """lin_pair.hip: one K-tile to more than the ring holds, whole and in splits, rows and outputs at and past a tile's edges, products per head, two
    segments with an epilogue. The products are summed in 32 bits: |error| <= 2^-24 K sum |x| |w|."""
    bf, c = torch.bfloat16, K.PAIR(nt, mt)
    assert K.GEMM_TILES[c] == (32 * nt, 32 * mt)
    for Kd, ks in ((61, 1), (64, 1), (130, 2), (256, 1), (257, 1), (320, 1), (700, 3), (1030, 8)):
        for M, N in ((1, 4), (32 * mt, 32 * nt), (32 * mt + 1, 32 * nt + 4), (48 * mt + 7, 40 * nt + 13)):
            x, w = rnd(M, Kd, seed=1).to(bf), rnd(N, Kd, seed=2).to(bf)
            y = torch.full((ks * M + 1, N), 7.0, device="cuda")
            L = K.LinLaunch([K.Seg(K.PackedLinear(w, False, "cuda"), act(x, K.act_ld(Kd)), y, slabs=ks, slab_rows=M)])
            L._cfg[M] = (True, c), ks
            assert L.run(M, st()) == ks and (y[ks * L.slab_rows:] == 7).all()
            if ks > 1 and L.slab_rows != M:
                continue
            got, want = y[:ks * M].view(ks, M, N).sum(0).cpu().double(), x.double() @ w.double().T
            bound = 2.0 ** -24 * (Kd + 8 + ks) * (x.double().abs() @ w.double().abs().T)
            assert ((got - want).abs() <= bound + 2.0 ** -23 * want.abs()).all(), (Kd, ks, M, N)
    M, Kd, G, N = 32 * mt + 5, 200, 3, 148
    x, wg, ws = rnd(M, G * 256, seed=3).to(bf), rnd(G, N, Kd, seed=4).to(bf), (rnd(2 * N, Kd, seed=5) * Kd ** -0.5).to(bf)
    x.view(M, G, 256)[:, :, Kd:] = 0
    yg, ys = torch.full((M + 1, G * (N + 8)), 7.0, device="cuda"), torch.full((M + 1, N), 7.0, dtype=bf, device="cuda")
    X = x.cuda()
    L = K.LinLaunch([K.Seg(K.PackedLinear(ws, False, "cuda"), X, ys[:M], "siluglu"), K.Seg(K.PackedLinear(wg, False, "cuda"), X, yg[:M], xgs=256, ygs=N + 8)])
    L._cfg[M] = (True, c), 1
    L.run(M, st())
    z = x[:, :Kd].double() @ ws.double().T
    assert relerr(ys[:M], torch.nn.functional.silu(z[:, 0::2]) * z[:, 1::2]) < 3e-3 and (ys[M] == 7).all()      # (bf16 outputs round to 2^-9)
    o = yg.view(M + 1, G, N + 8)
    for i in range(G):
        assert relerr(o[:M, i, :N], x[:, i * 256:i * 256 + Kd].double() @ wg[i].double().T) < 2e-6
    assert (o[:, :, N:] == 7).all() and (o[M] == 7).all()
    m = K.LinLaunch([K.Seg(K.PackedLinear(ws, False, "cuda"), X, ys[:M], "siluglu", xmap=torch.zeros(M, dtype=torch.int32, device="cuda"))])
    m._cfg[M] = (True, c), 1
    with pytest.raises(RuntimeError):
        m.run(M, st())                               # (row maps go to other tiles)


@pytest.mark.parametrize("T", [7, 32, 33, 200])
def test_padding_rows_are_not_routed(K, T):
    """Rows without keys get no entries, in both forms of the plan; none at all when every row is padding."""
    E, top = 8, 2
    z = rnd(T, E, seed=1).float()
    ctx = (torch.arange(T, dtype=torch.int32) % 3) * 5
    plan = K.MoePlan(T, E, top, 1, 1, 1.0, "cuda")
    for c in (ctx, torch.zeros_like(ctx)):
        plan.run(z.cuda(), T, st(), c.cuda())
        n = int(plan.ntiles[0])
        got = []
        for e, o, k, _ in plan.tiles[:n].tolist():
            rows = plan.rows[o:o + k].tolist()
            assert 1 <= k <= plan.bm(T) and all(plan.sel[r] == e for r in rows)
            got += rows
        assert sorted(got) == [i for i in range(T * top) if c[i // top] > 0]


@pytest.mark.parametrize("M,N,rows", [(300, 160, 1500), (600, 512, 1200), (700, 160, 1399)])
def test_tall_split(K, M, N, rows):
    """More rows than a slab was bound for: as many slabs as the buffer holds (4, 2, 1), apart by the launch's rows."""
    bf, Kd = torch.bfloat16, 4160
    x, w = rnd(M, Kd, seed=1).to(bf), (rnd(N, Kd, seed=2) * Kd ** -0.5).to(bf)
    y = torch.full((rows, N), 7.0, device="cuda")
    L = K.LinLaunch([K.Seg(K.PackedLinear(w, False, "cuda"), act(x, K.act_ld(Kd)), y, slabs=4, slab_rows=128)])
    n = L.run(M, st())
    assert n == min(4, rows // M) and (n == 1 or L.slab_rows == M)
    assert relerr(sum(y[i * M:(i + 1) * M].double() for i in range(n)), x.double() @ w.double().T) < 2e-6
    assert (y[n * M:] == 7).all()
    z = torch.zeros(M, N, device="cuda")
    K.norm_add(y, None, z, None, M, 1e-5, st(), slabs=n, slab_rows=L.slab_rows)
    assert relerr(z, x.double() @ w.double().T) < 2e-6


@pytest.mark.parametrize("N", [1030, 1031, 1032])
@pytest.mark.parametrize("M", [600, 601, 602, 603])
def test_tall_split_of_ragged_rows(K, M, N):
    """Row counts and widths that are no multiples of 4: the slabs stay where the residual's launch reads them, here and in a launch of
    a single slab behind it."""
    bf, Kd, rows = torch.bfloat16, 3200, 1300
    x, w = rnd(rows - 1, Kd, seed=1).to(bf), (rnd(N, Kd, seed=2) * Kd ** -0.5).to(bf)
    y = torch.full((rows, N), 7.0, device="cuda")
    L = K.LinLaunch([K.Seg(K.PackedLinear(w, False, "cuda"), act(x, K.act_ld(Kd)), y, slabs=8, slab_rows=128)])
    for m, splits in ((M, 2), (rows - 1, 1)):
        n = L.run(m, st())
        assert n == splits
        z = torch.zeros(m, N, device="cuda")
        K.norm_add(y, None, z, None, m, 1e-5, st(), slabs=n, slab_rows=L.slab_rows)
        assert relerr(z, x[:m].double() @ w.double().T) < 2e-6


@pytest.mark.parametrize("T,E", [(700, 3), (1100, 8)])
def test_phased_gemm_of_experts(K, T, E):
    """Experts' row lists in tiles of 256 rows: several tiles, part tiles, an expert without rows; both products and the choice."""
    bf, d, ff = torch.bfloat16, 192, 300
    x = rnd(T, d, seed=1).to(bf)
    z = rnd(T, E, seed=2).float()
    z[:, 1] = -9.0
    up, down = (rnd(E, ff, d, seed=3) * d ** -0.5).to(bf), (rnd(E, d, ff, seed=4) * ff ** -0.5).to(bf)
    plan = K.MoePlan(T, E, 2, 1, 1, 1.0, "cuda", tall=K.MoePlan.takes_tall(False, d, ff))
    assert plan.bm(T) == 256
    h, ye = torch.zeros(2 * T, K.act_ld(ff), dtype=bf, device="cuda"), torch.zeros(2 * T, d, device="cuda")
    U, D = K.PackedLinear(up, False, "cuda"), K.PackedLinear(down, False, "cuda")
    plan.run(z.cuda(), T, st())
    K.LinLaunch([K.Seg(U, act(x, K.act_ld(d)), h, "relu2", routed=(plan.rows, 2))], plan).run(T, st())
    K.LinLaunch([K.Seg(D, h, ye, routed=(plan.rows, 1))], plan).run(T, st())
    sel = plan.sel.view(T, 2).long().cpu()
    assert (z.topk(2, 1).indices.sort(1).values == sel.sort(1).values).all()
    for j in range(2):
        e = sel[:, j]
        hid = torch.zeros(T, ff, dtype=torch.float64)
        for k in range(E):
            hid[e == k] = torch.relu(x[e == k].double() @ up[k].double().T) ** 2
        assert relerr(h[j::2, :ff], hid) < 3e-3
        got = h[j::2, :ff].double().cpu()
        want = torch.stack([got[t] @ down[e[t]].double().T for t in range(T)])
        assert relerr(ye[j::2], want) < 2e-6


# heads, key heads, key and value columns: groups that do and do not divide 16, single heads, widths with a part of a block
@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("H,G,D", [(8, 2, 128), (6, 2, 20), (3, 3, 64), (20, 1, 32), (2, 1, 300), (1, 1, 600)])
@pytest.mark.parametrize("window,keep,sink", [(0, 0, False), (40, 5, True)])
def test_plain_attention_rows_of_many_sequences(K, dt, H, G, D, window, keep, sink):
    """Runs of several lengths beside single tokens and a padded row, more than 64 rows: a workgroup's tokens are of one sequence, of
    several, or end before the batch does."""
    d = {"f32": torch.float32, "bf16": torch.bfloat16}[dt]
    Dp, _ = K.head_pad(D)
    bs, scale = 16, 0.8 / math.sqrt(D)
    runs = [(0, 50), (33, 1), (100, 3), (0, 17), (7, 1), (15, 2)]            # first position, rows
    nb = 7
    T = sum(n for _, n in runs) + 1
    assert T > 64
    perm = torch.randperm(len(runs) * nb, generator=torch.Generator().manual_seed(5)).view(-1, nb)
    kc, vc = (torch.zeros(perm.numel() * bs, G, Dp, dtype=d) for _ in range(2))
    q = torch.zeros(T, H, Dp, dtype=d)
    q[..., :D] = rnd(T, H, D, seed=1).to(d)
    gate, want = rnd(T, H, seed=3).float(), torch.zeros(T, H, D, dtype=torch.float64)
    seq, ctx, t = torch.zeros(T, dtype=torch.int32), torch.zeros(T, dtype=torch.int32), 0
    for i, (p0, n) in enumerate(runs):
        N = p0 + n
        k, v = rnd(N, G, D, seed=10 + i).to(d), rnd(N, G, D, seed=50 + i).to(d)
        pos = torch.arange(N)
        slot = perm[i][pos // bs] * bs + pos % bs
        kc[slot, :, :D], vc[slot, :, :D] = k, v
        for p in range(p0, N):
            s = torch.einsum("hd,khd->hk", q[t, :, :D].double(), k.double().repeat_interleave(H // G, 1)) * scale
            see = (pos <= p) & ((p - pos < window) | (pos < keep) if window else torch.ones(N, dtype=torch.bool))
            s = s.masked_fill(~see, -math.inf)
            if sink:
                s = torch.cat([s, torch.zeros(H, 1, dtype=torch.float64)], 1)
            w = torch.softmax(s, 1)[:, :N]
            want[t] = torch.einsum("hk,khd->hd", w, v.double().repeat_interleave(H // G, 1)) * gate[t].double()[:, None]
            seq[t], ctx[t] = i, p + 1
            t += 1
    out = torch.full((T + 1, H * Dp), 7.0, dtype=d, device="cuda")
    part = tuple(torch.zeros(1, device="cuda") for _ in range(3))
    K.gqa_attention(q.view(T, -1).cuda(), kc.view(-1, G * Dp).cuda(), vc.view(-1, G * Dp).cuda(), gate.cuda(), out, part,
                    perm.int().cuda(), bs, seq.cuda(), ctx.cuda(), T, H, G, Dp, False, 1, scale, st(), window=window, keep=keep, sink=sink)
    o = out.view(T + 1, H, Dp)
    # f32: the sums of a row; bf16: the output's rounding
    assert relerr(o[:T, :, :D], want) < (2e-6 if dt == "f32" else 3e-3)
    assert (o[:T, :, D:] == 0).all() and (o[T - 1] == 0).all() and (o[T] == 7).all()


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("H,G,D,spread", [(8, 2, 128, 6), (6, 2, 20, 6), (4, 4, 64, 90), (2, 1, 300, 6), (1, 1, 600, 90)])
@pytest.mark.parametrize("window,keep", [(0, 0), (20, 3)])
def test_plain_attention_keeps_values_apart(K, dt, H, G, D, spread, window, keep):
    """An infinity and a NaN among one sequence's values reach the rows that see their keys, and no other: not those of other sequences,
    not earlier tokens of the same prompt, not tokens whose window has passed them. Runs of several tokens, single tokens, `spread` of
    them: workgroups with tokens of several sequences."""
    d = {"f32": torch.float32, "bf16": torch.bfloat16}[dt]
    Dp, _ = K.head_pad(D)
    bs, nb = 16, 5
    runs = [(0, 37), (30, 9)] + [(10 + i % 40, 1) for i in range(spread)] + [(0, 30)]
    T = sum(n for _, n in runs)
    assert T > 64
    perm = torch.randperm(len(runs) * nb, generator=torch.Generator().manual_seed(5)).view(-1, nb)
    kc, vc = (rnd(perm.numel() * bs, G * Dp, seed=s).to(d) for s in (1, 2))
    q, gate = rnd(T, H * Dp, seed=3).to(d), rnd(T, H, seed=4).float()
    seq = torch.tensor([i for i, (_, n) in enumerate(runs) for _ in range(n)], dtype=torch.int32)
    pos = torch.tensor([p + j for p, n in runs for j in range(n)])
    hit = {0: 33, 1: 36, 5: 2, len(runs) - 1: 0}               # sequence -> key with an infinity in column 1, a NaN in column 17
    bad = vc.clone()
    for i, k in hit.items():
        bad[perm[i][k // bs] * bs + k % bs, 1::Dp] = math.inf
        bad[perm[i][k // bs] * bs + k % bs, 17::Dp] = math.nan

    def run(v):
        out = torch.full((T, H * Dp), 7.0, dtype=d, device="cuda")
        part = tuple(torch.zeros(1, device="cuda") for _ in range(3))
        K.gqa_attention(q.cuda(), kc.cuda(), v.cuda(), gate.cuda(), out, part, perm.int().cuda(), bs, seq.cuda(), (pos + 1).int().cuda(),
                        T, H, G, Dp, False, 1, 0.8 / math.sqrt(D), st(), window=window, keep=keep, sink=False)
        return out.view(T, H, Dp).cpu()
    a, b = run(vc), run(bad)
    at = torch.tensor([hit.get(int(i), 1 << 30) for i in seq])
    see = (at <= pos) & ((pos - at < window) | (at < keep) if window else torch.ones(T, dtype=torch.bool))
    assert 0 < int(see.sum()) < T and a.isfinite().all()
    assert b[see][..., 1].isinf().all() and b[see][..., 17].isnan().all()
    # a row that is summed again takes its keys one after another: the sum of up to 50 products in another order, and the output's type
    tol = 2e-6 if dt == "f32" else 3e-3
    rest = [c for c in range(Dp) if c not in (1, 17)]
    assert relerr(b[~see], a[~see]) < tol and relerr(b[see][..., rest], a[see][..., rest]) < tol


@pytest.mark.parametrize("n", [1, 6, 7, 8, 14, 15, 50])
def test_rows_to_host(K, n):
    """Logits on their way through two pinned buffers of seven rows: fewer, exactly and more than they hold, wanted rows gathered."""
    from types import SimpleNamespace

    from nats_llm_studio_amd.engine.engine import Engine
    V = 33
    eng = SimpleNamespace(dev=torch.device("cuda:0"), STAGE_BYTES=7 * 4 * V + 5, _stage=None, max_logit_rows=64)
    for k in range(3):                                   # the buffers are used again
        src = rnd(n + 3, V, seed=k).float().cuda()
        for rows in (src[:n], src[list(range(n, 0, -1))]):
            dst = torch.zeros(n, V)
            Engine._rows_to_host(eng, rows, dst)
            assert (dst == rows.cpu()).all()
    assert len(eng._stage[0][0]) == 7


def test_rows_to_host_waits_on_the_engines_device(K, monkeypatch):
    """The buffers' events are recorded on the stream of the engine's device, not on that of whichever device is current."""
    from types import SimpleNamespace

    from nats_llm_studio_amd.engine.engine import Engine
    eng = SimpleNamespace(dev=torch.device("cuda:0"), STAGE_BYTES=1 << 10, _stage=None, max_logit_rows=64)
    asked, current = [], torch.cuda.current_stream
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: asked.append(device) or current(device))
    recorded, record = [], torch.cuda.Event.record
    monkeypatch.setattr(torch.cuda.Event, "record", lambda self, stream=None: recorded.append(stream) or record(self, stream))
    src, dst = rnd(9, 33).float().cuda(), torch.zeros(9, 33)
    Engine._rows_to_host(eng, src, dst)
    assert torch.equal(dst, src.cpu())
    assert len(recorded) == 2 and all(s == current(eng.dev) for s in recorded) and asked[:2] == [eng.dev] * 2


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("D", [60, 64, 128, 256])
def test_wkv_scan_loads(K, dt, D):
    """Runs around a staged chunk's 8 to 32 tokens, one that starts from a state, few heads and enough for the other split: rows on
    16-byte boundaries (8 values to a thread where D is the padded width) and rows that are not give the same bits, and so does
    a run in two pieces; against 64 bits sums of a run's n D products, each rounded a few times: 2^-24 (n + D) sums of their magnitudes."""
    H = 2 if D != 64 else 9
    lens, pos0 = [1, 31, 32, 33, 70, 40], [0, 0, 0, 0, 0, 5]
    n = sum(lens)
    r, k, v = (rnd(n, H * D, seed=i).to(dt) * 0.3 for i in range(3))
    w, u = torch.sigmoid(rnd(n, H * D, seed=4)).float(), rnd(H * D, seed=5).float()
    S0 = rnd(len(lens), H * D * D, seed=6).float() * 0.3

    def put(x, off):
        ld = H * D + (1 if off else 8)
        flat = torch.zeros(n * ld + 8, dtype=x.dtype, device="cuda")
        t = flat[off:off + n * ld].view(n, ld)[:, :H * D]
        t.copy_(x)
        return t

    def run(off, pieces):
        S, prev, x = S0.cuda(), torch.zeros(len(lens), 8, device="cuda"), torch.zeros(n, 8, device="cuda")
        o = torch.zeros(n, H * D, device="cuda")
        for lo, hi in pieces:
            rows, t = [], 0
            for s, (m, p) in enumerate(zip(lens, pos0)):
                a, b = int(m * lo), int(m * hi)
                rows.append([t + a, b - a, s, p + a])
                t += m
            K.wkv_scan(put(r, off), put(k, off), put(v, off), put(w, off), u.cuda(), o, S, x, prev,
                       torch.tensor(rows, dtype=torch.int32).cuda(), len(lens), H, D, st())
        return o.cpu(), S.cpu()
    o, S = run(0, [(0, 1)])
    for off, pieces in ((1, [(0, 1)]), (0, [(0, 0.5), (0.5, 1)]), (1, [(0, 0.3), (0.3, 1)])):
        o1, S1 = run(off, pieces)
        assert torch.equal(o, o1) and torch.equal(S, S1)
    t = 0
    for s, m in enumerate(lens):
        rr, kk, vv, ww = (x[t:t + m].double().view(m, H, D) for x in (r, k, v, w))
        uu = u.double().view(H, D, 1)
        Sd, Sa = (S0[s].double().view(H, D, D) * (pos0[s] > 0) for _ in range(2))
        Sa = Sa.abs()
        for i in range(m):
            kv = kk[i][:, :, None] * vv[i][:, None, :]
            want, mag = ((Sd + uu * kv) * rr[i][:, :, None]).sum(1), ((Sa + uu.abs() * kv.abs()) * rr[i].abs()[:, :, None]).sum(1)
            assert ((o[t + i].double().view(H, D) - want).abs() <= 2.0 ** -24 * (i + D + 8) * mag).all()
            Sd, Sa = ww[i][:, :, None] * Sd + kv, ww[i][:, :, None] * Sa + kv.abs()
        t += m


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("cfg", [0, 1, 2, 3, 5, 6, 8, 9, 10, 11])
def test_tile_steps(K, cfg, f32):
    """One to nineteen steps of K: fewer than the tile's stages, whole passes of them and every remainder, whole and in two splits. The
    products are summed in 32 bits: |error| <= 2^-24 K sum |x| |w|."""
    import ctypes
    M, N = 70, 200
    for steps in range(1, 20):
        Kd = steps * (32 if f32 else 64) - 3
        dt = torch.float32 if f32 else torch.bfloat16
        x, w = (rnd(n, Kd, seed=i).to(dt) for i, n in ((steps, M), (50, N)))
        xa = torch.zeros(M, K.act_ld(Kd), dtype=dt, device="cuda")
        xa[:, :Kd] = x
        y = torch.full((2 * M, N), 9.0, device="cuda")
        p = K.PackedLinear(w, f32, "cuda")
        a = K.LinLaunch([K.Seg(p, xa, y, slabs=2, slab_rows=M)]).a
        a.s[0].M = M
        want, bound = x.double() @ w.double().T, 2.0 ** -24 * (Kd + 8) * (x.double().abs() @ w.double().abs().T)
        for ks in (1, 2)[:min(2, p.nsub // 2)]:
            a.s[0].ks = ks
            K._check(K.lib().nls_lin_gemm(ctypes.byref(a), int(f32), cfg, st()), "gemm")
            got = y.view(2, M, N)[:ks].sum(0).cpu().double()
            assert ((got - want).abs() <= bound + 2.0 ** -23 * want.abs()).all(), (steps, ks)


@pytest.mark.parametrize("T,E", [(24, 4), (100, 8), (300, 8)])
def test_experts_of_one_and_of_several_tiles(K, T, E):
    """Experts' row lists in tiles of 64 rows: lists of one tile beside longer ones (their weights are fetched in different ways)."""
    bf, d, n = torch.bfloat16, 330, 200
    x, z, w = rnd(T, d, seed=1).to(bf), rnd(T, E, seed=2).float(), (rnd(E, n, d, seed=3) * d ** -0.5).to(bf)
    z[:, 1] += 2.0
    plan = K.MoePlan(T, E, 2, 1, 1, 1.0, "cuda")
    assert plan.bm(T) == 64
    y, W = torch.zeros(2 * T, n, device="cuda"), K.PackedLinear(w, False, "cuda")
    plan.run(z.cuda(), T, st())
    K.LinLaunch([K.Seg(W, act(x, K.act_ld(d)), y, routed=(plan.rows, 2))], plan).run(T, st())
    sel = plan.sel.cpu().long()
    rows = sel.bincount(minlength=E)
    assert T == 24 or (rows.max() > 64 and rows.min() <= 64)
    want = torch.stack([w[e].double() @ x[i // 2].double() for i, e in enumerate(sel.tolist())])
    assert relerr(y, want) < 2e-6


@pytest.mark.parametrize("f32", [False, True])
def test_fetch_of_one_and_of_two_row_tiles(K, f32):
    """Launches of one row tile fetch their weights with the non-temporal hint, those of more without: rows at and past a tile's edge. Inputs are
    exact in both types, products are summed in 32 bits."""
    x, w = (rnd(257, 150, seed=1) * 64).round() / 64, (rnd(300, 150, seed=2) * 64).round() / 64
    dt = torch.float32 if f32 else torch.bfloat16
    x, w = x.to(torch.bfloat16).double(), w.to(torch.bfloat16).double()
    xa = torch.zeros(257, K.act_ld(150), dtype=dt, device="cuda")
    xa[:, :150] = x.to(dt)
    p = K.PackedLinear(w, f32, "cuda")
    for cfg, (bn, bm) in K.GEMM_TILES.items():
        for M in (bm, bm + 1) if cfg != 7 else ():
            y = torch.full((M + 1, 300), 7.0, device="cuda")
            L = K.LinLaunch([K.Seg(p, xa, y)])
            L.config = lambda M, c=cfg: (True, c)
            L.run(M, st())
            assert relerr(y[:M], x[:M] @ w.T) < 2e-6 and (y[M] == 7).all(), (cfg, M)
