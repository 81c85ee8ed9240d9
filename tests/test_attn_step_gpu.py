"""Attention and a gated linear recurrence of single tokens in one launch: splits of the keys, padded rows, first tokens, both types."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("AH,AG,Dp,H,D,V", [(8, 2, 128, 3, 64, 128), (6, 1, 64, 2, 20, 28), (40, 2, 64, 2, 128, 128), (4, 4, 128, 5, 64, 64)])
@pytest.mark.parametrize("ctx", [[1], [1500], [0, 33, 500], [7, 90] * 9, [64] * 150], ids=lambda c: f"{len(c)}x{c[-1]}")
def test_attn_step(dtype, AH, AG, Dp, H, D, V, ctx):
    """States: the bits of gla_step. Outputs: |error| against 64 bits <= e of the magnitudes summed, e = 2^-7 in bf16 (a weight and
    the output round by 2^-9 each, the norm's scale is a mean of such sums), (keys + D + 64) 2^-22 in 32 bits."""
    from nats_llm_studio_amd.ops import stack as K
    f32, T, BS = dtype == torch.float32, len(ctx), 16
    if T > K.attn_step_fits(AH, AG, Dp, not f32, 0, H, D, V, f32):
        pytest.skip("more tokens than go together")
    g = torch.Generator().manual_seed(T + Dp)
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).cuda()
    nb = (max(ctx) + BS) // BS
    bt = torch.randperm(T * nb, generator=g).int().view(T, nb).cuda()
    kc, vc, aq = rnd(T * nb * BS, AG * Dp), rnd(T * nb * BS, AG * Dp), rnd(T, AH * Dp)
    ag = torch.rand(T, AH, generator=g).cuda()
    ts, cl = torch.arange(T).int().cuda(), torch.tensor(ctx).int().cuda()
    rank = 16
    lo = K.act_ld(H * (2 * D + V))
    buf = rnd(T, lo + 64)
    q, k, v, low = buf, buf[:, H * D:], buf[:, 2 * H * D:], buf[:, lo:]
    a2, a2b = rnd(H * D, rank), torch.randn(H * D, generator=g).cuda()
    norm, gate = torch.rand(H * V, generator=g).cuda(), rnd(T, H * V)
    S0 = torch.randn(T, H * D * V, generator=g).cuda()
    runs = torch.tensor([[i, 1, -1 if i % 7 == 5 else i, i % 3] for i in range(T)], dtype=torch.int32).cuda()
    st = torch.cuda.current_stream().cuda_stream
    groups = K.attn_groups(AH, AG)
    ns = max(1, min(64, 256 // (T * groups))) if not f32 else 1
    part = (torch.zeros(T * AH * ns * Dp).cuda(), torch.zeros(T * AH * ns * 2).cuda(), torch.zeros(T * groups, dtype=torch.int32).cuda())
    cat = torch.full((T, AH * Dp + K.act_ld(H * V)), 7.0, dtype=dtype).cuda()
    aout, out = cat[:, :AH * Dp], cat[:, AH * Dp:]
    S, ref, S1 = S0.clone(), torch.empty(T, H * V, dtype=dtype).cuda(), S0.clone()
    gi = (low, a2, a2b, 0.3)
    K.attn_step(aq, kc, vc, ag, aout, part, ns, bt, BS, ts, cl, T, AH, AG, Dp, 0.09, True, q, k, v, None, gi, 0.5, S, runs, norm, gate, out, H,
                D, V, 1e-5, st)
    K.gla_step(q, k, v, None, gi, 0.5, S1, runs, T, norm, gate, ref, H, D, V, 1e-5, st)
    assert torch.equal(S, S1) and (cat[:, AH * Dp + H * V:] == 7).all() and not part[2].any()
    e = 2.0 ** -7 if not f32 else (max(ctx) + D + 64) * 2.0 ** -22
    for t in range(T):
        n = ctx[t]
        slot = (bt[t].long() * BS)[:, None] + torch.arange(BS).cuda()
        slot = slot.view(-1)[:n]
        kk, vv = (x[slot].double().view(n, AG, Dp).repeat_interleave(AH // AG, 1) for x in (kc, vc))
        s = torch.einsum("hd,nhd->hn", aq[t].double().view(AH, Dp).cpu(), kk.cpu()) * 0.09
        p = torch.softmax(torch.cat([s, torch.zeros(AH, 1, dtype=torch.float64)], 1), 1)[:, :n]
        f = ag[t].double().cpu()[:, None]
        want, mag = (torch.einsum("hn,nhd->hd", p, x.cpu()) * f for x in (vv, vv.abs()))
        assert ((aout[t].double().view(AH, Dp).cpu() - want).abs() <= e * mag + 1e-30).all(), t
        if runs[t, 2] < 0:
            assert (out[t] == 7).all() and torch.equal(S[t], S0[t])
            continue
        o = (S1[t].double().view(H, D, V) * q[t, :H * D].double().view(H, D, 1) * 0.5)
        o, m = o.sum(1), o.abs().sum(1)
        sc = (norm.double() * gate[t].double()).view(H, V) / (o * o).mean(1, keepdim=True).add(1e-5).sqrt()
        err = (out[t, :H * V].double().view(H, V) - o * sc).abs()
        assert (err <= e * (m * sc.abs() + (o * sc).abs() * (m * m).mean(1, keepdim=True).sqrt() / (o * o).mean(1, keepdim=True).sqrt())).all(), t


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T", [1, 5])
def test_given_decays(dtype, T):
    """Decays per token and channel instead of the low-rank gate input: states and outputs of gla_step, attention of gqa_attention's width."""
    from nats_llm_studio_amd.ops import stack as K
    AH, AG, Dp, H, D, V, BS = 8, 2, 128, 6, 64, 128, 16
    f32 = dtype == torch.float32
    assert T <= K.attn_step_fits(AH, AG, Dp, not f32, 0, H, D, V, f32)
    g = torch.Generator().manual_seed(T)
    rnd = lambda *s: torch.randn(*s, generator=g).to(dtype).cuda()
    kc, vc, aq, z = rnd(T * 48, AG * Dp), rnd(T * 48, AG * Dp), rnd(T, AH * Dp), rnd(T, H * (2 * D + V))
    bt, ts = torch.arange(T * 3).int().view(T, 3).cuda(), torch.arange(T).int().cuda()
    cl, runs = torch.tensor([40 - i for i in range(T)]).int().cuda(), torch.tensor([[i, 1, i, i] for i in range(T)]).int().cuda()
    a, norm, gate = torch.rand(T, H * D, generator=g).cuda(), torch.rand(H * V, generator=g).cuda(), rnd(T, H * V)
    S0 = torch.randn(T, H * D * V, generator=g).cuda()
    part = (torch.zeros(T * AH * Dp).cuda(), torch.zeros(T * AH * 2).cuda(), torch.zeros(T * 2).int().cuda())
    st = torch.cuda.current_stream().cuda_stream
    q, k, v = z, z[:, H * D:], z[:, 2 * H * D:]
    S, S1, aout, out, aref, ref = S0.clone(), S0.clone(), *(torch.zeros(T, n, dtype=dtype, device="cuda") for n in (AH * Dp, H * V) * 2)
    K.attn_step(aq, kc, vc, None, aout, part, 1, bt, BS, ts, cl, T, AH, AG, Dp, 0.09, False, q, k, v, a, None, 0.5, S, runs, norm, gate, out, H, D, V,
                1e-5, st)
    K.gla_step(q, k, v, a, None, 0.5, S1, runs, T, norm, gate, ref, H, D, V, 1e-5, st)
    K.gqa_attention(aq, kc, vc, None, aref, part, bt, BS, ts, cl, T, AH, AG, Dp, not f32, 1, 0.09, st)
    assert torch.equal(S, S1) and (f32 or torch.equal(out, ref))
    o = S1.double().view(T, H, D, V) * q[:, :H * D].double().view(T, H, D, 1) * 0.5
    o, m = o.sum(2), o.abs().sum(2)
    sc = norm.double().view(H, V) * gate.double().view(T, H, V) / (o * o).mean(2, keepdim=True).add(1e-5).sqrt()
    bound = m * sc.abs() + (o * sc).abs() * ((m * m).mean(2, keepdim=True) / (o * o).mean(2, keepdim=True)).sqrt()
    # (32 bits: eight waves to a state here, four there, so sums of 64 products, and squares of them, in another order)
    assert ((out.double() - ref.double()).abs().view(T, H, V) <= 128 * 2.0 ** -22 * bound).all()
    # another number of waves adds up to 40 keys: a rounding of 2^-22 a key, then the output's
    e = 2.0 ** -7 if not f32 else 40 * 2.0 ** -22
    assert ((aout.double() - aref.double()).abs() <= e * vc.double().abs().max()).all()
