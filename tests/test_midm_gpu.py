"""Projections of 33 to some hundred rows (csrc/gemm_midm.hip): every tile, every epilogue, ragged rows and columns, waves without a chunk
of K — against the operators in fp64 on the same bf16 operands.  A result is one rounding of an fp32 sum of K products: off by at most half
a bf16 ulp plus the sum's error (K terms of the size of the result at most: 2e-6 of the row's absolute sum, far below an ulp), so by one ulp
where that sum lies on a rounding boundary."""
import pytest
import torch

from oracle import dafolorn_oracle as D
from oracle import glm4_moe_oracle as O
from oracle import napadra_oracle as N_
from util import assert_close_bf16

pytestmark = pytest.mark.gpu
BF = torch.bfloat16


@pytest.fixture(scope="module")
def ops():
    from nanovllm import hip_ops
    hip_ops.load_library()
    return hip_ops


def rnd(*shape, seed, scale=1.0):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * scale).to(BF)


def close(got, ref, what):
    """ref fp64, one rounding away."""
    assert_close_bf16(got.float().to(BF) if got.dtype == torch.float32 else got, ref.to(BF), 1, 0.05, atol=2 ** -9, what=what)


# silu(gate) * up has three rounding points in front of the last one (gate, up, silu): each may fall on the other side of a boundary, one ulp or
# 2^-7 of the value at most, and the last rounding adds one: 4 ulp.  Near zero of the gate the relative change of silu has no such bound, the
# absolute one is 2^-8 of the factors (of the order of one).
SILU = (4, 0.06, 2 ** -8)

# (rows, columns, K): split waves (K of one chunk, three waves without work, up to several rounds of the ring; the large tile of long
# reductions), then every tile of the shared ring, fewer chunks than stages and many, columns that end inside a tile, rows that end inside a
# block, and the tiled kernel's epilogues on 256-row blocks and on 128-row blocks
SIZES = [(33, 36, 64), (64, 100, 128), (65, 2048, 192), (97, 2052, 1088), (128, 264, 4096), (130, 4128, 8256),
         (211, 2112, 2048), (520, 1000, 1024), (300, 3000, 64), (130, 6404, 64), (129, 5700, 704), (33, 16420, 320), (64, 20000, 128), (256, 8200, 576),
         (1300, 2056, 128), (700, 264, 512), (4096, 64, 192), (4100, 60, 192),
         (1300, 6152, 128), (391, 14344, 64)]


@pytest.mark.parametrize("M,N,K", SIZES)
def test_plain(ops, M, N, K):
    x, w, b = rnd(M, K + 8, seed=1)[:, :K], rnd(N, K, seed=2, scale=K ** -0.5), rnd(N, seed=3)
    wp = ops.padded_weight(N, K, dtype=BF, device="cuda")
    wp.copy_(w)
    xd = torch.empty(M, K + 8, dtype=BF, device="cuda")[:, :K]
    xd.copy_(x)
    ref = x.double() @ w.double().T
    close(ops.gemm_bf16(xd, wp), ref, "plain")
    close(ops.gemm_bf16(xd, wp, b.cuda()), ref + b.double(), "bias")


@pytest.mark.parametrize("M,N,K", SIZES)
def test_activations(ops, M, N, K):
    """Act in the epilogue: per-column ones, xIELU, fp32 rows with and without a soft cap, rows into a wider buffer."""
    if N % 8:
        N += 4      # (fp32 rows and rows of a wider buffer are whole 16-byte pieces)
    x, w = rnd(M, K, seed=4), rnd(N, K, seed=5, scale=K ** -0.5)
    z = x.double() @ w.double().T
    cut = N // 3 // 8 * 8
    gate = torch.cat([z[:, :cut], torch.sigmoid(z[:, cut:])], 1)
    relu = torch.cat([z[:, :cut].clamp(min=0) ** 2, z[:, cut: 2 * cut], torch.sigmoid(z[:, 2 * cut:])], 1)
    p, q = torch.tensor(0.3).double(), torch.tensor(-0.4).double()
    xielu = (ops.ACT_XIELU, float(D.softplus(p)), float(0.5 + D.softplus(q)))
    xd, wd = x.cuda(), w.cuda()
    out = torch.full((M, N + 16), 7.0, dtype=BF, device="cuda")
    close(ops.linear_act(xd, wd, act=(ops.ACT_GATE, float(cut), 0.0), out=out[:, 8: 8 + N]), gate, "gate")
    assert torch.all(out[:, :8] == 7) and torch.all(out[:, 8 + N:] == 7)
    close(ops.linear_act(xd, wd, act=(ops.ACT_RELU2_GATE, float(cut), float(2 * cut))), relu, "relu^2 | pass | gate")
    close(ops.linear_act(xd, wd, act=xielu), D.xielu(z, p, q), "xielu")
    # fp32 rows: the sum's own error, K products of magnitude |x| |w|
    bound = 2.0 ** -23 * (x.double().abs() @ w.double().abs().T) * 8
    assert ((ops.linear_act(xd, wd, out_f32=True).cpu().double() - z).abs() <= bound + 1e-7).all()
    capped = ops.linear_act(xd, wd, act=(ops.ACT_SOFTCAP, 3.0, 0.0), out_f32=True).cpu().double()
    assert ((capped - N_.soft_cap(z, 3.0)).abs() <= bound + 2e-6).all()


@pytest.mark.parametrize("M,I,K", [(33, 24, 64), (65, 1000, 192), (97, 1408, 1088), (211, 4104, 576), (300, 264, 1024), (100, 3000, 128), (130, 3016, 64),
                                   (64, 9000, 192), (48, 1024, 1024), (64, 1032, 512), (95, 1368, 512), (64, 2048, 2048), (64, 2056, 2048), (64, 4096, 1024), (65, 4096, 64),
                                   (33, 384, 4096), (95, 448, 2688), (95, 448, 2736),
                                   (97, 40, 320), (97, 40, 384), (1000, 40, 512), (1001, 40, 512), (1001, 40, 576), (391, 7176, 128), (1300, 7176, 64)])
def test_gated(ops, M, I, K):
    x, w = rnd(M, K, seed=6), rnd(2 * I, K, seed=7, scale=K ** -0.5)
    g, u = (x.double() @ w.double().T).chunk(2, 1)
    close(ops.gated_glu(x.cuda(), w.cuda(), 2.0), N_.clamped_glu(g, u, 2.0), "clamped unit")
    act = ops.grouped_gemm_gateup_silu(x.cuda(), w.cuda().unsqueeze(0), None, None, M)
    assert_close_bf16(act, O.silu_and_mul(torch.cat([g, u], 1).to(BF)), *SILU, what="silu")
    d = rnd(K, I, seed=8, scale=I ** -0.5)
    y = ops.grouped_gemm_down(act, d.cuda().unsqueeze(0), None, None, 0)
    close(y, act.cpu().double() @ d.double().T, "down")


# 32 rows over eight waves: 16 columns (one round of the chip exactly, waves without a chunk at the least K) and 32 (exactly one round), one tile more
@pytest.mark.parametrize("M,N,K", [(33, 2048, 512), (64, 2044, 576), (97, 996, 1088), (33, 2052, 512), (128, 2048, 2048), (100, 1900, 576), (128, 2052, 512)])
def test_split_tiles_of_32_rows(ops, M, N, K):
    x, w, b = rnd(M, K + 8, seed=31)[:, :K], rnd(N, K, seed=32, scale=K ** -0.5), rnd(N, seed=33)
    xd = torch.empty(M, K + 8, dtype=BF, device="cuda")[:, :K]
    xd.copy_(x)
    out = torch.full((M + 2, N), 7.0, dtype=BF, device="cuda")
    ref = x.double() @ w.double().T
    close(ops.linear_act(xd, w.cuda(), b.cuda(), out=out[1: M + 1]), ref + b.double(), "bias")
    assert torch.all(out[0] == 7) and torch.all(out[-1] == 7)
    bound = 2.0 ** -23 * (x.double().abs() @ w.double().abs().T) * 8
    assert ((ops.linear_act(xd, w.cuda(), out_f32=True).cpu().double() - ref).abs() <= bound + 1e-7).all()


@pytest.mark.parametrize("T,nh,nkv,K", [(96, 4, 1, 512), (100, 12, 2, 512), (128, 16, 2, 576), (97, 14, 1, 1088)])
def test_split_tiles_of_32_rows_with_rope_store(ops, T, nh, nkv, K):
    """The fused QKV projection takes half a head per workgroup where the projection by itself takes 16 or 32 columns: bit for bit the same."""
    N = (nh + 2 * nkv) * 128
    x, w, b = rnd(T, K, seed=41).cuda(), rnd(N, K, seed=42, scale=K ** -0.5).cuda(), rnd(N, seed=43).cuda()
    pos = torch.randint(0, 512, (T,), generator=torch.Generator().manual_seed(44)).cuda()
    cs = O.build_cos_sin_cache(64, 512, 10000.0).reshape(512, 64).contiguous().cuda()
    q0, k0, v0 = ops.qkv_split_norm_rope_store(ops.gemm_bf16(x, w, b), nh, nkv, 128, pos, cs, 64, None, None, 1e-5, None, None, None, True)
    q1, k1, v1 = ops.gemm_qkv_rope_store(x, w, b, nh, nkv, 128, pos, cs, 64, None, None, None, True)
    assert torch.equal(q0, q1) and torch.equal(k0, k1) and torch.equal(v0, v1)


@pytest.mark.parametrize("T,E,k,H,I,shared", [(33, 3, 2, 192, 100, True), (97, 5, 3, 576, 72, False), (211, 8, 2, 128, 264, True), (64, 1, 1, 64, 40, False)])
def test_experts(ops, T, E, k, H, I, shared):
    """Groups of 24 to 95 rows on average, ragged ones among them (an expert without rows, one with more than a block of 64)."""
    G = E + int(shared)
    g = torch.Generator().manual_seed(T)
    idx = torch.stack([torch.randperm(max(E - 1, 1), generator=g)[: k] if t % 5 or E == 1 else torch.arange(k) for t in range(T)]).sort(-1).values
    wt = (torch.rand(T, k, generator=g) + 0.1).to(BF)
    offs, tok, scale, _ = ops.moe_align(idx.cuda(), wt.cuda(), E, shared)
    R = T * k + (T if shared else 0)
    assert 24 * G <= R < 96 * G
    x, w13, w2 = rnd(T, H, seed=20), rnd(G, 2 * I, H, seed=21, scale=H ** -0.5), rnd(G, H, I, seed=22, scale=I ** -0.5)
    I64 = I // 64 * 64 or 64
    act_in, w2 = rnd(R, I64, seed=23), rnd(G, H, I64, seed=22, scale=I64 ** -0.5)
    act = ops.grouped_gemm_gateup_silu(x.cuda(), w13.cuda(), offs, tok, R)
    y = ops.grouped_gemm_down(act_in.cuda(), w2.cuda(), offs, scale, E)
    o, s = offs.cpu().tolist(), scale.cpu()
    for e in range(G):
        if o[e + 1] > o[e]:
            rows = slice(o[e], o[e + 1])
            z = x[tok.cpu()[rows].long()].double() @ w13[e].double().T
            assert_close_bf16(act[rows], O.silu_and_mul(z.to(BF)), *SILU, what=f"act of expert {e}")
            d = (act_in[rows].double() @ w2[e].double().T).to(BF)
            assert_close_bf16(y[rows], (d.float() * s[rows, None].float()).to(BF) if e < E else d, 2, 0.06, atol=2 ** -8, what=f"y of expert {e}")


@pytest.mark.parametrize("T,E,k,H,I", [(300, 128, 6, 192, 512), (250, 80, 3, 4096, 832), (260, 128, 7, 448, 544)])
def test_many_experts_of_few_rows(ops, T, E, k, H, I):
    """Groups of 7 to 23 rows on average with column tiles for several rounds of the chip, one of them with more than a block of 64."""
    g = torch.Generator().manual_seed(T)
    idx = torch.stack([torch.randperm(E - 1, generator=g)[: k] if t % 3 else torch.arange(k) for t in range(T)]).sort(-1).values
    wt = (torch.rand(T, k, generator=g) + 0.1).to(BF)
    offs, tok, scale, _ = ops.moe_align(idx.cuda(), wt.cuda(), E, False)
    R, K2 = T * k, 64 * (I // 64)
    x, w13 = rnd(T, H, seed=20), rnd(E, 2 * I, H, seed=21, scale=H ** -0.5)
    act_in, w2 = rnd(R, K2, seed=23), rnd(E, H, K2, seed=22, scale=K2 ** -0.5)
    act = ops.grouped_gemm_gateup_silu(x.cuda(), w13.cuda(), offs, tok, R)
    y = ops.grouped_gemm_down(act_in.cuda(), w2.cuda(), offs, scale, E)
    o, s = offs.cpu().tolist(), scale.cpu()
    for e in (0, k - 1, k, E // 2, E - 2, E - 1):
        if o[e + 1] > o[e]:
            rows = slice(o[e], o[e + 1])
            z = x[tok.cpu()[rows].long()].double() @ w13[e].double().T
            assert_close_bf16(act[rows], O.silu_and_mul(z.to(BF)), *SILU, what=f"act of expert {e}")
            d = (act_in[rows].double() @ w2[e].double().T).to(BF)
            assert_close_bf16(y[rows], (d.float() * s[rows, None].float()).to(BF), 2, 0.06, atol=2 ** -8, what=f"y of expert {e}")


def test_experts_of_rows_far_apart(ops):
    """Gathered rows of an x longer than 32-bit byte offsets reach (rows 2 MiB apart: past 2 GiB from row 1024, past 4 GiB from row 2048): an
    expert of near rows, one of far ones, one of both, with a partial last block of 64."""
    H, I, T = 192, 72, 2100
    x = torch.empty(T, 1 << 20, dtype=BF, device="cuda")[:, :H]
    x.copy_(rnd(T, H, seed=63))
    tok = torch.cat([torch.arange(30), torch.arange(1023, 1053), torch.arange(0, T, 31)]).to(torch.int32)
    offs = [0, 30, 60, tok.numel()]
    w = rnd(3, 2 * I, H, seed=64, scale=H ** -0.5)
    act = ops.grouped_gemm_gateup_silu(x, w.cuda(), torch.tensor(offs, dtype=torch.int32).cuda(), tok.cuda(), tok.numel())
    for e in range(3):
        rows = slice(offs[e], offs[e + 1])
        z = rnd(T, H, seed=63)[tok[rows].long()].double() @ w[e].double().T
        assert_close_bf16(act[rows], O.silu_and_mul(z.to(BF)), *SILU, what=f"expert {e}")


@pytest.mark.parametrize("M,I,H", [(1, 1408, 512), (1, 10944, 512), (1, 10944, 1624), (1, 1024, 384), (1, 1024, 376), (1, 40, 64), (1, 416, 1024), (1, 408, 1024)])
def test_one_row_feed_forward(ops, M, I, H):
    """Either side of the K from which the GEMV body takes it (gate|up 256 + I / 8, down 384 + H / 32)."""
    x, w, d = rnd(M, H, seed=30), rnd(2 * I, H, seed=31, scale=H ** -0.5), rnd(H, I, seed=32, scale=I ** -0.5)
    act = ops.grouped_gemm_gateup_silu(x.cuda(), w.cuda().unsqueeze(0), None, None, M)
    assert_close_bf16(act, O.silu_and_mul((x.double() @ w.double().T).to(BF)), *SILU, what="silu")
    close(ops.grouped_gemm_down(act, d.cuda().unsqueeze(0), None, None, 0), act.cpu().double() @ d.double().T, "down")


@pytest.mark.parametrize("M", [1, 2])
def test_feed_forward_refuses_columns_off_four(ops, M):
    x, w = rnd(M, 64, seed=35).cuda(), rnd(12, 64, seed=36).cuda().unsqueeze(0)
    with pytest.raises(RuntimeError, match="N%4"):
        ops.grouped_gemm_gateup_silu(x, w, None, None, M)


@pytest.mark.parametrize("R", [1, 2, 40, 130])
def test_one_group_of_gathered_rows(ops, R):
    """No offsets, rows of a longer x by number: one row (the last of x) and more, on either side of every row count that picks a kernel."""
    T, H, I = 300, 192, 72
    x, w = rnd(T, H, seed=33), rnd(2 * I, H, seed=34, scale=H ** -0.5)
    tok = (T - 1 - 7 * torch.arange(R)) % T
    act = ops.grouped_gemm_gateup_silu(x.cuda(), w.cuda().unsqueeze(0), None, tok.to(torch.int32).cuda(), R)
    assert_close_bf16(act, O.silu_and_mul((x[tok].double() @ w.double().T).to(BF)), *SILU, what="silu")


@pytest.mark.parametrize("T,nh,nkv,K", [(97, 4, 1, 1024), (211, 6, 2, 640), (256, 2, 2, 512), (450, 6, 2, 576), (130, 40, 2, 128), (211, 96, 8, 320)])
def test_qkv_epilogue(ops, T, nh, nkv, K):
    """Split, rotation and cache rows in the projection's epilogue: the projection and the split kernel, bit for bit."""
    x, w, b = rnd(T, K, seed=9).cuda(), rnd((nh + 2 * nkv) * 128, K, seed=10, scale=K ** -0.5).cuda(), rnd((nh + 2 * nkv) * 128, seed=11).cuda()
    g = torch.Generator().manual_seed(12)
    pos = torch.randint(0, 500, (T,), generator=g).cuda()
    cs = O.build_cos_sin_cache(64, 512, 10000.0).reshape(512, 64).contiguous().cuda()
    slots = torch.randperm(512, generator=g)[:T].to(torch.int32)
    slots[::5] = -1
    caches = [torch.full((2, 256, nkv, 128), 3.0, dtype=BF, device="cuda") for _ in range(4)]
    q, k, v = ops.gemm_qkv_rope_store(x, w, b, nh, nkv, 128, pos, cs, 64, caches[0], caches[1], slots.cuda(), True)
    q2, k2, v2 = ops.qkv_split_norm_rope_store(ops.gemm_bf16(x, w, b), nh, nkv, 128, pos, cs, 64, None, None, 1e-5, caches[2], caches[3], slots.cuda(), True)
    assert torch.equal(q, q2) and torch.equal(k, k2) and torch.equal(v, v2)
    assert torch.equal(caches[0], caches[2]) and torch.equal(caches[1], caches[3])


@pytest.mark.parametrize("M,N,K", [(33, 100, 4096), (64, 2052, 6144), (95, 1000, 4608), (130, 2048, 8192), (211, 4096, 4096), (500, 2048, 6144), (400, 4096, 8192)])
def test_row_slices(ops, M, N, K):
    """Partial sums of K slices, out of wider rows: every slab its own slice's fp32 sum (K products of magnitude |x| |w|)."""
    xw, w = rnd(M, K + 16, seed=40), rnd(N, K, seed=41, scale=K ** -0.5)
    x = xw[:, 8: 8 + K]
    best = ops.row_slices(M, N, K)
    assert best >= 4 and ops.row_slices(M, N, K + 8) == 1 and ops.row_slices(32, N, K) == 1
    for ns in sorted({best, 2} if M < 96 else {best}):
        part = ops.gemm_bf16_partial(xw.cuda()[:, 8: 8 + K], w.cuda(), ns).part.cpu().double()
        assert part.shape == (ns, M, N)
        k = K // ns
        for s in range(ns):
            a, b = x[:, s * k: (s + 1) * k].double(), w[:, s * k: (s + 1) * k].double()
            assert ((part[s] - a @ b.T).abs() <= 2.0 ** -23 * 8 * (a.abs() @ b.abs().T) + 1e-7).all(), (ns, s)
    if M < 96:
        with pytest.raises(RuntimeError):
            ops.gemm_bf16_partial(x.cuda(), w.cuda(), 7)


def test_row_slices_only_where_they_are_taken(ops):
    """Where they pay (fewer K for more tiles); no count that gemm_bf16_partial refuses: tiled slabs of columns off eight, weights beyond 32-bit offsets with no kernel to fall back on."""
    assert ops.row_slices(700, 2056, 8192) > 1 and ops.row_slices(700, 2052, 8192) == 1
    assert ops.row_slices(1000, 2048, 5632) == 1 < ops.row_slices(1000, 2048, 6144) and ops.row_slices(1500, 2048, 4608) == 1 < ops.row_slices(1500, 2048, 5120)
    assert ops.row_slices(3000, 2048, 4096) > 1 and ops.row_slices(3000, 2048, 4032) == 1 and ops.row_slices(16384, 2048, 8192) == 1
    assert ops.row_slices(64, 4096, 65536) > 1 and ops.row_slices(64, 4096, 262144) == 1 and ops.row_slices(95, 2048, 262144) == 1


@pytest.mark.parametrize("M,N", [(40, 100), (700, 2052), (200, 2052), (64, 2048)])
def test_projection_and_norm_of_any_width(ops, M, N):
    """RowParallelLinear hands slices to the norm only where the norm adds them up (whole 16-byte pieces), rows otherwise."""
    from nanovllm.layers.layernorm import RMSNorm
    from nanovllm.layers.linear import RowParallelLinear
    K = 8192
    old = torch.get_default_dtype()
    torch.set_default_dtype(BF)
    try:
        with torch.device("cuda"):
            lin, norm = RowParallelLinear(K, N), RMSNorm(N, 1e-5)
    finally:
        torch.set_default_dtype(old)
    x, w, res = rnd(M, K, seed=60), rnd(N, K, seed=61, scale=K ** -0.5), rnd(M, N, seed=62)
    lin.weight.data.copy_(w)
    y = lin(x.cuda(), defer_reduce=True)
    assert isinstance(y, ops.PartialSum) == (N % 8 == 0)
    h, r = norm(y, res.cuda())
    # the projection's rounding is off by one of its ulps beside a boundary, 2^-5 at most below 8, which is what a sum near zero then differs by;
    # the norm divides by more than one and rounds twice more
    assert x.shape[0] * N < 1 << 22     # (so many normal values stay below 8)
    s = (x.double() @ w.double().T).to(BF).double() + res.double()
    assert_close_bf16(r, s.to(BF), 1, 0.05, atol=2 ** -5, what="residual")
    assert_close_bf16(h, (s * (s.pow(2).mean(-1, keepdim=True) + 1e-5).rsqrt()).to(BF), 2, 0.35, atol=2 ** -5, what="norm")


def test_feed_forward_gives_rows_unless_asked(ops):
    """A module's own caller (and its hooks) get a tensor; partial sums only where they are asked for, the same to a rounding."""
    from nanovllm.layers.dense_mlp import DenseMLP
    T, W, ff = 128, 1024, 4096
    m = DenseMLP(W, ff, BF)
    m.load({"up": rnd(ff, W, seed=65, scale=W ** -0.5), "down": rnd(W, ff, seed=66, scale=ff ** -0.5), "act": torch.zeros(2)}, "cuda")
    h = rnd(T, W, seed=67).cuda()
    y, parts = m(h), m(h, defer_reduce=True)
    assert isinstance(y, torch.Tensor) and y.shape == (T, W) and y.dtype == BF and isinstance(parts, ops.PartialSum)
    close(y, parts.part.cpu().double().sum(0), "rows and slabs")


@pytest.mark.parametrize("T,E,H,slices,gemm,split", [
    (191, 64, 1024, 4, False, False), (192, 64, 1024, 4, False, True), (255, 64, 512, 0, False, False), (256, 64, 512, 0, False, True), (257, 64, 512, 0, True, True),
    (300, 64, 1024, 3, True, True), (257, 40, 512, 4, False, False), (159, 128, 4096, 0, False, False), (160, 128, 4096, 0, True, True),
    (95, 128, 4096, 4, False, False), (96, 128, 4096, 4, False, True), (160, 128, 2048, 0, False, True), (48, 256, 2048, 4, True, True),
    (103, 152, 2048, 4, False, True), (128, 160, 2048, 0, True, True), (127, 160, 2048, 0, False, False), (700, 16, 512, 0, False, False),
    (1024, 16, 512, 0, True, True), (400, 60, 512, 4, False, False)])
def test_norm_router_and_bucketing_by_size(ops, monkeypatch, T, E, H, slices, gemm, split):
    """The norm behind a projection (its rows or its K slices), the router and the bucketing, on either side of every line between one launch and
    several and between the launch's own logits and a GEMM: norm and routing against the oracle, the bucketing as moe_align's contract, and all
    entry points alike — with the one launch too, wherever the logits are its own."""
    from test_hip_kernels import _check_align, _check_router
    k = 4
    assert ops.router_by_gemm(T, E, H) == gemm
    rows = rnd(T, H, seed=50)
    parts = torch.randn(max(slices, 1), T, H, generator=torch.Generator().manual_seed(51))
    res, nw, gw = rnd(T, H, seed=52), (1 + 0.1 * rnd(H, seed=53).float()).to(BF), rnd(E, H, seed=54, scale=H ** -0.5)
    bias = (torch.rand(E, generator=torch.Generator().manual_seed(55)) * 0.2 - 0.1).float()
    x = ops.PartialSum(parts.cuda()) if slices else rows.cuda()
    calls = []
    for name in ("add_rmsnorm", "add_rmsnorm_partial"):
        f = getattr(ops, name)
        monkeypatch.setattr(ops, name, lambda *a, f=f: (calls.append(1), f(*a))[1])
    args = (x, res.cuda(), nw.cuda(), 1e-5, gw.cuda(), bias.cuda(), k, 1.0)
    y, ro, idx, w, al = ops.add_rmsnorm_router_topk(*args, align_with_shared=True)
    assert bool(calls) == split
    # the sum's rounding: one ulp of a value below 8 beside a boundary (2^-5), which is what a residual near zero then differs by; the norm
    # divides by the root of a mean square above one and rounds twice more
    s = ((parts.double().sum(0).to(BF) if slices else rows).double() + res.double())
    assert s.abs().max() < 16 and s.pow(2).mean(-1).min() > 1
    assert_close_bf16(ro, s.to(BF), 1, 0.05, atol=2 ** -5, what="residual")
    ref = (s * (s.pow(2).mean(-1, keepdim=True) + 1e-5).rsqrt()).to(BF).double() * nw.double()
    assert_close_bf16(y, ref.to(BF), 2, 0.35, atol=2 ** -5, what="norm")
    _check_router(ops, y.cpu(), gw, bias, k, 1.0, f"{T} x {E}", allow_flip_rows=0.05)
    _check_align(*al, idx.cpu(), w.cpu(), E, True)
    idx2, w2 = ops.router_topk(y, gw.cuda(), bias.cuda(), k, 1.0)
    y3, ro3, idx3, w3 = ops.add_rmsnorm_router_topk(*args)
    assert torch.equal(idx, idx2) and torch.equal(w, w2) and all(torch.equal(a, b) for a, b in zip((y, ro, idx, w), (y3, ro3, idx3, w3)))
    if not gemm:
        for name in ("ROUTER_SPLIT_LOGITS", "ROUTER_SPLIT_LOGITS_SLABS", "ROUTER_SPLIT_LOGITS_MANY"):
            monkeypatch.setattr(ops, name, 1 << 40)
        del calls[:]
        y4, ro4, idx4, w4, al4 = ops.add_rmsnorm_router_topk(*args, align_with_shared=True)
        assert not calls and all(torch.equal(a, b) for a, b in zip((y, ro, idx, w), (y4, ro4, idx4, w4)))
        _check_align(*al4, idx4.cpu(), w4.cpu(), E, True)


@pytest.mark.parametrize("T", [64, 211, 300])
def test_layer_half_replayed(ops, T):
    """K slices, norm, router, bucketing and experts of a step in a HIP graph: every replay, on new rows and between eager work, is the eager result."""
    H, E, k, I, K = 1024, 64, 8, 192, 8192
    wo, gw, nw = rnd(H, K, seed=70, scale=K ** -0.5).cuda(), rnd(E, H, seed=71, scale=H ** -0.5).cuda(), (1 + 0.1 * rnd(H, seed=72).float()).to(BF).cuda()
    bias = (torch.rand(E, generator=torch.Generator().manual_seed(73)) * 0.2 - 0.1).cuda()
    w13, w2 = rnd(E + 1, 2 * I, H, seed=74, scale=H ** -0.5).cuda(), rnd(E + 1, H, I, seed=75, scale=I ** -0.5).cuda()
    x, res = torch.empty(T, K, dtype=BF, device="cuda"), torch.empty(T, H, dtype=BF, device="cuda")
    slices = ops.row_slices(T, H, K)
    assert slices > 1

    def step():
        y, ro, idx, w, (offs, tok, scale, pos) = ops.add_rmsnorm_router_topk(ops.gemm_bf16_partial(x, wo, slices), res, nw, 1e-5, gw, bias, k, 1.0, align_with_shared=True)
        rows = ops.grouped_gemm_down(ops.grouped_gemm_gateup_silu(y, w13, offs, tok, T * (k + 1)), w2, offs, scale, E)
        return y, ro, idx, w, ops.moe_combine(rows, pos, T, k, T * k)

    def fill(seed):
        x.copy_(rnd(T, K, seed=seed))
        res.copy_(rnd(T, H, seed=seed + 1))

    fill(80)
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = step()
    for i in range(4):
        fill(90 + 2 * i)
        want = [t.clone() for t in step()]
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(out, want)), i


@pytest.mark.parametrize("M,N,K", [(33, 4, 256), (64, 16, 320), (97, 64, 2048), (100, 132, 4096), (320, 380, 448), (2048, 64, 512), (8192, 12, 256), (341, 380, 256)])
@pytest.mark.parametrize("f32", [False, True])
def test_few_columns(M, N, K, f32):
    """32 rows x 16 columns over eight waves: ends of rows and columns, fewer chunks than waves, the largest grid of that tile and the next."""
    from nanovllm import hip_ops
    g = torch.Generator().manual_seed(M + N + K)
    x, w = torch.randn(M, K, generator=g).to(torch.bfloat16), (torch.randn(N, K, generator=g) * K ** -0.5).to(torch.bfloat16)
    out = torch.full((M, N + 8), 7.0, dtype=torch.float32 if f32 else torch.bfloat16, device="cuda")
    hip_ops.linear_act(x.cuda(), w.cuda(), out_f32=f32, out=out[:, :N])
    want = x.double() @ w.double().T
    err = (out[:, :N].cpu().double() - want).abs().max() / want.abs().max()
    assert err < (K * 2.0 ** -24 if f32 else 2.0 ** -8) and torch.all(out[:, N:] == 7)   # sums in fp32; the result's rounding


@pytest.mark.parametrize("M,N,K", [(512, 17, 256), (512, 208, 320), (900, 108, 4096), (1150, 100, 512), (1000, 128, 256), (4090, 20, 320), (2700, 36, 1088)])
@pytest.mark.parametrize("f32", [False, True])
def test_few_columns_row_block_by_row_block(M, N, K, f32):
    """Many rows of few columns: the order of the tiles is another one and nothing more, ends of the grid, rows and columns included."""
    from nanovllm import hip_ops
    N = N - N % 4
    g = torch.Generator().manual_seed(M + N + K)
    x, w = torch.randn(M, K, generator=g).to(torch.bfloat16).cuda(), (torch.randn(N, K, generator=g) * K ** -0.5).to(torch.bfloat16).cuda()
    out = torch.full((M + 40, N + 8), 7.0, dtype=torch.float32 if f32 else torch.bfloat16, device="cuda")
    hip_ops.linear_act(x, w, out_f32=f32, out=out[:M, :N])
    assert torch.all(out[:, N:] == 7) and torch.all(out[M:] == 7)
    for r in range(0, M, 480):      # so many rows go column tile by column tile
        n = min(480, M - r)
        if n > 32:
            assert torch.equal(out[r: r + n, :N], hip_ops.linear_act(x[r: r + n], w, out_f32=f32)), r
    want = x.cpu().double() @ w.cpu().double().T
    assert (out[:M, :N].cpu().double() - want).abs().max() / want.abs().max() < (K * 2.0 ** -24 if f32 else 2.0 ** -8)


@pytest.mark.parametrize("K,N,rows", [(320, 12288, (64, 128, 256)), (576, 8192, (128, 256)), (192, 24576, (64, 128))])
def test_shared_tiles_of_one_row_block(ops, K, N, rows):
    """Shared tiles with all rows in one block and the others of the same columns: every sum in the order of K, so a row
    is bit for bit the same whatever stands behind it."""
    x, w = rnd(max(rows), K, seed=61).cuda(), rnd(N, K, seed=62, scale=K ** -0.5).cuda()
    got = [(ops.linear_act(x[:M], w), ops.gated_glu(x[:M], w, 2.0), ops.grouped_gemm_gateup_silu(x[:M], w.unsqueeze(0), None, None, M)) for M in rows]
    close(got[-1][0], x.cpu().double() @ w.cpu().double().T, "plain")
    for y in got[:-1]:
        for a, b in zip(y, got[-1]):
            assert torch.equal(a, b[: a.shape[0]])


@pytest.mark.parametrize("K,N,rows", [(2048, 16384, (41, 64, 100, 128)), (1088, 32768, (64, 128))])
def test_large_weights_of_one_row_block_past_the_caches(ops, K, N, rows):
    """64 MiB of weights and more, which go past the caches where one block holds all rows, in every shared tile: bit for bit the same columns of fewer weights."""
    x, w = rnd(max(rows), K, seed=63).cuda(), rnd(N, K, seed=64, scale=K ** -0.5).cuda()
    n = N // 4 * 3               # (below the line, and still no round of the tiles whose K is split over the waves)
    few = torch.cat([w[: n // 2], w[N // 2: N // 2 + n // 2]])
    for M in rows:
        for _ in range(2):   # (the second time they are where the first left them)
            assert torch.equal(ops.linear_act(x[:M], w)[:, :n], ops.linear_act(x[:M], w[:n]))
            assert torch.equal(ops.gated_glu(x[:M], w, 2.0)[:, : n // 2], ops.gated_glu(x[:M], few, 2.0))
    close(ops.linear_act(x, w)[:, -64:], x.cpu().double() @ w[-64:].cpu().double().T, "plain")


@pytest.mark.parametrize("M,N,K", [(65, 2720, 512), (96, 2692, 576), (190, 2640, 1088), (330, 5300, 192), (161, 4168, 128), (350, 1352, 512)])
def test_column_tiles_whose_last_turn_is_not_every_xcds(ops, M, N, K):
    """A round of tiles that is more than one where every XCD counts as many column tiles as the first: they go in runs.  Every row and column, single and gated."""
    x, w, s = rnd(M, K, seed=81).cuda(), rnd(2 * N, K, seed=82, scale=K ** -0.5).cuda(), rnd(M, seed=83).cuda()
    z = x.cpu().double() @ w.cpu().double().T
    out = torch.full((M + 1, N + 4), 7.0, device="cuda", dtype=BF)
    ops.linear_act(x, w[:N], out=out[:M, :N])
    close(out[:M, :N].cpu(), z[:, :N], "plain")
    assert bool((out[M] == 7).all()) and bool((out[:, N:] == 7).all())
    close(ops.linear_act(x, w[:N], out_f32=True).cpu(), z[:, :N], "fp32")
    for n in (N, N // 8 * 4):
        g, u = z[:, :n], z[:, n: 2 * n]
        got = ops.grouped_gemm_gateup_silu(x, w[: 2 * n].unsqueeze(0), None, None, M).cpu()
        ref = (torch.nn.functional.silu(g.to(BF).double()).to(BF).double() * u.to(BF).double()).to(BF)
        assert_close_bf16(got, ref, SILU[0], SILU[1], atol=SILU[2], what=f"gate|up {n}")
    got = ops.grouped_gemm_down(x, w[:N].unsqueeze(0), None, s, 1).cpu()
    assert_close_bf16(got, (z[:, :N].to(BF).double() * s.cpu().double()[:, None]).to(BF), 2, 0.05, atol=2 ** -8, what="down")


def act64(kind, a, b, z, ops):
    n = torch.arange(z.shape[1])
    if kind == ops.ACT_SOFTCAP:
        return N_.soft_cap(z, a)
    if kind == ops.ACT_XIELU:
        return torch.where(z > 0, a * z * z + 0.5 * z, b * (torch.expm1(z) - z) + 0.5 * z)
    s = torch.sigmoid(z)
    if kind == ops.ACT_RELU2_GATE:
        return torch.where(n >= b, s, torch.where(n < a, torch.relu(z) ** 2, z))
    return torch.where(n >= a, s, z * s if kind == ops.ACT_SILU_GATE else z)


# rows that end in each 16-row piece of a tile, columns that end inside one: shared and split tiles, then the streaming kernels (few rows, K off the 64-wide chunks),
# then the tiled kernel: 256-row blocks in the lean and in the plain form, 128-row blocks in the plain form, several rounds of few rows
@pytest.mark.parametrize("M,N,K", [(65, 8200, 128), (81, 8200, 128), (97, 16424, 64), (128, 20000, 64), (113, 520, 576), (49, 40, 320), (300, 4104, 192),
                                   (2, 520, 512), (16, 4104, 768), (17, 9736, 512), (33, 520, 200), (49, 40, 72), (95, 136, 200), (200, 72, 264),
                                   (8500, 1032, 64), (8500, 1036, 64), (1300, 2052, 72), (1030, 15368, 64)])
def test_every_activation(ops, M, N, K):
    """Every kind, fp32 and bf16 rows.  fp32: of the sums that the same call without an activation stores, off by the functions' own error (a few ulp of the
    terms; xIELU's cancel: 2^-20 of the largest).  bf16: one rounding of that value."""
    x, w = rnd(M, K, seed=71).cuda(), rnd(N, K, seed=72, scale=K ** -0.5).cuda()
    x[M // 2, 0], x[M - 1, :2] = float("inf"), float("inf")       # infinite sums, and NaN where both signs meet
    z = ops.linear_act(x, w, out_f32=True).cpu().double()
    assert torch.isinf(z).any() and torch.isnan(z).any()
    for kind, a, b in ((ops.ACT_SOFTCAP, 3.0, 0.0), (ops.ACT_XIELU, 0.8, 0.7), (ops.ACT_GATE, N // 2, 0.0), (ops.ACT_SILU_GATE, N // 2, 0.0), (ops.ACT_SILU_GATE, N, 0.0),
                       (ops.ACT_RELU2_GATE, N // 2, N // 2 + 24)):
        ref, what = act64(kind, a, b, z, ops), f"kind {kind}"
        fine = torch.isfinite(z) & torch.isfinite(ref)
        y = ops.linear_act(x, w, act=(kind, float(a), float(b)), out_f32=True).cpu().double()
        assert ((y - ref).abs()[fine] <= 2.0 ** -20 * (1 + ref.abs() + z.abs())[fine]).all(), what
        y16 = ops.linear_act(x, w, act=(kind, float(a), float(b))).cpu()
        assert_close_bf16(y16.masked_fill(~fine, 0), ref.to(BF).masked_fill(~fine, 0), 1, 0.05, atol=2 ** -9, what=what)
        if kind in (ops.ACT_SOFTCAP, ops.ACT_GATE):   # of infinite sums: the cap, or gates of 0 and 1 (passed ones as they are)
            inf = torch.isinf(z)
            assert torch.equal(y[inf], ref[inf]) and torch.equal(y16.double()[inf], ref[inf])
            assert torch.isnan(y[torch.isnan(z) & torch.isnan(ref)]).all()
