"""Dafolorn on the GPU: every kernel against a plain evaluation, and the model through the engine's own scheduler, cache, state
and step function against oracle/dafolorn_oracle.py."""
import types

import pytest
import torch

from dafolorn_util import CONFIGS, LIMIT, config, distance, layer, make_model, run_cut, session, tokens
from oracle import dafolorn_oracle as O

pytestmark = [pytest.mark.gpu, pytest.mark.timeout(120)]
DT = {"float32": torch.float32, "bfloat16": torch.bfloat16}


def g(seed):
    return torch.Generator().manual_seed(seed)


def dev(t, dtype=None):
    return t.to("cuda", dtype) if dtype else t.to("cuda")


def i32(x):
    return torch.as_tensor(x, dtype=torch.int32, device="cuda")


# ---- kernels --------------------------------------------------------------------------------------------------------------
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("M,N,K", [(1, 40, 72), (3, 104, 264), (40, 520, 96), (100, 264, 136), (200, 72, 128), (300, 512, 1024)])
def test_linear_act(dtype, M, N, K):
    from nanovllm import hip_ops
    dt = DT[dtype]
    x, w, b = torch.randn(M, K, generator=g(1)).to(dt), (torch.randn(N, K, generator=g(2)) * K ** -0.5).to(dt), torch.randn(N, generator=g(3)).to(dt)
    z = x.double() @ w.double().T + b.double()
    p, q = torch.tensor(0.3).double(), torch.tensor(-0.8).double()
    xi = (hip_ops.ACT_XIELU, float(O.softplus(p)), float(0.5 + O.softplus(q)))
    for act, ref in ((hip_ops.NO_ACT, z), (xi, O.xielu(z, p, q)), ((hip_ops.ACT_SOFTCAP, 1.5, 0.0), O.soft_cap(z, 1.5))):
        for f32 in (False, True):
            y = hip_ops.linear_act(dev(x), dev(w), dev(b), act, out_f32=f32)
            tol = 2e-5 if y.dtype == torch.float32 else 1e-2
            assert torch.allclose(y.cpu().double(), ref, rtol=tol, atol=tol), (act[0], f32)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("width", [72, 76, 1040])
def test_embed_rows(dtype, width):
    from nanovllm import hip_ops
    wp = hip_ops.round8(width)
    table = torch.randn(50, width, generator=g(1)).to(DT[dtype])
    ids = torch.tensor([3, 49, 0, 3, 17])
    cat = torch.full((5, 2 * wp), 7.0, dtype=DT[dtype], device="cuda")
    x = hip_ops.embed_rows(dev(ids), dev(table), wp, cat[:, wp:]).cpu()
    assert torch.equal(x[:, :width], table[ids].float()) and torch.all(x[:, width:] == 0)
    assert torch.equal(cat[:, wp:].cpu().float(), x) and torch.all(cat[:, :wp] == 7)


def _portions(lens_per_step):
    """Steps of (sequence, start, length) -> metadata of glm_seq_norm."""
    at, par, steps = {}, {}, []
    for step in lens_per_step:
        pos, seq_of, qs, sin, sout = [], [], [0], [], []
        for s, (seq, n) in enumerate(step):
            a = at.get(seq, 0)
            pos += range(a, a + n)
            seq_of += [s] * n
            qs.append(qs[-1] + n)
            p = par.get(seq, 0)
            sin.append(2 * seq + p)
            sout.append(2 * seq + 1 - p)
            at[seq], par[seq] = a + n, 1 - p
        steps.append((step, types.SimpleNamespace(pos=i32(pos), seq_of=i32(seq_of), q_start=i32(qs), state_in=i32(sin), state_out=i32(sout))))
    return steps


@pytest.mark.parametrize("width,taps", [(64, 2), (76, 3), (200, 4), (1032, 5), (72, 8), (64, 13)])
@pytest.mark.parametrize("y_kind", ["none", "bf16", "f32", "slabs"])
def test_seq_norm(width, taps, y_kind):
    from nanovllm import hip_ops
    wp, tp, eps = hip_ops.round8(width), hip_ops.seq_norm_taps(taps), 1e-5
    L = {0: 700, 1: 41, 2: 9}
    pad = lambda t: torch.nn.functional.pad(t, (0, wp - width))  # noqa: E731
    x = {s: torch.randn(n, width, generator=g(s)) for s, n in L.items()}
    y = {s: torch.randn(n, width, generator=g(10 + s)).to(torch.bfloat16).float() for s, n in L.items()}
    gp, gq = 1 + 0.2 * torch.randn(width, generator=g(20)), 1 + 0.2 * torch.randn(width, generator=g(21))
    cw = torch.randn(width, taps, generator=g(22)).to(torch.bfloat16).float()
    conv = torch.zeros(tp, wp)
    conv[tp - taps:, :width] = cw.T
    ref_x = {s: (x[s].double() + O.unit_rms(y[s].double(), eps) * gp.double()) if y_kind != "none" else x[s].double() for s in L}
    ref_h = {s: O.canon(O.unit_rms(ref_x[s], eps) * gq.double(), cw.double()) for s in L}
    plans = [[[(0, 700), (1, 41), (2, 9)]],
             [[(0, 530), (1, 1)], [(1, 1), (0, 2), (2, 1)], [(1, 1), (2, 2)], [(0, 168), (2, 6), (1, 38)]],
             [[(2, 1)], [(2, 1), (1, 17)], [(1, 24), (2, 1)], [(2, 1)], [(2, 5), (0, 1)], [(0, 699)]]]
    outs = []
    for plan in plans:
        state = torch.full((6, max(tp - 1, 1), wp), float("nan"), device="cuda")
        at, got_h, got_x = {s: 0 for s in L}, {s: [] for s in L}, {s: [] for s in L}
        for step, meta in _portions(plan):
            cut = lambda t: torch.cat([pad(t[s][at[s]: at[s] + n]) for s, n in step])  # noqa: E731
            xs, ys = dev(cut(x)), cut(y)
            yk = {"none": None, "bf16": dev(ys, torch.bfloat16), "f32": dev(ys),
                  "slabs": hip_ops.PartialSum(dev(torch.stack([ys * 0.25, ys * 0.75])))}[y_kind]
            xo, h = hip_ops.seq_norm(xs, width, eps, y=yk, g_post=dev(pad(gp)), g_pre=dev(pad(gq)), conv=(dev(conv, torch.bfloat16), state), meta=meta,
                                     act_dtype=torch.float32)
            assert torch.all(h[:, width:] == 0)
            r = 0
            for s, n in step:
                got_h[s].append(h[r: r + n, :width].cpu())
                got_x[s].append(xo[r: r + n, :width].cpu())
                r, at[s] = r + n, at[s] + n
        got_h = {s: torch.cat(v) for s, v in got_h.items()}
        for s in L:
            n = got_h[s].shape[0]
            assert torch.allclose(got_h[s].double(), ref_h[s][:n], rtol=1e-5, atol=2e-5), s
            assert torch.allclose(torch.cat(got_x[s]).double(), ref_x[s][:n], rtol=1e-5, atol=1e-5)
        outs.append(got_h)
    for s in L:   # however the sequence was cut: beyond the order of a row's sum nothing may differ
        for o in outs[1:]:
            assert torch.allclose(o[s], outs[0][s][: o[s].shape[0]], rtol=1e-6, atol=2e-6)


@pytest.mark.parametrize("width,taps", [(72, 2), (520, 3), (1032, 4), (2056, 6), (4096, 8), (4104, 4)])
@pytest.mark.parametrize("lens", [[1] * 192, [1] * 193, [3, 1, 2, 5, 8, 1], [130, 1, 2, 59], [2, 0, 1]])
def test_seq_norm_is_one_launch_whatever_the_portions(width, taps, lens, monkeypatch):
    """The launch is chosen by what is known of the portions: rows, stream and state of all of them have the same bits."""
    from nanovllm import hip_ops
    wp, T, S = hip_ops.round8(width), sum(lens), len(lens)
    lib = hip_ops.load_library()
    start = [0, 1, 2, 40]   # (portions at the sequence's start need less of the state)
    pos = i32([start[s % 4] + p for s, n in enumerate(lens) for p in range(n)])
    meta = types.SimpleNamespace(pos=pos, seq_of=i32([s for s, n in enumerate(lens) for _ in range(n)]), q_start=i32([sum(lens[:s]) for s in range(S + 1)]),
                                 state_in=i32(list(range(S))), state_out=i32([S + s if s % 5 != 4 else -1 for s in range(S)]))
    x, gain, conv = torch.randn(T, wp, device="cuda"), torch.randn(wp, device="cuda"), torch.randn(taps, wp, device="cuda").bfloat16()
    state = torch.randn(2 * S, taps - 1, wp, device="cuda")
    for y in (hip_ops.PartialSum(torch.randn(2, T, wp, device="cuda")), torch.randn(T, wp, device="cuda").bfloat16(), hip_ops.PartialSum(torch.randn(7, T, wp, device="cuda"))):
        got = []
        for n_seq in (None, 0, max(1, T - 1)):

            class Library:
                def __getattr__(self, name):
                    return getattr(lib, name)

                def glm_seq_norm_step(self, *a):
                    return lib.glm_seq_norm_step(*a[:26], n_seq if n_seq is not None else a[26], *a[27:])

            monkeypatch.setattr(hip_ops, "load_library", Library)
            kept = state.clone()
            got.append(hip_ops.seq_norm(x, width, 1e-5, y=y, g_post=gain, g_pre=gain, conv=(conv, kept), meta=meta) + (kept,))
            monkeypatch.undo()
        for other in got[1:]:
            assert all(torch.equal(a, b) for a, b in zip(got[0], other))


@pytest.mark.parametrize("width,taps", [(64, 1), (72, 2), (520, 3), (1032, 4), (2048, 4), (4104, 4), (2056, 6), (4096, 8), (8192, 1)])
@pytest.mark.parametrize("lens", [[700, 1, 41, 2, 9, 600, 3, 1500], [4100]])
def test_seq_norm_stream_of_bf16(width, taps, lens):
    """Runs of rows with activations in bf16 (loads a row ahead, stores through buffers) against the form for fp32 rows: the same bits, h and the cast row rounded.  Rows of
    the cast start anywhere and what is around them stays; a launch without y, without h, without a cast and one of gathered rows."""
    from nanovllm import hip_ops
    wp, T, S = hip_ops.round8(width), sum(lens), len(lens)
    pos = i32([(40 if s % 3 == 1 else 0) + p for s, n in enumerate(lens) for p in range(n)])
    meta = types.SimpleNamespace(pos=pos, seq_of=i32([s for s, n in enumerate(lens) for _ in range(n)]), q_start=i32([sum(lens[:s]) for s in range(S + 1)]),
                                 state_in=i32(list(range(S))), state_out=i32([S + s if s % 5 != 4 else -1 for s in range(S)]))
    torch.manual_seed(width)
    x, gain, gp = torch.randn(T, wp, device="cuda"), torch.randn(wp, device="cuda"), torch.randn(wp, device="cuda")
    y = torch.randn(T, wp, device="cuda").bfloat16()
    state = torch.randn(2 * S, max(taps - 1, 1), wp, device="cuda")
    conv = (torch.randn(taps, wp, device="cuda").bfloat16(), state) if taps > 1 else None
    index = torch.randperm(T, device="cuda", dtype=torch.int32)
    for yv, g, shift, rows in [(y, gain, 0, None), (y, gain, 1, None), (y, gain, 4, None), (y, None, 8, None), (None, gain, None, None)] + ([(y, gain, None, index)] if taps == 1 else []):
        got = []
        for dtype in (torch.float32, torch.bfloat16):
            kept = state.clone()
            cast = torch.full((T, wp + 16), 7.0, device="cuda", dtype=dtype) if shift is not None else None
            xo, h = hip_ops.seq_norm(x, width, 1e-5, y=yv, g_post=gp, g_pre=g, conv=(conv[0], kept) if conv and g is not None else None, meta=meta, rows=rows, act_dtype=dtype,
                                     x_cast=cast[:, shift: shift + wp] if cast is not None else None)
            got.append([xo, kept] + ([] if h is None else [h.bfloat16()]) + ([] if cast is None else [cast.bfloat16()]))
        assert all(torch.equal(a, b) for a, b in zip(*got))
        if shift is not None:
            c = got[1][-1]
            assert bool((c[:, :shift] == 7).all()) and bool((c[:, shift + wp:] == 7).all()) and torch.equal(c[:, shift: shift + wp], got[1][0].bfloat16())


@pytest.mark.parametrize("width,taps", [(64, 1), (72, 2), (520, 3), (1032, 4), (2048, 4), (4104, 4), (200, 6), (2056, 6), (2048, 8), (4096, 8), (8192, 1)])
@pytest.mark.parametrize("more", [600, 2700, 9000])
def test_seq_norm_rows_alone_and_in_runs(width, taps, more):
    """Rows of a step of 300, each in a workgroup of its own, and the same rows in a longer step, in runs: the same bits in whatever the launch has, and in the state.
    Slabs in every number from one to nine."""
    from nanovllm import hip_ops
    wp, lens = hip_ops.round8(width), [3, 170, 1, 126]
    T, S = sum(lens), 5
    torch.manual_seed(width + taps)
    x, gain, gp = (torch.randn(*d, device="cuda") for d in ((T + more, wp), (wp,), (wp,)))
    x[:, width:] = 0
    state = torch.randn(2 * S, max(taps - 1, 1), wp, device="cuda")
    conv_w = torch.randn(taps, wp, device="cuda").bfloat16()
    y, slabs = torch.randn(T + more, wp, device="cuda"), torch.randn(9, T + more, wp, device="cuda") if more < 9000 else None
    kinds = [(None, torch.bfloat16), (y.bfloat16(), torch.bfloat16), (y.bfloat16(), torch.float32), (y, torch.float32)] + [(n, torch.bfloat16) for n in range(1, 10) if more < 9000]
    for kind, dtype in kinds:
        for cast, keep, norm in ((True, True, True), (False, False, True), (True, False, False), (False, True, True)):
            if not norm and taps > 1:
                continue
            got = []
            for ls in (lens, lens + [more]):
                n, meta_s = sum(ls), len(ls)
                meta = types.SimpleNamespace(pos=i32([(40 if s % 3 == 1 else 0) + p for s, c in enumerate(ls) for p in range(c)]), seq_of=i32([s for s, c in enumerate(ls) for _ in range(c)]),
                                             q_start=i32([sum(ls[:s]) for s in range(meta_s + 1)]), state_in=i32(list(range(meta_s))), state_out=i32([S + s for s in range(meta_s)]))
                kept, xc = state.clone(), torch.zeros(n, wp, device="cuda", dtype=dtype) if cast else None
                yk = hip_ops.PartialSum(slabs[:kind, :n].contiguous()) if isinstance(kind, int) else None if kind is None else kind[:n].contiguous()
                xo, h = hip_ops.seq_norm(x[:n].contiguous(), width, 1e-5, y=yk, g_post=gp, g_pre=gain if norm else None, conv=(conv_w, kept) if taps > 1 else None, meta=meta, act_dtype=dtype,
                                         x_cast=xc, keep_x=keep)
                got.append([None if t is None else t[:T] for t in (xo, h, xc)] + [kept[: S + 4]])
            for a, b in zip(*got):
                assert (a is None) == (b is None) and (a is None or torch.equal(a, b)), (dtype, cast, keep)


@pytest.mark.parametrize("n", [1, 3, 5, 6, 9, 16])
@pytest.mark.parametrize("T,width", [(1, 64), (7, 2048), (512, 520), (513, 520)])
def test_seq_norm_adds_slabs_in_their_order(n, T, width):
    from nanovllm import hip_ops
    x, g1 = dev(torch.randn(T, width, generator=g(1))), dev(1 + 0.2 * torch.randn(width, generator=g(2)))
    slabs = torch.randn(n, T, width, generator=g(3))
    total = slabs[0].clone()
    for s in slabs[1:]:
        total += s
    run = lambda y: hip_ops.seq_norm(x, width, 1e-5, y=y, g_post=g1, g_pre=g1, act_dtype=torch.float32)  # noqa: E731
    (xa, ha), (xb, hb) = run(hip_ops.PartialSum(dev(slabs))), run(dev(total))
    assert torch.equal(xa, xb) and torch.equal(ha, hb)


def _paged(rows, bs, n_blocks, seed):
    """Latent rows of several sequences scattered over pages; unused memory is NaN."""
    perm = torch.randperm(n_blocks, generator=g(seed)).tolist()
    cache = torch.full((n_blocks, bs, rows[0].shape[1]), float("nan"))
    width = max(-(-r.shape[0] // bs) for r in rows)
    bt = torch.full((len(rows), width), -1, dtype=torch.int32)
    for s, r in enumerate(rows):
        for b in range(-(-r.shape[0] // bs)):
            bt[s, b] = perm.pop()
            part = r[b * bs: (b + 1) * bs]
            cache[bt[s, b], : part.shape[0]] = part
    return cache, bt


def _standout(q, c, t, h, j, gain=40.0):
    """Make key j the one that row (t, h) sees, if it sees it: its score stands out by `gain`."""
    c[j] = q[t, h] / q[t, h].norm() ** 2 * gain


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("H,rank,vdim,window,bs", [(6, 40, 24, 50, 64), (1, 264, 72, 1, 32), (2, 64, 16, 100, 32), (32, 512, 128, 300, 64), (70, 24, 8, 33, 256),
                                                   (16, 1000, 40, 64, 64), (40, 576, 16, 129, 64)])
@pytest.mark.parametrize("n_q,splits", [(1, 0), (1, 1), (1, 5), (2, 0), (37, 3)])
def test_latent_attn(dtype, H, rank, vdim, window, bs, n_q, splits):
    from nanovllm import hip_ops
    dt, rp, S = DT[dtype], hip_ops.round8(rank), 4
    lens = [n_q, window + n_q + 70, window + n_q, 2 * bs + n_q]
    c = [torch.zeros(n, rp) for n in lens]
    for s, n in enumerate(lens):
        c[s][:, :rank] = torch.randn(n, rank, generator=g(s))
    q = torch.zeros(S, n_q, H, rp)
    q[..., :rank] = torch.randn(S, n_q, H, rank, generator=g(9)) * 0.5
    # a key just inside and one just outside the window of a row each, one at a page border
    for s, n in enumerate(lens):
        p = n - 1
        for h, j in ((0, p - window + 1), (H - 1, p - window), (H // 2, (p // bs) * bs)):
            if 0 <= j < n and (h == 0 or H > 2):
                _standout(q[s], c[s], n_q - 1, h, j)
    q, c = q.to(dt), [x.to(dt) for x in c]
    wuv = (torch.randn(H, vdim, rp, generator=g(5)) * rank ** -0.5).to(dt)
    wuv[..., rank:] = 0
    sink = torch.randn(H, generator=g(6)) * 2
    cache, bt = _paged([x.float() for x in c], bs, 64 if bs < 256 else 16, 7)
    pos = torch.cat([torch.arange(n - n_q, n) for n in lens])
    seq_of = torch.arange(S).repeat_interleave(n_q)
    tpt = min(hip_ops.latent_tokens_per_tile(rp, H), n_q)
    tok = [s * n_q + k for s in range(S) for k in range(0, n_q, tpt)]
    cnt = [min(tpt, n_q - k) for s in range(S) for k in range(0, n_q, tpt)]
    out = torch.full((S * n_q, H * vdim), float("nan"), dtype=dt, device="cuda")
    hip_ops.latent_attn(dev(q.reshape(S * n_q, H, rp)), dev(cache, dt), i32(tok), i32(cnt), tpt, i32(pos), i32(seq_of), i32(bt), window, 1.0,
                        dev(sink), dev(wuv), out, num_splits=splits)
    got = out.cpu().double().view(S, n_q, H, vdim)
    for s, n in enumerate(lens):
        vis = O.window_mask(n, window)[n - n_q:]
        for h in range(0, H, max(1, H // 5)):
            a = O.sink_softmax(q[s, :, h].double() @ c[s].double().T, vis, sink[h].double())
            ref = a @ c[s].double() @ wuv[h].double().T
            tol = 5e-5 if dtype == "float32" else 2e-2
            err = (got[s, :, h] - ref).abs().max() / max(1.0, float(ref.abs().max()))
            assert err < tol, (s, h, float(err))


@pytest.mark.parametrize("H,rank,vdim,window,bs,n_q,splits", [
    (16, 256, 128, 1024, 64, 1, 2), (16, 256, 136, 1024, 64, 1, 0), (5, 40, 24, 300, 64, 1, 1), (2, 64, 16, 2400, 32, 1, 1), (32, 256, 16, 600, 64, 1, 1),
    (4, 100, 16, 700, 64, 7, 2), (16, 384, 8, 2000, 128, 1, 7), (16, 512, 24, 1100, 64, 1, 3)])
@pytest.mark.parametrize("extra", [0, 64])
def test_latent_attn_long_ranges(H, rank, vdim, window, bs, n_q, splits, extra):
    """Ranges of six tiles per split and more, where the waves divide the keys: rings that go round, the block table's slice more than once,
    windows that start inside a stage, sequences shorter than a split, two row tiles (which do not); extra columns that make scores only."""
    from nanovllm import hip_ops
    vp, S = hip_ops.round8(rank), 4
    rp = vp + extra
    lens = [n_q, window + n_q + 77, window // 3 + n_q, window + n_q]
    c = [torch.zeros(n, rp) for n in lens]
    q = torch.zeros(S, n_q, H, rp)
    keep = [*range(rank), *range(vp, rp)]
    for s, n in enumerate(lens):
        c[s][:, keep] = torch.randn(n, len(keep), generator=g(s))
    q[..., keep] = torch.randn(S, n_q, H, len(keep), generator=g(9)) * 0.5
    for s, n in enumerate(lens):
        p = n - 1
        for h, j in ((0, p - window + 1), (H - 1, p - window), (H // 2, max(0, p - 100))):
            if 0 <= j < n and (h == 0 or H > 2):
                _standout(q[s], c[s], n_q - 1, h, j)
    bf = torch.bfloat16
    q, c = q.to(bf), [x.to(bf) for x in c]
    wuv = (torch.randn(H, vdim, vp, generator=g(5)) * rank ** -0.5).to(bf)
    wuv[..., rank:] = 0
    sink = torch.randn(H, generator=g(6)) * 2
    cache, bt = _paged([x.float() for x in c], bs, sum(-(-n // bs) for n in lens) + 3, 7)
    pos = torch.cat([torch.arange(n - n_q, n) for n in lens])
    seq_of = torch.arange(S).repeat_interleave(n_q)
    tpt = min(hip_ops.latent_tokens_per_tile(rp, H), n_q)
    tok = [s * n_q + k for s in range(S) for k in range(0, n_q, tpt)]
    cnt = [min(tpt, n_q - k) for s in range(S) for k in range(0, n_q, tpt)]
    out = torch.full((S * n_q, H * vdim), float("nan"), dtype=bf, device="cuda")
    gate = torch.randn(S * n_q, H * vdim, generator=g(8)).to(bf)
    hip_ops.latent_attn(dev(q.reshape(S * n_q, H, rp)), dev(cache, bf), i32(tok), i32(cnt), tpt, i32(pos), i32(seq_of), i32(bt), window, 1.0,
                        dev(sink), dev(wuv), out, num_splits=splits, gate=dev(gate) if extra else None)
    got = out.cpu().double().view(S, n_q, H, vdim)
    for s, n in enumerate(lens):
        vis = O.window_mask(n, window)[n - n_q:]
        for h in range(0, H, max(1, H // 5)):
            a = O.sink_softmax(q[s, :, h].double() @ c[s].double().T, vis, sink[h].double())
            ref = a @ c[s][:, :vp].double() @ wuv[h].double().T
            if extra:
                ref = ref * gate.view(S, n_q, H, vdim)[s, :, h].double()
            # roundings of the weights, the context and the result to bf16: 2 ** -9 each, summed up over what one row holds
            err = (got[s, :, h] - ref).abs().max() / max(1.0, float(ref.abs().max()))
            assert err < 2e-2, (s, h, float(err))


@pytest.mark.parametrize("H,vp,rp", [(16, 256, 256), (16, 512, 576), (5, 40, 48), (16, 384, 384), (16, 512, 512)])
@pytest.mark.parametrize("window,splits", [(1 << 30, 1), (1 << 30, 2), (290, 1), (1 << 30, 7)])
def test_latent_attn_by_the_length_of_a_range(H, vp, rp, window, splits):
    """Ranges around the tiles from which the waves divide the keys, in a block table for far longer ones: right, and the same bits as each sequence
    by itself in a table of its own length."""
    from nanovllm import hip_ops
    bf, vdim, lens = torch.bfloat16, 16, [1, 64, 257, 320, 321, 383, 384, 641, 645, 1300]
    S = len(lens)
    c = [torch.randn(n, rp, generator=g(s)).to(bf) for s, n in enumerate(lens)]
    q = (torch.randn(S, H, rp, generator=g(99)) * 0.3).to(bf)
    wuv, sink = (torch.randn(H, vdim, vp, generator=g(5)) * vp ** -0.5).to(bf), torch.randn(H, generator=g(6))
    cache, bt = _paged([x.float() for x in c], 64, 80, 7)
    wide = torch.full((S, 64), -1, dtype=torch.int32)
    wide[:, : bt.shape[1]] = bt

    def attend(rows, table):
        n = len(rows)
        out = torch.full((n, H * vdim), float("nan"), dtype=bf, device="cuda")
        hip_ops.latent_attn(dev(q[rows]), dev(cache, bf), i32(list(range(n))), i32([1] * n), 1, i32([lens[s] - 1 for s in rows]), i32(list(range(n))), i32(table), window, 1.0,
                            dev(sink), dev(wuv), out, num_splits=splits)
        return out.cpu()
    got = attend(list(range(S)), wide)
    for s, n in enumerate(lens):
        assert torch.equal(got[s], attend([s], bt[s: s + 1, : -(-n // 64)])[0]), n
        vis = O.window_mask(n, window)[n - 1:]
        for h in range(0, H, 4):
            ref = O.sink_softmax(q[s, h].double()[None] @ c[s].double().T, vis, sink[h].double()) @ c[s][:, :vp].double() @ wuv[h].double().T
            # roundings of the weights, the context and the result to bf16, as above
            assert (got[s].view(H, vdim)[h].double() - ref).abs().max() < 2e-2 * max(1.0, float(ref.abs().max())), (n, h)


@pytest.mark.parametrize("H,dk,dv,window", [(3, 24, 40, 50), (2, 128, 128, 200), (1, 136, 200, 1), (4, 64, 256, 64), (2, 200, 64, 1000), (2, 256, 256, 129)])
def test_window_attn_prefill(H, dk, dv, window):
    from nanovllm import hip_ops
    lens, hist = [300, 2, 129, 64], [0, min(window - 1, 77), window - 1, min(3, window - 1)]
    ks = [0]
    for n, h in zip(lens, hist):
        ks.append(ks[-1] + n + h)
    qs = [0]
    for n in lens:
        qs.append(qs[-1] + n)
    q = torch.randn(qs[-1], H, dk, generator=g(1)) * 0.7
    k, v = torch.randn(ks[-1], H, dk, generator=g(2)) * 0.7, torch.randn(ks[-1], H, dv, generator=g(3))
    for s in range(len(lens)):   # keys that stand out: just inside the window of the last row, just outside, the first key
        i = hist[s] + lens[s] - 1
        for h, j in ((0, i - window + 1), (H - 1, i - window), (H - 1, 0)):
            if 0 <= j:
                k[ks[s] + j, h] = q[qs[s + 1] - 1, h] / q[qs[s + 1] - 1, h].norm() ** 2 * 30
    q, k, v = (t.to(torch.bfloat16) for t in (q, k, v))
    sink = torch.randn(H, generator=g(4)) * 2
    tiles = [(s, o) for s, n in enumerate(lens) for o in range(0, n, 128)]
    kv = torch.cat([k.reshape(ks[-1], -1), v.reshape(ks[-1], -1)], 1).cuda()
    out = torch.full((qs[-1], H * dv), float("nan"), dtype=torch.bfloat16, device="cuda")
    hip_ops.window_attn_prefill(dev(q.reshape(qs[-1], -1)), kv[:, : H * dk], kv[:, H * dk:], out, i32(qs), i32(ks), i32([t[0] for t in tiles]),
                                i32([t[1] for t in tiles]), H, dk, dv, window, 1.0, dev(sink))
    got = out.cpu().double().view(-1, H, dv)
    for s, n in enumerate(lens):
        vis = O.window_mask(n + hist[s], window)[hist[s]:]
        for h in range(H):
            a = O.sink_softmax(q[qs[s]: qs[s + 1], h].double() @ k[ks[s]: ks[s + 1], h].double().T, vis, sink[h].double())
            ref = a @ v[ks[s]: ks[s + 1], h].double()
            assert (got[qs[s]: qs[s + 1], h] - ref).abs().max() < 4e-2, (s, h)


@pytest.mark.parametrize("H,dk,dv", [(2, 128, 128), (3, 24, 40), (2, 192, 128), (1, 256, 256), (2, 72, 104)])
def test_window_attn_prefill_gate(H, dk, dv):
    """Rows behind whole tiles and heads narrower than theirs, gates in rows of a pitch of their own."""
    from nanovllm import hip_ops
    lens, window = [129, 1, 64, 273], 90
    qs = [0, 129, 130, 194, 467]
    T = qs[-1]
    q, k, v = (torch.randn(T, H * d, generator=g(i)).to(torch.bfloat16) for i, d in ((1, dk), (2, dk), (3, dv)))
    sink, kv = dev(torch.randn(H, generator=g(4))), torch.cat([k, v], 1).cuda()
    wide = torch.randn(T, H * dv + 12, generator=g(5)).to(torch.bfloat16)
    gate = dev(wide)[:, 4: 4 + H * dv]
    tiles = [(s, o) for s, n in enumerate(lens) for o in range(0, n, 128)]
    got = []
    for gt in (None, gate):
        out = torch.full((T, H * dv + 4), float("nan"), dtype=torch.bfloat16, device="cuda")
        hip_ops.window_attn_prefill(dev(q), kv[:, : H * dk], kv[:, H * dk:], out[:, : H * dv], i32(qs), i32(qs), i32([t[0] for t in tiles]), i32([t[1] for t in tiles]), H, dk, dv,
                                    window, dk ** -0.5, sink, gate=gt)
        assert out[:, H * dv:].isnan().all()
        got.append(out[:, : H * dv].cpu().double())
    # the same sums in 32 bits, rounded to bf16 once in front of the factor (here) and once behind it: 2 ** -8 of the value each, at most
    ref = got[0] * wide[:, 4: 4 + H * dv].double()
    assert ((got[1] - ref).abs() <= 2 ** -7 * ref.abs() + 1e-30).all()


@pytest.mark.parametrize("H,dk,dv", [(2, 128, 128), (3, 24, 40), (2, 192, 128), (1, 256, 256)])
@pytest.mark.parametrize("scale", [-0.3, 0.0, -0.0, -1e-40, 1e-40])
def test_window_attn_prefill_any_scale(H, dk, dv, scale):
    """A scale below zero turns the scores round, with zero (or what is as good as zero) every visible key weighs the same: hidden keys stay hidden."""
    from nanovllm import hip_ops
    n, window, rotp = 300, 90, 8
    q, k, v = torch.randn(n, H, dk, generator=g(1)).bfloat16(), torch.randn(n, H, dk, generator=g(2)).bfloat16(), torch.randn(n, H, dv, generator=g(3)).bfloat16()
    sink, vis = torch.randn(H, generator=g(4)), O.window_mask(n, window)
    tiles = ([0, 0, 0], [0, 128, 256])
    for kr in (False, True):
        rot = {}
        if kr:      # the last columns of the keys in rows of their own (one head's for all), not turned
            k[:, :, dk - rotp:] = k[:, :1, dk - rotp:]
            rot = dict(kr=dev(k[:, 0, dk - rotp:].contiguous()), cs=torch.tensor([1.0, 0.0], device="cuda").repeat(n * rotp // 2).view(n, rotp))
        kk = k[:, :, : dk - rotp] if kr else k
        kv = torch.cat([kk.reshape(n, -1), v.reshape(n, -1)], 1).cuda()
        out = torch.full((n, H * dv), float("nan"), dtype=torch.bfloat16, device="cuda")
        hip_ops.window_attn_prefill(dev(q.reshape(n, -1)), kv[:, : kk.shape[1] * kk.shape[2]], kv[:, kk.shape[1] * kk.shape[2]:], out, i32([0, n]), i32([0, n]),
                                    i32(tiles[0]), i32(tiles[1]), H, dk, dv, window, scale, dev(sink), **rot)
        got = out.cpu().double().view(n, H, dv)
        for h in range(H):
            ref = O.sink_softmax(scale * (q[:, h].double() @ k[:, h].double().T), vis, sink[h].double()) @ v[:, h].double()
            # weights and result in bf16, 2 ** -9 each, of values around 1
            assert (got[:, h] - ref).abs().max() < 2e-2, (kr, h)


@pytest.mark.parametrize("H,dk,dv,rotp", [(3, 24, 40, 0), (2, 72, 40, 0), (2, 72, 40, 8), (2, 136, 200, 0), (1, 200, 136, 8), (2, 192, 128, 64)])
def test_window_attn_prefill_padding_is_zero(H, dk, dv, rotp):
    """What a head lacks of its tile's columns, and the keys behind the last one, count as zeros whatever the kernel before left in the shared memory: here not-a-numbers."""
    from nanovllm import hip_ops
    def run(q, kk, v, heads, dk, dv, n, **rot):
        kv = torch.cat([kk.reshape(n, -1), v.reshape(n, -1)], 1).cuda()
        out = torch.full((n, heads * dv), float("nan"), dtype=torch.bfloat16, device="cuda")
        tiles = list(range(0, n, 128))
        hip_ops.window_attn_prefill(dev(q.reshape(n, -1)), kv[:, : heads * (dk - rot_cols(rot))], kv[:, heads * (dk - rot_cols(rot)):], out, i32([0, n]), i32([0, n]),
                                    i32([0] * len(tiles)), i32(tiles), heads, dk, dv, 4096, 0.5 * dk ** -0.5, dev(torch.zeros(heads)), **rot)
        return out.cpu().double().view(n, heads, dv)
    rot_cols = lambda rot: rot["kr"].shape[1] if rot else 0  # noqa: E731
    n = 171
    q, k, v = (torch.randn(n, H, d, generator=g(i)).bfloat16() for i, d in ((1, dk), (2, dk), (3, dv)))
    rot = {}
    if rotp:
        k[:, :, dk - rotp:] = k[:, :1, dk - rotp:]
        rot = dict(kr=dev(k[:, 0, dk - rotp:].contiguous()), cs=torch.tensor([1.0, 0.0], device="cuda").repeat(n * rotp // 2).view(n, rotp))
    up = lambda d: next(t for t in (64, 128, 192, 256) if d <= t)  # noqa: E731
    for wk, wv in ((up(dk), up(dv)), (256, 256)):
        bad = torch.full((768, 64, wk), float("nan")).bfloat16()
        assert run(bad, bad, bad[:, :, :1].expand(-1, -1, wv), 64, wk, wv, 768).isnan().all()
        got = run(q, k[:, :, : dk - rotp] if rotp else k, v, H, dk, dv, n, **rot)
        for h in range(H):
            ref = O.sink_softmax(0.5 * dk ** -0.5 * (q[:, h].double() @ k[:, h].double().T), O.window_mask(n, 4096), torch.tensor(0.0).double()) @ v[:, h].double()
            # weights and result in bf16, 2 ** -9 each, of values up to about 4
            assert (got[:, h] - ref).abs().max() < 2e-2, (wk, wv, h)


# ---- the model through the engine -------------------------------------------------------------------------------------------
@pytest.fixture(scope="module", params=list(CONFIGS))
def model(request, tmp_path_factory):
    path = tmp_path_factory.mktemp(request.param)
    cfg, t = make_model(path, request.param, seed=len(request.param))
    toks = tokens(cfg, 420, 3)
    return types.SimpleNamespace(name=request.param, path=path, cfg=cfg, t=t, toks=toks, ref=O.forward(cfg, t, toks))


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_layers(model, dtype):
    """The residual stream after every layer run of one prompt."""
    from nanovllm.engine.sequence import Sequence
    from nanovllm.engine.step_batch import build_step
    ref = []
    O.forward(model.cfg, model.t, model.toks[:150], layers_out=ref)
    with session(model.path, dtype, 192) as s:
        r, sch = s.engine.model_runner, s.scheduler
        seq = Sequence(model.toks[:150])
        host, on_device, _ = build_step([sch.feed(seq, 150, [])], r.model, r.block_size)
        tap = []
        with torch.inference_mode():
            r.model(on_device(r._to_device(host)), residual_tap=tap)
        assert len(tap) == len(ref) == len(r.model.runs)
        for i, (a, b) in enumerate(zip(tap, ref)):
            assert distance(a.cpu(), b) < LIMIT[dtype], f"layer run {i}"


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_whole_against_cuts(model, dtype):
    """A whole prompt, portions of many sizes down to two tokens, token-by-token decoding: the same logits, at every position.
    Pages and slots are used again by every run."""
    with session(model.path, dtype, 448) as s:
        for cuts in ([420], [200, 1], [37, 64, 2, 2, 3, 130, 5, 1, 1, 40], [1, 2, 2, 17, 64, 1, 1, 96, 2, 33], [129]):
            assert distance(run_cut(s, model.toks, cuts), model.ref) < LIMIT[dtype], cuts


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_unequal_batches(model, dtype):
    """Up to four live requests, portions beside single tokens, requests that pause, end and make room for others."""
    ref = {n: O.forward(model.cfg, model.t, model.toks[o: o + n]) for n, o in ((1, 5), (23, 11), (150, 100), (97, 200), (260, 0), (61, 300))}
    off = {1: 5, 23: 11, 150: 100, 97: 200, 260: 0, 61: 300}
    plan = [{260: 90, 23: 2}, {260: 1, 23: 1, 150: 80}, {150: 2, 97: 64}, {260: 130, 150: 1, 97: 1, 23: 20}, {1: 1, 260: 2, 150: 40, 97: 30},
            {61: 50, 260: 1, 150: 1, 97: 2}, {61: 1, 260: 36}, {61: 10, 150: 26}]
    at, got = {n: 0 for n in ref}, {n: [] for n in ref}
    with session(model.path, dtype, 640, eager=False) as s:
        for step in plan:
            entries, end = [], []
            for n, k in step.items():
                entries.append({"id": n, "tokens": model.toks[off[n] + at[n]: off[n] + at[n] + k], "want": list(range(k))})
                at[n] += k
                if at[n] == n:
                    end.append(n)
            out, r = s.step(entries, end), 0
            for n, k in step.items():
                got[n].append(out[r: r + k])
                r += k
        bm = s.scheduler.block_manager
        assert len(bm.free_block_ids) + sum(b >= 0 for q in s.live.values() for b in q.block_table) == 10
    for n in ref:
        o = torch.cat(got[n])
        assert distance(o, ref[n][: o.shape[0]]) < LIMIT[dtype], n


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_long_decoding_graphs_and_eager(dtype, tmp_path):
    """Hundreds of decoded tokens: windows pass over decoded tokens and page borders, pages behind the windows are given back;
    the captured step replays between other work and equals the eager one."""
    cfg = config(64, 96, 4, [layer(4, 16, 24, 40, 70, 72), layer(3, 24, 16, 56, 5, 72)], (0, 2, 2), 10.0)
    cfg, t = make_model(tmp_path, cfg, 1)
    toks = tokens(cfg, 330, 2)
    ref = O.forward(cfg, t, toks)
    outs = []
    for eager in (True, False):
        with session(tmp_path, dtype, 192, eager=eager) as s:   # fewer pages than tokens: 330 tokens need the windows' trimming
            outs.append(run_cut(s, toks, [9, 1]))
            assert s.engine.model_runner.step_graphs if not eager else True
    assert distance(outs[0], ref) < LIMIT[dtype] and distance(outs[1], ref) < LIMIT[dtype]
    assert torch.equal(outs[0], outs[1])


def test_tiny_changes_show(model):
    """A window one token longer or shorter, a sink left out, a lost convolution input, a missing pass vector: planted in the
    plain evaluation, each is far outside the limit the other tests use."""
    import copy
    ref = model.ref[:200]
    for i in range(len(model.cfg["layers"])):
        for d in (-1, 1):
            c = copy.deepcopy(model.cfg)
            c["layers"][i]["mixer"]["mask"]["size"] += d
            if 0 < c["layers"][i]["mixer"]["mask"]["size"] < 190:
                assert distance(O.forward(c, model.t, model.toks[:200]), ref) > 10 * LIMIT["float32"], (i, d)
    for name, edit in (("l0.mix.sink", lambda v: v - 30), ("l0.canon1", lambda v: torch.cat([torch.zeros_like(v[:, :1]), v[:, 1:]], 1)),
                       ("l0.mlp.act", lambda v: v.flip(0))):
        t = dict(model.t)
        t[name] = edit(t[name])
        assert distance(O.forward(model.cfg, t, model.toks[:200]), ref) > 10 * LIMIT["float32"], name


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_generate(model, dtype):
    """Greedy generation through LLM.generate: own scheduler with a token budget smaller than the prompts, more requests than
    state slots, preemption for want of pages.  A token may differ from the plain evaluation's only within its rounding."""
    from nanovllm import LLM, SamplingParams
    prompts = [tokens(model.cfg, n, 50 + n) for n in (3, 130, 61, 200, 1, 77)]
    llm = LLM(str(model.path), dtype=dtype, max_num_seqs=3, max_num_batched_tokens=96, max_model_len=512, num_kvcache_blocks=7)
    try:
        out = llm.generate(prompts, SamplingParams(temperature=0.0, max_tokens=12, ignore_eos=True), use_tqdm=False)
        assert len(llm.scheduler.block_manager.free_block_ids) == 7 and len(llm.scheduler.state_manager.free_slots) == 3
    finally:
        llm.exit()
    torch.cuda.empty_cache()
    for p, o in zip(prompts, out):
        got = o["token_ids"]
        assert len(got) == 12
        lg = O.forward(model.cfg, model.t, p + got[:-1])[len(p) - 1:]
        gap = lg.max(-1).values - lg.gather(1, torch.tensor(got)[:, None])[:, 0]
        assert float(gap.max()) <= 6 * LIMIT[dtype] * float(lg.pow(2).mean().sqrt()), gap


def test_memory_sized_pool_and_sampling(tmp_path):
    """Without a given pool the engine sizes it by memory; temperatures above zero sample."""
    from nanovllm import LLM, SamplingParams
    cfg, t = make_model(tmp_path, "tail", 5)
    llm = LLM(str(tmp_path), max_num_seqs=5, max_num_batched_tokens=256, max_model_len=256, gpu_memory_utilization=0.05)
    try:
        assert llm.config.num_kvcache_blocks > 1000
        a, b = (llm.generate([tokens(cfg, 20, 1)], SamplingParams(temperature=x, max_tokens=24, ignore_eos=True), use_tqdm=False)[0]["token_ids"]
                for x in (0.0, 50.0))
        assert len(a) == len(b) == 24 and a != b
    finally:
        llm.exit()
    torch.cuda.empty_cache()
