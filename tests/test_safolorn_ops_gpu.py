"""Every kernel of the latent-attention decoders alone, in both element types, against float64 numpy."""
import numpy as np
import pytest
import torch

import safolorn_cases as C
from conftest import load_pkg
from oracle import safolorn_ref as R

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
DTYPES = [torch.bfloat16, torch.float32]


@pytest.fixture(scope="module")
def D(ops):
    return load_pkg("decoder_ops")


def tol(dt, f32=2e-6, b16=1.2e-2):
    return f32 if dt == torch.float32 else b16


def rnd(rng, *shape, std=1.0, dt=torch.float32):
    return torch.from_numpy(rng.normal(0, std, shape)).to(torch.bfloat16).to(dt).to(DEV)


def f64(t):
    return t.double().cpu().numpy()


def err(got, want):
    return float(np.abs(f64(got) - want).max() / np.abs(want).max())


def rows_of(act):
    return act if isinstance(act, torch.Tensor) else act.unpack()


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("T,H,Hp", [(1, 30, 32), (17, 104, 128), (70, 2100, 2112), (5, 5000, 5024), (3, 9000, 9024)])
def test_stream_norm(D, ops, dt, T, H, Hp):
    rng = np.random.default_rng(T)
    x, y, parts = (torch.zeros((*s, Hp), device=DEV) for s in ((T,), (T,), (2, T)))
    for t in (x, y, parts):
        t[..., :H] = rnd(rng, *t.shape[:-1], H, std=3.0)
    w = torch.zeros(Hp, dtype=dt, device=DEV)
    w[:H] = rnd(rng, H, dt=dt)
    x0 = f64(x)
    kp = ops.KSplitParts(parts.contiguous(), 3, Hp) if dt == torch.bfloat16 else None
    want = x0[:, :H] + (f64(parts).sum(0)[:, :H] if kp else 0) + R.rms(f64(y)[:, :H], 1e-3) * f64(w)[:H]
    frag = ops.FragActivation(T, Hp, DEV, dtype=dt) if dt == torch.bfloat16 else None
    row = torch.empty((T, Hp), dtype=dt, device=DEV)
    D.stream_norm(x, H, 1e-3, 1.7, kp, (y, w), out=frag, out_row=row)
    torch.cuda.synchronize()
    assert err(x[:, :H], want) < 2e-6 and float(x[:, H:].abs().sum()) == 0
    assert err(row[:, :H], R.rms(want, 1e-3) * 1.7) < tol(dt, b16=4e-3) and float(row[:, H:].abs().sum()) == 0
    if frag is not None:
        assert torch.equal(frag.unpack(), row)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("T,width,dim", [(1, 40, 5), (33, 104, 20), (300, 96, 20), (300, 96, 40), (4100, 72, 250), (16, 200, 70)])
def test_token_gate(D, ops, dt, T, width, dim):
    rng = np.random.default_rng(T)
    Hp, N, V = D.pad32(width), D.pad32(dim), 50
    x = torch.zeros((T, Hp), device=DEV)
    x[:, :width] = rnd(rng, T, width)
    Wr = rnd(rng, dim, width, std=2 * width ** -0.5, dt=dt)
    table = rnd(rng, V, 3 * dim, dt=dt)
    ids = torch.from_numpy(rng.integers(0, V, T).astype(np.int32)).to(DEV)
    xs, xa = f64(x)[:, :width], x
    if dt == torch.bfloat16:                              # the stream rounded to 16 bits, with what is pending added to it
        part = torch.zeros((2, T, Hp), device=DEV)
        part[..., :width] = rnd(rng, 2, T, width)
        xs = xs + f64(part).sum(0)[:, :width]
        xa = ops.FragActivation(T, Hp, DEV, dtype=dt)
        D.stream_norm(x, width, 1e-5, parts=ops.KSplitParts(part, 3, Hp), out=xa, raw=True)
        assert err(x[:, :width], xs) < 1e-6 and torch.equal(xa.unpack(), x.to(dt))
    out = rows_of(D.token_gate(xa, D.weight(D.padded(Wr, N, Hp)), table, dim, dim, ids))
    torch.cuda.synchronize()
    want = R.gelu_tanh(xs @ f64(Wr).T) * f64(table)[f64(ids).astype(int)][:, dim:2 * dim]
    assert err(out[:, :dim], want) < tol(dt) and float(out[:, dim:].abs().sum()) == 0


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("T,K,ff", [(1, 64, 64), (20, 96, 224), (64, 64, 96), (100, 64, 160), (4096, 64, 2048)])
def test_clipped_glu(D, ops, dt, T, K, ff):
    """T <= 64: the product as the GEMV's epilogue; 4096: as the persistent GEMM's; between: a launch of its own."""
    rng = np.random.default_rng(T)
    g, u = rnd(rng, ff, K, std=K ** -0.5, dt=dt), rnd(rng, ff, K, std=K ** -0.5, dt=dt)
    x = rnd(rng, T, K, std=2.0, dt=dt)
    gu = torch.cat([g, u])
    frag = dt == torch.bfloat16
    out = D.activation(T, ff, dt, DEV)
    D.gate_up_clipglu(ops.FragActivation.pack(x) if frag else x, D.weight(gu), ops.interleave_gate_up(gu) if frag else None, 1.5, 1.25, 1.702, out)
    torch.cuda.synchronize()
    gs, us = np.minimum(1.5 * f64(x) @ f64(g).T, 1.25), np.clip(1.5 * f64(x) @ f64(u).T, -1.25, 1.25)
    assert err(rows_of(out), gs / (1 + np.exp(-1.702 * gs)) * (us + 1)) < tol(dt)


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("T,H,K,N", [(1, 3, 32, 32), (18, 2, 64, 96), (50, 5, 96, 32), (300, 2, 64, 288)])
def test_head_linear(D, ops, dt, T, H, K, N):
    rng = np.random.default_rng(T)
    x = rnd(rng, T, H * K + 32, dt=dt)
    W = rnd(rng, H, N, K, std=K ** -0.5, dt=dt)
    out = torch.full((T, H, N + 32), 7.0, dtype=dt, device=DEV)
    D.head_linear(x, H * K + 32, K, D.weight(W.view(H * N, K)), H, T, K, N, out, H * (N + 32), N + 32, 0.5)
    want = 0.5 * np.einsum("thk,hnk->thn", f64(x)[:, : H * K].reshape(T, H, K), f64(W))
    torch.cuda.synchronize()
    assert err(out[..., :N], want) < tol(dt, b16=5e-3) and bool((out[..., N:] == 7.0).all())
    if dt == torch.bfloat16:
        f = ops.FragActivation(T, H * N, DEV, dtype=dt)
        D.head_linear(x, H * K + 32, K, D.weight(W.view(H * N, K)), H, T, K, N, f, 0, N, 0.5)
        assert torch.equal(f.unpack(), out[..., :N].reshape(T, H * N))


def latent_case(D, dt, ctxs, H, rank, rot, seed=0, n_extra=3):
    """A cache whose sequences have ctxs[i] tokens, pages scattered and the unused ones poisoned with large values."""
    rng = np.random.default_rng(seed)
    need = [-(-c // 16) for c in ctxs]
    n_pages = sum(need) + n_extra
    NB = D.pad32(rank) // 32 + D.pad32(rot) // 32
    order = rng.permutation(n_pages)
    bt = np.full((len(ctxs) + 1, max(need) + 1), -1, np.int32)
    lat = [rng.normal(size=(c, rank + rot)) for c in ctxs]
    dense = np.full((n_pages, 16, NB * 32), 1e4)
    dense[:, :, rank:D.pad32(rank)] = 0
    dense[:, :, D.pad32(rank) + rot:] = 0
    k = 0
    for i, c in enumerate(ctxs):
        lat[i] = torch.from_numpy(lat[i]).to(torch.bfloat16).double().numpy()
        for b in range(need[i]):
            p = bt[i + 1, b] = order[k]
            k += 1
            n = min(16, c - 16 * b)
            dense[p, :n, :rank] = lat[i][16 * b:16 * b + n, :rank]
            dense[p, :n, D.pad32(rank):D.pad32(rank) + rot] = lat[i][16 * b:16 * b + n, rank:]
    pages = torch.from_numpy(dense).to(dt).to(DEV).view(n_pages, 16, NB, 4, 8).permute(0, 2, 3, 1, 4).contiguous()
    return lat, pages, torch.from_numpy(bt).to(DEV), rng


def attn_want(lat, q, seq, pos, sink, scale, rank):
    T, H, _ = q.shape
    out = np.zeros((T, H, rank))
    for t in range(T):
        kv = lat[seq[t]][: pos[t] + 1]
        for h in range(H):
            s = kv @ q[t, h] * scale
            w = R.sink_softmax(s, sink[h]) if sink is not None else np.exp(s - s.max()) / np.exp(s - s.max()).sum()
            out[t, h] = w @ kv[:, :rank]
    return out


def put_queries(D, q, rank, rot, dt):
    T, H, _ = q.shape
    full = torch.zeros((T, H, D.pad32(rank) + D.pad32(rot)), dtype=dt, device=DEV)
    full[..., :rank] = torch.from_numpy(q[..., :rank]).to(dt)
    full[..., D.pad32(rank):D.pad32(rank) + rot] = torch.from_numpy(q[..., rank:]).to(dt)
    return full


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("H,rank,rot", [(1, 32, 8), (3, 72, 24), (16, 128, 40), (18, 256, 64), (20, 544, 16)])
@pytest.mark.parametrize("sunk", [True, False])
def test_latent_attention_decode(D, dt, H, rank, rot, sunk):
    ctxs = [1, 2, 15, 16, 17, 33, 200, 517]
    lat, pages, bt, rng = latent_case(D, dt, ctxs, H, rank, rot, seed=H)
    seq = list(range(len(ctxs)))
    q = torch.from_numpy(rng.normal(size=(len(ctxs), H, rank + rot))).to(torch.bfloat16).double().numpy()
    sink = rng.normal(2.0, 1.0, H).astype(np.float32) if sunk else None
    scale = 3.0 * (rank + rot) ** -0.5
    args = (put_queries(D, q, rank, rot, dt), pages, bt, torch.tensor([s + 1 for s in seq], dtype=torch.int32, device=DEV),
            torch.tensor([c - 1 for c in ctxs], dtype=torch.int32, device=DEV), torch.from_numpy(sink).to(DEV) if sunk else None, scale, rank, rot)
    want = attn_want(lat, q, seq, [c - 1 for c in ctxs], sink, scale, rank)
    for splits in ([1, 2, 5, 32] if dt == torch.bfloat16 else [1]):
        got = D.latent_attn(*args, max_ctx=max(ctxs), splits=splits)
        torch.cuda.synchronize()
        assert err(got[..., :rank], want) < tol(dt, b16=5e-3), splits
        assert float(got[..., rank:].abs().sum()) == 0
        if splits > 1:                                    # the same, merged on the way through W_uv
            uv = rnd(rng, H, 64, rank, std=rank ** -0.5, dt=dt)
            y = load_pkg("ops").FragActivation(len(ctxs), H * 64, DEV, dtype=dt)
            D.latent_attn_out(*args, splits, D.weight(D.padded(uv, H, 64, D.pad32(rank)).reshape(H * 64, D.pad32(rank))), 64, y)
            torch.cuda.synchronize()
            assert err(y.unpack().view(-1, H, 64), np.einsum("thr,hvr->thv", want, f64(uv))) < 8e-3, splits


@pytest.mark.parametrize("dt", DTYPES)
def test_latent_attention_single_keys_far_and_at_page_borders(D, dt):
    """One key stands out by its rotated part; its latent is what comes back - wherever it lies, and not one token later."""
    rank, rot, H, n = 64, 16, 2, 300
    lat, pages, bt, rng = latent_case(D, dt, [n], H, rank, rot, seed=5)
    spots = [0, 1, 15, 16, 17, 31, 32, 159, 160, 255, 256, 298, 299]
    NBr = D.pad32(rank)
    for j in spots:                                       # key j: rotated part 0 except one coordinate of its own
        v = np.zeros(rot)
        v[spots.index(j)] = 8.0
        lat[0][j, rank:] = v
        p = int(bt[1, j // 16])
        for d in range(rot):
            pages[p, (NBr + d) // 32, (NBr + d) % 32 // 8, j % 16, (NBr + d) % 8] = float(v[d])
    toks = [(j, pos) for j in spots for pos in (j - 1, j, j + 1, n - 1) if 0 <= pos < n]
    q = np.zeros((len(toks), H, rank + rot))
    for t, (j, _) in enumerate(toks):
        q[t, :, rank + spots.index(j)] = 8.0
    got = D.latent_attn(put_queries(D, q, rank, rot, dt), pages, bt, torch.ones(len(toks), dtype=torch.int32, device=DEV),
                        torch.tensor([p for _, p in toks], dtype=torch.int32, device=DEV), None, 1.0, rank, rot, max_ctx=n)
    torch.cuda.synchronize()
    for t, (j, pos) in enumerate(toks):
        e = float(np.abs(f64(got)[t, 0] - lat[0][j, :rank]).max())
        assert (e < 1e-2) if pos >= j else (e > 0.5), (j, pos)
    assert err(got[..., :rank], attn_want(lat, q, [0] * len(toks), [p for _, p in toks], None, 1.0, rank)) < tol(dt, b16=6e-3)


@pytest.mark.parametrize("H,rank,dim,rot,vdim", [(1, 32, 32, 8, 32), (3, 72, 40, 24, 48), (4, 512, 128, 64, 128), (2, 96, 100, 16, 64), (5, 64, 16, 40, 100)])
@pytest.mark.parametrize("scale,layout", [(1.0, "frag"), (-0.7, "rows")])
def test_latent_prefill(D, ops, H, rank, dim, rot, vdim, scale, layout):
    """Keys and values made from the latents: whole prompts, portions in the middle of one, several sequences, scattered pages;
    sharp scores, so that a key too many or too few shows."""
    parts = [(200, 200), (5, 5), (130, 517), (1, 64), (33, 65), (2, 18)]          # (new tokens, context after them)
    dt = torch.bfloat16
    lat, pages, bt, rng = latent_case(D, dt, [c for _, c in parts], H, rank, rot, seed=H)
    dp, vp, rp = D.pad32(dim), D.pad32(vdim), D.pad32(rank)
    T = sum(n for n, _ in parts)
    uk, uv = rnd(rng, H, dim, rank, std=2 * rank ** -0.5), rnd(rng, H, vdim, rank, std=rank ** -0.5)
    qkv = torch.zeros((T, D.pad32(H * dp + 7)), dtype=dt, device=DEV)
    qn = rnd(rng, T, H, dim)
    qkv[:, : H * dp] = D.padded(qn, T, H, dp).reshape(T, H * dp).to(dt)
    qr = rnd(rng, T, H, rot, std=0.5)
    sink = rng.normal(1.0, 1.0, H).astype(np.float32)
    pl = [[int(p) for p in bt[i + 1].tolist() if p >= 0] for i in range(len(parts))]
    plan = D.PrefillPlan([(pl[i], n, c) for i, (n, c) in enumerate(parts)], DEV)
    out = ops.FragActivation(T, H * vp, DEV, dtype=dt) if layout == "frag" else torch.empty((T, H * vp), dtype=dt, device=DEV)
    D.latent_prefill(plan, qkv, D.padded(qr, T, H, D.pad32(rot)).to(dt), pages, D.weight(D.padded(uk, H, dp, rp).reshape(H * dp, rp).to(dt)),
                     D.weight(D.padded(uv, H, vp, rp).reshape(H * vp, rp).to(dt)), torch.from_numpy(sink).to(DEV), scale, rank, dim, rot, vdim, out)
    torch.cuda.synchronize()
    got = f64(rows_of(out)).reshape(T, H, vp)
    bf = lambda a: torch.from_numpy(a).to(dt).double().numpy()
    want, t = np.zeros((T, H, vdim)), 0
    for i, (n, c) in enumerate(parts):
        for h in range(H):
            k, v = bf(lat[i][:, :rank] @ f64(uk)[h].T), bf(lat[i][:, :rank] @ f64(uv)[h].T)   # stored in 16 bits
            for j in range(n):
                pos = c - n + j
                s = (k[: pos + 1] @ f64(qn)[t + j, h] + lat[i][: pos + 1, rank:] @ f64(qr)[t + j, h]) * scale
                want[t + j, h] = R.sink_softmax(s, sink[h]) @ v[: pos + 1]
        t += n
    # a key whose 16-bit rounding falls to the other side moves a sharp softmax a little
    e = np.abs(got[..., :vdim] - want) / np.abs(want).max()
    assert np.quantile(e, 0.999) < 1e-2 and e.max() < 6e-2 and np.abs(got[..., vdim:]).max(initial=0) == 0


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("scaling", [None, C.YARN])
def test_latent_prep(D, dt, scaling):
    """Rotation of queries and key part, norm of the latent, and where they land; token rows of several sequences."""
    H, dim, rank, rot, T = 3, 40, 72, 24, 21
    c = C.rot(1000.0, 20, scaling)
    lat, pages, bt, rng = latent_case(D, dt, [40, 25], H, rank, rot)
    rotation = load_pkg("rotary").Rotation.from_config(c)
    cos, sin = (torch.from_numpy(t).to(DEV) for t in rotation.tables(rot, 64))
    seq = np.array([1] * 12 + [2] * 9, np.int32)
    pos = np.array(list(range(14, 26)) + list(range(16, 25)), np.int32)
    dp = 64
    ld = D.pad32(H * dp + H * rot + rank + rot)
    qkv = rnd(rng, T, ld, dt=dt)
    w = rnd(rng, rank, dt=dt)
    q = torch.full((T, H, D.pad32(rank) + 32), 9.0, dtype=dt, device=DEV)
    off = H * dp
    before = pages.clone()
    D.latent_prep(q, D.pad32(rank), pages, qkv, off, off + H * rot, off + H * rot + rank, 1.25, None, 1e-5, bt, torch.from_numpy(seq).to(DEV), torch.from_numpy(pos).to(DEV),
                  cos, sin, H, rank, rot)
    torch.cuda.synchronize()
    assert torch.equal(pages, before)                     # a layer that reads another layer's latents stores nothing
    D.latent_prep(q, D.pad32(rank), pages, qkv, off, off + H * rot, off + H * rot + rank, 1.25, w, 1e-5, bt, torch.from_numpy(seq).to(DEV), torch.from_numpy(pos).to(DEV),
                  cos, sin, H, rank, rot)
    torch.cuda.synchronize()
    x = 1.25 * f64(qkv)
    wq = R.rotate(f64(qkv)[:, off:off + H * rot].reshape(T, H, rot), pos, c)     # the gain is left to the scores' scale
    assert err(q[..., D.pad32(rank):D.pad32(rank) + rot], wq) < tol(dt, b16=5e-3)
    assert float(q[..., D.pad32(rank) + rot:].abs().sum()) == 0 and bool((q[..., :D.pad32(rank)] == 9.0).all())
    cw = R.rms(x[:, off + H * rot:off + H * rot + rank], 1e-5) * f64(w)
    kw = R.rotate(x[:, off + H * rot + rank:off + H * rot + rank + rot], pos, c)
    rows = pages.permute(0, 3, 1, 2, 4).reshape(pages.shape[0], 16, -1)
    at = np.array([int(bt[s, p // 16]) for s, p in zip(seq, pos)])
    got = f64(rows)[at, pos % 16]
    assert np.abs(got[:, :rank] - cw).max() < tol(dt, b16=1e-2) * 2 and np.abs(got[:, D.pad32(rank):D.pad32(rank) + rot] - kw).max() < tol(dt, b16=1e-2) * 2
    if dt == torch.bfloat16:                              # the same with the unrotated parts lifted beside it
        W = rnd(rng, H, D.pad32(rank), dp, std=dp ** -0.5, dt=dt)
        q2, p2 = torch.empty_like(q), before.clone()
        D.latent_prep(q2, D.pad32(rank), p2, qkv, off, off + H * rot, off + H * rot + rank, 1.25, w, 1e-5, bt, torch.from_numpy(seq).to(DEV),
                      torch.from_numpy(pos).to(DEV), cos, sin, H, rank, rot, D.weight(W.view(H * D.pad32(rank), dp)))
        torch.cuda.synchronize()
        assert torch.equal(p2, pages) and torch.equal(q2[..., D.pad32(rank):], q[..., D.pad32(rank):])
        assert err(q2[..., :D.pad32(rank)], np.einsum("thk,hrk->thr", f64(qkv)[:, :off].reshape(T, H, dp), f64(W))) < 5e-3
    changed = (pages != before).permute(0, 3, 1, 2, 4).reshape(pages.shape[0], 16, -1).any(-1).sum()
    assert int(changed) == T                              # every token one slot, no other slot


@pytest.mark.parametrize("dt", DTYPES)
@pytest.mark.parametrize("T,E,top", [(1, 1, 1), (1, 6, 3), (9, 70, 70), (37, 5, 1), (64, 130, 8), (700, 6, 4), (900, 16, 3)])
def test_experts(D, ops, dt, T, E, top):
    rng = np.random.default_rng(T + E)
    Wd, ff = 72, 40
    Hp = D.pad64(Wd)
    P = {"x.mlp.router": f64(rnd(rng, E, Wd, std=Wd ** -0.5)), "x.mlp.router.b": f64(rnd(rng, E))}
    for e in range(E):
        P[f"x.mlp.e{e}.up"], P[f"x.mlp.e{e}.down"] = f64(rnd(rng, ff, Wd, std=Wd ** -0.5)), f64(rnd(rng, Wd, ff, std=ff ** -0.5))
    x = torch.zeros((T, Hp), dtype=dt, device=DEV)
    x[:, :Wd] = rnd(rng, T, Wd, dt=dt)
    spec = load_pkg("feed_forward").MoeSpec(ff, E, top)
    t = lambda n: torch.from_numpy(P["x.mlp." + n])
    m = load_pkg("feed_forward").MoeRelu2(spec, {"router": t("router"), "router_b": t("router.b"), "up": [t(f"e{e}.up") for e in range(E)],
                                                 "down": [t(f"e{e}.down") for e in range(E)]}, Wd, 1.5, dt, DEV)
    # routing on given logits: exact choice, ties to the lower index
    z = torch.from_numpy(np.round(rng.normal(size=(T, D.pad32(E))) * 4) / 4).float().to(DEV)
    pick, w = D.moe_route(z, torch.zeros(E, device=DEV), 1.0, top, dt)
    zz = f64(z)[:, :E]
    order = np.argsort(-zz, -1, kind="stable")[:, :top]
    assert np.array_equal(pick.cpu().numpy(), order)
    ex = np.exp(np.take_along_axis(zz, order, -1))
    assert np.abs(f64(w) - ex / ex.sum(-1, keepdims=True)).max() < 1e-6
    # the plan covers every entry once, tiles hold one expert
    plan = D.MoePlan(pick, E, dt)
    torch.cuda.synchronize()
    tiles, perm = plan.tiles.view(-1, 4).cpu().numpy()[: int(plan.n_tiles[0])], plan.perm.cpu().numpy()
    used = int(plan.n_tiles[1])
    assert used <= plan.places and used % 16 == 0 and sorted(p for p in perm[:used] if p >= 0) == list(range(T * top))
    assert len(tiles) <= plan.max_tiles and tiles[:, 2].sum() == T * top
    flat = order.reshape(-1)
    for e, first, n, _ in tiles:
        assert 0 < n <= plan.tile_rows and first % 16 == 0 and (flat[perm[first:first + n]] == e).all()
    # the whole block; in bf16 on the router's own fp32 logits of the rounded input, so that choices agree
    resid = rnd(rng, T, Hp)
    before, kp, sums = f64(resid), None, None
    if dt == torch.bfloat16:
        part, sums = rnd(rng, 1, T, Hp), ops.FragActivation(T, Hp, DEV, dtype=dt)
        kp, before = ops.KSplitParts(part, 2, Hp), before + f64(part)[0]
    m.add_to(resid, ops.FragActivation.pack(x) if dt == torch.bfloat16 else x, x, kp, sums)
    torch.cuda.synchronize()
    assert sums is None or torch.equal(sums.unpack(), resid.to(dt))
    want = R.moe_ff(1.5 * f64(x)[:, :Wd], {"router": {"top": top}}, P, "x")
    gap = np.sort(1.5 * f64(x)[:, :Wd] @ P["x.mlp.router"].T + P["x.mlp.router.b"], -1)[:, ::-1]
    clear = np.ones(T, bool) if top == E else gap[:, top - 1] - gap[:, top] > 1e-3
    got = f64(resid) - before
    assert clear.mean() > 0.9 and np.abs(got[clear, :Wd] - want[clear]).max() / np.abs(want).max() < tol(dt, f32=5e-6)
    assert np.abs(got[:, Wd:]).max() < 1e-6


@pytest.mark.parametrize("T,K,N", [(1, 32, 20), (5, 96, 160), (40, 160, 72), (64, 64, 8224), (100, 96, 160), (300, 64, 224), (4096, 64, 4096), (16, 3072, 256)])
def test_bf16_linear(ops, T, K, N):
    """The linear kernels of the bfloat16 library: every shape class of the fp16 ones."""
    rng = np.random.default_rng(T)
    x, W = rnd(rng, T, K, dt=torch.bfloat16), rnd(rng, N, K, std=K ** -0.5, dt=torch.bfloat16)
    want = f64(x) @ f64(W).T
    Wp, xf = ops.PackedWeight(W), ops.FragActivation.pack(x)
    assert torch.equal(Wp.unpack(), W) and torch.equal(xf.unpack(), x)
    for y in (ops.linear(xf, Wp, out_dtype=torch.float32), ops.linear(x, Wp, out_dtype=torch.float32)):
        assert err(y, want) < 2e-6
    assert err(ops.linear(xf, Wp), want) < 4e-3
    acc = rnd(rng, T, N)
    a0 = f64(acc)
    parts = ops.linear_acc_ksplit(xf, Wp, acc, torch.empty(3 * T * N, device=DEV))
    tot = f64(acc) + (f64(parts.part[: (parts.ks - 1) * T * N].view(parts.ks - 1, T, N)).sum(0) if parts is not None else 0)
    assert np.abs(tot - a0 - want).max() < 2e-5


@pytest.mark.parametrize("T,K,N", [(1, 32, 20), (70, 96, 130), (200, 160, 64)])
def test_fp32_linear(ops, T, K, N):
    rng = np.random.default_rng(T)
    x, W = (torch.from_numpy(rng.normal(size=s)).float().to(DEV) for s in ((T, K), (N, K)))
    want = f64(x) @ f64(W).T
    assert err(ops.linear(x, W), want) < 1e-6
    acc = torch.from_numpy(rng.normal(size=(T, N))).float().to(DEV)
    a0 = f64(acc)
    ops.linear(x, W, out=acc, accumulate=True)
    assert err(acc, a0 + want) < 1e-6


@pytest.mark.parametrize("T,K,N", [(1, 16, 1), (16, 48, 31), (17, 208, 4100), (63, 2064, 70), (65, 80, 2050), (64, 16, 16400), (130, 48, 33000), (200, 112, 33001)])
def test_fp32_linear_forms(ops, T, K, N):
    """16, 64 and 128 rows per workgroup, ragged tokens, rows and K, stored 16 bytes at a time or by element.  Every product and every
    sum rounds once: at most K + 2 roundings of 2^-24 on what is added up."""
    rng = np.random.default_rng(K)
    x, W = (torch.from_numpy(rng.normal(size=s)).float().to(DEV) for s in ((T, K), (N, K)))
    want, room = x.double() @ W.double().T, x.abs().double() @ W.abs().double().T
    y = ops.linear(x, W)
    assert bool(((y.double() - want).abs() <= (K + 2) * 2.0 ** -24 * room).all())
    y0 = torch.from_numpy(rng.normal(size=(T, N))).float().to(DEV)
    y1 = ops.linear(x, W, out=y0.clone(), accumulate=True)
    torch.cuda.synchronize()
    assert torch.equal(y1, y0 + y)


@pytest.mark.parametrize("T,K,N", [(63, 2064, 70), (65, 16, 2050), (63, 208, 39), (130, 128, 4101), (65, 272, 8200), (20, 1040, 8201), (4, 1040, 32001)])
def test_fp32_linear_at_any_element(ops, T, K, N):
    """Operands that begin at any element give the bits of aligned ones, with 16, 64 (rings of two and of four stages, a K of one stage and of
    more) and 128 rows per workgroup; the rows of y likewise.  Rounding as in test_fp32_linear_forms."""
    rng = np.random.default_rng(K + N)
    x, W, y0 = (torch.from_numpy(rng.normal(size=s)).float().to(DEV) for s in ((T, K), (N, K), (T, N)))
    y = ops.linear(x, W)
    assert bool(((y.double() - x.double() @ W.double().T).abs() <= (K + 2) * 2.0 ** -24 * (x.abs().double() @ W.abs().double().T)).all())
    at = lambda t, i: torch.cat([t.new_zeros(i), t.reshape(-1), t.new_zeros(4 - i)])[i:i + t.numel()].view(t.shape)
    for i, j, k in ((1, 0, 2), (0, 2, 0), (3, 1, 1)):
        wide = torch.cat([x.new_zeros(T, i), x, x.new_zeros(T, 8 - i)], 1)[:, i:i + K]      # columns of a wider tensor
        out = at(y0, k)
        ops.linear(wide, at(W, j), out=out, accumulate=True)
        torch.cuda.synchronize()
        assert torch.equal(out, y0 + y), (i, j, k)


@pytest.mark.parametrize("T,n,H,rank,rot", [(300, 60, 3, 200, 40), (290, 50, 16, 512, 64), (260, 33, 2, 100, 24), (330, 33, 2, 100, 24), (301, 40, 2, 64, 16),
                                            (260, 40, 2, 60, 16), (100, 40, 17, 512, 64), (70, 40, 2, 512, 16), (2, 70, 18, 1600, 64), (70, 20, 1, 1560, 32),
                                            (270, 18, 1, 1560, 32), (200, 20, 3, 200, 40), (257, 18, 5, 250, 16), (5, 17, 3, 96, 16),
                                            (200, 20, 17, 512, 32), (450, 18, 1, 1560, 32)])
@pytest.mark.parametrize("sunk", [True, False])
def test_fp32_latent_attention_of_prompts(D, T, n, H, rank, rot, sunk):
    """Four, eight and sixteen waves, outputs of 64 to 512 dims and in parts, queries that do not fit LDS, a second tile of heads."""
    dt = torch.float32
    lat, pages, bt, rng = latent_case(D, dt, [n], H, rank, rot, seed=T)
    pos = rng.integers(0, n, T)
    q = torch.from_numpy(rng.normal(size=(T, H, rank + rot))).to(torch.bfloat16).double().numpy()
    sink = rng.normal(2.0, 1.0, H).astype(np.float32) if sunk else None
    scale = 3.0 * (rank + rot) ** -0.5
    got = D.latent_attn(put_queries(D, q, rank, rot, dt), pages, bt, torch.ones(T, dtype=torch.int32, device=DEV),
                        torch.from_numpy(pos.astype(np.int32)).to(DEV), torch.from_numpy(sink).to(DEV) if sunk else None, scale, rank, rot, max_ctx=n)
    torch.cuda.synchronize()
    assert err(got[..., :rank], attn_want(lat, q, [0] * T, pos, sink, scale, rank)) < tol(dt)
    assert float(got[..., rank:].abs().sum()) == 0


@pytest.mark.parametrize("glu", [False, True])
@pytest.mark.parametrize("counts", [[300], [257, 0, 64], [1, 16, 17, 64, 65, 255, 256], [511, 0, 0, 240, 241], [128] * 10, [700, 1, 1, 900, 33, 48, 49],
                                    [256, 512, 768]])
def test_experts_over_ragged_tiles(D, counts, glu):
    """Tiles of 256 places with few, some and all of their fragments, one to nine of them (bands of three, whole and cut), in each of the three
    epilogues.  The hidden values round once to bf16 (2^-9; gate and up beforehand as well: |silu| and |silu'| are at most |g| and 1.1), the
    results once more; the fp32 sums are far below that."""
    dt, E, K, ff, N, T = torch.bfloat16, len(counts), 128, 320, 288, sum(counts)
    rng = np.random.default_rng(T)
    pick = rng.permutation(np.repeat(np.arange(E), counts))
    plan = D.MoePlan(torch.from_numpy(pick.astype(np.int32)).to(DEV).view(T, 1), E, dt)
    assert plan.tile_rows == 256
    x, up, down = rnd(rng, T, K, dt=dt), rnd(rng, E, ff * (2 if glu else 1), K, std=K ** -0.5, dt=dt), rnd(rng, E, N, ff, std=ff ** -0.5, dt=dt)
    mid = D.moe_linear(x, D.weight(up.view(-1, K)), plan, ff, K, D.MOE_UP, D.ACT_GLU if glu else D.ACT_RELU2)
    got = f64(D.moe_linear(mid, D.weight(down.view(-1, ff)), plan, N, ff, D.MOE_DOWN))
    torch.cuda.synchronize()
    for e in range(E):
        rows = pick == e
        v = f64(x)[rows] @ f64(up)[e].T
        g, u = v[:, :ff], v[:, -ff:]
        h, room = (g / (1 + np.exp(-g)) * u, 2 * np.abs(g * u)) if glu else (np.maximum(g, 0) ** 2,) * 2
        want = h @ f64(down)[e].T
        assert (np.abs(got[rows] - want) <= 2.0 ** -8 * (room @ np.abs(f64(down)[e]).T + np.abs(want)) + 1e-6).all(), e


@pytest.mark.parametrize("counts", [[300, 1, 65, 130], [16, 17, 0, 33], [64, 128, 64]])
@pytest.mark.parametrize("K,N", [(272, 72), (128, 4100), (272, 8200), (208, 12290)])
def test_fp32_experts_over_ragged_tiles(D, counts, K, N):
    """One to four token tiles of 16 per workgroup, rows gathered from tokens and scattered to entries, with 16 and 64 weight rows, ragged
    ones and a ragged K; K + 3 roundings of 2^-24 on what is added up, twice that for the square."""
    dt, E, top = torch.float32, len(counts), 2
    rng = np.random.default_rng(K + N)
    pick = rng.permutation(np.repeat(np.arange(E), np.array(counts) * top)).astype(np.int32)
    T = sum(counts)
    plan = D.MoePlan(torch.from_numpy(pick).to(DEV).view(T, top), E, dt)
    torch.cuda.synchronize()
    perm = plan.perm[: int(plan.n_tiles[1])].long()
    places = (perm >= 0).nonzero().view(-1)
    entry = perm[places]
    x, rows, W = (torch.from_numpy(rng.normal(size=s).astype(np.float32)).to(DEV) for s in ((T, K), (plan.places, K), (E, N, K)))
    up = D.moe_linear(x, W.view(-1, K), plan, N, K, D.MOE_UP, D.ACT_RELU2)
    down = D.moe_linear(rows, W.view(-1, K), plan, N, K, D.MOE_DOWN)
    eps = (K + 3) * 2.0 ** -24
    for e in range(E):
        at = places[torch.from_numpy(pick).to(DEV)[entry] == e]
        src, w = x[perm[at] // top].double(), W[e].double()
        v, room = src @ w.T, src.abs() @ w.abs().T
        assert bool(((up[at].double() - v.clamp(min=0) ** 2).abs() <= 2 * eps * room ** 2).all()), e
        v, room = rows[at].double() @ w.T, rows[at].double().abs() @ w.abs().T
        assert bool(((down[perm[at]].double() - v).abs() <= eps * room).all()), e


@pytest.mark.parametrize("glu", [False, True])
@pytest.mark.parametrize("top,ff,N", [(7, 224, 240), (9, 224, 240), (15, 256, 272)])
def test_experts_of_a_few_entries_with_four_row_tiles(D, glu, top, ff, N):
    """Tiles of 16 entries on both sides of what takes four row tiles per workgroup (eight entries per expert), rows that are and are not whole
    blocks of them.  Bounds as for the large tiles."""
    dt, E, K, T = torch.bfloat16, 512, 96, 512
    rng = np.random.default_rng(top)
    pick = np.argsort(rng.random((T, E)), -1)[:, :top].astype(np.int32)
    plan = D.MoePlan(torch.from_numpy(pick).to(DEV), E, dt)
    assert plan.tile_rows == 16
    x, up, down = rnd(rng, T, K, dt=dt), rnd(rng, E, ff * (2 if glu else 1), K, std=K ** -0.5, dt=dt), rnd(rng, E, N, ff, std=ff ** -0.5, dt=dt)
    mid = D.moe_linear(x, D.weight(up.view(-1, K)), plan, ff, K, D.MOE_UP, D.ACT_GLU if glu else D.ACT_RELU2)
    got = f64(D.moe_linear(mid, D.weight(down.view(-1, ff)), plan, N, ff, D.MOE_DOWN)).reshape(T, top, N)
    torch.cuda.synchronize()
    X, U, Dn = f64(x), f64(up), f64(down)
    for e in range(E):
        t, j = np.nonzero(pick == e)
        v = X[t] @ U[e].T
        g, u = v[:, :ff], v[:, -ff:]
        h, room = (g / (1 + np.exp(-g)) * u, 2 * np.abs(g * u)) if glu else (np.maximum(g, 0) ** 2,) * 2
        want = h @ Dn[e].T
        assert (np.abs(got[t, j] - want) <= 2.0 ** -8 * (room @ np.abs(Dn[e]).T + np.abs(want)) + 1e-6).all(), e


@pytest.mark.parametrize("E,T,top,K,N,stage", [(128, 64, 4, 1056, 528, "gated"), (128, 64, 2, 2048, 560, "gated"), (128, 300, 4, 1056, 1040, "down"),
                                               (128, 300, 4, 544, 1072, "up"), (16, 100, 2, 4128, 528, "down"), (16, 100, 2, 4128, 528, "up"),
                                               (64, 300, 3, 2080, 2064, "gated")])
def test_experts_with_four_row_tiles_over_many_steps(D, E, T, top, K, N, stage):
    """Four row tiles per workgroup with two to seventeen steps of 32 k in a wave, not the same number in each, and rows that end in one, two or three of
    a workgroup's tiles.  fp32 sums of exact products: K + 8 roundings of 2^-24 on what is added up; then one rounding to bf16 (2^-8 of a
    place's size), of gate and up beforehand as well, |silu| and |silu'| being at most |g| and 1.1."""
    dt = torch.bfloat16
    g = torch.Generator(device=DEV).manual_seed(K + N)
    rand = lambda *sh: torch.randn(*sh, generator=g, device=DEV)
    pick = torch.argsort(rand(T, E), -1)[:, :top].to(torch.int32).contiguous()
    plan = D.MoePlan(pick, E, dt)
    assert plan.tile_rows == 16
    rows = 2 * N if stage == "gated" else N
    W = (rand(E, rows, K) * K ** -0.5).to(dt)
    x = rand(plan.places if stage == "down" else T, K).to(dt)
    act = {"gated": D.ACT_GLU, "up": D.ACT_RELU2, "down": D.ACT_NONE}[stage]
    y = D.moe_linear(x, D.weight(W.view(-1, K)), plan, N, K, D.MOE_DOWN if stage == "down" else D.MOE_UP, act)
    torch.cuda.synchronize()
    perm, u, eps = plan.perm.long(), 2.0 ** -8, (K + 8) * 2.0 ** -24
    places = (perm[:int(plan.n_tiles[1])] >= 0).nonzero().view(-1)
    of = pick.view(-1)[perm[places]]
    for e in range(E):
        at = places[of == e]
        if at.numel() == 0:
            continue
        src, w = (x[at] if stage == "down" else x[perm[at] // top]).double(), W[e].double()
        v, err = src @ w.T, eps * (src.abs() @ w.abs().T)
        if stage == "gated":
            v, err = [v[:, :N], v[:, N:]], [err[:, :N] + u * v[:, :N].abs(), err[:, N:] + u * v[:, N:].abs()]
            want = v[0] * torch.sigmoid(v[0]) * v[1]
            bound = 1.1 * err[0] * (v[1].abs() + err[1]) + v[0].abs() * err[1]
        elif stage == "up":
            want, bound = v.clamp(min=0) ** 2, 2 * v.abs() * err + err ** 2
        else:
            want, bound = v, err
        got = (y[perm[at]] if stage == "down" else y[at]).double()
        assert bool(((got - want).abs() <= (1 + u) * bound + u * want.abs() + 2.0 ** -30).all()), e


@pytest.mark.parametrize("T,K,N", [(17, 2048, 64), (33, 1040, 100), (100, 2048, 36), (299, 512, 128), (70, 16, 4100), (70, 48, 4100), (130, 80, 8200), (65, 144, 2052),
                                   (300, 2064, 2052), (299, 208, 20004)])
@pytest.mark.parametrize("shift", [0, 1])
def test_fp32_linear_token_blocks_and_row_lengths(ops, T, K, N, shift):
    """Few weight rows in blocks of 16, 32 and 64 tokens, and rows whose last 64 k are not whole on each of the other forms, x beginning at any
    column of a wider tensor: K additions and products of fp32."""
    g = torch.Generator(device=DEV).manual_seed(T + K + N)
    x = torch.randn((T, K + 16), generator=g, device=DEV)[:, shift:shift + K]
    W = torch.randn((N, K), generator=g, device=DEV) * K ** -0.5
    want, room = x.double() @ W.double().T, x.double().abs() @ W.double().abs().T
    y = ops.linear(x, W)
    acc = torch.ones((T, N), device=DEV)
    ops.linear(x, W, out=acc, accumulate=True)
    assert bool(((y.double() - want).abs() <= (K + 2) * 2.0 ** -24 * room).all())
    assert bool(((acc.double() - 1 - want).abs() <= (K + 3) * 2.0 ** -24 * (room + 1)).all())


@pytest.mark.parametrize("T,K,N", [(1, 2048, 2048), (4, 2048, 11264), (24, 2048, 5632), (40, 1024, 5632), (16, 5632, 11264), (299, 2048, 2048), (299, 2048, 11264),
                                   (24, 2048, 32000)])
@pytest.mark.parametrize("shift", [0, 1])
def test_fp32_linear_adds_in_eight_sums(ops, T, K, N, shift):
    """The products of an output are added in at least eight chains, whatever the rows per workgroup: beside 1, at any place of K, one product in
    four is 2^-24 (1 + 2^-10), at most one in an MFMA, and what follows 1 in its chain rounds up to 2^-23 each time.  K / 32 such products in a
    chain, seven sums of chains, alpha."""
    n, tiny = torch.arange(N, device=DEV), 2.0 ** -24 * (1 + 2.0 ** -10)
    W = torch.zeros((N, K // 16, 16), device=DEV)
    W[:, :, :4] = tiny
    W.view(N, K)[n, n % (K // 16) * 16 + n // (K // 16) % 4] = 1.0
    y = ops.linear(torch.ones((T, K + 4), device=DEV)[:, shift:shift + K], W.view(N, K))
    want = 1.0 + (K // 4 - 1) * tiny
    assert float((y.double() - want).abs().max()) <= (K // 32 + 8) * 2.0 ** -24 * want
