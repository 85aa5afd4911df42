"""The mechanisms of the packed decoder step one by one (``penroz.ops.packed``, the state manager) against the
plain oracle: on the CPU their torch forms, with ``gpu`` the HIP kernels in fp32 and bf16."""
import math

import pytest
import torch

import latent_oracle as O
from penroz.models.kv_cache import SequenceState
from penroz.models.layers import fresh_batch
from penroz.ops import packed as P

TARGETS = [pytest.param(("cpu", torch.float32), id="cpu-fp32"),
           pytest.param(("cuda", torch.float32), id="gpu-fp32", marks=pytest.mark.gpu),
           pytest.param(("cuda", torch.bfloat16), id="gpu-bf16", marks=pytest.mark.gpu)]
TOL = {torch.float32: 1e-5, torch.bfloat16: 1.2e-2}


def rand(*shape, seed=0, scale=1.0, dtype=torch.float32):
    t = torch.randn(*shape, generator=torch.Generator().manual_seed(seed + 17 * len(shape) + shape[0])) * scale
    return t.to(dtype)


def near(got, want, dtype, tol=None):
    e = (got.double().cpu() - want.double()).abs().max() / want.double().abs().max()
    assert float(e) < (tol or TOL[dtype]), float(e)


# --------------------------------------------------------------------------- norms, residual, convolution
@pytest.mark.parametrize("target", TARGETS)
@pytest.mark.parametrize("C,groups", [(96, 3), (100, 5), (60, 30), (7, 1), (2048, 4), (4096, 1), (4100, 2)])
def test_grouped_norm(target, C, groups):
    dev, dt = target
    x, w = rand(5, C, scale=3), rand(C, seed=1)
    x[:, :C // groups] *= 100  # one part far larger: its scale must not reach the others
    ref = torch.stack([O.grouped_norm(r, w.double(), groups, 1e-3) for r in x.double()])
    near(P.row_norm(x.to(dev), w.to(dev), groups, 1e-3, dt), ref, dt)
    rows = torch.tensor([4, 0, 4], dtype=torch.int32, device=dev)
    near(P.row_norm(x.to(dev), w.to(dev), groups, 1e-3, dt, rows=rows), ref[[4, 0, 4]], dt)
    # residual add, plain and as the weighted sum of expert rows
    b = fresh_batch(1, 5, torch.device(dev))
    y, pw = rand(5, 3, C, seed=2, dtype=dt), rand(5, 3, seed=3).abs()
    base = rand(5, C, seed=4)
    got, h = P.residual_conv(b, dt, x=base.to(dev), y=y[:, 0].contiguous().to(dev), norm=(w.to(dev), groups, 1e-3))
    want = base.double() + torch.stack([O.grouped_norm(r, w.double(), groups, 1e-3) for r in y[:, 0].double()])
    assert h is None
    near(got, want, torch.float32)
    got, _ = P.residual_conv(b, dt, x=base.to(dev), y=y.reshape(15, C).to(dev), pair_w=pw.to(dev),
                             norm=(w.to(dev), groups, 1e-3))
    ys = (y.double() * pw.double().unsqueeze(-1)).sum(1)
    near(got, base.double() + torch.stack([O.grouped_norm(r, w.double(), groups, 1e-3) for r in ys]), torch.float32)


@pytest.mark.parametrize("target", TARGETS)
@pytest.mark.parametrize("C,taps", [(96, 3), (37, 4), (64, 1), (512, 7), (5000, 2)])
def test_convolution_in_portions(target, C, taps):
    """Three sequences cut differently, two tokens or fewer than the taps at a time, their slots taken in
    another order than their rows; then a new sequence in a used slot."""
    dev, dt = target
    cw = rand(C, taps, scale=0.5)
    st = SequenceState([], [(C, taps)], [], dt, dev, slots=1)
    conv = (cw.t().contiguous().to(dev), None)
    xs = {n: rand(11, C, seed=i) for i, n in enumerate("abc")}
    cuts = {"a": [1, 2, 1, 1, 6], "b": [5, 1, 2, 1, 2], "c": [2, 2, 4, 1, 2]}
    slots = {n: st.acquire() for n in "cab"}
    got, at = {n: [] for n in xs}, dict.fromkeys(xs, 0)

    def step(entries):
        b = st.begin([(slots[n], k) for n, k in entries])
        x = torch.cat([xs[n][at[n]:at[n] + k] for n, k in entries]).to(dev)
        _, h = P.residual_conv(b, dt, x=x, conv=(conv[0], st.conv[0]))
        for (n, k), part in zip(entries, h.split([k for _, k in entries])):
            got[n].append(part)
            at[n] += k

    for i in range(5):
        step([(n, cuts[n][i]) for n in ("abc" if i % 2 else "bca")])
    for n in xs:
        near(torch.cat(got[n]), O.time_conv(xs[n].double(), cw.double()), dt)
    st.release(slots["b"])
    xs["d"], got["d"], at["d"] = rand(6, C, seed=9), [], 0
    slots["d"] = st.acquire()
    assert slots["d"] == slots["b"]
    for k in (1, 1, 2, 1, 1):
        step([("d", k)])
    near(torch.cat(got["d"]), O.time_conv(xs["d"].double(), cw.double()), dt)


@pytest.mark.gpu
@pytest.mark.parametrize("y_dt,dt", [(torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32),
                                     (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("C,groups,taps,top,cuts", [
    (512, 2, 4, 0, [[1, 5, 6, 2], [3, 1, 7, 12], [40, 2, 3, 1]]), (1536, 6, 3, 0, [[4, 9, 14], [1, 1, 30]]),
    (512, 1, 1, 0, [[7, 6], [2, 2]]), (2048, 4, 4, 0, [[1, 6700, 3], [2, 3, 29]]), (2048, 4, 2, 0, [[1, 2, 19000]]),
    (5120, 10, 4, 0, [[9, 1, 70], [5, 2, 3]]), (2048, 8, 1, 0, [[3, 30]]), (1536, 6, 3, 2, [[4, 9, 14], [1, 1, 30]]),
    (512, 2, 5, 0, [[7, 6], [2, 2]]), (768, 6, 4, 0, [[7, 6], [2, 2]])])
def test_norm_and_convolution_in_one_pass(C, groups, taps, top, cuts, y_dt, dt):
    """Residual add, norm and convolution of prompts as the step-by-step form computes them. In one pass (x left as it
    was): at the edges of the wave's spans (5 rows, and one round or two of longer ones), every sequence in portions, 1 to
    4 taps, groups of 256 and 512, fewer of them than a workgroup has waves and more. One kernel after the other (x
    updated in place): expert rows, 5 taps, other groups, and an output of another type than the sublayer's."""
    one_pass = top == 0 and taps <= 4 and C // groups in (256, 512) and y_dt == dt
    g = torch.Generator().manual_seed(C + taps)
    w, cw = torch.rand(C, generator=g) + 0.5, torch.randn(taps, C, generator=g)
    state = {d: SequenceState([], [(C, taps)], [], dt, d, slots=len(cuts[0])) for d in ("cpu", "cuda")}
    slots = {d: [st.acquire() for _ in cuts[0]][::-1] for d, st in state.items()}
    for counts in cuts:
        N = sum(counts)
        x0, y = torch.randn(N, C, generator=g), torch.randn(N * max(top, 1), C, generator=g).to(y_dt)
        pw = torch.rand(N, top, generator=g) if top else None
        out = {}
        for d, st in state.items():
            b, x = st.begin(list(zip(slots[d], counts))), x0.clone().to(d)
            out[d] = P.residual_conv(b, dt, x=x, y=y.to(d), pair_w=None if pw is None else pw.to(d),
                                     norm=(w.to(d), groups, 1e-5), conv=(cw.to(d), st.conv[0]))
        assert (out["cuda"][0].data_ptr() != x.data_ptr()) == one_pass
        near(out["cuda"][0], out["cpu"][0], torch.float32)
        near(out["cuda"][1], out["cpu"][1], dt)
        for a, c in zip(slots["cuda"], slots["cpu"]):
            if taps > 1:
                near(state["cuda"].conv[0][a], state["cpu"].conv[0][c], torch.float32)


@pytest.mark.parametrize("target", TARGETS)
def test_embedding_rows_start_the_residual(target):
    dev, dt = target
    table, toks = rand(19, 24, dtype=dt), torch.tensor([3, 18, 0])
    st = SequenceState([], [(24, 3)], [], dt, dev)
    b = st.begin([(st.acquire(), 3)])
    cw = rand(24, 3)
    x, h = P.residual_conv(b, dt, embed=(toks.to(dev), table.to(dev)), conv=(cw.t().contiguous().to(dev), st.conv[0]))
    assert x.dtype == torch.float32 and torch.equal(x.cpu(), table[toks].float())
    near(h, O.time_conv(table[toks].double(), cw.double()), dt)


# --------------------------------------------------------------------------- rotation
def test_rotation_table_matches_single_rotations():
    tab = P.rotation_table(300.0, 6, 2000, "cpu")
    v = rand(6)
    for pos in (0, 1, 77, 1999):
        near(P._rotate(v, tab[pos]), O.rotate(v.double(), pos, 300.0), torch.float32)


# --------------------------------------------------------------------------- latent attention
SIZES = {  # heads, dim, rot, vdim, rank
    "tiny": (1, 8, 2, 8, 8), "padded": (3, 12, 6, 10, 20), "small": (4, 48, 16, 40, 72), "mid": (5, 64, 64, 128, 136),
    "deep": (2, 128, 64, 128, 512), "many-heads": (33, 32, 32, 64, 264), "wide-rot": (2, 96, 128, 136, 384),
    "beyond-mfma": (2, 200, 136, 264, 520),
}


def latent_case(name, T, seed=0, scale=None, sharp=1.0, C=64, dt=torch.float32):
    H, d, r, vd, R = SIZES[name]
    s = P.LatentSizes(H, d, r, vd, R, scale or (d + r) ** -0.5, 1e4, 1e-4)
    w = {k: rand(*sh, seed=seed + i, scale=sh[1] ** -0.5 * (sharp if k == "q" else 1.0), dtype=dt)
         for i, (k, sh) in enumerate({"q": (H * (d + r), C), "dkv": (R + r, C), "uk": (H * d, R), "uv": (H * vd, R)}.items())}
    nw, h = 1 + 0.2 * rand(R, seed=seed + 9), rand(T, C, seed=seed + 11, dtype=dt)
    cfg = {"heads": H, "dim": d, "rot_dim": r, "vdim": vd, "kv_rank": R, "scale": s.scale, "rot": {"base": 1e4}}
    return s, w, nw, h, cfg


def pack(s, w, dev):
    eye = torch.eye(s.heads * s.vdim, dtype=w["q"].dtype)
    return {k: v.to(dev) for k, v in P.pack_latent(s, w["q"], w["dkv"], w["uk"], w["uv"], eye).items()}


def unpad(out, s):
    return out.view(-1, s.heads, s.v8)[:, :, :s.vdim].reshape(-1, s.heads * s.vdim)


def oracle_latent(w, nw, h, cfg, s):
    D = {k: v.double() for k, v in w.items()}
    D["o"] = torch.eye(s.heads * s.vdim, dtype=torch.float64)
    c, k = O.latent(h.double(), D["dkv"], nw.double(), s.rank, 1e4, s.eps)
    return O.attend(h.double(), c, k, D, cfg)


@pytest.mark.parametrize("target", TARGETS)
@pytest.mark.parametrize("name", list(SIZES))
@pytest.mark.parametrize("cuts", [[150], [70, 80], [150 - 9] + [1] * 9, [64, 2, 5, 1, 64, 3, 1, 10]])
def test_latent_attention(target, name, cuts):
    """Prompts, portions down to two tokens and decoded tokens of one layer; a second layer with its own
    projections attends over the first one's cache."""
    dev, dt = target
    s, w, nw, h, cfg = latent_case(name, 150, dt=dt, sharp=2.0)
    s2, w2, _, _, _ = latent_case(name, 1, seed=50, dt=dt, sharp=2.0)
    pk, pk2 = pack(s, w, dev), pack(s2, {**w2, "dkv": None}, dev)
    D = {k: v.double() for k, v in w.items()}
    D2 = {**{k: v.double() for k, v in w2.items()}, "o": torch.eye(s.heads * s.vdim, dtype=torch.float64)}
    c, k = O.latent(h.double(), D["dkv"], nw.double(), s.rank, 1e4, s.eps)
    st = SequenceState([s.cache_width], [], [(s.base, s.rot)], dt, dev, slots=2, capacity=40)
    other, slot = st.acquire(), st.acquire()  # the sequence does not sit in slot 0
    got, got2, at = [], [], 0
    for n in cuts:
        b = st.begin([(slot, n)])
        x = h[at:at + n].to(dev)
        tab = st.tables[(s.base, s.rot)]
        got.append(P.latent_attention(s, pk, P.linear(x, pk["z"]), st.latent[0], nw.to(dev), tab, b))
        got2.append(P.latent_attention(s2, pk2, P.linear(x, pk2["z"]), st.latent[0], None, tab, b))
        at += n
    near(unpad(torch.cat(got), s), oracle_latent(w, nw, h, cfg, s), dt, 2e-2 if dt == torch.bfloat16 else None)
    near(unpad(torch.cat(got2), s), O.attend(h.double(), c, k, D2, cfg), dt, 2e-2 if dt == torch.bfloat16 else None)


@pytest.mark.parametrize("target", TARGETS)
@pytest.mark.parametrize("name", ["small", "deep", "padded"])
def test_one_loud_key_at_every_border(target, name):
    """Unequal sequences whose latents are small but for one loud key, placed around tile, key-range and
    sequence borders, asked for by decoded tokens (several key ranges) and by a prompt's rows: with the key
    left out the oracle's output differs clearly."""
    dev, dt = target
    s, w, nw, _, cfg = latent_case(name, 1, dt=dt)
    H, R, r = s.heads, s.rank, s.rot
    lens = [700, 1, 33, 257]
    D = {k: v.double() for k, v in w.items()}
    D["o"] = torch.eye(H * s.vdim, dtype=torch.float64)
    pk = pack(s, {**w, "dkv": None}, dev)
    hq = rand(64, 64, seed=5, scale=12, dtype=dt)
    places = (0, 1, 31, 32, 63, 64, 127, 128, 255, 256, 257, 511, 512, 640, 699)
    for place in places if dev == "cuda" else places[::5]:
        st = SequenceState([s.cache_width], [], [(s.base, r)], dt, dev, slots=4, capacity=704)
        rows, keep = [], []
        for i, n in enumerate(lens):
            c, k = rand(n, R, seed=20 + i, scale=0.05, dtype=dt), rand(n, r, seed=30 + i, scale=0.05, dtype=dt)
            if place < n:
                c[place] = rand(R, seed=40 + i, scale=1.5, dtype=dt)
            slot = st.acquire()
            st.latent[0][slot].fill_(float("nan"))  # nothing behind a sequence's end may be read into it
            st.latent[0][slot, :n] = 0
            st.latent[0][slot, :n, :R] = c.to(dev)
            st.latent[0][slot, :n, s.R8:s.R8 + r] = k.to(dev)
            rows.append(slot)
            keep.append((c.double(), k.double(), n))
        tab = st.tables[(s.base, r)]

        def run(counts):
            for slot, (_, _, n), m in zip(rows, keep, counts):
                st._len[slot] = n - m
            b = st.begin([(slot, m) for slot, m in zip(rows, counts)])
            x = torch.cat([hq[:m] for m in counts]).to(dev)
            return unpad(P.latent_attention(s, pk, P.linear(x, pk["z"]), st.latent[0], None, tab, b), s), counts

        for out, counts in (run([1, 1, 1, 1]), run([64, 1, 20, 64])):
            at = 0
            for i, ((c, k, n), m) in enumerate(zip(keep, counts)):
                got, at = out[at:at + m], at + m
                full = torch.cat([torch.zeros(n - m, 64, dtype=torch.float64), hq[:m].double()])
                ref = O.attend(full, c, k, D, cfg, start=n - m)
                near(got, ref, dt, 6e-2 if dt == torch.bfloat16 else 2e-5)
                if place < n - m and n > 1:
                    c2 = c.clone()
                    c2[place] = 0
                    assert float((O.attend(full, c2, k, D, cfg, start=n - m) - ref).abs().max() / ref.abs().max()) > 0.2
            assert not torch.isnan(out).any()


@pytest.mark.gpu
@pytest.mark.parametrize("rows,heads,length", [(1, 4, 5000), (1, 64, 1), (16, 16, 1025), (70, 5, 333)])
def test_key_ranges_agree(rows, heads, length):
    """The decode kernel split over any number of key ranges (also more than there are tiles) gives the plain
    kernel's result."""
    from penroz.ops._ext import kernels
    K, R8, r8 = kernels(), 136, 32
    g = torch.Generator(device="cuda").manual_seed(1)
    dev = dict(device="cuda")
    qa = (torch.randn(rows, heads, R8 + r8, generator=g, **dev) * 2).bfloat16()
    cache = torch.randn(rows, length, R8 + r8, generator=g, **dev).bfloat16()
    i32 = dict(dtype=torch.int32, **dev)
    slot, pos = torch.arange(rows, **i32).flip(0).contiguous(), torch.randint(0, length, (rows,), generator=g, **i32)
    pos[0] = length - 1
    wuv = torch.randn(heads, 40, R8, generator=g, **dev).bfloat16() * R8 ** -0.5
    ref = torch.empty(1, rows, heads, R8, **dev)
    K.latent_attn_row(qa, cache, slot, pos, R8, 0.1, ref)
    want = torch.empty(rows, heads * 40, dtype=torch.bfloat16, **dev)
    K.latent_uv(ref, None, wuv, want)
    for n in {1, 2, 7, 64, P.key_ranges(rows, heads, length)}:
        ol = torch.full((n, rows, heads, R8), float("nan"), **dev)
        ml = torch.full((n, rows, heads, 2), float("nan"), **dev)
        K.latent_decode(qa, cache, slot, pos, R8, 0.1, ol, ml)
        out = torch.empty_like(want)
        K.latent_uv(ol, ml, wuv, out)
        near(out, want.cpu(), torch.bfloat16)


# --------------------------------------------------------------------------- experts
@pytest.mark.parametrize("target", TARGETS)
@pytest.mark.parametrize("N,E,top,C", [(3, 6, 2, 64), (1, 1, 1, 32), (80, 16, 3, 96), (5, 130, 7, 40), (2, 5, 5, 33)])
def test_router(target, N, E, top, C):
    dev, dt = target
    h, wr = rand(N, C, dtype=dt), rand(E, C, seed=1, scale=3 * C ** -0.5, dtype=dt)
    ids, wts = P.route(h.to(dev), wr.to(dev), top)
    for t in range(N):
        e, w = O.route(h[t].double(), wr.double(), top)
        assert ids[t].tolist() == e
        near(wts[t], torch.tensor(w), torch.float32, 1e-4)
    ids2, wts2 = P.route(h.to(dev), wr.to(dev), top, renorm=True)
    assert torch.equal(ids, ids2) and torch.allclose(wts2.sum(-1).cpu(), torch.ones(N), atol=1e-5)


@pytest.mark.parametrize("target", TARGETS)
@pytest.mark.parametrize("E,C", [(64, 2048), (65, 2056), (81, 4104), (200, 512)])
def test_router_of_wide_rows(target, E, C):
    """Logits in the kernel's spans of 2048 columns with a remainder, and experts in several rounds of its waves."""
    dev, dt = target
    h, wr = rand(3, C, dtype=dt), rand(E, C, seed=1, scale=3 * C ** -0.5, dtype=dt)
    ids, wts = P.route(h.to(dev), wr.to(dev), 6)
    for t in range(3):
        e, w = O.route(h[t].double(), wr.double(), 6)
        assert ids[t].tolist() == e
        near(wts[t], torch.tensor(w), torch.float32, 1e-4)


@pytest.mark.parametrize("target", TARGETS)
@pytest.mark.parametrize("N,E,top,C,F", [(3, 6, 2, 64, 48), (1, 1, 1, 32, 20), (40, 5, 4, 96, 96), (5, 9, 3, 40, 33),
                                         (400, 7, 3, 64, 80), (300, 3, 4 - 1, 160, 32), (1100, 40, 1, 32, 64)])
@pytest.mark.parametrize("spread", ["random", "one"])
def test_experts(target, N, E, top, C, F, spread):
    """Few pairs, more pairs than the few-pairs kernel takes, a single expert with all of them."""
    dev, dt = target
    limit = 0.7
    h = rand(N, C, dtype=dt)
    g, u, d = (rand(E, *sh, seed=i, scale=2 * sh[1] ** -0.5, dtype=dt) for i, sh in enumerate([(F, C), (F, C), (C, F)]))
    ids = torch.stack([torch.randperm(E, generator=torch.Generator().manual_seed(i))[:top] for i in range(N)])
    if spread == "one":
        ids[:, 0] = E - 1
    w = {k: v.to(dev) for k, v in P.pack_experts(g, u, d).items()}
    y = P.experts(h.to(dev), ids.int().to(dev), w, 1, limit).cpu().view(N, top, C)
    for e in range(E):
        ref = O.expert_ff(h.double(), {"gate": g[e].double(), "up": u[e].double(), "down": d[e].double()}, limit)
        sel = ids == e
        if sel.any():
            near(y[sel], ref[sel.nonzero()[:, 0]], dt)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("dt,N", [(torch.float32, 300), (torch.bfloat16, 300), (torch.bfloat16, 1300)])
def test_gated_activations_over_the_whole_range(kind, dt, N):
    """Gates down to where exp(-g) is the largest finite value: every result within what fp32 exp, add and divide round
    (a reciprocal there is subnormal, which the hardware's approximate one returns as zero)."""
    z = torch.linspace(-88.5, 30, N).to(dt).float() / (1.702 if kind else 1.0)
    h = torch.zeros(N, 32)
    h[:, 0], h[:, 1] = z, 1.0
    h = h.to(dt)
    z = h[:, 0].double()
    g, u, d = torch.zeros(1, 32, 32), torch.zeros(1, 32, 32), torch.eye(32)[None]
    g[:, :, 0], u[:, :, 1] = 1.0, 1.0  # every product one term: exact
    limit = 40.0
    s = 1.702 * z if kind else z
    want = (z * torch.sigmoid(s) * (2 if kind else 1))[:, None]
    bound = (2 * s.abs() + 8)[:, None] * 2.0 ** -24 + (0 if dt == torch.float32 else 2.0 ** -8)
    w = {k: v.cuda() for k, v in P.pack_experts(g.to(dt), u.to(dt), d.to(dt)).items()}
    got = [P.experts(h.cuda(), torch.zeros(N, 1, dtype=torch.int32, device="cuda"), w, kind, limit)]
    if kind == 1:
        got.append(P.gated_linear(h.cuda(), torch.cat([g[0], u[0]]).to(dt).cuda(), kind, limit))
    for y in got:
        e = (y.double().cpu() - want).abs() / want.abs().clamp_min(1e-300)
        e[z == 0] = 0
        assert bool((e <= bound).all()), (e / bound).max()


@pytest.mark.gpu
def test_gelu_of_grouped_experts_is_rounded_like_erff():
    """The prompts' gelu at 786432 values of (-3, 0]: of x (1 + erff(x / sqrt 2)) / 2 in fp32, about 1.2e-4 of them round
    to another bf16 than the exact value does (by its relative error, up to 1.2e-5 at -3); no more here."""
    dt, dev = torch.bfloat16, "cuda"
    a, b, f = torch.arange(192) / 64, torch.arange(16) * 17 / 2 ** 22, torch.arange(256) / 2 ** 14
    h = torch.zeros(192, 16, 256)
    h[..., 0], h[..., 1], h[..., 2] = -a[:, None], -b, 1.0
    h = h.view(-1, 256)
    up, down = torch.zeros(1, 256, 256), torch.eye(256)[None]
    up[0, :, 0], up[0, :, 1], up[0, :, 2] = 1.0, 1.0, -f  # sums of three terms, exact in fp32
    x = h.double() @ up[0].double().t()
    want = (0.5 * x * torch.erfc(-x / math.sqrt(2))).to(dt)
    w = {k: v.to(dev) for k, v in P.pack_experts(None, up.to(dt), down.to(dt)).items()}
    y = P.experts(h.to(dt).to(dev), torch.zeros(h.shape[0], 1, dtype=torch.int32, device=dev), w, P.UNGATED, 0.0)
    assert (y.cpu() != want).double().mean() < 1.3e-4


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [0, 1, P.UNGATED])
@pytest.mark.parametrize("C,F", [(544, 288), (576, 512)])
def test_experts_in_large_tiles(kind, C, F):
    """Enough pairs for the 256-wide tiles, with experts of every tile height (1 to 4 times 64 pairs, one pair, one
    short of a tile, none) and a reduction that ends in half a step (C, F = 32 mod 64)."""
    dev, E, few = "cuda", 10, [1, 63, 64, 65, 129, 193, 257, 511, 0]
    ids = torch.cat([torch.full((n,), e) for e, n in enumerate(few + [81920 - sum(few)])])
    ids = ids[torch.randperm(ids.numel(), generator=torch.Generator().manual_seed(1))].to(dev)
    h = rand(ids.numel(), C, dtype=torch.bfloat16).to(dev)
    g, u, d = (rand(E, *sh, seed=i, scale=2 * sh[1] ** -0.5, dtype=torch.bfloat16).to(dev)
               for i, sh in enumerate([(F, C), (F, C), (C, F)]))
    w = P.pack_experts(None if kind == P.UNGATED else g, u, d)
    y = P.experts(h, ids.int()[:, None], w, kind, 0.7)
    for e in range(E):
        x = h[ids == e].float()
        a = P.expert_activation(None if kind == P.UNGATED else x @ g[e].float().t(), x @ u[e].float().t(), kind, 0.7)
        if x.numel():
            near(y[ids == e], (a @ d[e].float().t()).cpu(), torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [1, P.UNGATED])
@pytest.mark.parametrize("C,F", [(32, 64), (96, 160), (192, 96), (224, 256)])
def test_experts_in_large_tiles_of_few_steps(kind, C, F):
    """Reductions of half a step to four (a tile's last three steps bring the next tile's rows), several choices per token, workgroups
    with several tiles of unequal heights, and an expert that few chose."""
    dev, E, N, top = "cuda", 10, 50000, 3
    g = torch.Generator().manual_seed(3)
    ids = torch.stack([torch.randperm(E - 1, generator=g)[:top] for _ in range(500)]).repeat(N // 500, 1)
    ids[7, 1] = E - 1
    ids = ids.to(dev)
    h = rand(N, C, dtype=torch.bfloat16).to(dev)
    wg, u, d = (rand(E, *sh, seed=i, scale=2 * sh[1] ** -0.5, dtype=torch.bfloat16).to(dev)
                for i, sh in enumerate([(F, C), (F, C), (C, F)]))
    w = P.pack_experts(None if kind == P.UNGATED else wg, u, d)
    y = P.experts(h, ids.int(), w, kind, 0.7).view(N, top, C)
    for e in range(E):
        tok, k = (ids == e).nonzero(as_tuple=True)
        x = h[tok].float()
        a = P.expert_activation(None if kind == P.UNGATED else x @ wg[e].float().t(), x @ u[e].float().t(), kind, 0.7)
        near(y[tok, k], (a @ d[e].float().t()).cpu(), torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [1, P.UNGATED])
@pytest.mark.parametrize("E,C,F", [(512, 1024, 64), (512, 992, 32), (40, 96, 160), (20, 512, 544), (20, 544, 512),
                                   (20, 1056, 1024), (70, 992, 512), (70, 992, 544)])
def test_experts_of_few_pairs(kind, E, C, F):
    """Few pairs at both widths of the second product's workgroups (64 weight rows from 1024 workgroups of 32, F up to
    512), with an odd number of them, and at widths that end in half of one; reductions of one round of loads (4 or 8 steps of 32 per
    wave), of one step more and of less."""
    dev, N, top = "cuda", 130, 4
    h = rand(N, C, dtype=torch.bfloat16).to(dev)
    ids = torch.stack([torch.randperm(E, generator=torch.Generator().manual_seed(i))[:top] for i in range(N)]).to(dev)
    ids[:40, 0] = 3
    g, u, d = (rand(E, *sh, seed=i, scale=2 * sh[1] ** -0.5, dtype=torch.bfloat16).to(dev)
               for i, sh in enumerate([(F, C), (F, C), (C, F)]))
    w = P.pack_experts(None if kind == P.UNGATED else g, u, d)
    y = P.experts(h, ids.int(), w, kind, 0.7).view(N, top, C)
    x = h.float()[:, None, :, None]
    for k in range(top):
        e = ids[:, k]
        a = P.expert_activation(None if kind == P.UNGATED else (g[e].float() @ x[:, 0])[..., 0],
                                (u[e].float() @ x[:, 0])[..., 0], kind, 0.7)
        near(y[:, k], (d[e].float() @ a.unsqueeze(-1))[..., 0].cpu(), torch.bfloat16)


@pytest.mark.gpu
@pytest.mark.parametrize("N,E", [(1023, 2), (5461, 700), (5462, 700), (6827, 3), (30000, 1000)])
def test_experts_of_many_pairs(N, E):
    """Sorting at the edges of its two forms (16384 pairs) and of their workgroups (4096), with experts of no pair, of
    one and of most: every pair's result, where an expert's weights are its number."""
    dev, C, top = "cuda", 32, 3 if E > 3 else 1
    g = torch.Generator().manual_seed(N)
    ids = torch.randint(0, E, (N, top), generator=g)
    ids[::2, 0] = E - 1
    h = torch.zeros(N, C, dtype=torch.bfloat16)
    h[:, 0] = torch.randint(1, 9, (N,), generator=g)
    u, d = torch.zeros(E, 32, C, dtype=torch.bfloat16), torch.zeros(E, C, 32, dtype=torch.bfloat16)
    u[:, 0, 0] = 16.0  # gelu(16 x) = 16 x for x >= 1
    d[:, 0, 0], d[:, 1, 0] = torch.arange(E) % 31, torch.arange(E) // 31
    w = {k: v.to(dev) for k, v in P.pack_experts(None, u, d).items()}
    y = P.experts(h.to(dev), ids.int().to(dev), w, P.UNGATED, 0.0).cpu().view(N, top, C).float()
    x = 16 * h[:, :1].float()
    for col, of in ((0, ids % 31), (1, ids // 31)):
        assert torch.equal(y[..., col], (x * of).bfloat16().float())  # one product each, rounded once


@pytest.mark.parametrize("target", TARGETS)
@pytest.mark.parametrize("N", [1, 4, 16, 30, 90])
def test_dense_feed_forward(target, N):
    dev, dt = target
    C, F = 64, 48
    p = {k: rand(*sh, seed=i, scale=sh[1] ** -0.5, dtype=dt)
         for i, (k, sh) in enumerate({"gate": (F, C), "up": (F, C), "down": (C, F)}.items())}
    h = rand(N, C, dtype=dt)
    a = P.gated_linear(h.to(dev), torch.cat([p["gate"], p["up"]]).to(dev), 0)
    near(P.linear(a, p["down"].to(dev)), O.dense_ff(h.double(), {k: v.double() for k, v in p.items()}), dt, 2e-2
         if dt == torch.bfloat16 else None)


# --------------------------------------------------------------------------- state manager
def test_state_manager_slots_and_growth():
    st = SequenceState([24, 16], [(8, 3)], [(1e4, 8)], torch.float32, "cpu", slots=1, capacity=4)
    a = st.acquire()
    st.begin([(a, 3)])
    st.latent[0][a, :3] = 7.0
    st.conv[0][a] = 5.0
    b = st.acquire()  # grows the slots, keeps what a holds
    assert a != b and st.slots == 2 and float(st.latent[0][a, :3].min()) == 7.0 and float(st.conv[0][a].min()) == 5.0
    d = st.begin([(b, 2), (a, 2)])  # a outgrows the capacity
    assert st.capacity >= 5 and float(st.latent[0][a, :3].min()) == 7.0
    assert st.tables[(1e4, 8)].shape[0] == st.capacity
    assert d.slot.tolist() == [b, b, a, a] and d.pos.tolist() == [0, 1, 3, 4] and d.first.tolist() == [0, 0, 2, 2]
    assert d.cu.tolist() == [0, 2, 4] and d.lens == [2, 5] and not d.single and not d.fresh
    assert d.query_blocks(2).tolist() == [[1, 0], [0, 0]]
    assert d.key_rows()[0].tolist() == [0, 2, 7]
    st.release(a)
    assert st.acquire() == a and st.length(a) == 0 and st.length(b) == 2
    assert st.begin([(a, 1), (b, 1)]).single
    with pytest.raises(ValueError):
        st.begin([(a, 1), (a, 1)])
    with pytest.raises(ValueError):
        st.begin([(a, 0)])
    st.clear()
    assert st.seq_len() == 0


def test_key_ranges_fill_the_gpu_without_tiny_ranges():
    for rows, heads, n in [(1, 4, 10), (1, 16, 4096), (64, 16, 4096), (1, 128, 100000), (1000, 8, 512)]:
        p = P.key_ranges(rows, heads, n)
        assert 1 <= p <= P.MAX_KEY_RANGES and (p == 1 or n / p >= 32)
        assert p == 1 or rows * math.ceil(heads / 32) * (p - 1) < P.DECODE_WORKGROUPS


def test_upload_is_no_part_of_a_graph(monkeypatch):
    """Refused before anything reaches the device or the host's allocator, where a capture would keep the pinned block's address."""
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    monkeypatch.setattr(torch.Tensor, "pin_memory", lambda t: pytest.fail("pinned under capture"))
    with pytest.raises(RuntimeError, match="captured graph"):
        P.upload([1, 2], torch.int32, torch.device("cuda"))
    assert torch.equal(P.upload([1, 2], torch.int32, torch.device("cpu")), torch.tensor([1, 2], dtype=torch.int32))


@pytest.mark.gpu
@torch.inference_mode()  # (as decoders capture; torch's generator state of a process is of the first capture's mode)
def test_upload_refused_under_capture():
    dev = torch.device("cuda")
    x = P.upload([3, 4], torch.int64, dev)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        with pytest.raises(RuntimeError, match="captured graph"):
            P.upload([1, 2], torch.int64, dev)
        y = x + 1
    for _ in range(3):
        assert torch.equal(P.upload([5, 6], torch.int64, dev).cpu(), torch.tensor([5, 6]))
        graph.replay()
        assert torch.equal(y.cpu(), torch.tensor([4, 5]))
