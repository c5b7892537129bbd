"""Workloads of the 5-view disparity path, through its public entry points.

A case says which entry point is called, with how many rigs of which sizes and
which options.  `prepare` makes the inputs and the handle that a program keeps,
`run` is one call, `work` the bytes and integer operations a call cannot do
without, `exact` the same outputs from plain torch arithmetic.

  entry "class"   SisterMultiviewDisparities.compute_disparities: host arrays
                  in, the three maps out
  entry "host"    Context.compute_rig: host arrays, every output
  entry "device"  Context.run_device: views and outputs in HBM
  entry "graph"   a batch captured once, replayed by graph_launch
  entry "serve"   a burst of device-resident requests to the serving loop
"""
import weakref

import numpy as np
import torch

import sister_amd

# sizes and disparity counts of the repository's mixed batch
MIXED_SIZES = ((640, 480), (1280, 720), (1920, 1080), (2048, 1536))
MIXED_DISPS = (64, 128, 192, 256)
# what a stream of small cameras sends
BURST_SIZES = ((320, 240), (640, 480), (800, 600))
BURST_DISPS = (32, 64)

# integer lane-ops per padded cell of one multiview pass: 4 costs x 5, 8 LR-check
# argmins, the weighted sum 4, 8 paths x 8, the winner 1
OPS_STEREO, OPS_SUM, OPS_SGM = 28, 4, 65


def _case(name, entry, w, h, d, rigs=1, modes=1, subpix=False, pitch=0, mix=""):
    return {"name": name, "entry": entry, "rigs": rigs, "w": w, "h": h, "d": d, "modes": modes,
            "subpix": subpix, "pitch": pitch, "mix": mix}


def listed():
    return [
        # a thumbnail rig through the class: the floor of a call (latency, launches, copies)
        _case("class_64x48_d16", "class", 64, 48, 16, modes=7),
        # the plain rig of the command-line tool: VGA through the class, three maps
        _case("class_640x480_d64", "class", 640, 480, 64, modes=7),
        # a camera that is no multiple of anything, D past 192, every output the host form has
        _case("host_1244x700_d200", "host", 1244, 700, 200, modes=7, subpix=True),
        # a small rig already in HBM: launches and synchronisations alone
        _case("device_96x64_d24", "device", 96, 64, 24),
        # one VGA frame set in HBM, with the sub-pixel map: the ordinary latency call
        _case("device_640x480_d64", "device", 640, 480, 64, subpix=True),
        # one full-HD frame set: the rig the benchmark calls plain
        _case("device_1920x1080_d192", "device", 1920, 1080, 192),
        # the largest rig of the benchmark (D = 384: a workspace of 44 GB)
        _case("device_4096x3000_d384", "device", 4096, 3000, 384),
        # the two pair modes over a few rigs, views inside wider rows, D not a multiple of 16
        _case("device8_1000x620_d136_pairs", "device", 1000, 620, 136, rigs=8, modes=6, pitch=24),
        # a captured batch of one camera model, replayed
        _case("graph16_1920x1080_d192", "graph", 1920, 1080, 192, rigs=16),
        # the headline batch, issued eagerly
        _case("device64_1920x1080_d192", "device", 1920, 1080, 192, rigs=64),
        # a captured batch of mixed cameras, 640x480 D=64 .. 2048x1536 D=256
        _case("graph16_mixed", "graph", 2048, 1536, 256, rigs=16, mix="cameras"),
        # a burst of small requests to the serving loop, waited for
        _case("serve24_small", "serve", 800, 600, 64, rigs=24, mix="burst"),
    ]


def draw(rng):
    """One more case: sizes over their logarithm, widths and heights any
    multiple of 4 and D any multiple of 8, as the entry points take them."""
    entry = rng.choice(("class", "host", "device", "device", "device", "graph"))
    w = 4 * round(2 ** rng.uniform(4, 9))                       # 64 .. 2048
    h = max(16, 4 * round(w * rng.uniform(0.5, 0.9) / 4))
    d = 8 * max(1, min(48, round(w * rng.uniform(0.06, 0.2) / 8)))
    cells = (w + 2 * d) * (h + 2 * d) * d
    rigs = 1
    if entry in ("device", "graph"):
        most = int(min(32, max(1, 6e9 / cells)))
        rigs = max(1, round(2 ** rng.uniform(0, np.log2(most + 0.5))))
    modes = 7 if entry == "class" else rng.choice((1, 1, 7, 6))
    sub = entry != "class" and bool(modes & 1) and rng.random() < 0.5
    pitch = rng.choice((0, 0, 4, 28)) if entry in ("device", "graph") else 0
    c = _case("", entry, w, h, d, rigs, modes, sub, pitch)
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# inputs: textured scenes, a slanted plane with raised boxes, the neighbours
# warped from the centre view, sensor noise
# ---------------------------------------------------------------------------
def shapes(case):
    """(W, H, D) of every rig.  The mixes are part of the case, not of the seed."""
    n = case["rigs"]
    if case["mix"]:
        sizes, disps = (MIXED_SIZES, MIXED_DISPS) if case["mix"] == "cameras" else (BURST_SIZES, BURST_DISPS)
        r = np.random.default_rng(1000)
        return [(*sizes[int(r.integers(len(sizes)))], disps[int(r.integers(len(disps)))]) for _ in range(n)]
    return [(case["w"], case["h"], case["d"])] * n


def _blur(img, sigma):
    k = torch.arange(-6, 7, device=img.device, dtype=torch.float32)
    k = torch.exp(-0.5 * (k / sigma) ** 2)
    k = k / k.sum()
    x = img[None, None]
    x = torch.nn.functional.conv2d(torch.nn.functional.pad(x, (6, 6, 0, 0), mode="reflect"), k.view(1, 1, 1, -1))
    x = torch.nn.functional.conv2d(torch.nn.functional.pad(x, (0, 0, 6, 6), mode="reflect"), k.view(1, 1, -1, 1))
    return x[0, 0]


def _views(W, H, D, seed, device):
    """Five H x W uint8 views (center, right, top, left, bottom)."""
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    rs = np.random.RandomState(seed % (1 << 32))
    img = torch.rand((H, W), generator=g, device=device)
    img = _blur(img, 1.5)
    img = torch.round((img - img.min()) / (img.max() - img.min()) * 255.0)
    d = (0.1 * D + 0.2 * D * torch.arange(W, device=device, dtype=torch.float32) / (W - 1)).expand(H, W).clone()
    for _ in range(5):
        bw, bh = (int(rs.randint(max(4, s // 10), max(5, s // 3))) for s in (W, H))
        x, y = int(rs.randint(0, W - bw + 1)), int(rs.randint(0, H - bh + 1))
        d[y:y + bh, x:x + bw] = float(rs.uniform(0.3, 0.9)) * D
    ys = torch.arange(H, device=device, dtype=torch.float32)[:, None]
    xs = torch.arange(W, device=device, dtype=torch.float32)[None, :]
    out = [img]
    for sx, sy in ((1, 0), (0, -1), (-1, 0), (0, 1)):
        fx, fy = (xs + sx * d).clamp(0, W - 1), (ys + sy * d).clamp(0, H - 1)
        x0, y0 = fx.floor(), fy.floor()
        ax, ay = fx - x0, fy - y0
        x0, y0 = x0.long(), y0.long()
        x1, y1 = (x0 + 1).clamp(max=W - 1), (y0 + 1).clamp(max=H - 1)
        v = (img[y0, x0] * (1 - ax) + img[y0, x1] * ax) * (1 - ay) + (img[y1, x0] * (1 - ax) + img[y1, x1] * ax) * ay
        out.append(v + 2.0 * torch.randn((H, W), generator=g, device=device))
    return torch.stack([torch.round(v).clamp(0, 255).to(torch.uint8) for v in out])


def _inputs(case, seed, device):
    return [_views(W, H, D, seed * 1009 + i, device) for i, (W, H, D) in enumerate(shapes(case))]


# One handle per workload, kept as long as a state of it lives (a program keeps
# one).  A context holds one captured batch, so each captured state has its own.
_handles = weakref.WeakValueDictionary()


def _handle(case):
    key = (case["entry"], case["rigs"], case["w"], case["h"], case["d"], case["mix"])
    if case["entry"] == "graph":
        return sister_amd.Context()
    ctx = _handles.get(key)
    if ctx is None:
        ctx = sister_amd.Context()
        if case["entry"] == "serve":
            ctx.serve_start(4)
        _handles[key] = ctx
    return ctx


def _names(case):
    names = [n for bit, n in ((1, "multiview"), (2, "horizontal"), (4, "vertical")) if case["modes"] & bit]
    if case["modes"] & 1 and case["entry"] != "class":
        names += ["disp"] + (["subpix"] if case["subpix"] else [])
    return names


def prepare(case, seed):
    ctx = _handle(case)
    imgs = _inputs(case, seed, "cuda")
    if case["entry"] in ("class", "host"):
        return {"case": case, "ctx": ctx, "views": [v.cpu().numpy() for v in imgs[0]]}
    # each output of all rigs in one buffer, rig after rig (16-bit maps as
    # their bit patterns in int16)
    npx = [W * H for W, H, _ in shapes(case)]
    outs = {n: torch.zeros(sum(npx), device="cuda", dtype=torch.float32 if n == "subpix" else torch.int16)
            for n in _names(case)}
    rigs, at = [], 0
    for (W, H, D), n, v in zip(shapes(case), npx, imgs):
        if case["pitch"]:
            wide = torch.zeros((5, H, W + case["pitch"]), dtype=torch.uint8, device="cuda")
            wide[:, :, :W] = v
            v = wide[:, :, :W]
        mine = {k: o[at:at + n].view(H, W) for k, o in outs.items()}
        rigs.append((sister_amd.Context.rig_struct(list(v), D, mine), v))
        at += n
    state = {"case": case, "ctx": ctx, "rigs": [r for r, _ in rigs], "views": [v for _, v in rigs], "outs": outs}
    if case["entry"] == "graph":
        torch.cuda.synchronize()
        ctx.graph_capture(state["rigs"], case["modes"])
    return state


def run(state):
    case, ctx = state["case"], state["ctx"]
    if case["entry"] == "class":
        return sister_amd.SisterMultiviewDisparities(*state["views"], context=ctx).compute_disparities(case["d"])
    if case["entry"] == "host":
        return ctx.compute_rig(state["views"], case["d"], modes=case["modes"], disp=True, subpix=case["subpix"])
    if case["entry"] == "device":
        ctx.run_device(state["rigs"], case["modes"])
    elif case["entry"] == "graph":
        ctx.graph_launch()
    else:
        for t in [ctx.submit(r, case["modes"], device=True) for r in state["rigs"]]:
            ctx.wait(t)
    return state["outs"]


def work(case):
    sums = sum((case["modes"] >> m) & 1 for m in range(3))
    nbytes = flops = 0
    for W, H, D in shapes(case):
        nbytes += 5 * W * H + sum(W * H * (4 if n == "subpix" else 2) for n in _names(case))
        flops += (OPS_STEREO + sums * (OPS_SUM + OPS_SGM)) * (W + 2 * D) * (H + 2 * D) * D
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------------------
# the same maps from plain torch integers, written from the definitions
# ---------------------------------------------------------------------------
EXACT_CELLS = 1.2e9    # padded cells of all rigs, times the modes (about 3 seconds)


def _popcount(x):
    x = x - ((x >> 1) & 0x5555555555555555)
    x = (x & 0x3333333333333333) + ((x >> 2) & 0x3333333333333333)
    x = (x + (x >> 4)) & 0x0F0F0F0F0F0F0F0F
    return ((x * 0x0101010101010101) >> 56) & 0x7F


def _census(img):
    R, C = img.shape
    code = torch.zeros((R, C), dtype=torch.int64, device=img.device)
    core, last = torch.zeros((R - 6, C - 8), dtype=torch.int64, device=img.device), None
    for y in range(-3, 4):
        for x in range(-4, 5):
            a = img[3 + y:R - 3 + y, 4 + x:C - 4 + x]
            b = img[3 - y:R - 3 - y, 4 - x:C - 4 - x]
            last = (a > b).long()
            core = (core << 1) | last
    # the 64th bit is the last test of the pixel before, in raster order
    carry = torch.cat([torch.zeros(1, dtype=torch.int64, device=img.device), last.reshape(-1)[:-1]]).view_as(core)
    code[3:R - 3, 4:C - 4] = (core & 0x7FFFFFFFFFFFFFFF) | (carry << 63)
    return code


def _to_frame(p, F):
    return (p, p.flip(0, 1).t(), p.flip(1), p.flip(1).t())[F]


def _from_frame(a, F):
    return (a, a.t().flip(0, 1), a.flip(1), a.t().flip(1))[F]


def _median_in_place(maps):
    """3x3 median of [K, R, C] maps, rows above already replaced: the window of
    flat position q is out[q-C-1 .. q-C+1] and in[q-1 .. q+1, q+C-1 .. q+C+1]."""
    K, R, C = maps.shape
    n = R * C
    src = maps.reshape(K, n)
    out = src.clone()
    for r in range(1, R):
        lo, hi = r * C, min((r + 1) * C, n - C - 4)
        if lo >= hi:
            break
        q = torch.arange(lo, hi, device=maps.device)
        win = lambda j: torch.stack([out[:, j - C - 1], out[:, j - C], out[:, j - C + 1], src[:, j - 1], src[:, j],  # noqa: E731
                                     src[:, j + 1], src[:, j + C - 1], src[:, j + C], src[:, j + C + 1]]).sort(0)[0][4]
        vals = win(q)
        if r == 1:
            vals[:, 0] = 0
        out[:, lo:hi] = vals
        if hi == (r + 1) * C:    # the last column's window holds column 0 of its own row
            out[:, hi - 1] = win(torch.tensor([hi - 1], device=maps.device))[:, 0]
    return out.view(K, R, C)


def _sgm_step(m, prev, pmin, p1=7, p2=100):
    """One step of every chain: m and prev [..., D] (guards beyond 0 and D-1)."""
    up = torch.nn.functional.pad(prev[..., :-1], (1, 0), value=1 << 20)
    dn = torch.nn.functional.pad(prev[..., 1:], (0, 1), value=1 << 20)
    best = torch.minimum(torch.minimum(prev, torch.minimum(up, dn) + p1), (pmin + p2)[..., None])
    cur = m + best - pmin[..., None]
    return cur, cur.amin(-1)


def _exact_rig(views, D, modes):
    dev = views.device
    H, W = views.shape[1:]
    Hp, Wp = H + 2 * D, W + 2 * D
    yy = (torch.arange(Hp, device=dev) - D).clamp(0, H - 1)
    xx = (torch.arange(Wp, device=dev) - D).clamp(0, W - 1)
    pad = [v.to(torch.int32)[yy][:, xx] for v in views]
    codes = [(_census(_to_frame(pad[0], F)), _census(_to_frame(pad[1 + F], F))) for F in range(4)]
    best = []
    for CC, CN in codes:
        L = torch.full(CC.shape, 1 << 30, dtype=torch.int64, device=dev)
        Rr = L.clone()
        C = CC.shape[1]
        for d in range(D):
            if d >= C:
                break
            key = _popcount(CC[:, d:] ^ CN[:, :C - d]) * 512 + d
            L[:, d:] = torch.minimum(L[:, d:], key)
            Rr[:, :C - d] = torch.minimum(Rr[:, :C - d], key)
        best.append((L & 511, Rr & 511))
    masks = [None] * 4
    for pair in ((0, 2), (1, 3)):
        med = _median_in_place(torch.stack([m for F in pair for m in best[F]]))
        for k, F in enumerate(pair):
            L, Rr = med[2 * k], med[2 * k + 1]
            c = torch.arange(L.shape[1], device=dev)[None, :].expand_as(L)
            back = torch.gather(Rr, 1, (c - L).clamp(min=0))
            masks[F] = (L >= 1) & (L <= c) & ((L - back).abs() <= 5) & (c >= D)
    res = {}
    for m, name, frames in ((0, "multiview", (0, 1, 2, 3)), (1, "horizontal", (0, 2)), (2, "vertical", (1, 3))):
        if not (modes >> m) & 1:
            continue
        M = torch.zeros((D, Hp, Wp), dtype=torch.int16, device=dev)
        for F in frames:
            CC, CN = codes[F]
            C = CC.shape[1]
            for d in range(D):
                cost = torch.zeros(CC.shape, dtype=torch.int16, device=dev)
                cost[:, d:] = _popcount(CC[:, d:] ^ CN[:, :C - d]).to(torch.int16)
                M[d] += _from_frame(cost * masks[F], F)
        M = M.permute(1, 2, 0).contiguous()                      # [y, x, d]
        S = torch.zeros((H, W, D), dtype=torch.int32, device=dev)
        crop = M[D:D + H]
        for xs in (range(Wp), range(Wp - 1, -1, -1)):            # rows, restarted at each border
            cur = None
            for x in xs:
                c = crop[:, x].to(torch.int32)
                cur, cmin = (c, c.amin(-1)) if cur is None else _sgm_step(c, cur, cmin)
                if D <= x < D + W:
                    S[:, x - D] += cur
        for ys in (range(Hp), range(Hp - 1, -1, -1)):            # columns and both diagonals
            cur = None
            for y in ys:
                c = M[y].to(torch.int32)
                if cur is None:                                  # the first line takes its costs
                    cur = c.expand(3, Wp, D)
                    cmin = cur.amin(-1)
                    continue
                prev = torch.full((3, Wp, D), 1 << 20, dtype=torch.int32, device=dev)
                pmin = torch.zeros((3, Wp), dtype=torch.int32, device=dev)
                prev[0], pmin[0] = cur[0], cmin[0]
                prev[1, 1:], pmin[1, 1:] = cur[1, :-1], cmin[1, :-1]
                prev[2, :-1], pmin[2, :-1] = cur[2, 1:], cmin[2, 1:]
                cur, cmin = _sgm_step(c, prev, pmin)
                if D <= y < D + H:
                    S[y - D] += cur[:, D:D + W].sum(0, dtype=torch.int32)
        d = (S * 512 + torch.arange(D, device=dev, dtype=torch.int32)).amin(-1).long() & 511
        res[name] = (d * 255).clamp(max=65535)
        if m == 0:
            at = lambda k: torch.gather(S, 2, k.clamp(0, D - 1)[..., None])[..., 0].double()  # noqa: E731
            sm, s0, sp = at(d - 1), at(d), at(d + 1)
            den = sm - 2 * s0 + sp
            ok = (d > 0) & (d < D - 1) & (den > 0)
            res["disp"] = d
            res["subpix"] = d.double() + torch.where(ok, (sm - sp) / (2 * torch.where(ok, den, torch.ones_like(den))), torch.zeros_like(den))
        del M, S
    return res


def exact(case, seed):
    sums = sum((case["modes"] >> m) & 1 for m in range(3))
    if sums * sum((W + 2 * D) * (H + 2 * D) * D for W, H, D in shapes(case)) > EXACT_CELLS:
        return None
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    rigs = [_exact_rig(v, D, case["modes"]) for v, (_, _, D) in zip(_inputs(case, seed, dev), shapes(case))]
    if case["entry"] == "class":
        return tuple(rigs[0][n] for n in _names(case))
    if case["entry"] == "host":
        return {n: rigs[0][n] for n in _names(case)}
    return {n: torch.cat([r[n].reshape(-1) for r in rigs]) for n in _names(case)}
