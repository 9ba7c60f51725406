"""CPU emulation of the one-launch SOR (k_sor_res.hip): the cut into boxes, the
column of every thread, the LDS copy with its halo ring, the side a cell's
in-row neighbour lies on, the halo words every block sends and receives, the
walls, the periodic rows of even and odd jm and the ghosts iteration 1 reads.
Every index is checked against its buffer, every word a block waits for against
being written, once, in that sweep, and the iterates against plain
red-black iterations of the reference's loop (press.f95:89-111 with boundp1
after each colour and boundp2 after both) bit for bit in FP32."""
import numpy as np
import pytest

NT, PLANE, WORDS = 512, 832, 8
f32 = np.float32


def reference(p, rhs, c2, c3, lev, omega, iters):
    """p (im+2, jm+2, km+2) with the entry ghosts; the reference's loop."""
    p = p.copy()
    im, jm, km = (n - 2 for n in p.shape)
    sums = []
    i, j, k = np.meshgrid(np.arange(1, im + 1), np.arange(1, jm + 1), np.arange(1, km + 1), indexing="ij")
    c4l, c4s, cn = (lev[n][None, None, :] for n in range(3))
    for _ in range(iters):
        s = 0.0
        for col in (1, 0):
            m = ((i + j + k) & 1) == col
            q = p[1:-1, 1:-1, 1:-1]
            x = (c2 * p[2:, 1:-1, 1:-1] + c2 * p[:-2, 1:-1, 1:-1] + c3 * p[1:-1, 2:, 1:-1] + c3 * p[1:-1, :-2, 1:-1]
                 + c4l * p[1:-1, 1:-1, 2:] + c4s * p[1:-1, 1:-1, :-2] - rhs)
            rel = np.where(m, omega * (cn * x - q), f32(0))
            p[1:-1, 1:-1, 1:-1] = q + rel
            s += float((rel.astype(np.float64) ** 2).sum())
            p[0], p[-1] = p[1], p[-2]
            p[:, 0], p[:, -1] = p[:, -2], p[:, 1]
        p[:, :, 0], p[:, :, -1] = p[:, :, 1], p[:, :, -2]
        sums.append(s)
    return p[1:-1, 1:-1, 1:-1], sums


class Box:
    def __init__(self, sh, bid):
        self.bid = bid
        self.bx, self.by, self.bz = bid % sh.ntx, bid // sh.ntx % sh.nty, bid // (sh.ntx * sh.nty)
        cut = lambda n, m, q: (q * n // m, (q + 1) * n // m)  # noqa: E731
        self.t0, t1 = cut(sh.nt, sh.ntx, self.bx)
        j0, j1 = cut(sh.jm, sh.nty, self.by)
        k0, k1 = cut(sh.km, sh.ntz, self.bz)
        self.tpn, self.tjn, self.nlev = t1 - self.t0, j1 - j0, k1 - k0
        self.j0, self.k0 = 1 + j0, 1 + k0
        assert 0 < self.tpn <= sh.tp and 0 < self.tjn <= sh.tj and 0 < self.nlev <= sh.kl


class Shape:
    def __init__(self, im, jm, km, ntx, nty, ntz):
        self.im, self.jm, self.km, self.ntx, self.nty, self.ntz = im, jm, km, ntx, nty, ntz
        self.nt = (im + 1) // 2
        up = lambda a, b: -(-a // b)  # noqa: E731
        self.tp, self.tj, self.kl = up(self.nt, ntx), up(jm, nty), up(km, ntz)
        self.nb = ntx * nty * ntz
        self.NI = self.tj * self.kl if ntx > 1 else 0
        self.NJ = self.tp * self.kl
        self.NT, self.nthr = NT, max(64, -(-max(self.tp * self.tj, -(-(2 * self.NI + 2 * self.NJ) // WORDS)) // 64) * 64)
        self.nq = -(-(2 * self.NI + 2 * self.NJ) // self.nthr)
        self.iw = self.nq * self.nthr + 2 * NT
        self.W = self.tp + 2
        self.odd = jm & 1
        # the limits of res_shape
        assert self.nthr <= NT and self.nq <= WORDS
        assert self.W * (self.tj + 2 + (4 if self.odd else 0)) < PLANE


def solve(sh, p, rhs, c2, c3, lev, omega, iters, zero=False):
    """The launch: p (im+2, jm+2, km+2), rhs (im, jm, km)."""
    im, jm, W, BK = sh.im, sh.jm, sh.W, -(-sh.kl // 4) * 4
    inbox = [np.full((sh.nb, sh.iw), np.nan, f32) for _ in range(2)]
    tag = [np.zeros((sh.nb, sh.iw), int) for _ in range(2)]
    P = np.zeros((im + 3, jm + 2, sh.km + 2), f32)  # the padded field: i = im+1 exists, im+2 too
    P[:im + 2] = p
    if zero:
        P[:] = 0
    boxes = []
    for bid in range(sh.nb):
        b = Box(sh, bid)
        tid = np.arange(NT)
        b.row, b.t = tid // b.tpn, tid % b.tpn
        b.act = b.row < b.tjn
        b.tg, b.j = b.t0 + b.t, b.j0 + b.row
        b.par = (b.j + b.k0) & 1
        b.cen = np.where(b.act, (b.row + 1) * W + b.t + 1, W + 1)
        b.side = np.where(b.par == 1, 1, -1)
        wlo, whi = b.tg == 0, b.tg == sh.nt - 1
        b.wl = [np.where(b.par == 1, whi, wlo), np.where(b.par == 1, wlo, whi)]
        last = whi & bool(im & 1)
        b.inv = [last & (b.par == 1), last & (b.par == 0)]
        b.wrl = bool(sh.odd) & (b.by == 0) & (b.row == 0)
        b.wrh = bool(sh.odd) & (b.by == sh.nty - 1) & (b.row == b.tjn - 1)
        b.S = np.full((BK, PLANE), np.nan, f32)
        b.v = np.zeros((2, BK, NT), f32)
        b.rh = np.zeros((2, BK, NT), f32)
        b.hlo, b.hhi = np.zeros((2, NT), f32), np.zeros((2, NT), f32)
        a = np.flatnonzero(b.act)
        tg, j = b.tg[a], b.j[a]
        for kk in range(b.nlev):
            k = b.k0 + kk
            pr = ((b.par[a] + kk) & 1) != 0
            x, y = P[2 * tg + 1, j, k], P[2 * tg + 2, j, k]
            b.v[1, kk, a], b.v[0, kk, a] = np.where(pr, y, x), np.where(pr, x, y)
            for c in (0, 1):
                i = 2 * tg + 1 + ((1 + j + k + c) & 1)
                b.rh[c, kk, a] = np.where(i <= im, rhs[np.minimum(i, im) - 1, j - 1, k - 1], f32(7))
            b.S[kk, b.cen[a]] = b.v[0, kk, a]
            for hi in (0, 1):
                pp = np.arange(b.tpn)
                tt, je = b.t0 + pp, b.j0 + b.tjn - 1 if hi else b.j0
                jn = je + 1 if hi else je - 1
                i = 2 * tt + 1 + ((1 + je + k + 1) & 1)
                if sh.odd and (je == jm if hi else je == 1):
                    b.S[kk, (sh.tj + 4 + hi) * W + pp + 1] = P[i, jn, k]
                    ib = 2 * tt + 1 + ((1 + je + k) & 1)
                    b.S[kk, (sh.tj + 2 + hi) * W + pp + 1] = np.where(ib > im, f32(0), P[ib, 1 if hi else jm, k])
                else:
                    b.S[kk, (b.tjn + 1 if hi else 0) * W + pp + 1] = P[i, jn, k]
                r = np.arange(b.tjn)
                b.S[kk, (r + 1) * W + (b.tpn + 1 if hi else 0)] = P[2 * (b.t0 + b.tpn) + 1 if hi else 2 * b.t0,
                                                                  b.j0 + r, k]
        k1 = b.k0 + b.nlev - 1
        for c in (0, 1):
            b.hlo[c, a] = P[2 * tg + 1 + ((1 + j + b.k0 + c) & 1), j, b.k0 - 1]
            b.hhi[c, a] = P[2 * tg + 1 + ((1 + j + k1 + c) & 1), j, k1 + 1]
        # the halo words: e, the box sent to, source, destination, colour stride
        b.words = []
        for e in range(sh.nq * sh.nthr):
            to, so, de, wrap = bid, 0, PLANE - 1, 0
            if e < 2 * sh.NI:
                hi = int(e >= sh.NI)
                r, kk = divmod(e - sh.NI * hi, sh.kl)
                to = bid - b.bx + (b.bx + (sh.ntx - 1 if hi else 1)) % sh.ntx
                if r < b.tjn and kk < b.nlev:
                    so = kk * PLANE + (r + 1) * W + (1 if hi else b.tpn)
                    if (b.bx < sh.ntx - 1) if hi else (b.bx > 0):
                        de = kk * PLANE + (r + 1) * W + (b.tpn + 1 if hi else 0)
            elif e < 2 * sh.NI + 2 * sh.NJ:
                f = e - 2 * sh.NI
                hi = int(f >= sh.NJ)
                kk, pp = divmod(f - sh.NJ * hi, sh.tp)
                to = b.bx + sh.ntx * ((b.by + (sh.nty - 1 if hi else 1)) % sh.nty + sh.nty * b.bz)
                if pp < b.tpn and kk < b.nlev:
                    so = kk * PLANE + (1 if hi else b.tjn) * W + pp + 1
                    wrap = int(sh.odd and (b.by == sh.nty - 1 if hi else b.by == 0))
                    de = kk * PLANE + (sh.tj + 2 + hi if wrap else b.tjn + 1 if hi else 0) * W + pp + 1
            st = 2 * W * wrap
            assert 0 <= so < 65536 and 0 <= de + st < min(65536, BK * PLANE)
            assert de == PLANE - 1 or (de + st) // PLANE == de // PLANE
            assert 0 <= to < sh.nb and e < sh.iw - 2 * sh.NT
            b.words.append((e, to, so, de, st))
        boxes.append(b)
    sums = []
    for it in range(1, iters + 1):
        s = 0.0
        for c in (1, 0):
            later = it > 1 or zero
            n = 2 * it + c
            for b in boxes:
                bel = b.v[c, 0] if b.bz == 0 and later else b.hlo[c]
                wall = [b.wl[c ^ 1] & (later or c == 0), b.wl[c] & (later or c == 0)]
                new = b.v[c].copy()
                for kk in range(b.nlev):
                    ai = (kk & 1) ^ (c ^ 1)
                    own, oth = b.v[c, kk], b.v[c ^ 1, kk]
                    au, ad = b.cen - W, b.cen + W
                    if sh.odd:
                        xr = b.cen + (sh.tj + 2 + 2 * c - 1 - b.row) * W
                        au, ad = np.where(b.wrl, xr, au), np.where(b.wrh, xr + W, ad)
                    la = b.cen + (b.side if ai == 0 else -b.side)
                    for x in (au, ad, la):
                        assert x.min() >= 0 and x.max() < PLANE
                    lat = np.where(wall[kk & 1], own, b.S[kk, la])
                    if im & 1:
                        oth = np.where(b.inv[ai ^ 1] & (later or c == 0), own, oth)
                    pkm = bel if kk == 0 else b.v[c ^ 1, kk - 1]
                    pkp = (own if b.bz == sh.ntz - 1 and later else b.hhi[c]) if kk == b.nlev - 1 else b.v[c ^ 1,
                                                                                                           kk + 1]
                    k = b.k0 + kk - 1
                    x = (c2 * lat + c2 * oth + c3 * b.S[kk, ad] + c3 * b.S[kk, au] + lev[0][k] * pkp + lev[1][k] * pkm
                         - b.rh[c, kk])
                    rel = omega * (lev[2][k] * x - own)
                    if im & 1:
                        rel = np.where(b.inv[ai], f32(0), rel)
                    assert np.isfinite(rel[b.act]).all()
                    s += float((rel[b.act].astype(np.float64) ** 2).sum())
                    new[kk] = own + rel
                b.v[c] = np.where(b.act, new, b.v[c])
            for b in boxes:  # the copy, the faces
                a = np.flatnonzero(b.act)
                for kk in range(b.nlev):
                    b.S[kk, b.cen[a]] = b.v[c, kk, a]
                base = sh.nq * sh.nthr
                per = sh.ntx * sh.nty
                for cond, to, e, val in ((b.bz > 0, b.bid - per, base + sh.NT, b.v[c, 0]),
                                         (b.bz < sh.ntz - 1, b.bid + per, base, b.v[c, b.nlev - 1])):
                    if cond:
                        x = np.arange(sh.nthr)
                        assert (tag[c][to, e + x] != n).all() and (e + x).max() < sh.iw
                        inbox[c][to, e + x], tag[c][to, e + x] = val[:sh.nthr], n
                flat = b.S.reshape(-1)
                for e, to, so, de, st in b.words:
                    if sh.nb == 1:
                        flat[de + st * c] = flat[so]
                    else:
                        assert tag[c][to, e] != n
                        inbox[c][to, e], tag[c][to, e] = flat[so], n
            for b in boxes:
                a = np.flatnonzero(b.act)
                base = sh.nq * sh.nthr
                for cond, e, dst in ((b.bz > 0, base, b.hlo), (b.bz < sh.ntz - 1, base + sh.NT, b.hhi)):
                    if cond:  # every thread of the block waits for its words
                        assert (tag[c][b.bid, e + np.arange(sh.nthr)] == n).all()
                        dst[c ^ 1, a] = inbox[c][b.bid, e + a]
                flat = b.S.reshape(-1)
                if sh.nb > 1:
                    for e, to, so, de, st in b.words:
                        assert tag[c][b.bid, e] == n
                        flat[de + st * c] = inbox[c][b.bid, e]
        sums.append(s)
    out = np.full((im, jm, sh.km), np.nan, f32)
    for b in boxes:
        a = np.flatnonzero(b.act)
        tg, j = b.t0 + b.cen[a] % W - 1, b.j0 + b.cen[a] // W - 1
        assert (tg == b.tg[a]).all() and (j == b.j[a]).all()
        for kk in range(b.nlev):
            k = b.k0 + kk
            for c in (0, 1):
                i = 2 * tg + 1 + ((1 + j + k + c) & 1)
                ok = i <= im
                assert np.isnan(out[i[ok] - 1, j[ok] - 1, k - 1]).all()
                out[i[ok] - 1, j[ok] - 1, k - 1] = b.v[c, kk, a][ok]
    return out, sums


CASES = [
    (24, 20, 16, 1, 1, 1, 1.0), (23, 20, 9, 1, 1, 1, 1.0), (24, 9, 5, 1, 1, 2, 1.0),
    (24, 20, 16, 2, 2, 3, 1.0), (25, 21, 13, 3, 2, 4, 1.0), (12, 7, 5, 2, 3, 2, 1.5),
    (31, 2, 6, 4, 1, 2, 1.0), (2, 2, 2, 1, 1, 1, 1.0), (3, 3, 3, 2, 1, 3, 1.2),
    (9, 5, 4, 5, 5, 4, 1.0), (40, 12, 11, 3, 4, 1, 1.0), (200, 5, 3, 2, 1, 1, 1.0),
]


@pytest.mark.parametrize("zero", [False, True], ids=["entry", "zero"])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c[:3])) + "-boxes" + "x".join(map(str, c[3:6])))
def test_boxes_give_the_reference_iterates(case, zero):
    im, jm, km, ntx, nty, ntz, om = case
    rng = np.random.default_rng(im * 1000 + jm * 10 + km)
    p = np.zeros((im + 2, jm + 2, km + 2), f32) if zero else rng.uniform(-1, 1, (im + 2, jm + 2, km + 2)).astype(f32)
    rhs = rng.uniform(-1, 1, (im, jm, km)).astype(f32)
    lev = [rng.uniform(0.1, 0.3, km).astype(f32) for _ in range(3)]
    c2, c3, om = f32(0.0625), f32(0.11), f32(om)
    want, ws = reference(p, rhs, c2, c3, lev, om, 4)
    got, gs = solve(Shape(im, jm, km, ntx, nty, ntz), p, rhs, c2, c3, lev, om, 4, zero)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    np.testing.assert_allclose(gs, ws, rtol=1e-12)
