"""The exact sequential sums of the device CDF (cdf_step.hip, exact_seq_sum), restated in Python
step for step and checked against the plain sequential f64 sum they must reproduce.

The device sums a row's non-negative terms without forming them one after the other: while the
running sum s stays in one binade, s = T u on the grid u = 2^(E-52) and fl(s + x) = (T + a) u
with a = round(x / u), half to the side that makes T + a even.  Segments of 256 terms (a wave's,
four a lane) are counted on a binade that the segment sums guess, their ties settled from the
parity of T on 64-bit lane masks (odd_before, odd_behind, wave_ties, grid_count); one wave then
adds runs of up to 64 counts (chain) and takes the other segments in rounds up to each crossing
or NaN (exact_segment).  The functions below have the device's names and do its operations,
prefix sums in its order of adds included, so a flaw in the method (a wrong mask, a missed tie, a
wrong crossing test, the subnormal grid, the -0.0 start) fails here on the CPU, on inputs built to
hit each case; the GPU tests then check the kernel against the host CDF bit for bit.
"""
import math

import numpy as np
import pytest

LANES, TERMS = 64, 4             # kTerms terms a lane
SEG = LANES * TERMS              # kSegTerms
WINDOW, SLOTS = 256, 24          # kWinSegs segments of a window, kSlots of them in LDS
ALL = (1 << 64) - 1
NO_GRID = 0


def sequential(x, s0):
    s = np.float64(s0)
    for v in x:
        s = np.float64(s + np.float64(v))
    return s


def same(a, b):
    return (math.isnan(a) and math.isnan(b)) or np.float64(a).view(np.uint64) == np.float64(b).view(np.uint64)


def bits(v):
    return np.asarray(v, np.float64).view(np.uint64)


def ballot(lanes):
    return sum(1 << i for i, v in enumerate(lanes) if v)


def lanes(mask):
    return np.array([mask >> i & 1 for i in range(LANES)], bool)


def wave_incl_sum(v):
    """The DPP scan: shifts of 1, 2, 4, 8 within rows of 16, then row 0 / 2's last lane into rows
    1 / 3 and lane 31 into rows 2 and 3."""
    v = np.array(v, np.float64).reshape(4, 16)
    for k in (1, 2, 4, 8):
        v = v + np.concatenate([np.zeros((4, k)), v[:, :-k]], 1)
    v = v + np.array([[0.0], [v[0, 15]], [0.0], [v[2, 15]]])
    v = v + np.array([[0.0], [0.0], [v[1, 15]], [v[1, 15]]])
    return v.reshape(LANES)


# ---- ties on 64-bit masks ----

def odd_before(H, P):
    x = P << 1 & ALL
    for k in (1, 2, 4, 8, 16, 32):
        x ^= x << k & ALL
    other = ~H & ALL
    return x ^ (((x & H) << 1) + other & ALL ^ other)


def odd_behind(H, P):
    frm = ALL << H.bit_length() - 1 & ALL if H else ALL
    return bin(P & frm).count("1") & 1


def grid_term(q):
    """The count, the remainder and the count's parity of q on the grid (arrays)."""
    m = q + 2.0 ** 52
    a = m - 2.0 ** 52
    return a, q - a, (bits(m) & np.uint64(1)).astype(bool)


def unit_step(mask, d):
    return np.where(lanes(mask), np.where(np.signbit(d), -1.0, 1.0), 0.0)


def wave_ties(d, odd):
    """d, odd: [TERMS][LANES].  The masks of the device's WaveTies."""
    x = seen = first_x = 0
    step, lead = [], []
    for j in range(TERMS):
        tie = ballot(np.abs(d[j]) == 0.5)
        lead.append(tie & ~seen)
        step.append(tie & seen & x)
        first_x |= lead[j] & x
        seen |= tie
        x = (x ^ ballot(odd[j])) & ~tie
    w_odd = odd_before(seen, x) ^ first_x
    first = seen & -seen
    step = [step[j] | (lead[j] & w_odd & ~first) for j in range(TERMS)]
    return step, lead, first, w_odd, odd_behind(seen, x)


def lane_sum(a):
    return (a[0] + a[1]) + (a[2] + a[3])


def by_lane(x):
    """A segment's terms as [TERMS][LANES] (lane L: terms 4 L ..), zeros past its end."""
    return np.concatenate([x, np.zeros(SEG - len(x))]).reshape(LANES, TERMS).T


def grid_count(fx, ks):
    """(count, tie bits) of a segment on the grid 2^-ks."""
    with np.errstate(over="ignore", invalid="ignore"):
        a, d, odd = grid_term(fx * math.ldexp(1.0, ks))
        mine, ties = lane_sum(a), 0
        if (np.abs(d) == 0.5).any():
            step, lead, first, w_odd, behind = wave_ties(d, odd)
            down = 0
            for j in range(TERMS):
                mine = mine + unit_step(step[j], d[j])
                down |= lead[j] & ballot(d[j] < 0.0)
            ties = 1 | (2 if w_odd & first else 0) | behind << 2 | (8 if down & first else 0)
        total = wave_incl_sum(mine)[63]
        return total, ties or int(bits(total + 2.0 ** 52) & np.uint64(1)) << 2


# ---- rounds, runs of counts, windows ----

def ldexp(v, k):
    with np.errstate(over="ignore", under="ignore", invalid="ignore"):
        return np.ldexp(np.float64(v), k)


def exact_segment(fx, s):
    """s after a segment's terms, in rounds up to each crossing or NaN; and the rounds."""
    fx, rounds = np.array(fx), 0
    while True:
        if not s < 2.0 ** 52:
            return s, rounds
        rounds += 1
        sub = s < 2.0 ** -1022
        ks = 1074 if sub else 1075 - int(bits(s) >> np.uint64(52))
        top = 2.0 ** 52 if sub else 2.0 ** 53
        T0 = ldexp(s, ks)
        with np.errstate(over="ignore", invalid="ignore"):
            q = np.ldexp(fx, ks)
            bad = ~(q < 2.0 ** 52)
            a, d, odd = grid_term(np.where(bad, 0.0, q))
        if (np.abs(d) == 0.5).any():
            step, lead, first, w_odd, _ = wave_ties(d, odd)
            t_odd = bool(int(bits(T0 + 2.0 ** 52 if sub else T0)) & 1)
            first = first if bool(w_odd & first) != t_odd else 0
            a = np.stack([a[j] + unit_step(step[j] | (lead[j] & first), d[j]) for j in range(TERMS)])
        incl = wave_incl_sum(lane_sum(a))
        end = T0 + incl[63]
        if not bad.any() and end < top:
            return ldexp(end, -ks), rounds
        c = np.cumsum(a, 0)
        base = T0 + np.concatenate([[0.0], incl[:-1]])
        hit = bad | (base + c >= top)
        src = int(np.argmax(hit.any(0)))
        at = int(np.argmax(hit[:, src]))
        t_ev = base[src] + c[at - 1, src] if at else base[src]
        s = ldexp(t_ev, -ks) + fx[at, src]
        fx = np.where(np.arange(LANES) * TERMS + np.arange(TERMS)[:, None] <= src * TERMS + at, 0.0, fx)


def classify(seg, s):
    """Each segment's grid 2^-grid, or NO_GRID (the prefix sums in the device's order)."""
    grid = [NO_GRID] * len(seg)
    with np.errstate(invalid="ignore", over="ignore"):
        v = seg[np.minimum(np.arange(WINDOW), len(seg) - 1)].reshape(LANES, TERMS).T
        at = s + np.concatenate([[0.0], wave_incl_sum(lane_sum(v))[:-1]])
        for j in range(TERMS):
            lo = bits(at * (1.0 - 2.0 ** -30)) >> np.uint64(52)
            at = at + v[j]
            hi = bits(at * (1.0 + 2.0 ** -30)) >> np.uint64(52)
            for L in range(LANES):
                i, e = L * TERMS + j, int(lo[L])
                if i < len(seg) and e == int(hi[L]) and 1023 - 900 <= e < 1023 + 52:
                    grid[i] = 1075 - e
    return grid


def run_of_counts(count, ties, T0):
    """T behind each member of a run of up to 64 counted segments."""
    c = np.zeros(LANES)
    c[:len(count)] = count
    t = list(ties) + [0] * (LANES - len(ties))
    H = ballot(v & 1 for v in t)
    if H:
        t_odd = ALL if int(bits(T0)) & 1 else 0
        low = H & -H
        before = odd_before(H, ballot(v & 4 for v in t)) ^ (t_odd & (low | low - 1))
        step = H & (before ^ ballot(v & 2 for v in t))
        c = c + np.where(lanes(step), np.where([bool(v & 8) for v in t], -1.0, 1.0), 0.0)
    return T0 + wave_incl_sum(c)


def device_sum(x, s0, seg=None, window=WINDOW, stats=None):
    """The row's sum as k_cdf_sums forms it.  seg: the segment sums that guide it (by default the
    terms', any order); stats: segments added as counts ("used"), counted in vain ("refused"),
    taken in rounds without a count ("rounds"), and the longest run."""
    x = np.asarray(x, np.float64)
    parts = [x[k:k + SEG] for k in range(0, len(x), SEG)]
    if seg is None:
        seg = np.array([p.sum() for p in parts])
    s, st = np.float64(s0), {"used": 0, "refused": 0, "rounds": 0, "run": 0}
    for w0 in range(0, len(parts), window):
        fx = [by_lane(p) for p in parts[w0:w0 + window]]
        m = len(fx)
        grid = classify(np.asarray(seg[w0:w0 + window], np.float64), s)
        counts = [grid_count(f, g) if g != NO_GRID else (0.0, 0) for f, g in zip(fx, grid)]
        i = 0
        if w0 == 0:                         # the row's first segment in order
            assert grid[0] == NO_GRID
            s, i = sequential(x[:SEG], s), 1
        while i < m:
            if math.isnan(s):
                break
            ks = NO_GRID - 1 if s < 2.0 ** -1022 or not s < 2.0 ** 52 else 1075 - int(bits(s) >> np.uint64(52))
            run = 0
            while run < LANES and i + run < m and grid[i + run] == ks:
                run += 1
            if run:
                T = run_of_counts([c for c, _ in counts[i:i + run]], [t for _, t in counts[i:i + run]], ldexp(s, ks))
                ok = T[:run] < 2.0 ** 53
                take = run if ok.all() else int(np.argmin(ok))
                if take:
                    s = ldexp(T[take - 1], -ks)
                st["used"] += take
                st["run"] = max(st["run"], take)
                i += take
                if take == LANES or i >= m:
                    continue
            st["refused" if grid[i] != NO_GRID else "rounds"] += 1
            s, _ = exact_segment(fx[i], s)
            i += 1
    if stats is not None:
        stats.update(st)
    return s


def rounds_sum(x, s0):
    """Every segment in rounds."""
    s = np.float64(s0)
    for k in range(0, len(x), SEG):
        s, _ = exact_segment(by_lane(np.asarray(x[k:k + SEG], np.float64)), s)
    return s


def check(x, s0=0.0):
    want = sequential(x, s0)
    # (the rounds add to +0: the device starts each row in order, which turns -0 into +0)
    assert same(rounds_sum(x, abs(s0)), want)
    # behind a start of its own, so that the terms meet counted segments and not only the start
    assert same(device_sum(x, s0), want)
    shifted = np.concatenate([np.zeros(SEG), x])
    assert same(device_sum(shifted, s0), want)


# ---- the pieces ----

def parity_walk(H, P, t):
    """T's parity before each of 64 members, and behind them, one by one."""
    before = 0
    for i in range(64):
        before |= t << i
        t = P >> i & 1 if H >> i & 1 else t ^ (P >> i & 1)
    return before, t


def random_masks(n):
    rng = np.random.default_rng(1)
    for _ in range(n):
        H, P = (int.from_bytes(rng.bytes(8), "little") for _ in range(2))
        for _ in range(int(rng.integers(0, 7))):       # sparser and sparser
            H &= int.from_bytes(rng.bytes(8), "little")
        yield H, P
    for k in range(64):
        yield 1 << k, ALL
        yield ALL ^ 1 << k, ALL
    yield from ((0, ALL), (ALL, ALL), (ALL, 0), (1 | 1 << 63, ALL))


def test_parity_masks_are_the_sequential_parity():
    for H, P in random_masks(5000):
        before, behind = parity_walk(H, P, 0)
        assert odd_before(H, P) == before, (H, P)
        assert odd_behind(H, P) == behind, (H, P)
        # from an odd T: flipped up to the first tie, the same behind it (as run_of_counts has it)
        low = H & -H
        assert odd_before(H, P) ^ (ALL if H == 0 else low | low - 1) == parity_walk(H, P, 1)[0], (H, P)


def tie_terms(rng, n, share):
    """Values in units of the grid: whole, halves (ties) and others."""
    q = rng.integers(0, 6, n).astype(np.float64)
    kind = rng.random(n)
    q += np.where(kind < share, 0.5, np.where(kind < share + 0.1, rng.random(n), 0.0))
    return q


def test_ties_of_a_wave_settled_from_masks():
    rng = np.random.default_rng(2)
    for k in range(300):
        q = by_lane(tie_terms(rng, SEG, [0.0, 0.01, 0.1, 0.5, 0.9][k % 5]))
        total, ties = grid_count(q, 0)
        for t0 in (2 ** 52, 2 ** 52 + 1):
            s = sequential(q.T.reshape(-1), float(t0))         # grid 1: u = 1
            got = run_of_counts([total], [ties], float(t0))[0]
            assert same(got, s), (k, t0)
        behind = int(bits(sequential(q.T.reshape(-1), 2.0 ** 52))) & 1
        assert ties >> 2 & 1 == behind


def test_runs_of_64_counted_segments():
    rng = np.random.default_rng(3)
    for k in range(12):
        segs = [by_lane(tie_terms(rng, SEG, rng.choice([0.0, 0.0, 0.002, 0.3]))) for _ in range(64)]
        counts = [grid_count(q, 0) for q in segs]
        for t0 in (2.0 ** 52, 2.0 ** 52 + 1):
            T = run_of_counts([c for c, _ in counts], [t for _, t in counts], t0)
            s = t0
            for i, q in enumerate(segs):
                s = sequential(q.T.reshape(-1), s)
                assert same(T[i], s), (k, t0, i)


def test_a_wrong_mask_is_caught(monkeypatch):
    # planted mistakes: odd_before without the reset behind a tie, and a first tie that takes
    # an even T for granted
    def no_reset(H, P):
        x = P << 1 & ALL
        for k in (1, 2, 4, 8, 16, 32):
            x ^= x << k & ALL
        return x

    monkeypatch.setitem(globals(), "odd_before", no_reset)
    with pytest.raises(AssertionError):
        test_ties_of_a_wave_settled_from_masks()
    monkeypatch.undo()
    real = run_of_counts
    monkeypatch.setitem(globals(), "run_of_counts", lambda c, t, T0: real(c, [v & ~3 for v in t], T0))
    with pytest.raises(AssertionError):
        test_runs_of_64_counted_segments()


# ---- whole sums ----

@pytest.mark.parametrize("seed", range(6))
def test_exp_rows(seed):
    rng = np.random.default_rng(seed)
    logits = rng.standard_normal(3000) * [0.1, 1, 3, 8, 30, 300][seed]
    e = np.exp(logits - logits.max())
    check(e)
    p = (e * (1.0 / sequential(e, 0.0))).astype(np.float32).astype(np.float64)
    check(p, -0.0)


def test_ties_round_to_even():
    # s = 1 (grid 2^-52): a term of exactly half a grid step ties; the result depends on the
    # parity of s's last bit, which alternates as odd steps are added
    half = 2.0 ** -53
    check([1.0, half, half, 2.0 ** -52, half, 3 * half, half, 2.0 ** -52 + half, half] * 20)
    # ties on a coarser grid and just below a binade top
    check([2.0 ** 10] + [2.0 ** -43, 2.0 ** -42 * 3] * 100 + [2.0 ** 11 - 2.0 ** 10 - 2.0 ** -42] + [2.0 ** -43] * 50)


def test_crossings_every_few_terms():
    check([2.0 ** k for k in range(-30, 20)] + [1.0] * 500 + [2.0 ** -60] * 100)


def test_subnormal_grid_and_zero_starts():
    tiny = 2.0 ** -1074
    check([0.0, 0.0, tiny, 3 * tiny, 2.0 ** -1030, 2.0 ** -1022, tiny, 1e-300, 0.0, 1.0])
    check([0.0, 0.0], -0.0)                                        # -0.0 + 0.0 = +0.0
    check([0.0], -0.0)
    check([tiny] * 300, -0.0)
    check([2.0 ** -1022 - tiny] + [tiny] * 600)                    # up into the normal numbers


def test_nan_propagates():
    x = [0.5, 0.25, float("nan"), 0.125]
    check(x)
    check([0.5] * 700 + x + [1.0] * 700)


@pytest.mark.parametrize("window", [1, 3, 64])
def test_window_size_does_not_matter(window):
    rng = np.random.default_rng(11)
    x = np.exp(rng.standard_normal(5100) * 4)
    assert same(device_sum(x, 0.0, window=window), sequential(x, 0.0))


@pytest.mark.parametrize("n", [1, 255, 256, 257, 511, 512, 513, 1024])
def test_a_sequential_head_then_segments(n):
    # the row's first segment is added in order; ties and crossings sit on both sides of its end
    rng = np.random.default_rng(n)
    half = 2.0 ** -53
    x = np.concatenate([np.exp(rng.standard_normal(240) * 3), [1.0] + [half, 2.0 ** -52] * 20,
                        np.exp(rng.standard_normal(2000))])[:n]
    for s0 in (0.0, -0.0):
        check(x, s0)
    check((x * (1.0 / sequential(x, 0.0))).astype(np.float32).astype(np.float64), -0.0)


def test_a_missed_tie_is_caught():
    # planted mistake: rounding ties up instead of to even changes these sums, so the
    # tie rule is what makes the method exact
    half = 2.0 ** -53
    x = [1.0] + [half, 2.0 ** -52] * 10

    def ties_up(x, s0):
        s = float(s0)
        for v in x:
            t = np.float64(s) + np.float64(v)
            # round-half-up on the grid of s
            u = 2.0 ** (math.frexp(s)[1] - 53) if s >= 2.0 ** -1022 else 2.0 ** -1074
            q = (v / u) if s else None
            if q is not None and q - math.floor(q) == 0.5:
                t = s + (math.floor(q) + 1) * u
            s = float(t)
        return s

    assert not same(ties_up(x, 0.0), sequential(x, 0.0))
    check(x)


# ---- segments counted apart, on a right and on a wrong guess ----

@pytest.mark.parametrize("spread,least", [(0.0, 55), (1.0, 55), (4.0, 55), (60.0, 1)])
def test_segments_counted_apart(spread, least):
    # (at spread 60 the largest term is nearly the whole sum, which then stays within 2^-30 of
    # 1, the edge of a binade: no count behind it)
    rng = np.random.default_rng(int(spread))
    logits = rng.standard_normal(20000) * spread
    e, st = np.exp(logits - logits.max()), {}
    s = device_sum(e, 0.0, stats=st)
    assert same(s, sequential(e, 0.0))
    # about one segment a doubling of the sum goes without a count, and a good guess is never refused
    assert st["used"] >= least and st["refused"] == 0 and st["used"] + st["rounds"] == 78, st
    p = (e * (1.0 / s)).astype(np.float32).astype(np.float64)
    assert same(device_sum(p, -0.0, stats=st), sequential(p, -0.0)) and st["used"] >= least, st
    half = np.tile([2.0 ** -53, 3 * 2.0 ** -53, 2.0 ** -52], 7000)     # ties beside a sum of 1.5
    t = np.concatenate([[1.5], half])
    assert same(device_sum(t, 0.0, stats=st), sequential(t, 0.0))
    assert st["used"] == len(t) // SEG and st["run"] == 64, st


def test_segments_with_a_wrong_guess_or_a_nan():
    rng = np.random.default_rng(3)
    x = np.exp(rng.standard_normal(8000) * 2)
    want = sequential(x, 0.0)
    right = np.array([x[k:k + SEG].sum() for k in range(0, 8000, SEG)])
    st = {}
    assert same(device_sum(x, 0.0, right, stats=st), want) and st["used"] >= 20 and st["refused"] == 0, st
    # a guess of another binade: counts are formed on a grid that is not s's, and refused; one of
    # no binade: none is formed
    for wrong, refused in ((right * 2, True), (right / 2, True), (right * 0, False), (right * np.nan, False),
                           (np.full(len(right), 7.0), True), (right[::-1].copy(), None), (right * 2.0 ** 60, False)):
        assert same(device_sum(x, 0.0, wrong, stats=st), want)
        if refused is not None:
            assert (st["refused"] > 0) == refused, (st, wrong[:3])
    # a guess that stays in the binade s leaves: the counts that take T to 2^53 are refused
    flat = np.concatenate([np.full(SEG, 1.0 / SEG), np.full(4 * SEG, 2.0 ** -9)])     # 1, then 0.5 a segment
    assert same(device_sum(flat, 0.0, np.array([1.2] + [0.0] * 4), stats=st), sequential(flat, 0.0))
    assert st["used"] > 0 and st["refused"] > 0, st
    x[1234] = np.nan
    assert math.isnan(device_sum(x, 0.0, right))
