"""Fits the price formulas of the tile kernels and of the W4A16 decode kernel to the timings of scan.py, and says how good
the plans are that they choose.

    python profiles/plan_prices/fit.py fp8_tile|w4_tile|w4sub_tile|w8_tile|w8g64_tile|w8g32_tile|w4_decode|w4_regs TIMINGS.csv[.gz] [...] [--fit]

Without --fit: the constants of the sources, read from them.  The formulas are those of `tile_plan_us` in
vllm_amd/csrc/tile_plan.h, `decode2_us` in vllm_amd/csrc/w4a16_decode2.hip and `regs_us` in vllm_amd/csrc/w4a16_regs.hip.
"""
from __future__ import annotations

import ctypes
import re
import sys
from pathlib import Path

import numpy as np

sys.path.insert(0, str(Path(__file__).resolve().parent.parent.parent))
from vllm_amd import _lib  # noqa: E402

CSRC = Path(__file__).resolve().parent.parent.parent / "vllm_amd" / "csrc"
CUS = 256


def numbers(text: str) -> list[float]:
    return [float(x) for x in re.findall(r"-?\d+\.?\d*(?:e-?\d+)?", text)]


def source_table(file: str, name: str) -> list[float]:
    """The numbers of `constexpr ... name = {...};` (or `name[] = {...}`)."""
    text = re.sub(r"//.*", "", (CSRC / file).read_text())
    body = re.search(re.escape(name) + r"(?:\[\])?\s*=\s*\{(.*?)\};", text, re.S).group(1)
    return numbers(body)


# ------------------------------------------------------------------------------------------------------- tile kernels

class Tiles:
    def __init__(self, kind):
        self.kind = kind
        fp8 = kind == "fp8_tile"
        file = "fp8_scaled_mm.hip" if fp8 else "w4a16_prefill.hip"
        prefix = kind.split("_")[0].upper()
        g64, prefix = prefix == "W8G64", "W8" if prefix == "W8G64" else prefix      # (the table of 8-bit codes, less one slot)
        rows = np.array(source_table(file, f"{prefix}_TILE_SHAPES")).reshape(-1, 10)
        if g64:
            rows[rows[:, 0] == 41, 4] = 1
        self.ids = rows[:, 0].astype(int)
        self.shape = rows[:, 1:5]                        # bm, bn, nw, slots
        self.p_shape = rows[:, 5:]                       # base, step, load, shared, out
        self.p_costs = np.array(source_table(file, f"{prefix}_TILE_COSTS"))
        self.few_rows = 512 if prefix in ("W4", "W8") else 0
        self.bytes = 0.5 if prefix.startswith(("W4", "LDS")) else 1.0

    def pack(self):
        return np.concatenate([self.p_shape.ravel(), self.p_costs])

    def unpack(self, p):
        self.p_shape, self.p_costs = p[:self.p_shape.size].reshape(self.p_shape.shape), p[self.p_shape.size:]

    def load(self, files):
        """Every file is a set of problems of its own (the formats were timed on the same ones)."""
        parts, problems = [], 0
        for file in files:
            d = np.loadtxt(file, delimiter=",", ndmin=2)
            d = d[np.isin(d[:, 3], self.ids)]
            order = np.lexsort((d[:, 6], d[:, 5], d[:, 4], d[:, 3], d[:, 2], d[:, 1], d[:, 0]))
            d = d[order]
            first = np.ones(len(d), bool)
            first[1:] = (d[1:, :6] != d[:-1, :6]).any(1)
            d = d[first]
            key = np.unique(d[:, :3], axis=0, return_inverse=True)[1].ravel() + problems
            problems = key.max() + 1
            parts.append((d, key))
        d, self.key = (np.concatenate(x) for x in zip(*parts))
        self.k, self.n, self.m, ident, self.sk, self.tail, self.us = d.T
        self.which = np.searchsorted(self.ids, ident, sorter=np.argsort(self.ids))
        self.which = np.argsort(self.ids)[self.which]

    def price(self, p_shape, p_costs):
        bm, bn, _, slots = self.shape[self.which].T
        base, step, load, shared, out = p_shape[self.which].T
        few = np.where((self.ids[self.which] == 48) & (self.m <= self.few_rows), 1.03, 1.0)      # (TILE256_FEW_ROWS_PRICE)
        base, step, load = base * few, step * few, load * few
        weight_mb, handover, part_cost, handover_mb, sum_mb = p_costs[:5]
        tiles = np.ceil(self.m / bm) * np.ceil(self.n / bn)
        steps = self.k // 64
        tail = self.tail > 0
        split = np.where(tail, tiles % CUS, tiles)
        cap = CUS * slots
        rounds = np.where(tail, tiles // CUS, tiles * self.sk // cap)
        rest = np.where(tail, split * self.sk, tiles * self.sk % cap) / CUS
        part = steps / self.sk
        whole = np.where(tail, steps, part)
        us = rounds * (base + whole * (step + load * slots + np.where(slots > 1, shared, 0)))
        us = us + (rest > 0) * (base + part * (step + load * rest + np.where(rest > 1, shared, 0)))
        mem = weight_mb * 1e-6 * self.bytes * self.k * self.n
        us = (us ** 4 + mem ** 4) ** 0.25 + 2.0 + out * 2e-6 * self.m * self.n
        us = us + (self.sk > 1) * (handover + self.sk * (part_cost + 4e-6 * bm * bn * (handover_mb * split + sum_mb)))
        return us

    def prices(self, p=None):
        if p is None:
            return self.price(self.p_shape, self.p_costs)
        return self.price(p[:self.p_shape.size].reshape(self.p_shape.shape), p[self.p_shape.size:])

    def allowed(self):
        """The plans that the planner weighs (its limits on the K split)."""
        steps = self.k // 64 if self.kind == "fp8_tile" else self.k // 128
        bm, bn, _, _ = self.shape[self.which].T
        tiles = np.ceil(self.m / bm) * np.ceil(self.n / bn)
        fp8 = self.kind == "fp8_tile"
        whole = (self.sk == 1) | ((steps // self.sk >= (8 if fp8 else 3)) & (tiles * self.sk * 10 <= CUS * (23 if fp8 else 24)))
        tail = steps // self.sk >= (16 if fp8 else 8)
        return np.where(self.tail > 0, tail, whole)


def report(price, us, key, allowed, groups):
    """How the cheapest plan compares with the fastest one, per group of problems."""
    n = key.max() + 1
    best = np.full(n, np.inf)
    np.minimum.at(best, key, us)
    masked = np.where(allowed, price, np.inf)
    cheapest = np.full(n, np.inf)
    np.minimum.at(cheapest, key, masked)
    took = np.full(n, np.nan)
    at = (masked == cheapest[key]) & np.isfinite(masked)
    took[key[at]] = us[at]
    loss = took / best
    print(f"{len(us)} plans of {n} problems; rms error of the price {np.sqrt(np.mean(np.log(price / us) ** 2)):.3f}")
    for name, mask in groups.items():
        rows = np.zeros(n, bool)
        rows[key[mask]] = True
        l = loss[rows & np.isfinite(loss)]
        if len(l):
            print(f"  {name:34s} {len(l):5d} problems, chosen / fastest: mean {np.exp(np.mean(np.log(l))):.3f}  "
                  f"90 % {np.quantile(l, .9):.3f}  99 % {np.quantile(l, .99):.3f}  worst {l.max():.2f}")
    return loss


def fit(prices, p0, us, key, accuracy, sharp=0.05):
    """Constants (positive ones of `p0` are moved) that make the cheapest plan a fast one: the mean of log(time / fastest time)
    over a problem's plans, weighted by exp(-log(price) / sharp), plus `accuracy` times the rms error of the price (each
    problem counts the same, plans of 1.7 times the fastest one and more a fifth)."""
    from scipy.optimize import minimize
    problems = key.max() + 1
    best = np.full(problems, np.inf)
    np.minimum.at(best, key, us)
    lost = np.log(us / best[key])
    weight = np.where(lost < np.log(1.7), 1.0, 0.2) / np.bincount(key)[key]
    weight /= weight.sum()
    at = np.flatnonzero(p0 > 0)
    start = np.log(p0[at])

    def full(q):
        p = p0.copy()
        p[at] = np.exp(q)
        return p

    def objective(q):
        log_price = np.log(prices(full(q)))
        cheapest = np.full(problems, np.inf)
        np.minimum.at(cheapest, key, log_price)
        w = np.exp((cheapest[key] - log_price) / sharp)
        chosen = np.bincount(key, w * lost) / np.bincount(key, w)
        error = log_price - np.log(us)
        return chosen.mean() + accuracy * np.sqrt((weight * error * error).sum()) + 1e-4 * ((q - start) ** 2).sum()
    r = minimize(objective, start, method="L-BFGS-B", bounds=[(x - 4, x + 2) for x in start], options=dict(maxiter=150, maxfun=50000))
    return full(r.x)


# ------------------------------------------------------------------------------------------------- W4A16 decode kernel

TABLES = ("W8", "SUB", "W8_MB2", "SUB_MB2", "MB34", "ROWS_W8", "ROWS_SUB", "ROWS")


def lds_bytes(wks, groups, mr, mb):
    act = (wks * groups * 256 * mr * mb + 1023) // 1024 * 1024 + np.where(wks == 1, 1024, 0)
    red = np.where(wks > 1, np.where(mb == 2, 16 - 16 // wks, 16) * mb * 1024, 0)
    sums = np.where(mb >= 2, wks * groups * mb * 64, 0)
    return np.where(mb > 2, np.maximum(act, red) + sums, act + red + sums)


def wg_slots(waves, lds):
    return np.maximum(1, np.minimum(16 // waves, 160 * 1024 // lds))


def pick_wn(nt, sk, wks, lds):
    best = np.ones_like(nt)
    best_rounds = np.full(nt.shape, np.inf)
    best_waves = np.full(nt.shape, np.inf)
    for wn in range(1, 17):
        ok = wn <= 16 // wks
        slots = wg_slots(np.where(ok, wks * wn, 1), lds)
        per_cu = np.ceil(np.ceil(nt / wn) * sk / CUS)
        rounds = np.ceil(per_cu / slots)
        waves = np.minimum(per_cu, slots) * wn * wks
        take = ok & ((rounds < best_rounds) | ((rounds == best_rounds) & (waves < best_waves)))
        best, best_rounds, best_waves = (np.where(take, a, b) for a, b in ((wn, best), (rounds, best_rounds), (waves, best_waves)))
    return best.astype(int)


def tile_prices(k, n, m, any_shape):
    """What the cheapest plan of the W4A16 tile kernel with weights through LDS is priced at, which the decode kernels are weighed
    against; `any_shape`: the 128 x 256 tiles are built for the format."""
    t = Tiles("lds_tile")
    best = np.full(len(k), np.inf)
    t.k, t.n, t.m = k, n, m
    for i, ident in enumerate(t.ids):
        t.which = np.full(len(k), i)
        bm, bn = t.shape[i][:2]
        tiles = np.ceil(m / bm) * np.ceil(n / bn)
        for sk, tail in [(s, 0) for s in range(1, 9)] + [(s, 1) for s in (2, 3, 4)]:
            t.sk, t.tail = np.full(len(k), sk), np.full(len(k), tail)
            ok = t.allowed() & ((ident != 13) | any_shape)
            if tail:
                ok &= (ident == 20) & (tiles > CUS) & (tiles % CUS > 0) & (tiles % CUS * sk <= CUS)
            best = np.minimum(best, np.where(ok, t.prices(), np.inf))
    return best


class Decode:
    """Plans of workgroups of all rows (kind 0) and of 16 rows (1) of the decode kernel, and what the tile kernel takes (2)."""

    def __init__(self):
        self.p = {t: np.array(source_table("w4a16_decode2.hip", f"D2_COST_{t}")) for t in TABLES}      # in the order of Decode2Cost

    def load(self, files):
        self.load_rows(np.concatenate([np.loadtxt(f, delimiter=",", ndmin=2) for f in files]))

    def load_rows(self, d):
        self.k, self.n, self.m, self.sub, self.w8, self.kind, self.gs, self.wks, self.wn = d[:, :9].T.astype(int)
        self.us = d[:, 9]
        tile = self.kind == 2
        self.gs, self.wks = np.maximum(self.gs, 1), np.maximum(self.wks, 1)
        self.tpg = np.where(self.w8 == 1, 2, 1)
        g = self.k // 128 * self.tpg
        rows = self.kind == 1
        self.sk = -(-g // (self.wks * self.gs))
        self.copies = np.where(rows, -(-self.m // 16), 1)
        self.mb = np.where(rows, 1, -(-self.m // 16))
        self.mr = np.where(rows, 16, np.where(self.m == 1, 1, np.where(self.m <= 4, 4, 16)))
        self.lds = lds_bytes(self.wks, np.maximum(self.gs // self.tpg, 1), self.mr, self.mb)
        auto = pick_wn(self.n // 16, self.sk, self.wks, self.lds)
        self.wn = np.where(self.wn == 0, auto, self.wn)
        self.key = np.unique(d[:, :5], axis=0, return_inverse=True)[1].ravel()
        plain = (self.sub == 1) & (self.w8 == 0)
        self.table = np.where(tile, -1, np.where(rows, np.where(self.w8 == 1, 5, np.where(plain, 7, 6)),
                                                 np.where(self.w8 == 1, np.where(self.m > 16, 2, 0),
                                                          np.where(plain, 4, np.where(self.m > 16, 3, 1)))))
        self.tile_us = np.full(len(self.us), np.nan)
        self.tile_us[tile] = tile_prices(*(a[tile].astype(float) for a in (self.k, self.n, self.m)), plain[tile]) * np.where((self.w8[tile] == 1) & (self.m[tile] <= 64), 1.06, 1.0)
        # workgroups of three and four m-blocks: by the rule, the price only weighs them against the other kinds
        self.by_rule = np.ones(len(self.us), bool)
        lib, plan = _lib.load(), (ctypes.c_double * 6)()
        for i in np.flatnonzero(self.table == 4):
            lib.vaq_w4a16_decode_plan(int(self.m[i]), int(self.n[i]), int(self.k[i]), 1, 0, 1, plan)
            self.by_rule[i] = (self.gs[i], self.wks[i], self.wn[i]) == tuple(int(x) for x in plan[:3])

    def price(self, t, at):
        base, round_, fill_kb, mem_mb, again, reduce_, handover, part, part_mb = t[:9]
        latency, work, sub_work, chain, last, pair, spread = t[9:12], t[12:15], t[15:18], t[18], t[19], t[20], t[21]
        k, n, m, gs, wks, wn, sk, mr, mb, copies, tpg = (a[at] for a in (self.k, self.n, self.m, self.gs, self.wks, self.wn, self.sk,
                                                                       self.mr, self.mb, self.copies, self.tpg))
        sub = self.sub[at]
        ri = np.where(mr == 1, 0, np.where(mr <= 8, 1, 2))
        slots = wg_slots(wks * wn, self.lds[at])
        per_cu = np.ceil(np.ceil(n // 16 / wn) * sk * copies / CUS)
        side, rounds = np.minimum(per_cu, slots), np.ceil(per_cu / slots)
        rounds = np.where(rounds > 1, per_cu / slots + last * (rounds - per_cu / slots), rounds)
        whole = (mr <= 4) & (gs <= np.where(sub > 1, 4, 8))
        flight = np.where(whole | (gs < 3), gs, 3)
        si = np.where(sub == 4, 2, sub - 1)
        tile = ((latency[ri] / flight) ** 4 + (side * wks * wn * work[ri] * sub_work[si]) ** 4) ** 0.25 + chain * sub_work[si]
        fill = fill_kb * side * (wks * gs // tpg) * (mr * mb * 0.25)
        slow = np.where((wks * wn == 2) & (per_cu > 4), pair, 1.0)
        core = slow * rounds * (round_ / slots + fill + gs * tile + reduce_ * np.log2(wks))
        mem = mem_mb * 0.5e-6 * k * n * tpg * (1 + again * (copies - 1))
        us = base + (core ** 3 + mem ** 3) ** (1 / 3)
        xcds = 8 // np.gcd(-(-(n // 16) // wn), 8)
        us = us + spread * (np.minimum(copies, xcds) - 1) / 7.0
        return us + (sk > 1) * (handover + sk * (part + part_mb * 4e-6 * m * n))

    def prices(self, p=None):
        out = self.tile_us.copy()
        for i, t in enumerate(TABLES):
            at = self.table == i
            if at.any():
                out[at] = self.price((p or self.p)[t], at)
        return out

    def allowed(self):
        four = (self.mb == 2) & (self.sub == 4) & (self.gs == 4) & (self.w8 == 0)
        split = (self.sk > 1) & ((self.k <= 2048) | (self.sk * (self.n // 16) * self.mb * 1024 > 16 << 20))
        return (self.kind == 2) | (self.by_rule & ~four & ~split & ~((self.kind == 1) & (self.wks * self.wn < 4)))


# --------------------------------------------------------------------- W4A16 kernel with activations in registers

class Regs:
    TABLES = ("W4_4ROWS", "W4", "W4_64", "W4_32", "W8", "W8_64", "W8_32")

    def __init__(self):
        self.p = np.array([source_table("w4a16_regs.hip", f"REGS_COST_{t}") for t in self.TABLES])      # in the order of RegsCost

    def load(self, files):
        self.load_rows(np.concatenate([np.loadtxt(f, delimiter=",", ndmin=2) for f in files]))

    def load_rows(self, d):
        """`other`: the time of what takes each problem without this kernel (nan: not timed)."""
        key = np.unique(d[:, :7], axis=0, return_inverse=True)[1].ravel()
        other = np.full(key.max() + 1, np.nan)
        other[key[d[:, 7] == 0]] = d[d[:, 7] == 0, 11]
        d, key = d[d[:, 7] > 0], key[d[:, 7] > 0]
        self.key = np.unique(key, return_inverse=True)[1].ravel()
        self.other = other[np.unique(key)]
        self.k, self.n, self.m, self.sub, self.w8, self.zp, self.fp16, self.nw, self.j, self.mb, self.sk = d[:, :11].T.astype(int)
        self.us = d[:, 11]
        at = np.where(self.sub == 1, 0, np.where(self.sub == 2, 1, 2))
        self.table = np.where(self.w8 == 1, 4 + at, np.where((at == 0) & (self.m <= 4), 0, 1 + at))

    def prices(self, p=None):
        (base, round_, latency, row, tile, tile_mb, kb, mem_mb, last, meet, meet_wave, out, handover, part, part_mb, again, alone, copies,
         k1024) = (self.p if p is None else p)[self.table].T
        k, n, m, sub, nw, j, mb, sk = self.k, self.n, self.m, self.sub, self.nw, self.j, self.mb, self.sk
        planes, mr, rb = 1 + self.w8, np.where((m <= 4) & (mb == 1), 4, 16), -(-m // (16 * mb))
        registers = 8 * j * planes + 4 * j * mb + 16 * mb + 4 * planes * mb + (4 + sub) * mb + np.where(sub == 4, 65, 45)
        lds = np.maximum(nw * (mb * mr * 256 + 2 * sub * 256), j * mb * nw * 1024)
        slots = np.maximum(1, np.minimum(np.clip(512 // registers, 1, 8) * 4 // nw, 160 * 1024 // lds))
        per_cu = -(-(-(-(n // 16) // j) * rb * sk) // CUS)
        side, waves = np.minimum(per_cu, slots), np.minimum(per_cu, slots) * nw / 4
        rounds = np.where(per_cu > slots, per_cu / slots + last * (-(-per_cu // slots) - per_cu / slots), 1.0)
        tiles = -(-(-(-(k // 128) // sk)) // nw)
        work = waves * (row * mb * np.where(sub == 4, 2, 1) + j * planes * (tile + tile_mb * mb))
        work = work * np.where(registers > 256, copies, 1.0) * np.where(waves <= 1, alone, 1.0)
        moved = kb * side * nw * (mb * mr / 4 + j * planes)
        each = (latency ** 3 + work ** 3 + moved ** 3) ** (1 / 3) * np.where(k % 1024 == 0, k1024, 1.0)
        core = rounds * (round_ + tiles * each + j * mb * (meet + meet_wave * side * nw))
        mem = mem_mb * 0.5e-6 * k * n * planes * (1 + again * (rb - 1))
        us = base + (core ** 3 + mem ** 3) ** (1 / 3) + out * 2e-6 * m * n
        return us + (sk > 1) * (handover + sk * (part + part_mb * 4e-6 * rb * 16 * mb * n))

    def allowed(self):
        units = -(-(self.n // 16) // self.j) * (-(-self.m // (16 * self.mb)))
        return (self.sk == 1) | ((self.k // 128 // self.sk >= self.nw) & (units < CUS) & (units * self.sk <= 2 * CUS))


def show(values, per):
    for i in range(0, len(values), per):
        print("    {" + ", ".join(f"{v:.3g}" for v in values[i:i + per]) + "},")


def main():
    kind, files, refit = sys.argv[1], [a for a in sys.argv[2:] if a != "--fit"], "--fit" in sys.argv
    t = Decode() if kind == "w4_decode" else Regs() if kind == "w4_regs" else Tiles(kind)
    t.load(files)
    size = t.k * t.n
    groups = {"ordinary (K 1024-14336, N <= 28672)": (t.k >= 1024) & (t.k <= 14336) & (t.n >= 1024) & (t.n <= 28672),
              "K > 14336": t.k > 14336, "N > 28672": t.n > 28672, "K < 1024 or N < 1024": (t.k < 1024) | (t.n < 1024),
              "K N < 2^22": size < 2 ** 22, "all": size > 0}
    if kind not in ("w4_decode", "w4_regs"):
        for a, b in ((9, 32), (33, 64), (65, 128), (129, 256), (257, 512), (513, 1024), (1025, 2048), (2049, 8192)):
            groups[f"{a} .. {b} rows"] = (t.m >= a) & (t.m <= b)
    else:
        for sub in (1, 2, 4):
            for w8 in (0, 1):
                for a, b in ((1, 4), (5, 16), (17, 32), (33, 64), (65, 256)):
                    groups[f"groups of {128 // sub}, {8 if w8 else 4} bits, {a} .. {b} rows"] = \
                        (t.sub == sub) & (t.w8 == w8) & (t.m >= a) & (t.m <= b)
    if refit and kind == "w4_decode":
        ok = t.allowed()
        # the kinds that a number of rows has the choice of, together (the tile kernel at its own price)
        for names, tile in ((("W8",), False), (("SUB",), False), (("W8_MB2", "ROWS_W8"), True), (("SUB_MB2", "ROWS_SUB"), True),
                            (("MB34", "ROWS"), True)):
            tables = [TABLES.index(x) for x in names]
            here = np.isin(t.table, tables) & ok
            if tile:
                here |= (t.kind == 2) & np.isin(t.key, t.key[here])
            at = np.flatnonzero(here)
            where = [np.flatnonzero(t.table[at] == i) for i in tables]

            def prices(p, at=at, where=where):
                out = t.tile_us[at]
                for j, w in enumerate(where):
                    out[w] = t.price(p[22 * j:22 * j + 22], at[w])
                return out
            p = fit(prices, np.concatenate([t.p[x] for x in names]), t.us[at], np.unique(t.key[at], return_inverse=True)[1], 0.15)
            for j, name in enumerate(names):
                t.p[name] = p[22 * j:22 * j + 22]
                print(name, ", ".join(f"{v:.3g}" for v in t.p[name]))
    elif refit and kind == "w4_regs":
        for i, name in enumerate(Regs.TABLES):
            at = (t.table == i) & t.allowed()

            def prices(p, at=at, i=i):
                full = t.p.copy()
                full[i] = p
                return t.prices(full)[at]
            t.p[i] = fit(prices, t.p[i], t.us[at], np.unique(t.key[at], return_inverse=True)[1], 0.5)
            print(name, ", ".join(f"{v:.3g}" for v in t.p[i]))
    elif refit:
        at = t.allowed()
        key = np.unique(t.key[at], return_inverse=True)[1]
        t.unpack(fit(lambda p: t.prices(p)[at], t.pack(), t.us[at], key, 0.15 if kind == "fp8_tile" else 0.3))
        show(t.p_shape.ravel(), 5)
        show(t.p_costs, len(t.p_costs))
    report(t.prices(), t.us, t.key, t.allowed(), groups)


if __name__ == "__main__":
    main()
