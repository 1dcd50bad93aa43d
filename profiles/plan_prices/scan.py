"""Times every plan of random problems, for the price formulas that choose among them (fit.py).

    python profiles/plan_prices/scan.py fp8_tile|w4_tile|w8_tile|w4g64z_tile|w4g32_tile|w4g32z_tile|w4g32zh_tile|w8g64_tile|w8g32_tile|w8g32h_tile|w4_decode|w4_regs SECONDS SEED OUT.csv

Runs on the GPU; the *.csv.gz beside it are what it wrote on an MI355X, but for the rows of kernels that changed or came after a file was written: those are what it wrote then, scaled to
the file as said below by a step that is not kept here, so that their ratios to a problem's other rows count and not their us.  A problem is a layer (K, N) and a number of rows; a plan is forced through the `_tuned` entry points
(vllm_amd/csrc/vaq_tuning.h).  Weights are cold: a graph of launches walks over copies of the layer (640 MB of them, at most
400).  One line per plan, with the time of a launch in us:

    fp8_tile, w4_tile (4-bit codes in groups of 128 rows with zero points), w8_tile (8-bit codes), and both in groups of 64 / 32 rows,
    z with zero points, h fp16 instead of bf16:  k, n, m, tile id, parts of K, 1 if only the tiles of the last round are in parts, us
                        (tile id 48, the 256 x 256 tiles of w4a16_tile256_kernel.h, was timed later, on the files' problems of more than 128 rows: its times are
                        scaled by what the fastest plan of the problem took then and takes in the file; the same with the tile ids 42 (not in groups of 32), 43, 44 and
                        46 of 8-bit codes, whose activation reads changed: twice to four times each where within 1.35 of the fastest plan, geometric mean, the others by the
                        mean ratio of their id)
    w4_decode:          k, n, m, groups of 128 rows (1, 2, 4), 8-bit codes, kind, gs, wks, wn (0: by the planner), us
                        kind 0 workgroups of all rows, 1 of 16 rows, 2 the tile kernel by the plan of the shapes with weights
                        through LDS (gs, wks, wn 0), at whose price the decode kernels are weighed
    w4_regs:            k, n, m, groups of 128 rows, 8-bit codes, zero points, fp16, wavefronts, n-tiles, m-blocks, parts of K, us: the kernel
                        with activations in registers (8-bit codes timed again after their planes became one operand, scaled by what the problem takes without this
                        kernel then and in the file); wavefronts 0: what takes the problem without it.  (The file's last
                        problems, vocabulary layers and ordinary K and N, have the library's plan alone.)
"""
from __future__ import annotations

import ctypes
import random
import sys
import time
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent.parent))
from vllm_amd import _lib  # noqa: E402

CUS = 256
POOL, MOST_COPIES = 640_000_000, 400


class Layer:
    """Operands of one layer: views of one pool of random bytes (finite e4m3 codes) and of one of scales."""
    pool = scales = None

    def __init__(self, fp8: bool, k: int, n: int, most_m: int, bits: int = 4, group: int = 128, zeros: bool | None = None,
                 dtype: torch.dtype = torch.bfloat16):
        if Layer.pool is None:
            p = torch.randint(0, 256, (1_500_000_000,), dtype=torch.uint8, device="cuda")
            Layer.pool = torch.where((p & 0x7f) == 0x7f, p ^ 1, p)
            Layer.scales = (torch.rand(150_000_000, device="cuda") * 1e-2 + 1e-3).to(torch.bfloat16)
        self.fp8, self.k, self.n, self.bits, self.group = fp8, k, n, bits, group
        self.zeros = bits == 4 and group == 128 if zeros is None else zeros      # uint4 with zero points, else uint4b8
        self.bytes = k * n if fp8 else k * n * bits // 8
        self.copies = max(2, min(MOST_COPIES, POOL // self.bytes))
        self.tag = _lib.VAQ_F16 if dtype == torch.float16 else _lib.VAQ_BF16
        x = torch.randn(most_m, k, device="cuda", dtype=dtype)
        self.a = x.to(torch.float8_e4m3fn) if fp8 else x
        self.sa, self.sb = torch.rand(most_m, device="cuda"), torch.rand(n, device="cuda")
        self.out = torch.empty(most_m, n, device="cuda", dtype=dtype)
        self.counters = torch.zeros(1 << 20, dtype=torch.int32, device="cuda")
        self.tmp = torch.empty(1 << 20, device="cuda")

    def fits(self) -> bool:
        return self.copies * self.bytes <= self.pool.numel()

    def launch(self, lib, m, i, tune, path):
        c, stream = i % self.copies, torch.cuda.current_stream().cuda_stream
        w = self.pool.data_ptr() + c * self.bytes // 256 * 256
        tmp, tmp_bytes = self.tmp.data_ptr(), self.tmp.numel() * 4
        if self.fp8:
            return lib.vaq_fp8_scaled_mm_ws_tuned(
                self.a.data_ptr(), self.k, w, self.k, self.sa.data_ptr(), m, self.sb.data_ptr(), self.n, None, self.out.data_ptr(), self.n,
                _lib.VAQ_BF16, m, self.n, self.k, tmp, tmp_bytes, self.counters.data_ptr(), self.counters.numel(), stream, tune)
        scale_count = self.n * (self.k // self.group)
        at = c * scale_count % max(1, self.scales.numel() - scale_count) // 64 * 64
        wtype = _lib.VAQ_WTYPE_U8B128 if self.bits == 8 else _lib.VAQ_WTYPE_U4 if self.zeros else _lib.VAQ_WTYPE_U4B8
        z = self.pool.data_ptr() + self.pool.numel() - (c + 1) * (scale_count // 2) // 64 * 64 - scale_count if self.zeros else None
        return lib.vaq_w4a16_gemm_tuned(
            self.a.data_ptr(), self.k, w, self.scales.data_ptr() + 2 * at, z, None, None, self.out.data_ptr(), tmp, tmp_bytes, None,
            self.counters.data_ptr(), self.counters.numel(), m, self.n, self.k, self.group, self.tag, wtype, path, stream, tune)

    def scratch(self, lib, m, tune) -> bool:
        t, a, n = ctypes.c_size_t(), ctypes.c_size_t(), ctypes.c_size_t()
        if self.fp8:
            rc = lib.vaq_fp8_scaled_mm_workspace_tuned(m, self.n, self.k, ctypes.byref(t), ctypes.byref(n), tune)
        else:
            rc = lib.vaq_w4a16_gemm_workspace_tuned(m, self.n, self.k, 0, 0, ctypes.byref(t), ctypes.byref(a), ctypes.byref(n), tune)
        if rc or n.value > self.counters.numel() or t.value > 4 << 30:
            return False
        if t.value > self.tmp.numel() * 4:
            self.tmp = torch.empty(t.value // 4, device="cuda")
        return True

    def time(self, lib, m, path=0, **fields):
        """us per launch, None where the library refuses the plan."""
        tuning = _lib.VaqTuning()
        for name, value in fields.items():
            if name == "exp":
                for i, v in value.items():
                    tuning.exp[i] = v
            else:
                setattr(tuning, name, value)
        tune = ctypes.byref(tuning)
        if not self.scratch(lib, m, tune) or self.launch(lib, m, 0, tune, path):
            return None
        marks = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
        marks[0].record()
        for i in range(2):
            self.launch(lib, m, i, tune, path)
        marks[1].record()
        marks[1].synchronize()
        guess = marks[0].elapsed_time(marks[1]) * 500
        count = max(2, min(self.copies, int(4000 / guess)))
        graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            graph.capture_begin()
            for i in range(count):
                self.launch(lib, m, i, tune, path)
            graph.capture_end()
        torch.cuda.current_stream().wait_stream(side)
        best = 1e9
        for i in range(3 if guess < 2000 else 2):
            marks[0].record()
            graph.replay()
            marks[1].record()
            marks[1].synchronize()
            if i:
                best = min(best, marks[0].elapsed_time(marks[1]) * 1e3 / count)
        return best


def log(rng, low, high, step):
    return max(step, round(low * (high / low) ** rng.random() / step) * step)


def shape(rng, step_n, most):
    """Half of the problems of an ordinary model's sizes, half of a much wider range (vocabularies, very long or short K)."""
    while True:
        if rng.random() < 0.5:
            k, n = log(rng, 1024, 14336, 128), log(rng, 1024, 28672, step_n)
        else:
            k, n = log(rng, 256, 28672, 128), log(rng, 256, 152064, step_n)
        if k * n <= most:
            return k, n


TILES = {"fp8_tile": {13: (128, 128), 14: (64, 128), 15: (64, 64), 16: (128, 64), 17: (128, 256), 19: (256, 128), 1: (256, 256), 10: (256, 384)},
         "w4_tile": {12: (128, 128), 14: (64, 128), 15: (128, 64), 16: (256, 128), 13: (128, 256), 20: (256, 256),
                     41: (32, 128), 51: (32, 64), 42: (64, 128), 52: (64, 64), 43: (96, 128), 44: (128, 128), 46: (128, 256), 66: (128, 256),
                     48: (256, 256)},
         "w8_tile": {12: (128, 128), 14: (64, 128), 15: (128, 64), 16: (256, 128), 20: (256, 256), 41: (32, 128), 51: (32, 64), 42: (64, 128),
                     52: (64, 64), 43: (96, 128), 44: (128, 128), 46: (128, 256), 48: (256, 256)}}
FORMATS_OF = {"w4_tile": (4, 128, True), "w8_tile": (8, 128, False),      # bits, rows of a group, zero points, activations
              "w4g32zh_tile": (4, 32, True, torch.float16), "w8g32h_tile": (8, 32, False, torch.float16)}
TILES["w4g32zh_tile"] = TILES["w8g32h_tile"] = TILES["w8_tile"]
for _bits in (4, 8):
    for _group in (64, 32):
        for _zeros in ("", "z") if _bits == 4 else ("",):
            FORMATS_OF[f"w{_bits}g{_group}{_zeros}_tile"] = (_bits, _group, _zeros == "z")
            TILES[f"w{_bits}g{_group}{_zeros}_tile"] = TILES["w8_tile"]


def tile_plans(kind, k, n, m):
    steps = k // 64 if kind == "fp8_tile" else k // 128
    for ident, (bm, bn) in TILES[kind].items():
        if ident == 10 and n % 384:
            continue
        tiles = -(-m // bm) * -(-n // bn)
        rest = tiles % CUS
        # (shapes that leave most of every tile empty, or of the device, are never the fastest)
        if bm > 64 and bm >= 2 * m:
            continue
        for sk in range(1, 9):
            if sk == 1 or (steps // sk >= (6 if kind == "fp8_tile" else 3) and tiles * sk <= CUS * 3):
                yield ident, sk, 0
        if ident in (1, 20, 48) and tiles > CUS and rest:
            for sk in (2, 3, 4):
                if rest * sk <= CUS and steps // sk >= (12 if kind == "fp8_tile" else 6):
                    yield ident, sk, 1


def scan_tiles(lib, kind, rng, until, out):
    fp8 = kind == "fp8_tile"
    while time.time() < until:
        k, n = shape(rng, 64, 700_000_000 if fp8 else 1_300_000_000)
        rows = [m for m in (log(rng, 9 if fp8 else 17, 8192, 1) for _ in range(3)) if 2.0 * m * n * k < 2e12 and m * n < 6e8]
        if not rows:
            continue
        layer = Layer(fp8, k, n, max(rows), *(() if fp8 else FORMATS_OF[kind]))
        if not layer.fits():
            continue
        for m in rows:
            for ident, sk, tail in tile_plans(kind, k, n, m):
                exp = {6: sk} if tail else {10: 1}
                split = 0 if tail else sk
                us = layer.time(lib, m, fp8_path=2, fp8_tile_cfg=ident, fp8_split=split, exp=exp) if fp8 else \
                    layer.time(lib, m, path=2, prefill_tile=ident + 1, prefill_split=split, exp=exp)
                if us is not None:
                    print(k, n, m, ident, sk, tail, f"{us:.2f}", sep=",", file=out)
        print(kind, k, n, rows, flush=True)
        out.flush()


FORMATS = [(128, 4), (128, 4), (64, 4), (32, 4), (128, 8), (64, 8), (32, 8)]


def decode_plans(k, n, m, group, bits):
    """(rows over workgroups, gs, wks, wn) that the planner may choose from."""
    sub, per = 128 // group, bits // 4
    g, nt = k // 128 * per, n // 16
    if group == 128 and bits == 4 and m <= 32:
        return      # (by rule, not by price)
    for rows in (0, 1):
        if rows and not 16 < m <= 256 or not rows and m > (64 if group == 128 and bits == 4 else 32):
            continue
        mb, mr = (1, 16) if rows else (-(-m // 16), 1 if m == 1 else 4 if m <= 4 else 16)
        most = 512 // (mr * mb) * per
        for gs in (1, 2, 4, 7, 8, 14, 16):
            if (sub > 1 and gs & (gs - 1)) or (bits == 8 and gs % 2):
                continue
            for wks in (1, 2, 4, 8, 16):
                sk = -(-g // (wks * gs))
                if wks * gs > most or (wks > 1 and gs > 2 and wks * gs >= 2 * g) or sk > (1 if rows else 8):
                    continue
                yield rows, gs, wks, nt


def scan_decode(lib, rng, until, out):
    while time.time() < until:
        k, n = shape(rng, 64, 700_000_000)
        group, bits = rng.choice(FORMATS)
        rows = [log(rng, 1, 16, 1), log(rng, 17, 64, 1), log(rng, 17, 256, 1)]
        layer = Layer(False, k, n, max(rows), bits, group)
        if not layer.fits():
            continue
        for m in rows:
            us = None
            if m > 16:      # (the plan whose price the decode kernels are weighed against, not the strips that may take its place)
                plan = (ctypes.c_double * 4)()
                lib.vaq_w4a16_tile_plan(m, n, k, 128 // group, int(bits == 8), 1, plan)
                ident, sk, tail = int(plan[0]), int(plan[1]), plan[2] > 0
                us = layer.time(lib, m, path=2, prefill_tile=ident + 1, prefill_split=0 if tail else sk, exp={6: sk} if tail else {10: 1})
            if us is not None:
                print(k, n, m, 128 // group, int(bits == 8), 2, 0, 0, 0, f"{us:.2f}", sep=",", file=out)
            for split, gs, wks, nt in decode_plans(k, n, m, group, bits):
                wns = [w for w in range(1, 17) if 4 <= w * wks <= 16] if split else [0]
                for wn in rng.sample(wns, min(4, len(wns))):
                    fields = dict(decode_impl=1, decode2_gs=gs, decode2_wks=wks, decode2_wn=wn)
                    us = layer.time(lib, m, path=0 if split else 1, exp={2: 2 if split else 1}, **fields)
                    if us is not None:
                        print(k, n, m, 128 // group, int(bits == 8), split, gs, wks, wn, f"{us:.2f}", sep=",", file=out)
        print("w4_decode", k, n, group, bits, rows, flush=True)
        out.flush()


def regs_plans(rng, k, n, m, sub, w8):
    """Up to 24 launch shapes and K splits of a problem: those that fill the device most evenly, and some others."""
    plans = []
    for mb, nw, j in ((mb, nw, j) for mb in (1, 2, 3) for nw in (4, 8) for j in range(1, 9)):
        if (mb > 1 and m <= 16 * (mb - 1)) or not ((j <= 4 and not (w8 and sub == 4 and mb * j == 12)) if nw == 8 else 3 <= j <= (6 if w8 else 8)):
            continue
        rb = -(-m // (16 * mb))
        for sk in range(1, 9):
            units = -(-n // 16 // j) * rb * sk
            if sk > 1 and (k // 128 // sk < nw or units > 690 or sk * n * rb * mb * 64 > 16 << 20 or n // 16 * rb * mb > max(4096, n // 4)):
                continue
            rounds = units / CUS
            idle = -(-units // CUS) / rounds if rounds < 3 else 1
            read = k // sk * 32 * mb + j * 16 * k // sk * (1 if w8 else 0.5)
            plans.append((idle * (1 + 0.15 * rng.random()) * (read * rounds) ** 0.5, nw, j, mb, sk))
    plans.sort()
    return [p[1:] for p in plans[:16] + rng.sample(plans[16:], min(8, max(0, len(plans) - 16)))]


def scan_regs(lib, rng, until, out):
    while time.time() < until:
        k, n = shape(rng, 64, 400_000_000)
        group, bits = rng.choice(FORMATS + [(128, 4)])
        zeros, dtype = bits == 4 and rng.random() < 0.5, torch.float16 if rng.random() < 0.33 else torch.bfloat16
        rows = sorted({log(rng, 1, 200, 1) for _ in range(3)})
        layer = Layer(False, k, n, max(rows), bits, group, zeros, dtype)
        if not layer.fits():
            continue
        for m in rows:
            head = (k, n, m, 128 // group, int(bits == 8), int(zeros), int(dtype == torch.float16))
            us = layer.time(lib, m, exp={8: 1})
            if us is not None:
                print(*head, 0, 0, 0, 0, f"{us:.2f}", sep=",", file=out)
            for nw, j, mb, sk in regs_plans(rng, k, n, m, 128 // group, int(bits == 8)):
                us = layer.time(lib, m, exp={8: j | mb << 4 | nw << 8 | sk << 12})
                if us is not None:
                    print(*head, nw, j, mb, sk, f"{us:.2f}", sep=",", file=out)
        print("w4_regs", k, n, rows, flush=True)
        out.flush()


if __name__ == "__main__":
    what, seconds, seed, path = sys.argv[1], float(sys.argv[2]), int(sys.argv[3]), sys.argv[4]
    library, numbers, end = _lib.load(), random.Random(seed), time.time() + float(sys.argv[2])
    with open(path, "w") as f:
        if what in ("w4_decode", "w4_regs"):
            (scan_decode if what == "w4_decode" else scan_regs)(library, numbers, end, f)
        else:
            scan_tiles(library, what, numbers, end, f)
