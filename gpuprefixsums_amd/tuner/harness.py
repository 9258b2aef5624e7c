"""Exhaustive autotuning harness: times every candidate configuration of each
workload on the GPU. Its output is both the cost model's training data and
the judge of the model's regret; for a workload the model does not cover it
is the fallback.

    python -m gpuprefixsums_amd.tuner.harness --out times.jsonl [--sweep c5|stall|extra] [--start 0 --count 512]
                                              [--configs name,name,...]

One JSON line per workload: {"wid", "n", "dtype", "segments", "times_ms": {config: ms}}.
Each time is the median of a few brackets of events on the launch stream, each
around enough back-to-back runs to last BRACKET_MS (fewer for long runs).
"""
from __future__ import annotations

import argparse
import json
import statistics
import sys
import time
from pathlib import Path
from typing import Dict

from .space import (Config, Workload, c5_workloads, candidates, default_config, extra_workloads, stall_workloads,
                    with_default)


# A single run between two events reads up to 2 us too long or too short, more
# than most configurations differ at a few microseconds.
BRACKET_MS = 0.2
MAX_RUNS = 32


class Runner:
    """Device buffers for the largest workload and one handle per configuration."""

    def __init__(self, max_n: int = 1 << 30, max_segments: int = 1 << 14):
        import torch

        import gpuprefixsums_amd as gps
        self.torch, self.gps = torch, gps
        self.max_n = max_n
        dev = "cuda"
        self.u32 = torch.empty(max_n, dtype=torch.int32, device=dev)
        gps.fill_random_u32(self.u32, max_n, seed=6, bits=32)
        g = torch.Generator(device=dev)
        g.manual_seed(6)
        self.f32 = torch.randn(max_n, dtype=torch.float32, device=dev, generator=g)
        self.bf16 = self.f32.to(torch.bfloat16).view(torch.int16)
        self.out = torch.empty(max_n, dtype=torch.int32, device=dev)
        self.off = torch.empty(max_segments + 1, dtype=torch.int64, device=dev)
        self.handles: Dict[tuple, object] = {}
        torch.cuda.synchronize()

    def handle(self, c: Config, stall_period: int = 0):
        gps = self.gps
        key = (c, c.plain, stall_period)
        h = self.handles.get(key)
        if h is None:
            algo, kw = c.handle_args()
            if stall_period:
                kw["stall_period"] = stall_period
            h = gps.ScanHandle(algo, self.max_n, **kw)
            self.handles[key] = h
        return h

    def stage(self, w: Workload) -> None:
        import numpy as np
        self.off[: w.segments + 1].copy_(self.torch.from_numpy(w.offsets.view(np.int64)))

    def run(self, w: Workload, c: Config) -> None:
        h = self.handle(c, w.stall_period)
        if w.dtype == "u32":
            if c.kind == "batched":
                h.segmented(self.u32, self.out, self.off, w.segments, w.n, False)
            else:
                h.segmented_per_segment(self.u32, self.out, w.offsets, False)
        else:
            src = self.f32 if w.dtype == "f32" else self.bf16
            if c.kind == "batched_fp":
                h.segmented_fp(src, self.out, self.off, w.segments, w.n, bf16=w.dtype == "bf16", compensated=True)
            else:
                h.fp_per_segment(src, self.out, w.offsets, bf16=w.dtype == "bf16", compensated=True)

    def time(self, w: Workload, c: Config, best_so_far: float = float("inf")) -> float:
        torch = self.torch
        st = torch.cuda.current_stream()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)

        def bracket(runs: int) -> float:
            e0.record(st)
            for _ in range(runs):
                self.run(w, c)
            e1.record(st)
            e1.synchronize()
            return e0.elapsed_time(e1) / runs

        self.run(w, c)  # warm-up
        runs = min(max(int(BRACKET_MS / max(bracket(1), 1e-3)), 1), MAX_RUNS)
        reps, out = 5, []
        for r in range(reps):
            ms = bracket(runs)
            out.append(ms)
            # long or clearly losing configurations need fewer repetitions;
            # "clearly losing" is judged on the fastest run so far, so one
            # transiently slow run cannot end the timing of a fast one
            if ms > 20.0 or (r >= 1 and min(out) > 4.0 * best_so_far):
                break
        return statistics.median(out)

    def time_all(self, w: Workload, only=None, passes: int = 2) -> Dict[str, float]:
        """Times every candidate of w (or only those named in `only`), the one
        that stands for the default as a default handle: the lower of `passes`
        medians, each pass over all candidates in turn, so a transient slowdown
        of the device during one configuration's timing (seen once to make a
        20.8 us configuration read 36.9 us) is not taken for its speed."""
        self.stage(w)
        res: Dict[str, float] = {}
        best = float("inf")
        cands = with_default(candidates(w.dtype, w.stall_period),
                             default_config(w.dtype, w.segments, w.n, w.stall_period))
        for _ in range(passes):
            for c in cands:
                if only is not None and c.name not in only:
                    continue
                t = self.time(w, c, best)
                best = min(best, t)
                res[c.name] = min(res.get(c.name, float("inf")), t)
        for h in self.handles.values():
            if h.device_error():
                raise RuntimeError(f"device error on workload {w.wid}")
        return res


def main(argv=None) -> int:
    ap = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    ap.add_argument("--out", required=True)
    ap.add_argument("--sweep", choices=("c5", "stall", "extra"), default="c5")
    ap.add_argument("--start", type=int, default=0)
    ap.add_argument("--count", type=int, default=1 << 20, help="time at most this many workloads")
    ap.add_argument("--seed", type=int, default=None)
    ap.add_argument("--configs", default=None, help="comma list: time only these configurations")
    args = ap.parse_args(argv)
    if args.sweep == "c5":
        ws = c5_workloads(6 if args.seed is None else args.seed)
    elif args.sweep == "extra":
        ws = extra_workloads(8 if args.seed is None else args.seed)
    else:
        ws = stall_workloads(7 if args.seed is None else args.seed)
    ws = ws[args.start:args.start + args.count]
    only = set(args.configs.split(",")) if args.configs else None
    if only is not None:
        ws = [w for w in ws if any(c.name in only for c in candidates(w.dtype, w.stall_period))]
    runner = Runner(max_n=max(w.n for w in ws) if ws else 1 << 10)
    path = Path(args.out)
    path.parent.mkdir(parents=True, exist_ok=True)
    t0 = time.time()
    with path.open("a") as f:
        for w in ws:
            res = runner.time_all(w, only)
            f.write(json.dumps({"wid": w.wid, "n": w.n, "dtype": w.dtype, "segments": w.segments,
                                "stall_period": w.stall_period, "times_ms": res}) + "\n")
            f.flush()
            print(f"[harness] workload {w.wid} n={w.n} {w.dtype} S={w.segments} best "
                  f"{min(res, key=res.get)} {min(res.values()):.4f} ms ({time.time() - t0:.0f} s)",
                  file=sys.stderr, flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
