"""The launch choice for layers nobody has tuned, measured: the config that ``config.untuned_config``
picks beside the bucket's default, and its modelled time beside the measured one, on random layers.

Usage (needs the GPU)::

    python bench_probes/launch_choice.py time SEED SECONDS > launch_choice.log
    python bench_probes/launch_choice.py tiles N K GROUP M [M ...] >> launch_choice.log
    python bench_probes/launch_choice.py summary launch_choice.log   # profiles/untuned_launch_choice.md

``time`` draws layers (N 256 .. 32768 in steps of 8, K 256 .. 16384 in steps of 128, groups of 32, 64 and
128) and eight M from 1 to 8000 each, until SECONDS have passed. ``tiles`` times every tile and K split of
the model's candidates on one layer, one JSON line each: the data a refit of the model needs. Times are
the median of 7 replays, in turn, of HIP graphs that launch once per copy of the layer, the copies
together 640 MB (at most 40), so weights come from HBM.
"""

from __future__ import annotations

import json
import math
import os
import random
import statistics
import sys
import tempfile
import time
from dataclasses import replace
from pathlib import Path

ROOT = Path(__file__).resolve().parents[1]
SUMMARY = ROOT / "profiles" / "untuned_launch_choice.md"
RANGES = ((1, 1), (2, 4), (5, 8), (9, 16), (17, 128), (129, 1024), (1025, 4096), (4097, 8000))


def _setup():  # type: ignore[no-untyped-def]
    sys.path.insert(0, str(ROOT))
    os.environ["TOKENFORGE_CACHE_DIR"] = tempfile.mkdtemp()
    import torch

    from tokenforge.kernels import autotune, config
    from tokenforge.kernels.hip.w4a16 import w4a16_gemm

    dev = torch.device("cuda")

    def layers(n: int, k: int, group: int) -> list:
        copies = max(3, min(40, (640 << 20) // (n * k // 2)))
        first = autotune.synthetic_layer(n, k, group, dev)
        return [first] + [tuple(t.clone() for t in first) for _ in range(copies - 1)]

    def times(cfgs: list, m: int, k: int, group: int, copies: list) -> list[float]:
        x = torch.randn((m, k), device=dev).to(torch.float16)
        graphs = []
        for cfg in cfgs:
            w4a16_gemm(x, *copies[0], group, cfg)
            torch.cuda.synchronize()
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph, stream=torch.cuda.Stream()):
                for layer in copies:
                    w4a16_gemm(x, *layer, group, cfg)
            graph.replay()
            graphs.append(graph)
        us: list[list[float]] = [[] for _ in cfgs]
        for r in range(7):
            for i in range(len(graphs)):
                j = (i + r) % len(graphs)
                start, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
                start.record()
                graphs[j].replay()
                end.record()
                end.synchronize()
                us[j].append(start.elapsed_time(end) * 1e3 / len(copies))
        return [round(statistics.median(t), 2) for t in us]

    return config, layers, times


def _name(cfg) -> str:  # type: ignore[no-untyped-def]
    return f"{cfg.kernel} {cfg.block_m}x{cfg.block_n} k{cfg.block_k} w{cfg.num_warps} s{cfg.num_stages} split {cfg.split_k}"


def _cost(config, cfg, group: int):  # type: ignore[no-untyped-def]
    return dict((c.variant(), cost) for c, cost in config._model_tiles(group, True)).get(cfg.variant())


def time_random(seed: int, seconds: float) -> None:
    config, layers, times = _setup()
    rng = random.Random(seed)
    end = time.time() + seconds
    while time.time() < end:
        n = int(math.exp(rng.uniform(math.log(256), math.log(32768)))) // 8 * 8
        n = n // 16 * 16 if rng.random() < 0.75 else n
        k = max(256, int(math.exp(rng.uniform(math.log(256), math.log(16384)))) // 128 * 128)
        group = rng.choice((128, 128, 64, 32))
        copies = layers(n, k, group)
        for m in sorted({min(int(math.exp(rng.uniform(0, math.log(8000)))), (140 << 30) // (n * k)) for _ in range(8)}):
            bucket = min(config.m_bucket(min(m, config.MAX_BUCKET_M)), config.MAX_BUCKET_M)
            default, chosen = config.default_config(bucket, n, k, group), config.untuned_config(m, n, k, group)
            default, chosen = (  # the operators' guard above the largest bucket
                replace(c, split_k=1) if m > config.MAX_BUCKET_M and
                -(-m // c.block_m) * -(-n // c.block_n) >= config.NUM_CUS else c for c in (default, chosen))
            us = times([default, chosen] if default != chosen else [chosen], m, k, group, copies)
            cost = _cost(config, chosen, group)
            print(json.dumps({"m": m, "n": n, "k": k, "group": group, "default": [us[0], _name(default)],
                              "chosen": [us[-1], _name(chosen)],
                              "modelled": round(config._model_us(chosen, cost, m, n, k), 2) if cost else None}),
                  flush=True)


def time_tiles(n: int, k: int, group: int, ms: list[int]) -> None:
    config, layers, times = _setup()
    copies = layers(n, k, group)
    for m in ms:
        for cfg, cost in config._model_tiles(group, config.ksplit_applies(n, k)):
            for split in (1, 2, 3, 4, 6, 8):
                if split > 1 and split * 2 > k // 128:
                    break
                c = replace(cfg, split_k=split)
                us = times([c], m, k, group, copies)[0]
                print(json.dumps({"m": m, "n": n, "k": k, "group": group, "tile": [us, _name(c)],
                                  "modelled": round(config._model_us(c, cost, m, n, k), 2)}), flush=True)


def summary(log: str) -> None:
    rows = [json.loads(ln) for ln in Path(log).read_text().splitlines() if ln.startswith("{")]
    rows = [r for r in rows if "chosen" in r]
    out = [
        "# The launch choice for untuned layers: the chosen config beside the bucket's default",
        "",
        "Commands (on the MI355X box):",
        "",
        "```",
        "R=<repo root>",
        "python $R/bench_probes/launch_choice.py time SEED SECONDS > launch_choice.log",
        "python $R/bench_probes/launch_choice.py summary launch_choice.log",
        "```",
        "",
        f"{len(rows)} calls on {len({(r['n'], r['k'], r['group']) for r in rows})} random layers, cold weights,",
        "plain epilogue. Ratios are chosen / default, the mean geometric. Modelled / measured: where the",
        "time model made the choice (evaluated at the call's own M), mean and standard deviation of its log.",
        "",
        "| M | calls | mean ratio | slower by over 3% | largest ratio | modelled / measured |",
        "|---|---:|---:|---:|---:|---:|",
    ]
    for lo, hi in RANGES:
        part = [r for r in rows if lo <= r["m"] <= hi]
        if not part:
            continue
        ratio = [r["chosen"][0] / r["default"][0] for r in part]
        logs = [math.log(r["modelled"] / r["chosen"][0]) for r in part if r["modelled"]]
        model = (f"{math.exp(statistics.fmean(logs)):.2f} (± {statistics.pstdev(logs):.2f})" if logs else "—")
        out.append(f"| {lo if lo == hi else f'{lo}..{hi}'} | {len(part)} | {math.exp(statistics.fmean(map(math.log, ratio))):.3f} "
                   f"| {sum(q > 1.03 for q in ratio)} | {max(ratio):.3f} | {model} |")
    worst = sorted(rows, key=lambda r: r["default"][0] / r["chosen"][0])[:12]
    out += ["", "The calls that lose most:", "", "| layer | group | M | default us | chosen us |", "|---|---:|---:|---|---|"]
    out += [f"| {r['n']} x {r['k']} | {r['group']} | {r['m']} | {r['default'][0]} ({r['default'][1]}) | "
            f"{r['chosen'][0]} ({r['chosen'][1]}) |" for r in worst]
    SUMMARY.write_text("\n".join(out) + "\n")
    print(f"wrote {SUMMARY}")


def main(argv: list[str]) -> None:
    if argv[:1] == ["time"] and len(argv) == 3:
        time_random(int(argv[1]), float(argv[2]))
    elif argv[:1] == ["tiles"] and len(argv) >= 5:
        n, k, group, *ms = map(int, argv[1:])
        time_tiles(n, k, group, ms)
    elif argv[:1] == ["summary"] and len(argv) == 2:
        summary(argv[1])
    else:
        raise SystemExit(__doc__)


if __name__ == "__main__":
    main(sys.argv[1:])
