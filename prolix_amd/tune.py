"""Autotuner for the pair kernels' build-time settings.

The settings are the unroll depth of the Born, force and chain passes' loops
over an item's rows of patches, the XCD-aware item order, and a minimum
occupancy the three kernels' registers must fit (0: none for the Born and chain
passes, the force pass's own choice for it). They are
compile-time constants of ``csrc/prx_pair_dev.h`` (the pair passes' device
code, compiled into ``prx_pair.hip``'s kernels); the chosen ones live in
``csrc/prx_tuned.h``, which that header includes before its defaults.

Candidates come from coordinate descent around the current settings: each
setting in turn takes each of its other values while the rest stay put. Every
candidate is timed on the 256-system batched mix, in a process of its own,
as mean wall time per step of the captured step graph.

Three commands, because the GPU runs what was compiled beforehand:

    python -m prolix_amd.tune build           # compile one library per candidate (no GPU needed)
    python -m prolix_amd.tune run  RESULTS    # time every built candidate on the GPU, one JSON line each
    python -m prolix_amd.tune pick RESULTS    # write csrc/prx_tuned.h from the fastest candidate

``pick`` keeps the current settings unless a candidate is faster by more
than ``NOISE`` (same-process timings vary by a few tenths of a percent).
"""

from __future__ import annotations

import json
import os
import pickle
import re
import subprocess
import sys
import tempfile
import time
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
TUNED = CSRC / "prx_tuned.h"
TUNE_DIR = PKG / "lib" / "tune"

# Each setting's values, and its default in prx_pair_dev.h.
KNOBS = {
    "PRX_UNROLL_BORN": (1, 2),
    "PRX_UNROLL_FORCE": (1, 2),
    "PRX_UNROLL_CHAIN": (1, 2),
    "PRX_XCD_MAP": (0, 1),
    "PRX_MIN_WAVES": (0, 6),
}
DEFAULTS = {"PRX_UNROLL_BORN": 1, "PRX_UNROLL_FORCE": 1, "PRX_UNROLL_CHAIN": 1, "PRX_XCD_MAP": 1,
            "PRX_MIN_WAVES": 0}
NOISE = 0.005


def parse_tuned(text: str | None = None) -> dict:
    """The settings a prx_tuned.h defines."""
    if text is None:
        text = TUNED.read_text() if TUNED.exists() else ""
    return {m.group(1): int(m.group(2)) for m in re.finditer(r"^#define (PRX_\w+) (-?\d+)\s*$", text, re.M)}


def current() -> dict:
    s = dict(DEFAULTS)
    s.update({k: v for k, v in parse_tuned().items() if k in KNOBS})
    return s


def name_of(settings: dict) -> str:
    short = {"PRX_UNROLL_BORN": "ub", "PRX_UNROLL_FORCE": "uf", "PRX_UNROLL_CHAIN": "uc", "PRX_XCD_MAP": "x",
             "PRX_MIN_WAVES": "mw"}
    return "_".join(f"{short[k]}{settings[k]}" for k in KNOBS)


def plan(base: dict | None = None) -> list[dict]:
    """The current settings first, then every one-setting change of them."""
    base = dict(base or current())
    out = [base]
    for k, values in KNOBS.items():
        for v in values:
            if v != base[k]:
                c = dict(base)
                c[k] = v
                out.append(c)
    return out


def header(settings: dict, note: str = "") -> str:
    lines = ["// Generated by prolix_amd/tune.py -- pair-kernel settings measured fastest on",
             "// the 256-system batched mix (mean ms per captured step)."]
    lines += [f"// {l}" for l in note.splitlines() if l.strip()]
    lines.append("#pragma once")
    # guarded, so a -D on the compiler line (a tuning candidate) takes precedence
    for k, value in settings.items():
        lines += [f"#ifndef {k}", f"#define {k} {value}", "#endif"]
    return "\n".join(lines) + "\n"


def build(candidates: list[dict] | None = None) -> list[Path]:
    """Compile prx_pair.hip once per candidate and link it with the other
    objects of the current build (prolix_amd.build must have run)."""
    from prolix_amd import build as B

    objdir = B.PKG / "lib" / "obj"
    others = [objdir / (s + ".o") for s in B.SOURCES if s != "prx_pair.hip"]
    missing = [str(o) for o in others if not o.exists()]
    if missing:
        raise RuntimeError(f"build the engine first (python -m prolix_amd.build): missing {missing}")
    cc = B.hipcc()
    out = []
    for c in candidates or plan():
        d = TUNE_DIR / name_of(c)
        d.mkdir(parents=True, exist_ok=True)
        # every setting explicitly, so the candidate does not depend on prx_tuned.h
        defines = [f"-D{k}={v}" for k, v in c.items()]
        obj = d / "prx_pair.o"
        subprocess.run([cc, *B.HIP_FLAGS, *defines, f"-I{B.ROOT / 'include'}", f"-I{B.CSRC}", "-c",
                        str(B.CSRC / "prx_pair.hip"), "-o", str(obj)], check=True,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
        subprocess.run([cc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(d / "libprolix_gb.so"), str(obj),
                        *map(str, others)], check=True, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
        (d / "settings.json").write_text(json.dumps(c))
        out.append(d)
        print(f"built {d.name}", flush=True)
    return out


def _measure(lib: str, mix_file: str, steps: int) -> dict:
    """One candidate, in its own process (the library is loaded once per process)."""
    from prolix_amd import _native as N

    N.LIB_PATH = Path(lib)
    import torch

    from prolix_amd.engine import GBEngine, Langevin
    from prolix_amd.minimize import minimize

    with open(mix_file, "rb") as fh:
        systems, temps = pickle.load(fh)
    eng = GBEngine(systems)
    x = minimize(eng, [s["positions"] for s in systems], steps=200)
    eng.init(x, [Langevin(1.0, float(temps[k]), 1.0, seed=1000 + k, safety_caps=True) for k in range(len(systems))])
    eng.steps(50)
    torch.cuda.synchronize()
    t = time.perf_counter()
    eng.steps(steps)
    torch.cuda.synchronize()
    ms = (time.perf_counter() - t) / steps * 1e3
    passes = eng.profile_steps(20)
    eng.close()
    return {"ms_per_step": ms, "pass_ms": passes}


def run(results: str, steps: int = 300, n_systems: int = 256) -> None:
    """Time every built candidate; one JSON line per candidate in ``results``."""
    from prolix_amd import synth

    dirs = sorted(p for p in TUNE_DIR.iterdir() if (p / "libprolix_gb.so").exists()) if TUNE_DIR.exists() else []
    if not dirs:
        raise RuntimeError("no candidates: run `python -m prolix_amd.tune build` first")
    # the mix is generated here, before any process touches the GPU
    prots, temps = synth.batch_mix(n_systems, 300, 5000, seed=2)
    with tempfile.TemporaryDirectory() as tmp:
        mix_file = os.path.join(tmp, "mix.pkl")
        with open(mix_file, "wb") as fh:
            pickle.dump(([p.system_dict() for p in prots], list(temps)), fh)
        with open(results, "w") as out:
            for d in dirs:
                settings = json.loads((d / "settings.json").read_text())
                print(f"[tune] {d.name}", flush=True)
                r = subprocess.run([sys.executable, "-m", "prolix_amd.tune", "_measure", str(d / "libprolix_gb.so"),
                                    mix_file, str(steps)], capture_output=True, text=True, timeout=600)
                if r.returncode != 0:
                    raise RuntimeError(f"candidate {d.name} failed:\n{r.stdout[-2000:]}\n{r.stderr[-2000:]}")
                line = json.loads(r.stdout.strip().splitlines()[-1])
                line.update({"name": d.name, "settings": settings})
                out.write(json.dumps(line) + "\n")
                out.flush()
                print(f"[tune] {d.name}: {line['ms_per_step']:.4f} ms/step", flush=True)


def pick(results: str, write: bool = True) -> tuple[dict, str]:
    """The fastest candidate's settings (the current ones unless beaten by more
    than NOISE) and a markdown table of the results; writes prx_tuned.h."""
    rows = [json.loads(l) for l in Path(results).read_text().splitlines() if l.strip()]
    if not rows:
        raise ValueError(f"{results}: no results")
    base = current()
    base_rows = [r for r in rows if r["settings"] == base]
    best = min(rows, key=lambda r: r["ms_per_step"])
    chosen = base
    if not base_rows or best["ms_per_step"] < base_rows[0]["ms_per_step"] * (1.0 - NOISE):
        chosen = best["settings"]
    table = ["| candidate | ms/step | Born | force | chain (ms, in-graph) |", "|---|---:|---:|---:|---:|"]
    for r in sorted(rows, key=lambda r: r["ms_per_step"]):
        p = r.get("pass_ms", {})
        mark = " (chosen)" if r["settings"] == chosen else ""
        table.append(f"| `{r['name']}`{mark} | {r['ms_per_step']:.4f} | {p.get('born_pairs', float('nan')):.4f} | "
                     f"{p.get('force_pairs', float('nan')):.4f} | {p.get('chain_pairs', float('nan')):.4f} |")
    note = "\n".join(f"{r['name']}: {r['ms_per_step']:.4f}" for r in sorted(rows, key=lambda r: r["ms_per_step"]))
    if write:
        TUNED.write_text(header(chosen, note))
    return chosen, "\n".join(table)


def main(argv: list[str]) -> int:
    if not argv or argv[0] not in ("build", "run", "pick", "_measure"):
        print(__doc__)
        return 2
    cmd = argv[0]
    if cmd == "build":
        build()
    elif cmd == "run":
        run(argv[1] if len(argv) > 1 else "tune_results.jsonl")
    elif cmd == "pick":
        chosen, table = pick(argv[1] if len(argv) > 1 else "tune_results.jsonl")
        print(table)
        print(f"chosen: {name_of(chosen)} -> {TUNED}")
    else:
        print(json.dumps(_measure(argv[1], argv[2], int(argv[3]))), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main(sys.argv[1:]))
