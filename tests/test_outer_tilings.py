"""The outer update of a batch in 128-tiles against its members alone in
64-tiles: that these sizes take the two forms (host code, on the CPU), and that
they give the same bits (on the GPU)."""

import json
import shutil
import subprocess
from pathlib import Path

import pytest

from tests.helpers import make_prior, small_problem

ROOT = Path(__file__).resolve().parent.parent
# odd and even numbers of block rows (25 and 26)
BATCHES = {mode: [1600 + 50 * (k % 2) - k for k in range(count)]
           for mode, count in [("fp64", 8), ("fp32", 8), ("bf16", 7)]}


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_batches_take_128_tiles_and_their_members_64(tmp_path):
    exe = tmp_path / "check"
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", str(ROOT / "probit_amd/csrc"),
                    str(ROOT / "tests/native/outer_schedule_check.cpp"), "-o", str(exe)],
                   check=True)
    table = json.loads((ROOT / "probit_amd/tune_table.json").read_text())
    for op, mode in enumerate(("fp64", "fp32", "bf16")):
        G = table["gfx950"][mode][1]["superstep"]
        nbs = sorted(((N + 63) // 64 for N in BATCHES[mode]), reverse=True)

        def wide(members):
            r = subprocess.run([str(exe), str(op), str(G), *map(str, members)], check=True,
                               capture_output=True, text=True, timeout=60)
            return [int(v) for v in r.stdout.split()]

        assert sum(wide(nbs)) >= 1, mode
        assert all(sum(wide([nb])) == 0 for nb in set(nbs)), mode


@pytest.mark.gpu
@pytest.mark.parametrize("mode", list(BATCHES))
def test_batch_and_members_agree(mode):
    import torch

    import probit_amd as P
    from probit_amd.serving import ServingEngine
    probs = [small_problem(200 + k, N, 2, "probit", "EQ", noise=0.5)
             for k, N in enumerate(BATCHES[mode])]
    eng = ServingEngine(precision=mode, capacity=8)
    for tag, (X, y, theta, lp, _) in enumerate(probs):
        assert eng.submit(tag, X, y, "EQ", theta[0], theta[1], "probit", lp[0], lp[1])
    out = {}
    while eng.in_flight:
        for c in eng.step():
            out[c.tag] = c
    eng.close()
    for tag, (X, y, theta, lp, _) in enumerate(probs):
        gp = P.LaplaceGP(data=(X, y), prior=make_prior("EQ"), precision_mode=mode,
                         log_likelihood=P.log_probit_likelihood)
        w, p = gp.approximate_posterior((theta, lp))
        assert torch.equal(w, out[tag].weight) and torch.equal(p, out[tag].precision), tag
