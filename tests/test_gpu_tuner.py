"""What the launch-form cache says is what runs: where it holds a faster
register form the batch takes it, else the blocked RRQR, and a tuning run takes
the path of the later runs that read its file."""
import json
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SCRIPT = r"""
import json, sys
sys.path.insert(0, {root!r})
import numpy as np
import spaqr_public_amd as sq
from spaqr_public_amd import gen
A, _ = sq.colscale(gen.config_matrix("advdiff3d_16"))
t = sq.Tree(sq.default_levels(A.shape[1]), 0, sq.FP64)
t.set_scale(1)
t.set_tol(1e-2)
t.set_square(1)
t.set_tensor_coordinates(16, 3)
t.kernel_timing(True)
t.partition(A)
t.assemble(A)
t.factorize()
b = np.random.default_rng(0).standard_normal(A.shape[0])
print(json.dumps(dict(families=sorted(f for f in t.kernel_stats() if f.startswith(("qp3r", "rrqrp"))),
                      ranks=t.sparsified()[:, 4].tolist(), x=t.solve(b).tolist())))
"""


def run(path, tune):
    env = dict(os.environ, SPAQR_TUNE=str(tune), SPAQR_TUNE_FILE=str(path))
    r = subprocess.run([sys.executable, "-c", SCRIPT.format(root=ROOT)], env=env, capture_output=True, text=True,
                       timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    return json.loads(r.stdout.strip().splitlines()[-1])


def test_recorded_choice_runs(gpu_lib, tmp_path):
    path = tmp_path / "tune.json"
    tuning = run(path, 1)
    rec = json.load(open(path))
    assert rec["entries"] and all(e["blocked"] > 0 for e in rec["entries"])
    again = run(path, 0)
    assert again == tuning  # families, ranks and bits of x

    def with_entries(change):
        out = json.loads(json.dumps(rec))
        for e in out["entries"]:
            change(e)
        # one entry per line, as the library writes them
        path.write_text('{"arch": "gfx950", "entries": [\n' + ",\n".join(json.dumps(e) for e in out["entries"]) + "\n]}\n")
        return run(path, 0)

    def register(e):
        e["choice"], e["blocked"] = 48, 1e6

    def blocked(e):
        e["blocked"] = 0.0

    assert with_entries(register)["families"] == ["qp3r256_48"]
    got = with_entries(blocked)["families"]
    assert got and all(f.startswith("rrqrp") for f in got)
    assert with_entries(lambda e: e.pop("blocked"))["families"] == got  # an older file
