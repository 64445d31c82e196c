"""Empty sizes are reported, not fatal: every workspace query answers them, and the calls refuse them."""
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

QUERY = """
import itertools, sys
from holodeck_amd import _lib
name, nargs = sys.argv[1], int(sys.argv[2])
for args in itertools.product((0, 1, 5), repeat=nargs):
    _lib.size(name, *args)
for args in itertools.product((-1, 0, 3), repeat=nargs):
    _lib.size(name, *args)
"""


def _queries():
    from holodeck_amd import _lib
    return [(n, len(args)) for n, (_, args) in _lib.SIGNATURES.items()
            if n.endswith("_workspace_size") and not n.startswith("hd_mlp")]     # (that one takes a network)


@pytest.mark.parametrize("name,nargs", _queries())
def test_workspace_queries_answer_empty_sizes(name, nargs):
    """In a process of its own: an integer division by zero ends the process."""
    run = subprocess.run([sys.executable, "-c", QUERY, name, str(nargs)], cwd=ROOT, capture_output=True, text=True)
    assert run.returncode == 0, (run.returncode, run.stderr[-500:])


@pytest.mark.gpu
@pytest.mark.parametrize("B,F,R", [(0, 3, 5), (100, 0, 4), (100, 3, 0)])
@pytest.mark.parametrize("given", [True, False])
def test_empty_realizations_are_refused(gpu, B, F, R, given):
    import torch
    from holodeck_amd import _lib, engine
    new = lambda *s: torch.ones(s, dtype=torch.float64, device="cuda")
    order = torch.arange(B, device="cuda")
    print(f"[empty realize B={B} F={F} R={R} given={given}]", flush=True)
    with pytest.raises(_lib.HoloHipError):
        engine.realize(new(B, F), new(B, F), R, 2, _lib.HD_SEL_SORTED, order=order,
                       counts=new(B, F, R) if given else None)
