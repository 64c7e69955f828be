"""Small selects on a workspace that holds the number of the launch to come: brackets that are not the state's,
marks of workgroups that have not finished, counters of any size.  The count of launches starts with the process,
so a process of its own knows the numbers ahead; whatever the memory held, the outputs are the same."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

_PROGRAM = r"""
import torch
from oracle import select as SEL
from sga_amd import _lib as L
from sga_amd.fused_step import FusedSparseStep
from sga_amd.selection import read_result
from tests.util import student_t
dev, count = torch.device("cuda"), 0


def held(ws, how):
    # words of 64 bits, and their halves: (a bracket's end, the number), (the number, an end), the number alone
    number = (2 * count + 1) * 0x9E3779B1 & 0xFFFFFFFF
    pair = {"low end": (0x3F000000, number), "high end": (0x7F000000, number), "zero": (0, number),
            "marks": (number, 0x3F000000), "all": (number, number)}[how]
    words = torch.tensor([x - (x >> 31 << 32) for x in pair], dtype=torch.int32, device=ws.device)
    n = ws.numel() // 8
    ws[:n * 8].view(torch.int32).view(n, 2).copy_(words.expand(n, 2))


redone = 0
for n in (5, 4097, 300_001, 1_300_001, 4_100_000, 5_000_001):
    ws = torch.empty(int(L.raw("sga_select_workspace_bytes", n)), dtype=torch.uint8, device=dev)
    mask, res = torch.empty(n, dtype=torch.uint8, device=dev), torch.empty(8, dtype=torch.int32, device=dev)
    for how in ("low end", "high end", "zero", "marks", "all"):
        sc = student_t(n, count).abs()
        k = max(1, n // 100)
        want, thresh = SEL.select_topk_flat(sc, k)
        sd = sc.to(dev)
        held(ws, how)
        print(n, how, flush=True)
        L.call("sga_select_topk", L.ptr(sd), n, k, L.TIE_LOWEST_INDEX, L.ptr(mask), L.ptr(res), L.ptr(ws), ws.numel(),
               L.stream())
        count += 1
        r = read_result(res)
        assert (r.n_selected, r.thresh) == (k, thresh) and torch.equal(mask.cpu().bool(), want), (n, how)
        redone += n >= 1 << 20 and r.path == 0
assert redone > 0, "no memory made the finish go over the data again"
segs = [dict(start=0, n=200_000, lr=1e-4, b1=0.9, b2=0.95, eps=1e-8, wd=0.1),
        dict(start=200_000, n=100_001, lr=2e-4, b1=0.8, b2=0.99, eps=1e-6, wd=0.0)]
n = 300_001
for score in ("abs_g", "update"):
    ends = []
    for how in (None, "low end", "zero", "marks", "all"):
        fs = FusedSparseStep(n, segs, dev, values_dtype=torch.float32, want_mask=True)
        gen = torch.Generator().manual_seed(1)
        state = [torch.zeros(n, device=dev), (torch.randn(n, generator=gen) * 0.02).to(dev),
                 (torch.randn(n, generator=gen) * 1e-4).to(dev), torch.full((n,), 1e-8, device=dev)]
        fs.ws.zero_() if how is None else held(fs.ws, how)
        print(score, how, flush=True)
        idx, val = fs.step(student_t(n, 5).to(dev), *state, 1, ratio_percent=1.0, score=score)
        count += 1
        ends.append([idx.clone(), val.clone(), fs.mask.clone(), *state])
    assert all(torch.equal(a, b) for e in ends[1:] for a, b in zip(ends[0], e)), score
print("done")
"""


def test_memory_that_holds_the_launch_number(dev):
    r = subprocess.run([sys.executable, "-c", _PROGRAM], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and r.stdout.endswith("done\n"), (r.returncode, r.stdout[-500:], r.stderr[-2000:])
