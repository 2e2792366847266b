"""CPU checks of the plan of PQ2_0 products of many tokens (csrc/pq2_mx_plan.hpp):
the scratch that a call reserves holds its own plan's need and every smaller
batch's on the same matrix (a stream capture must not allocate, and is prepared
by one call at the largest batch)."""
import shutil
import subprocess
from pathlib import Path

import pytest

import pq2data

SRC = Path(__file__).resolve().parent / "cpp" / "test_pq2_plan.cpp"


@pytest.fixture(scope="module")
def plan_exe(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not found")
    exe = tmp_path_factory.mktemp("plan") / "test_pq2_plan"
    subprocess.run([gxx, "-O2", "-Wall", "-std=c++17", str(SRC), "-o", str(exe)], check=True)
    return exe


def test_scratch_grows_with_tokens(plan_exe):
    res = subprocess.run([str(plan_exe)], capture_output=True, text=True, timeout=120)
    print(res.stdout)
    assert res.returncode == 0 and "0 failures" in res.stdout, res.stdout


@pytest.mark.parametrize("shape,plan", pq2data.MX_CASES)
def test_products_reach_their_form(plan_exe, shape, plan):
    """The shapes of the block-scaled products' GPU tests are cut as their list
    says: a change of the plan's constants can't move one to another kernel
    unnoticed."""
    res = subprocess.run([str(plan_exe), *map(str, shape)], capture_output=True, text=True, check=True)
    assert tuple(map(int, res.stdout.split())) == plan


_CAPTURE_SCRIPT = r'''
import sys
import torch
sys.path.insert(0, sys.argv[1])
from conftest import load_bonsai
bh = load_bonsai()
dev = torch.device("cuda:0")
ne0, n_rows = 5120, 17408
tab = torch.randint(0, 256, (n_rows, ne0 // 128, 34), device=dev, dtype=torch.uint8)
tab[..., 0], tab[..., 1] = 0x11, 0x22  # one finite scale
tab = tab.view(-1)
xs = {t: torch.randn((t, ne0), device=dev) for t in (65, 33, 17, 5)}
s = torch.cuda.Stream(device=dev)
torch.cuda.synchronize()
bh.pq2_matmul_n(tab, ne0, n_rows, xs[65], stream=s)  # the largest batch, once, eagerly
torch.cuda.synchronize()
for t in (33, 17, 5):
    y = torch.empty((t, n_rows), device=dev)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g, stream=s):
        bh.pq2_matmul_n(tab, ne0, n_rows, xs[t], out=y, stream=s)
    want = bh.pq2_matmul_n(tab, ne0, n_rows, xs[t])
    torch.cuda.synchronize()
    for rep in range(3):
        y.fill_(float("nan"))
        xs[t].mul_(1.0)  # eager work between replays
        torch.cuda.synchronize()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want), (t, rep)
# a matrix never called before, which would reserve more than there is now and
# needs less: the capture takes what is there
n_rows = 20000
tab = tab[:34].repeat(n_rows * ne0 // 128)
x, y, s = torch.randn((100, ne0), device=dev), torch.empty((100, n_rows), device=dev), torch.cuda.Stream(device=dev)
torch.cuda.synchronize()
g = torch.cuda.CUDAGraph()
with torch.cuda.graph(g, stream=s):
    bh.pq2_matmul_n(tab, ne0, n_rows, x, out=y, stream=s)
g.replay()
torch.cuda.synchronize()
assert torch.equal(y, bh.pq2_matmul_n(tab, ne0, n_rows, x))
print("capture ok")
'''


@pytest.mark.gpu
def test_smaller_batch_captured_after_largest(dev):
    """One eager call at 65 tokens prepares the capture of 33, 17 and 5 tokens
    on the same matrix, whose plans have more parts than its own.  Runs in a
    fresh process so no earlier call has grown the scratch."""
    import sys
    here = Path(__file__).resolve().parent
    res = subprocess.run([sys.executable, "-c", _CAPTURE_SCRIPT, str(here)], capture_output=True,
                         text=True, timeout=100)
    print(res.stdout[-2000:], res.stderr[-2000:])
    assert res.returncode == 0 and "capture ok" in res.stdout
