"""CPU check of the sequential sum of squares of a whole row by turns over
lanes (csrc/seqsum.hpp), which the fused gather + RMSNorm uses to reproduce
the reference's loop (src/kernels.rs:65-68) bit for bit: random scales, ties,
sums that stop moving, whole-number sums, and rows of 1 to 150 blocks in
windows of 64, 40 and 7 lanes (tests/cpp/test_seqturns.cpp)."""
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

SRC = Path(__file__).resolve().parent / "cpp" / "test_seqturns.cpp"


@pytest.mark.parametrize("rcp_ulp", [0, -1, 1])
def test_row_by_turns_matches_sequential_loop(tmp_path, rcp_ulp):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not found")
    exe = tmp_path / "test_seqturns"
    subprocess.run([gxx, "-O2", "-std=c++17", "-ffp-contract=off", f"-DRCP_ULP={rcp_ulp}",
                    str(SRC), "-o", str(exe)], check=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    print(res.stdout)
    assert res.returncode == 0, res.stdout
    assert " 0 mismatches" in res.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("ne0", [256, 1272, 5120, 64 * 128, 70 * 128])
@pytest.mark.parametrize("n_ids", [1, 5, 700])
def test_gather_rms_row_kernel(bh, oracle, dev, ne0, n_ids):
    """One workgroup per row: rows of 2 blocks, a partial last block on rows
    that start on 4 bytes only, exactly one window of 64 blocks and a second
    one of 6, with code-3 blocks (added by hand), zero and non-finite scales
    among the runs; both outputs bit for bit where the row is finite."""
    import torch
    rng = np.random.default_rng(ne0 + n_ids)
    rows, nblk = 60, -(-ne0 // 128)
    codes = rng.choice(4, size=(rows, nblk, 32, 4), p=[0.3, 0.4, 0.29, 0.01]).astype(np.uint8)
    codes[::2][codes[::2] == 3] = 2  # every other row has closed-form blocks only
    scales = rng.integers(0x0400, 0x5000, size=(rows, nblk)).astype(np.uint16)
    scales[rng.random((rows, nblk)) < 0.05] = 0
    scales[7, 0], scales[9, nblk - 1] = 0x7c00, 0x7e01
    table = np.empty((rows, nblk, 34), np.uint8)
    table[..., 0], table[..., 1] = scales & 0xff, scales >> 8
    table[..., 2:] = codes[..., 0] | codes[..., 1] << 2 | codes[..., 2] << 4 | codes[..., 3] << 6
    table = table.reshape(rows, nblk * 34)
    ids = rng.integers(0, rows, size=n_ids).astype(np.uint32)
    w = rng.standard_normal(ne0).astype(np.float32)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    e, n = bh.pq2_embed_gather(t(table), ne0, rows, t(ids), w=t(w), eps=1e-6)
    ref_e, ref_n = oracle.embed_gather(table, ne0, rows, ids, w, 1e-6)
    finite = np.all((scales[ids] & 0x7c00) != 0x7c00, axis=1)
    ge, gn = e.cpu().numpy(), n.cpu().numpy()
    assert np.array_equal(ge.view(np.uint32), ref_e.view(np.uint32))
    assert np.array_equal(gn[finite].view(np.uint32), ref_n[finite].view(np.uint32))
    assert np.array_equal(np.isnan(gn), np.isnan(ref_n))
