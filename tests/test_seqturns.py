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
@pytest.mark.parametrize("n_ids", [1, 5, 700, 2500])  # 2500: more than 8 a CU, 128 lanes for short rows
def test_gather_rms_row_kernel(bh, oracle, dev, ne0, n_ids):
    """One workgroup per row: rows of 2 blocks, a partial last block on rows
    that start on 4 bytes only, exactly one window of 64 blocks and a second
    one of 6, with code-3 blocks (two squares; by hand at a binade's end), zero and non-finite scales
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


def _landing_rows(n_rows, nblk, seed):
    """Scale bits and counts of codes other than 1 of rows whose second run
    ends exactly on the upper end of the sum's binade: its square is rounded
    up to m units of the sum, and m divides the units left in the binade."""
    rng = np.random.default_rng(seed)
    half = np.arange(0x7c00, dtype=np.uint16).view(np.float16).astype(np.float32)
    scales = np.zeros((n_rows, nblk), np.uint16)
    runs = np.zeros((n_rows, nblk), np.int64)
    scales[0, :3], runs[0, :3] = (0x3c45, 0x2d55, 0x2d55), (1, 124, 77)
    r = 1
    while r < n_rows:
        e = int(rng.integers(9, 18))
        h0, n0 = (e << 10) | int(rng.integers(1024)), int(rng.integers(1, 101))
        s = np.float32(0)
        for _ in range(n0):
            s = s + half[h0] * half[h0]
        unit = np.float64(np.spacing(s))
        gap = int((2.0 ** (np.floor(np.log2(np.float64(s))) + 1) - np.float64(s)) / unit)
        cand = np.arange((e - 6) << 10, (e + 1) << 10)
        xu = np.float64(half[cand] * half[cand]) / unit
        m = np.rint(xu).astype(np.int64)
        ok = (m == np.floor(xu) + 1) & (xu - np.floor(xu) != 0.5)
        ok &= (gap % np.maximum(m, 1) == 0) & (gap <= 128 * m)
        if not ok.any():
            continue
        i = int(rng.choice(np.flatnonzero(ok)))
        scales[r, :2], runs[r, :2] = (h0, cand[i]), (n0, gap // int(m[i]))
        scales[r, 2:] = ((e - rng.integers(0, 6, nblk - 2)) << 10) | rng.integers(0, 1024, nblk - 2)
        runs[r, 2:] = rng.integers(0, 129, nblk - 2)
        r += 1
    return scales, runs


@pytest.mark.gpu
@pytest.mark.parametrize("nblk", [4, 40])
def test_gather_rms_run_ends_on_binade(bh, oracle, dev, nblk):
    """Rows whose runs end exactly on a power of two, which their next runs
    have to leave in the next binade's units: bit for bit in a short batch (the
    sum by turns) and in a long one (the sum walked a lane per row)."""
    import torch
    rows, ne0 = 64, nblk * 128
    scales, runs = _landing_rows(rows, nblk, 11 + nblk)
    codes = np.ones((rows, nblk, 128), np.uint8)
    codes[np.arange(128) < runs[..., None]] = 2
    codes = codes.reshape(rows, nblk, 32, 4)
    table = np.empty((rows, nblk, 34), np.uint8)
    table[..., 0], table[..., 1] = scales & 0xff, scales >> 8
    table[..., 2:] = codes[..., 0] | codes[..., 1] << 2 | codes[..., 2] << 4 | codes[..., 3] << 6
    table = table.reshape(rows, nblk * 34)
    w = np.ones(ne0, np.float32)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    for n_ids in (rows, 16 * torch.cuda.get_device_properties(0).multi_processor_count):
        ids = (np.arange(n_ids) % rows).astype(np.uint32)
        _, n = bh.pq2_embed_gather(t(table), ne0, rows, t(ids), w=t(w), eps=1e-6)
        _, ref = oracle.embed_gather(table, ne0, rows, ids[:rows], w, 1e-6)
        got = n.cpu().numpy().reshape(-1, rows, ne0)
        assert np.array_equal(got.view(np.uint32), np.broadcast_to(ref.view(np.uint32), got.shape))


@pytest.mark.gpu
def test_gather_rms_code_3_rows_cost(bh, dev):
    """Rows of four codes cost about what rows of three do (their blocks are
    summed in closed form too, but for those that leave a binade): a table's
    codes must not decide the call's time.  Weight by weight they took 30
    times as long; six leaves room for the clock."""
    import torch
    g = torch.Generator(device=dev)
    g.manual_seed(3)
    rows, nblk = 64, 40
    w = torch.ones(nblk * 128, device=dev)
    ids = torch.arange(rows, device=dev, dtype=torch.int32)
    us = {}
    for top in (3, 4):
        table = torch.randint(0, top, (rows, nblk, 34, 4), device=dev, generator=g, dtype=torch.uint8)
        table = table[..., 0] | table[..., 1] << 2 | table[..., 2] << 4 | table[..., 3] << 6
        d = (torch.randn((rows, nblk), device=dev, generator=g) * 0.02).abs().to(torch.float16)
        table[..., :2] = d.view(torch.uint8).view(rows, nblk, 2)
        table = table.contiguous().view(-1)
        times = []
        for _ in range(5):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(50):
                bh.pq2_embed_gather(table, nblk * 128, rows, ids, w=w, eps=1e-6)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b) * 20)
        us[top] = min(times)
    print(us, flush=True)
    assert us[4] <= 6 * us[3]
