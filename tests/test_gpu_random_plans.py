"""Seeded random plans against the oracle, for every task form and both widths.

Each seed draws a matrix shape (ragged row counts, tail SWs), a degree mix (empty rows, short rows,
rows long enough to split an SW into several tasks, rows touching one row group or several), value
magnitudes and X statistics, and checks Y against the oracle's double sum of the same TF32
products, with the completion counters back at zero. The golden cases pin specific edges; these
cover the combinations between them.

The bound is the north-star tolerance plus the summation-conditioning term of the c5 check
(16 x 2^-24 x sum|terms|, gpu_cases.assert_close_conditioned), needed by at most 1e-3 of the
elements: A values up to 1e3 against x100 outlier features on rows of thousands of terms cancel
so far that no FP32 summation order meets 1e-3 absolute on a few elements (seed 1 at F256: a
row-order FP32 sum of the same products misses it on 19 elements, this kernel on 3)."""
import numpy as np
import pytest

import tcc_spmm_amd as T
from gpu_cases import assert_close_conditioned, features, gpu_prepare

pytestmark = pytest.mark.gpu


def _random_csr(seed):
    rng = np.random.default_rng(seed)
    rows = int(rng.integers(1, 1500))
    cols = int(rng.integers(1, 12000))
    kind = rng.random(rows)
    deg = np.where(kind < 0.15, 0,                                   # empty rows
                   np.where(kind < 0.92, rng.integers(1, 40, rows),  # ordinary rows
                            rng.integers(40, 4000, rows)))           # long rows
    if rng.random() < 0.7:  # a heavy SW: several long rows in one 32-row window, split into tasks
        sw = int(rng.integers(0, (rows + 31) // 32))
        heavy = sw * 32 + rng.choice(min(32, rows - sw * 32), size=min(4, rows - sw * 32),
                                     replace=False)
        deg[heavy] = rng.integers(2000, 9000, heavy.size)
    offsets = np.zeros(rows + 1, np.uint32)
    sources, values = [], []
    band = int(rng.integers(1, cols + 1))
    for r in range(rows):
        d = min(int(deg[r]), cols)
        if d and rng.random() < 0.5:  # columns near the row, as in a banded graph
            lo = max(0, min(r, cols - 1) - band // 2)
            c = rng.integers(lo, min(cols, lo + band), d)
        else:
            c = rng.integers(0, cols, d)
        c = np.unique(c).astype(np.uint32)
        v = rng.uniform(-1.0, 1.0, c.size).astype(np.float32) * np.float32(10.0 ** rng.integers(-3, 4))
        v[v == 0] = 0.5
        sources.append(c)
        values.append(v)
        offsets[r + 1] = offsets[r] + c.size
    src = np.concatenate(sources) if sources else np.zeros(0, np.uint32)
    val = np.concatenate(values) if values else np.zeros(0, np.float32)
    return rows, cols, offsets, src.astype(np.uint32), val.astype(np.float32)


@pytest.mark.parametrize("waves", ["1", "2", "4", "8"])
@pytest.mark.parametrize("seed", range(12))
def test_random_plans_against_the_oracle(oracle, gpu, seed, waves, launch_overrides):
    launch_overrides(task_waves=int(waves))
    import torch
    from tcc_spmm_amd.device import TorchDeviceMatrix
    rows, cols, off, src, val = _random_csr(1000 + seed)
    feats = 128 if seed % 2 == 0 else 256
    print(f"random plan seed {seed}: {rows}x{cols}, nnz {src.size}, F{feats}, waves {waves}", flush=True)
    csr = T.make_canonical_csr(rows, cols, off, src, val)
    fmt = T.convert_csr_to_sw32(rows, cols, csr)
    x = features(cols, feats, seed=seed, stddev=float(2.0 ** (seed % 5 - 2)), outlier_fraction=0.02,
                 outlier_scale=100.0)
    packed, scale, _, sc, pk = gpu_prepare(x, gpu)
    dm = TorchDeviceMatrix(fmt, feats, device=gpu)
    if dm.partials is not None:
        dm.partials.fill_(float("nan"))
    y = torch.full((rows, feats), float("nan"), device=gpu)
    dm.spmm(packed, scale, y)
    torch.cuda.synchronize()
    if dm.counters is not None:
        assert int(dm.counters.abs().sum()) == 0
    of = oracle.sw32(rows, cols, *csr.views())
    windows = np.arange(len(fmt.window_offsets) - 1, dtype=np.uint32)
    y_ref, y_abs = of.spmm_windows_f64(pk, sc, windows, with_abs=True)
    relaxed = assert_close_conditioned(y.cpu().numpy(), y_ref[:rows], y_abs[:rows],
                                       f"seed {seed} F{feats} waves {waves}")
    assert relaxed <= rows * feats * 1e-3, f"{relaxed} elements needed the conditioning term"
