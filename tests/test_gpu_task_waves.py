"""Y at both sides of every line of the rule that picks a task's waves and its workgroup order.

With `slots` wave slots, a plan takes 8 waves per task up to slots / 8 tasks, 4 up to 5/8 slots, 2 up to 8
slots at F128 and 3 at F256, and 1 above. Plans whose waves fill at most 3/4 of the slots, or all of them with
8 waves and no split SW, skip the range search and the tail window: the lines are at 3/32 (8 waves) and 3/16
(4 waves) of the slots. The plans have short tasks of few panels (waves without any panel), split SWs (chunks
merged by the workgroup's waves) and a last SW with missing rows.
"""
import hashlib
import os
import subprocess
import sys

import numpy as np
import pytest

import tcc_spmm_amd as T
from conftest import ROOT
from gpu_cases import ATOL, RTOL, features, gpu_prepare

pytestmark = pytest.mark.gpu


def _matrix(tasks, rng, hubs=None):
    """A matrix whose plan has exactly `tasks` tasks: SWs of a few panels and, among them, one row of
    7,000 entries (876 panels, three tasks) per 400 tasks, or `hubs` such rows."""
    hubs = max(1, tasks // 400) if hubs is None else hubs
    sws = tasks - 2 * hubs
    rows, cols = 32 * sws - 5, 9000
    degree = rng.integers(0, 4, rows)
    if hubs:
        degree[rng.choice(sws, hubs, replace=False) * 32 + rng.integers(0, 27, hubs)] = 7000
    lists = [np.sort(rng.choice(cols, d, replace=False)) if d else np.zeros(0, np.int64)
             for d in degree]
    off = np.concatenate([[0], np.cumsum(degree)]).astype(np.uint32)
    src = np.concatenate(lists).astype(np.uint32)
    val = rng.uniform(-1, 1, src.size).astype(np.float32)
    return T.make_canonical_csr(rows, cols, off, src, val)


@pytest.mark.parametrize("feats", [128, 256])
@pytest.mark.parametrize("num,den,extra", [(1, 32, 0), (3, 32, 0), (3, 32, 1), (1, 8, 0), (1, 8, 1),
                                           (5, 8, 0), (5, 8, 1), (3, 1, 0), (3, 1, 1)])
def test_spmm_at_the_lines_of_the_waves_rule(oracle, gpu, feats, num, den, extra):
    import torch
    from tcc_spmm_amd.device import TorchDeviceMatrix
    slots = torch.cuda.get_device_properties(gpu).multi_processor_count * 4 * (4 if feats == 128 else 2)
    tasks = slots * num // den + extra
    csr = _matrix(tasks, np.random.default_rng(tasks + feats))
    fmt = T.convert_csr_to_sw32(csr.rows, csr.cols, csr)
    assert len(fmt.tasks) == tasks and fmt.partial_count > 0
    packed, scale, _, sc, pk = gpu_prepare(features(csr.cols, feats, seed=tasks), gpu)
    dm = TorchDeviceMatrix(fmt, feats, device=gpu)
    y = torch.full((csr.rows, feats), float("nan"), device=gpu)
    dm.partials.fill_(float("nan"))
    for _ in range(2):  # the second launch finds the counters as the first left them
        dm.spmm(packed, scale, y)
    assert int(dm.counters.abs().sum()) == 0
    ofmt = oracle.sw32(csr.rows, csr.cols, *csr.views())
    # A sum of n FP32 additions of exact products is off by at most n * 2^-24 of the sum of their
    # magnitudes; over the 7,000 terms of a hub row that is covered by the oracle's conditioned bound.
    st = ofmt.check_full(pk, sc, y.cpu().numpy(), ATOL, RTOL, cond=16.0, threads=8)
    assert st["checked"] == y.numel() and st["bad"] == 0, st


def _line_matrix(tasks, rng):
    """A matrix like _matrix's, drawn without a loop over rows: up to three entries per row, and rows of 7,000
    (the sum over such a row rounds differently in every task form)."""
    hubs = max(1, tasks // 400)
    sws = tasks - 2 * hubs
    rows, cols = 32 * sws - 5, 9000
    degree = rng.integers(0, 4, rows)
    hub_rows = rng.choice(sws, hubs, replace=False) * 32 + rng.integers(0, 27, hubs)
    degree[hub_rows] = 7000
    off = np.concatenate([[0], np.cumsum(degree)])
    at = np.arange(off[-1]) - np.repeat(off[:-1], degree)
    src = np.repeat(rng.integers(0, cols // 3, rows), degree) + cols // 3 * at
    for r in hub_rows:
        src[off[r]:off[r] + 7000] = np.sort(rng.choice(cols, 7000, replace=False))
    return T.make_canonical_csr(rows, cols, off.astype(np.uint32), src.astype(np.uint32),
                                rng.uniform(-1, 1, src.size).astype(np.float32))


@pytest.mark.parametrize("feats,num,den,extra,waves,other", [
    (f, n, d, e, w, o) for f in (128, 256) for n, d, e, w, o in (
        (3, 32, 0, 8, 4), (3, 32, 1, 8, 4), (1, 8, 0, 8, 4), (1, 8, 1, 4, 8), (3, 16, 0, 4, 2),
        (3, 16, 1, 4, 2), (5, 8, 0, 4, 2), (5, 8, 1, 2, 4), (3, 1, 0, 2, 1))
] + [(256, 3, 1, 1, 1, 2), (128, 3, 1, 1, 2, 1), (128, 8, 1, 0, 2, 1), (128, 8, 1, 1, 1, 2)])
def test_spmm_takes_the_form_of_the_waves_rule(oracle, gpu, feats, num, den, extra, waves, other):
    """The launch's own choice is `waves`, and not the form on the line's other side: its Y is that form's bit
    for bit."""
    import torch
    from tcc_spmm_amd.device import TorchDeviceMatrix, launch_overrides
    slots = torch.cuda.get_device_properties(gpu).multi_processor_count * 4 * (4 if feats == 128 else 2)
    tasks = slots * num // den + extra
    csr = _line_matrix(tasks, np.random.default_rng(tasks + feats))
    fmt = T.convert_csr_to_sw32(csr.rows, csr.cols, csr)
    assert len(fmt.tasks) == tasks and fmt.partial_count > 0
    packed, scale, _, sc, pk = gpu_prepare(features(csr.cols, feats, seed=tasks), gpu)
    dm = TorchDeviceMatrix(fmt, feats, device=gpu)
    y = dm.spmm(packed, scale)
    with launch_overrides(task_waves=waves):
        assert torch.equal(y.view(torch.int32), dm.spmm(packed, scale).view(torch.int32))
    with launch_overrides(task_waves=other):
        assert not torch.equal(y.view(torch.int32), dm.spmm(packed, scale).view(torch.int32))
    st = oracle.sw32(csr.rows, csr.cols, *csr.views()).check_full(pk, sc, y.cpu().numpy(), ATOL, RTOL,
                                                                  cond=16.0, threads=8)
    assert st["checked"] == y.numel() and st["bad"] == 0, st


@pytest.mark.parametrize("feats", [128, 256])
@pytest.mark.parametrize("num,den,extra", [(3, 32, 0), (3, 32, 1), (1, 8, 0), (1, 8, 1),
                                           (3, 16, 0), (3, 16, 1)])
def test_spmm_unsplit_plans_at_the_lines_of_the_order_rule(oracle, gpu, feats, num, den, extra):
    """Plans without split SWs take their tasks in list order up to slots / 8 tasks (eight waves each)
    and, with four waves, up to 3/16 slots; above the lines by ranges and size classes."""
    import torch
    from tcc_spmm_amd.device import TorchDeviceMatrix
    slots = torch.cuda.get_device_properties(gpu).multi_processor_count * 4 * (4 if feats == 128 else 2)
    tasks = slots * num // den + extra
    csr = _matrix(tasks, np.random.default_rng(tasks), hubs=0)
    fmt = T.convert_csr_to_sw32(csr.rows, csr.cols, csr)
    assert len(fmt.tasks) == tasks and fmt.partial_count == 0
    packed, scale, _, sc, pk = gpu_prepare(features(csr.cols, feats, seed=tasks), gpu)
    y = torch.full((csr.rows, feats), float("nan"), device=gpu)
    TorchDeviceMatrix(fmt, feats, device=gpu).spmm(packed, scale, y)
    st = oracle.sw32(csr.rows, csr.cols, *csr.views()).check_full(pk, sc, y.cpu().numpy(), ATOL, RTOL,
                                                                  threads=8)
    assert st["checked"] == y.numel() and st["bad"] == 0, st


@pytest.mark.parametrize("feats", [128, 256])
@pytest.mark.parametrize("waves", [0, 1, 2, 4, 8])
def test_spmm_odd_walks_ignore_the_first_source(oracle, gpu, feats, waves):
    """A walk of an odd number of panels fills its last pair with an empty panel, whose metadata reads as
    source 0. No row references source 0 here, so its scale and features may be anything."""
    from tcc_spmm_amd.device import TorchDeviceMatrix, launch_overrides
    rng = np.random.default_rng(feats + waves)
    rows, cols = 32 * 9, 600
    # SW i: one row of 8 (i + 1) - 3 entries: i + 1 panels of one exclusive bucket
    lists = [np.zeros(0, np.int64)] * rows
    for i in range(9):
        lists[32 * i + (i % 4) * 8] = np.sort(rng.choice(np.arange(1, cols), 8 * (i + 1) - 3, replace=False))
    off = np.concatenate([[0], np.cumsum([len(c) for c in lists])]).astype(np.uint32)
    src = np.concatenate(lists).astype(np.uint32)
    csr = T.make_canonical_csr(rows, cols, off, src, rng.uniform(-1, 1, src.size).astype(np.float32))
    packed, scale, _, sc, pk = gpu_prepare(features(cols, feats, seed=7), gpu)
    dm = TorchDeviceMatrix(T.convert_csr_to_sw32(rows, cols, csr), feats, device=gpu)
    with launch_overrides(task_waves=waves):
        want = dm.spmm(packed, scale).clone()
        for bad in (float("nan"), float("inf"), -float("inf")):
            scale[0] = bad
            got = dm.spmm(packed, scale)
            assert bool((got == want).all()), bad
    ref = oracle.sw32(rows, cols, *csr.views()).spmm_f64(pk, sc)
    assert np.abs(want.cpu().numpy() - ref).max() < 1e-3


def test_task_waves_from_the_environment(gpu):
    """TCC_SPMM_TASK_WAVES=8 is the form that forcing 8 gives, bit for bit (the order of the additions
    differs between the forms), and not another one."""
    from tcc_spmm_amd.device import TorchDeviceMatrix, launch_overrides
    csr = _matrix(64, np.random.default_rng(3))
    packed, scale, *_ = gpu_prepare(features(csr.cols, 128, seed=3), gpu)
    dm = TorchDeviceMatrix(T.convert_csr_to_sw32(csr.rows, csr.cols, csr), 128, device=gpu)
    forms = {}
    for waves in (1, 2, 4, 8):
        with launch_overrides(task_waves=waves):
            forms[waves] = hashlib.sha256(dm.spmm(packed, scale).cpu().numpy().tobytes()).hexdigest()
    assert len(set(forms.values())) == 4
    code = """
import hashlib, sys
import numpy as np
sys.path[:0] = ["tests", "."]
import tcc_spmm_amd as T
from gpu_cases import features, gpu_prepare
from tcc_spmm_amd.device import TorchDeviceMatrix
from test_gpu_task_waves import _matrix
csr = _matrix(64, np.random.default_rng(3))
packed, scale, *_ = gpu_prepare(features(csr.cols, 128, seed=3), "cuda")
dm = TorchDeviceMatrix(T.convert_csr_to_sw32(csr.rows, csr.cols, csr), 128, device="cuda")
print(hashlib.sha256(dm.spmm(packed, scale).cpu().numpy().tobytes()).hexdigest())
"""
    res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, cwd=ROOT,
                         env=dict(os.environ, TCC_SPMM_TASK_WAVES="8"), timeout=100)
    assert res.returncode == 0, res.stderr
    assert res.stdout.split()[-1] == forms[8]


def _shared_entry_csr():
    """22 SWs: SW i has i % 3 and (i // 3) % 2 exclusive panels of two row groups (its shared part starts in
    the middle of a pair or not), then 1 to 3 panels in each of two shared buckets, the first of them bucket
    i % 11 of the eleven (those before it empty), the second further on or missing."""
    from itertools import combinations
    rng = np.random.default_rng(23)
    shared = [sum(1 << g for g in c) for n in (2, 3, 4) for c in combinations(range(4), n)]
    rows_of = []
    nxt = 0
    for i in range(22):
        panels = {1 << (i % 4): i % 3, 1 << ((i + 1) % 4): (i // 3) % 2, shared[i % 11]: 1 + i % 3}
        if i % 11 < 10:
            panels[shared[10 - (i * 7) % (10 - i % 11)]] = 1 + (i + 1) % 3
        lists = [[] for _ in range(32)]
        for mask, n in panels.items():
            for s in range(nxt, nxt + 8 * n):
                for g in range(4):
                    if mask >> g & 1:
                        lists[8 * g + int(rng.integers(0, 8))].append(s)
            nxt += 8 * n
        rows_of += lists
    off = np.concatenate([[0], np.cumsum([len(r) for r in rows_of])]).astype(np.uint32)
    src = np.concatenate([np.sort(np.array(r, np.uint32)) for r in rows_of])
    return T.make_canonical_csr(len(rows_of), nxt, off, src, rng.uniform(0.1, 1, src.size).astype(np.float32))


@pytest.mark.parametrize("feats", [128, 256])
@pytest.mark.parametrize("waves,wide", [(1, False), (2, False), (4, False), (8, False), (1, True)])
def test_spmm_walks_that_enter_the_shared_buckets_anywhere(oracle, gpu, feats, waves, wide):
    from tcc_spmm_amd.device import TorchDeviceMatrix, launch_overrides
    csr = _shared_entry_csr()
    fmt = T.convert_csr_to_sw32(csr.rows, csr.cols, csr)
    per = np.diff(fmt.bucket_offsets.reshape(-1, 17).astype(np.int64), axis=1)
    assert set((per[:, 5:] > 0).argmax(axis=1)) == set(range(11))  # every bucket is some SW's first shared one
    assert set(per[:, 1:5].sum(axis=1) % 2) == {0, 1}
    packed, scale, _, sc, pk = gpu_prepare(features(csr.cols, feats, seed=5), gpu)
    with launch_overrides(task_waves=waves, force_wide=wide):
        y = TorchDeviceMatrix(fmt, feats, device=gpu).spmm(packed, scale).cpu().numpy()
    st = oracle.sw32(csr.rows, csr.cols, *csr.views()).check_full(pk, sc, y, ATOL, RTOL, threads=8)
    assert st["checked"] == y.size and st["bad"] == 0, st
