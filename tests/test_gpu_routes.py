"""The plain kernels on grids that the plan still gives them: shapes of one to
four heads, which most parity tests use, run key groups or split-KV.  Each case
asserts its route (on 256 CUs), then checks sampled rows of O and the LSE
against the fp64 oracle and the emulated reference kernel.  Also key groups of
one step, whose ragged only tile must not depend on a spread test."""
from __future__ import annotations

import ctypes
import math

import numpy as np
import pytest
import torch

import abi_ctypes as A
from helpers import LSE_TOL, MAX_ABS_TOL, case_seed, err_stats, make_qkv, to_np32
from test_gpu_parity import _check_against_oracle, _fwd, _sample_rows, _scale_keys

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(scope="module")
def lib():
    return A.load()


def _assert_route(lib, q, causal, rows, groups=0):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    pl = A.FaFwdPlan()
    p = A.params_from_tensors(q, q, q, q, causal=causal)
    assert lib.fa_fwd_plan(ctypes.byref(p), cus, ctypes.byref(pl)) == A.FA_OK
    if cus == 256:
        assert (pl.block_rows, pl.key_groups, pl.n_items) == (rows, groups, 0)
        assert pl.key_halves == (4 if groups == 4 else 1)


def _inputs(H, N, D, dtype, seed, sigma, pattern):
    q, k, v = make_qkv(1, H, N, D, dtype, seed=case_seed(seed), qk_sigma=sigma, device="cpu")
    if pattern:
        k = _scale_keys(k, pattern).to(k.dtype)
    return q, k, v


CASES = [
    # H, N, D, causal, block rows, Q/K scale, jump pattern
    (20, 2049, 128, False, 256, 1.0, "jump"),  # 8 waves, one ragged row
    (20, 2049, 128, False, 256, 1.0, "huge"),
    (20, 2300, 64, False, 256, 1.0, "ramp"),
    (20, 2300, 128, False, 256, 1.0, "drop"),
    (20, 2300, 64, False, 256, 3.0, None),
    (24, 2100, 128, False, 256, 1.0, None),    # 6 of the last 8 waves past N
    (40, 1000, 128, False, 128, 3.0, None),    # 4 waves: hand-over of the first tile
    (40, 1000, 64, False, 128, 3.0, None),
    (40, 930, 128, False, 128, 1.0, "jump"),   # 2 of the last 4 waves past N
    (40, 930, 64, False, 128, 1.0, "huge"),
    (96, 960, 64, False, 128, 1.0, None),      # waves past N compute (D = 64, 3 per CU)
    (64, 1100, 128, True, 128, 1.0, "jump"),   # 4 waves, causal
    (64, 1100, 64, True, 128, 3.0, None),
]


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("H,N,D,causal,rows,sigma,pattern", CASES)
def test_plain_grids_vs_oracle(fa, oracle, lib, H, N, D, causal, rows, sigma, pattern, dtype):
    print(f"case route H={H} N={N} D={D} {dtype} causal={causal} {sigma} {pattern}", flush=True)
    q, k, v = _inputs(H, N, D, dtype, 1500 + N + D, sigma, pattern)
    qd = q.to(DEV)
    _assert_route(lib, qd, causal, rows)
    o, lse = _fwd(fa, qd, k.to(DEV), v.to(DEV), causal)
    assert torch.isfinite(o).all() and torch.isfinite(lse).all()
    scale = 1.0 / math.sqrt(D)
    rng = np.random.default_rng(1500 + N + D)
    _, sel_bh, sel_row = _sample_rows(N, H, rng, n_random=24)
    qn, kn, vn = (to_np32(t) for t in (q, k, v))
    ref_o, ref_lse = oracle.attn_rows_f64(qn, kn, vn, scale, causal, sel_bh, sel_row)
    emu_o, _ = oracle.kernel_numerics_rows(qn, kn, vn, scale, causal, sel_bh, sel_row,
                                           oracle.BF16 if dtype == "bf16" else oracle.F16)
    got = to_np32(o[0])[sel_bh, sel_row]
    got_lse = to_np32(lse[0])[sel_bh, sel_row].astype(np.float64)
    mx, mean = err_stats(got, ref_o)
    emx, emean = err_stats(emu_o, ref_o)
    lse_err = float(np.abs(got_lse - ref_lse).max())
    print(f"  {len(sel_row)} rows: max_abs={mx:.3e} mean_abs={mean:.3e} "
          f"(ref-kernel emu {emx:.3e}/{emean:.3e}) lse={lse_err:.3e}", flush=True)
    # the bars of the other non-contract cases (_check_against_oracle)
    bar = MAX_ABS_TOL if dtype == "fp16" else MAX_ABS_TOL * max(1.0, float(np.abs(ref_o).max()))
    assert mx <= bar
    assert mx <= 2 * emx + 1e-6 and mean <= 2 * emean + 1e-6
    assert lse_err <= LSE_TOL


@pytest.mark.parametrize("H,N,rows", [(20, 2300, 256), (40, 1000, 128), (40, 930, 128)])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("sigma", [1.0, 3.0])
def test_bf16_output_same_with_and_without_lse(fa, lib, H, N, rows, D, sigma):
    """The two forms of the bf16 plain kernels: O does not depend on the LSE's
    sum."""
    q, k, v = (t.to(DEV) for t in _inputs(H, N, D, "bf16", 1580, sigma, None))
    _assert_route(lib, q, False, rows)
    o1 = fa.forward(q, k, v)
    o2, lse = fa.forward(q, k, v, return_lse=True)
    torch.cuda.synchronize()
    assert torch.isfinite(lse).all() and torch.equal(o1, o2)


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("N", [193, 200, 225, 255, 256])
@pytest.mark.parametrize("sigma", [1.0, 3.0])
def test_one_step_key_groups_vs_oracle(fa, oracle, lib, N, sigma, dtype):
    """Four groups, four key tiles: the last group has the ragged one only."""
    print(f"case one step N={N} {sigma} {dtype}", flush=True)
    q, k, v = _inputs(8, N, 64, dtype, 1590 + N, sigma, None)
    qd = q.to(DEV)
    _assert_route(lib, qd, False, 64, groups=4)
    o, lse = _fwd(fa, qd, k.to(DEV), v.to(DEV), False)
    _check_against_oracle(oracle, q, k, v, o, lse, False, 1.0 / 8.0, dtype, contract=False)
