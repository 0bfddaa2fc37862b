"""fa_kg_kernel (key groups: the waves of a workgroup share its q-tile's keys)
against the fp64 oracle and the emulated reference kernel, at the edges of its
tiles and of the plan rule that picks it: ragged rows and keys, causal rows
whose later groups see no key, one to many steps, rows whose maximum jumps
between groups, strided views, with and without an LSE."""
from __future__ import annotations

import ctypes
import math

import pytest
import torch

import abi_ctypes as A
from helpers import case_seed, make_qkv
from test_gpu_parity import _check_against_oracle

pytestmark = pytest.mark.gpu

DEV = "cuda"


@pytest.fixture(scope="module")
def lib():
    return A.load()


def _plan(lib, q, causal):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    pl = A.FaFwdPlan()
    p = A.params_from_tensors(q, q, q, q, None, causal)
    assert lib.fa_fwd_plan(ctypes.byref(p), cus, ctypes.byref(pl)) == A.FA_OK
    return pl, cus


# (B, H, N, D, causal, q-tile rows): 64 rows are four groups, 128 two
CASES = [
    (1, 4, 65, 64, True, 64), (1, 4, 128, 128, True, 64),      # groups without a visible key
    (1, 8, 200, 64, False, 64), (2, 3, 129, 128, False, 64),   # ragged last rows and keys
    (1, 5, 511, 64, True, 64), (1, 8, 513, 128, True, 64),     # one key past a step of groups
    (2, 6, 577, 128, False, 64), (1, 16, 1024, 64, False, 64), # the last: a workgroup on every CU
    (1, 17, 1023, 64, False, 128), (2, 9, 1025, 128, False, 128),
    (1, 16, 2048, 128, False, 128),                            # two groups at the end of their range
]


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("B,H,N,D,causal,rows", CASES)
def test_key_groups_vs_oracle(fa, oracle, lib, B, H, N, D, causal, rows, dtype):
    print(f"case key groups {B}x{H}x{N}x{D} {dtype} causal={causal}", flush=True)
    q, k, v = make_qkv(B, H, N, D, dtype, seed=case_seed(1300 + N + D), device=DEV)
    pl, cus = _plan(lib, q, causal)
    if cus == 256:
        assert pl.block_rows == rows and pl.key_groups == 256 // rows
        assert pl.n_items == 0 and pl.workspace_bytes == 0
    o, lse = fa.forward(q, k, v, causal=causal, return_lse=True)
    o2 = fa.forward(q, k, v, causal=causal)  # without an LSE: the same O
    o3 = fa.forward(q, k, v, causal=causal, split_kv=False)
    torch.cuda.synchronize()
    assert torch.equal(o, o2) and torch.equal(o, o3)
    _check_against_oracle(oracle, q, k, v, o, lse, causal, 1.0 / math.sqrt(D), dtype)


@pytest.mark.parametrize("dtype", ["fp16", "bf16"])
@pytest.mark.parametrize("H,N,D,key,by,causal,groups", [
    # the maximum in another group's first tile
    (4, 500, 64, 70, 6.0, False, 4), (4, 500, 64, 70, 6.0, True, 4),
    (4, 500, 128, 40, 6.0, False, 4), (4, 500, 128, 40, 6.0, True, 4),
    # far above it, in a later step: the group's offset is derived again
    (8, 900, 64, 600, 30.0, False, 4), (8, 900, 64, 600, 30.0, True, 4),
    (8, 900, 128, 600, 30.0, False, 4), (8, 900, 128, 600, 30.0, True, 4),
    (20, 900, 64, 600, 30.0, False, 2), (20, 900, 128, 600, 30.0, False, 2),
])
def test_key_groups_score_jumps_vs_oracle(fa, oracle, lib, H, N, D, key, by, causal, groups, dtype):
    """One key scaled far above the others: the groups' offsets lie far
    apart, so all but one group's share of a row vanishes in the combine."""
    print(f"case key groups jump N={N} D={D} key={key} {dtype} causal={causal}", flush=True)
    q, k, v = make_qkv(1, H, N, D, dtype, seed=case_seed(1350 + N + D), device="cpu")
    k = k.clone()
    k[:, :, key] = (k[:, :, key].float() * by).to(k.dtype)
    q, k, v = q.to(DEV), k.to(DEV), v.to(DEV)
    pl, cus = _plan(lib, q, causal)
    assert cus != 256 or pl.key_groups == groups
    o, lse = fa.forward(q, k, v, causal=causal, return_lse=True)
    _check_against_oracle(oracle, q, k, v, o, lse, causal, 1.0 / math.sqrt(D), dtype,
                          contract=False)


def test_key_groups_strided_views(fa, lib):
    """[B, N, H, D] views and a padded output give the contiguous result; the
    padding is not written."""
    B, H, N, D = 2, 4, 300, 64
    q, k, v = make_qkv(B, H, N, D, "fp16", seed=case_seed(1390), device=DEV)
    pl, cus = _plan(lib, q, False)
    assert cus != 256 or pl.key_groups == 4
    ref = fa.forward(q, k, v)
    qs, ks, vs = (t.permute(0, 2, 1, 3).contiguous().permute(0, 2, 1, 3) for t in (q, k, v))
    buf = torch.full((B, H, N, D + 8), 7.0, dtype=q.dtype, device=DEV)
    fa.forward(qs, ks, vs, buf[..., :D])
    torch.cuda.synchronize()
    assert torch.equal(buf[..., :D], ref) and bool((buf[..., D:] == 7.0).all().item())
