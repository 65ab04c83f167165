"""Plans of the planner on both sides of its lines (rows, K rounds of the 4x4x4 GEMV, K of the 8-bit
GEMV, K splits and columns of the column-block kernel), through the entry points and against the
oracle, in both code layouts, which have to agree to the bit.

The bars are the contract's: 2e-3 of the largest output after removing the final rounding, and at
least 98% (bf16) or 90% (f16) of outputs equal to the correctly rounded reference."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import metile_amd as mt
from metile_amd import tuning
from oracle import affine as O
from tests.helpers import act_to_torch, affine_to_torch, torch_to_act

TOL = 2e-3
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16}

# K, N, bits, group, dtype, projections, rows
CASES = [
    (64, 32, 4, 64, "bf16", 1, (1, 2, 3, 4, 5)),         # one partial round, one column group
    (3584, 96, 4, 64, "f16", 1, (2, 3, 4)),              # seven rounds: strips from three rows on
    (3648, 800, 4, 64, "bf16", 2, (1, 3, 4)),            # eight rounds, the last partial
    (12288, 160, 4, 128, "f16", 1, (1, 2, 4)),           # 24 rounds, three a wave
    (12352, 64, 4, 64, "bf16", 1, (1, 4)),               # 25 rounds: strips
    (8192, 96, 8, 64, "bf16", 1, (1, 2, 3)),             # the 8-bit GEMV's longest K
    (8256, 64, 8, 64, "f16", 2, (1, 2)),                 # beyond it
    (192, 32, 8, 32, "f16", 1, (1, 2, 3)),               # group of 32, 12 code chunks a column
    (1088, 2016, 8, 64, "bf16", 1, (2, 3, 16)),          # columns below the block kernel's line
    (1088, 2048, 8, 64, "f16", 1, (3, 16, 17, 32)),      # and at it
    (6144, 2048, 8, 128, "bf16", 2, (5, 32)),            # 96 K steps: unsplit
    (6208, 2048, 8, 64, "f16", 1, (5, 17)),              # 97: four splits
    (128, 9216, 8, 64, "bf16", 1, (4, 20)),              # strips as many as CUs
    (128, 9248, 8, 64, "f16", 1, (4, 20)),               # twice as many
    (128, 18464, 8, 64, "bf16", 2, (3,)),                # one a 32-column strip
    (4608, 160, 4, 64, "bf16", 2, (1, 2, 4)),            # nine rounds, three waves of three
    (5120, 3072, 4, 64, "f16", 2, (1, 3, 4)),            # ten, five of two; two column groups
    (5632, 96, 4, 64, "bf16", 2, (2,)),                  # eleven: uneven waves
    (8192, 3104, 4, 128, "bf16", 2, (1, 4)),             # sixteen, eight waves: four groups
    (1536, 9600, 4, 64, "bf16", 2, (1, 2)),              # 600 workgroups of four groups: two all the same
    (8256, 2528, 4, 64, "f16", 1, (2, 3)),               # 17 rounds, columns beside five for eight CUs
    (8256, 2560, 4, 64, "bf16", 1, (2, 4)),
    (8256, 5088, 4, 64, "f16", 1, (3,)),                 # the most columns of three rounds a wave
    (8256, 5120, 4, 64, "bf16", 1, (2, 4)),
    (6208, 3040, 8, 64, "bf16", 1, (5, 8)),              # K split, columns below its line
    (6208, 3072, 8, 64, "f16", 1, (5, 17)),              # and at it
    (1536, 2048, 8, 64, "f16", 2, (3, 17)),              # short K: from 2048 columns
    (1600, 4576, 8, 64, "bf16", 1, (3, 8)),              # longer: columns beside 18 per CU
    (1600, 4608, 8, 64, "f16", 1, (3, 8, 16)),
    (1600, 4608, 8, 64, "bf16", 2, (3, 17)),
    (1600, 6112, 8, 64, "f16", 1, (16,)),                # and 24 with more than 16 rows
    (1600, 6144, 8, 64, "bf16", 1, (8, 17)),
    (192, 4576, 8, 64, "f16", 2, (4, 32)),               # two projections below two blocks per CU
    (192, 4608, 8, 64, "bf16", 2, (3, 16)),              # and at them: nine columns a block
    (128, 20480, 8, 64, "f16", 2, (5,)),                 # forty
    (128, 20512, 8, 64, "bf16", 2, (5,)),
]


@pytest.fixture
def clean_plans():
    tuning.clear_plans()
    yield
    tuning.clear_plans()


@pytest.mark.parametrize("k,n,bits,g,dtype,nproj,rows", CASES)
def test_planner_plans_are_valid_candidates(k, n, bits, g, dtype, nproj, rows, clean_plans):
    for m in rows:
        plan = tuning.qmv_plan(m, k, n, g, bits, nproj, DTYPES[dtype])
        bucket = tuning.row_bucket(m)
        if bucket == m:
            assert plan in tuning.qmv_plan_candidates(m, k, n, g, bits, nproj)
        else:  # accepted at the bucket the dispatch belongs to
            tuning.install_qmv_plan(m, k, n, g, bits, nproj, DTYPES[dtype], plan)


@pytest.mark.gpu
@pytest.mark.parametrize("k,n,bits,g,dtype,nproj,rows", CASES)
def test_planner_plans_meet_the_contract(k, n, bits, g, dtype, nproj, rows, clean_plans):
    if not torch.cuda.is_available():
        pytest.skip("no ROCm device")
    weights = [O.make_affine_weight(n, k, bits, g, 67, 10 + 2 * p, dtype=dtype)
               for p in range(nproj)]
    triples = [affine_to_torch(w, dtype) for w in weights]
    packed = [(mt.affine_repack(w, bits=bits), s, b) for w, s, b in triples]
    op = mt.affine_swiglu if nproj == 2 else mt.affine_qmv
    same = []
    for m in rows:
        print(f"[planner] {m}x{k}x{n} bits={bits} g={g} {dtype} nproj={nproj}", flush=True)
        x = O.make_activations(m, k, 67, dtype=dtype)
        xt = act_to_torch(x, dtype)
        got, again = (op(xt, *[t for w in ws for t in w], group_size=g, bits=bits)
                      for ws in (triples, packed))
        if nproj == 2:
            ref = O.affine_swiglu(x, *weights, g, bits, dtype=dtype)
        else:
            ref = O.affine_qmv(x, *weights[0], g, bits, dtype=dtype)
        y = torch_to_act(got, dtype)
        rounded = O.to_f32(O.from_f32(ref.astype(np.float32), dtype), dtype)
        same.append((O.to_f32(y, dtype) == rounded).ravel())
        assert O.tolerance_error(y, ref, dtype) <= TOL
        assert torch.equal(got, again)
    assert np.mean(np.concatenate(same)) >= (0.98 if dtype == "bf16" else 0.90)
