"""GPU parity of the Gated-DeltaNet matrix form for few sequences (front, state
and norm launches; src/engine.cpp:2600-2716) at the edges of its blocks,
sequence counts and workspace segments, and of the persistent matrix form at
the ranges that test_gpu_deltanet_ranges.py now reaches only through the
few-sequence form.  The oracle and the fp32 bars are those files'."""
import numpy as np
import pytest

import kvc
from gpu_util import say
from test_gpu_deltanet import run_case
from test_gpu_deltanet_ranges import check_all, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_tok,n_seqs,in_dtype,out_dtype", [
    (9, 1, kvc.DTYPE_BF16, kvc.DTYPE_F32),    # shortest: one block of 9
    (10, 4, kvc.DTYPE_F32, kvc.DTYPE_F32),    # shortest of 4 sequences
    (16, 1, kvc.DTYPE_BF16, kvc.DTYPE_BF16),  # one whole block
    (17, 3, kvc.DTYPE_F32, kvc.DTYPE_BF16),   # a second block of one token
    (95, 2, kvc.DTYPE_BF16, kvc.DTYPE_F32),   # more blocks than LDS buffers, ragged end
    (33, 5, kvc.DTYPE_BF16, kvc.DTYPE_F32),   # 3 blocks: first call length of 5 sequences
    (65, 7, kvc.DTYPE_F32, kvc.DTYPE_F32),    # 5 blocks: the most sequences
    (64, 7, kvc.DTYPE_BF16, kvc.DTYPE_F32),   # one block fewer: the persistent kernel
])
def test_few_sequences(n_tok, n_seqs, in_dtype, out_dtype):
    say(f"deltanet, {n_seqs} sequences of {n_tok} tokens, in {in_dtype} out {out_dtype}")
    run_case(in_dtype, out_dtype, n_tok=n_tok, n_seqs=n_seqs, seed=12000 + 7 * n_tok + n_seqs)


def test_few_sequences_over_workspace_segments():
    """4 sequences of 700 tokens need 44 blocks of workspace each where 40 fit,
    so the call runs as two segments of blocks."""
    say("deltanet, 4 sequences of 700 tokens in two workspace segments")
    run_case(kvc.DTYPE_BF16, kvc.DTYPE_F32, n_tok=700, n_seqs=4, seed=12900)


@pytest.mark.parametrize("case", [
    dict(a_range=(1e-4, 1e-3)), dict(a_range=(20.0, 50.0)), dict(beta_raw=60.0),
    dict(proj_scale=100.0, state_scale=1.0), dict(small_rows=[(3, 5), (31, 127)], zero_rows=[(7, 9)]),
])
def test_persistent_kernel_ranges(case):
    say(f"deltanet ranges, 8 sequences of 48 tokens: {case}")
    out, states, ref_out, ref_states = run(48, 8, 13000 + len(case), **case)
    assert np.isfinite(out).all()
    check_all(out, states, ref_out, ref_states, str(case))
