"""GPU parity of the Gated-DeltaNet matrix form for few sequences (front, state
and norm launches; src/engine.cpp:2600-2716) at the edges of its blocks,
sequence counts and workspace segments; of the kernels that calls of more
sequences run, in the types, math modes and ranges that test_gpu_deltanet.py and
test_gpu_deltanet_ranges.py, with few sequences, reach only through other
kernels; and of short calls against one-token steps, bit for bit.  The oracle
and the fp32 bars are those files'."""
import numpy as np
import pytest

import _oracle as O
import kvc
from gpu_util import say
from test_gpu_deltanet import ctx_ssm, run_case, state_bufs
from test_gpu_deltanet_ranges import check_all, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_tok,n_seqs,in_dtype,out_dtype", [
    (13, 1, kvc.DTYPE_BF16, kvc.DTYPE_F32),   # shortest: one block of 13
    (13, 4, kvc.DTYPE_F32, kvc.DTYPE_F32),    # shortest of 4 sequences
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


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("n_seqs", [1, 2, 3, 4, 17])
@pytest.mark.parametrize("n_tok", [2, 8, 9, 10, 11, 12])
def test_short_calls_have_the_bits_of_token_steps(n_tok, n_seqs, exact):
    """Up to 12 tokens, however few the sequences, the arithmetic is fp32
    throughout and the same as token by token: outputs and state bit for bit."""
    say(f"deltanet, {n_seqs} sequences of {n_tok} tokens against token steps, exact {exact}")
    h = kvc.hip()
    rng = np.random.default_rng(12500 + 10 * n_tok + n_seqs)
    OUT = O.SSM_NV * O.SSM_DV
    w = [0.5 * rng.standard_normal((4, O.SSM_C)), rng.standard_normal(O.SSM_NV), -rng.uniform(0.05, 1.0, O.SSM_NV),
         rng.uniform(0.5, 1.5, O.SSM_DV)]
    proj = rng.standard_normal((n_seqs, n_tok, O.SSM_PROJ)).astype(np.float32)
    in_dtype = kvc.DTYPE_F32 if n_seqs % 2 else kvc.DTYPE_BF16
    if in_dtype == kvc.DTYPE_BF16:
        proj = O.f32_to_bf16(proj)
    S0 = (0.05 * rng.standard_normal(OUT * O.SSM_DK)).astype(np.float32)
    got = []
    with ctx_ssm(max_seqs=2 * n_seqs, flags=kvc.FLAG_EXACT_MATH if exact else 0) as ctx:
        bufs = [kvc.to_device(x.astype(np.float32)) for x in w]
        for step in (n_tok, 1):
            seqs = [ctx.seq_create() for _ in range(n_seqs)]
            for s in seqs:
                state_bufs(ctx, s, 0)[0].upload(S0)
            out = np.empty((n_seqs, n_tok, OUT), np.float32)
            for t in range(0, n_tok, step):
                pb, ob = kvc.to_device(np.ascontiguousarray(proj[:, t:t + step])), h.malloc(n_seqs * step * OUT * 4)
                ctx.deltanet_step(0, seqs, step, pb, *bufs, ob, in_dtype=in_dtype)
                ctx.sync()
                out[:, t:t + step] = ob.download(np.float32, (n_seqs, step, OUT))
                pb.free()
                ob.free()
            got.append([out] + [b.download(np.float32, (b.nbytes // 4,)) for s in seqs for b in state_bufs(ctx, s, 0)])
        for b in bufs:
            b.free()
    for a, b in zip(*got):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def test_few_sequences_over_workspace_segments():
    """4 sequences of 700 tokens need 44 blocks of workspace each where 40 fit,
    so the call runs as two segments of blocks."""
    say("deltanet, 4 sequences of 700 tokens in two workspace segments")
    run_case(kvc.DTYPE_BF16, kvc.DTYPE_F32, n_tok=700, n_seqs=4, seed=12900)


@pytest.mark.parametrize("n_tok,n_seqs,in_dtype,out_dtype,exact", [
    # the persistent matrix form: every type and math mode
    (16, 8, kvc.DTYPE_BF16, kvc.DTYPE_BF16, False),
    (33, 8, kvc.DTYPE_BF16, kvc.DTYPE_BF16, True),
    (37, 8, kvc.DTYPE_BF16, kvc.DTYPE_F32, True),
    (20, 9, kvc.DTYPE_F32, kvc.DTYPE_BF16, False),
    (37, 8, kvc.DTYPE_F32, kvc.DTYPE_BF16, True),
    (17, 8, kvc.DTYPE_F32, kvc.DTYPE_F32, True),
    (13, 5, kvc.DTYPE_F32, kvc.DTYPE_F32, False),
    # the blocked kernel's two-block form
    (9, 5, kvc.DTYPE_F32, kvc.DTYPE_F32, True),
    (12, 8, kvc.DTYPE_F32, kvc.DTYPE_BF16, False),
    (12, 5, kvc.DTYPE_BF16, kvc.DTYPE_BF16, True),
    # the one-token kernel's 512-thread form
    (1, 17, kvc.DTYPE_F32, kvc.DTYPE_F32, False),
    (1, 17, kvc.DTYPE_F32, kvc.DTYPE_BF16, True),
    (1, 18, kvc.DTYPE_BF16, kvc.DTYPE_BF16, True),
])
def test_many_sequences(n_tok, n_seqs, in_dtype, out_dtype, exact):
    say(f"deltanet, {n_seqs} sequences of {n_tok} tokens, in {in_dtype} out {out_dtype} exact {exact}")
    run_case(in_dtype, out_dtype, n_tok=n_tok, n_seqs=n_seqs, seed=12700 + 7 * n_tok + n_seqs, exact=exact)


def test_persistent_kernel_long_call_with_almost_no_decay():
    say("deltanet ranges: 8 sequences of 512 tokens, decays near 1")
    check_all(*run(512, 8, 13100, a_range=(1e-4, 1e-3)), "512 tokens, weak decay")


@pytest.mark.parametrize("case", [
    dict(a_range=(1e-4, 1e-3)), dict(a_range=(20.0, 50.0)), dict(beta_raw=60.0),
    dict(proj_scale=100.0, state_scale=1.0), dict(small_rows=[(3, 5), (31, 127)], zero_rows=[(7, 9)]),
])
def test_persistent_kernel_ranges(case):
    say(f"deltanet ranges, 8 sequences of 48 tokens: {case}")
    out, states, ref_out, ref_states = run(48, 8, 13000 + len(case), **case)
    assert np.isfinite(out).all()
    check_all(out, states, ref_out, ref_states, str(case))
