"""GPU parity of the prefill's work splits: 16- and 32-row workgroups, keys cut
into pieces that a second launch folds, and launches that mix one-piece and
many-piece row blocks, against the oracle's causal attention
(src/engine.cpp:2892-2924), and the prefill step through 32-row launches
against its two-call form, bit for bit.  test_prefill_split.py checks on the CPU
that each case takes the route given here.

Bars: max |diff| <= 2e-2 and relative RMS <= 5e-3 (bf16 weights in P.V: about
1e-3 measured, whatever the split)."""
import numpy as np
import pytest

import _oracle as O
import kvc
from gpu_util import D, NKV, NQ, ROW, Mirror, fill_seq, say
from test_gpu_prefill_step import run_pair

pytestmark = pytest.mark.gpu

CASES = [
    # prefixes, n_q, (rows per workgroup, keys in pieces): what the launch exercises
    ((0,), 1, (16, False)),           # one row, one key
    ((0,), 17, (16, False)),          # two 16-row blocks, the second with one row
    ((63,), 32, (16, False)),         # a tile that the first rows do not see at all
    ((64, 0), 33, (16, False)),       # three 16-row blocks, the last with one row
    ((300,), 32, (16, True)),         # pieces of one tile, last tile ragged
    ((2047,), 16, (16, True)),        # last key ends a tile's first block
    ((4001,), 32, (16, True)),        # many pieces, more than one fold batch
    ((1, 5000), 20, (16, True)),      # one sequence in one piece beside a long one
    ((900, 0, 31), 130, (16, True)),  # empty prefixes in one piece, odd unit count
    ((0,), 500, (16, False)),         # a first prompt, blocks dealt to all XCDs
    ((7000,), 96, (16, True)),        # several row blocks of many pieces
    ((3000, 2500, 100), 100, (32, True)),         # a last block of 4 rows, one sequence in one piece
    (tuple(range(20, 1940, 120)), 17, (32, True)),  # one piece to six, blocks of 17 rows
    ((0,) * 33, 17, (32, False)),     # one round where 16 rows need two
    ((16,) * 13, 100, (32, False)),   # the same with four blocks, the last of 4 rows
]


@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("prefix,n_q", [c[:2] for c in CASES])
def test_prefill_work_splits(prefix, n_q, gated):
    say(f"prefill split: prefixes {prefix}, {n_q} rows, gated {gated}")
    h = kvc.hip()
    n = len(prefix)
    seed = 8100 + 13 * n_q + sum(prefix)
    with kvc.Context(n_attn_layers=1, n_ssm_layers=0, max_seqs=n, max_seq_len=max(prefix) + n_q + 32,
                     pool_blocks=sum((p + n_q) // 32 + 2 for p in prefix) + 8, snapshot_slots=0,
                     alloc_seed=seed) as ctx:
        m = Mirror(1)
        seqs = [ctx.seq_create() for _ in prefix]
        for s, p in zip(seqs, prefix):
            if p:
                fill_seq(ctx, m, [s], p, seed=seed + p)
        k = O.normal_bf16(n * n_q * ROW, seed + 1).reshape(n, n_q, ROW)
        v = O.normal_bf16(n * n_q * ROW, seed + 2).reshape(n, n_q, ROW)
        q = O.normal_bf16(n * n_q * NQ * D, seed + 3).reshape(n, n_q, NQ * D)
        g = O.normal_bf16(n * n_q * NQ * D, seed + 4).reshape(n, n_q, NQ * D)
        bufs = [kvc.to_device(x) for x in (k, v, q, g)]
        ob = h.malloc(n * n_q * NQ * D * 4)
        ctx.reserve(seqs, n_q)
        ctx.append(0, seqs, n_q, bufs[0], bufs[1])
        ctx.prefill_attn(0, seqs, n_q, bufs[2], ob, gate=bufs[3] if gated else None)
        ctx.sync()
        out = ob.download(np.float32, (n, n_q, NQ * D))
        for b in bufs + [ob]:
            b.free()
    for i, p in enumerate(prefix):
        kk, vv = m.get(seqs[i], 0)
        ref = O.prefill_attn(q[i], np.concatenate([kk, k[i]]), np.concatenate([vv, v[i]]), p, n_q,
                             gate=g[i] if gated else None)
        O.assert_attn_close(out[i], ref.reshape(n_q, NQ * D), rel_rms=5e-3, what=f"seq {i} prefix {p}")


@pytest.mark.parametrize("in_dtype", [kvc.DTYPE_BF16, kvc.DTYPE_F32])
@pytest.mark.parametrize("prefix,n_q", [c[:2] for c in CASES if c[2][0] == 32])
def test_prefill_step_work_splits(prefix, n_q, in_dtype):
    say(f"prefill step vs two launches, 32-row workgroups: prefixes {prefix}, {n_q} rows, in_dtype {in_dtype}")
    run_pair(list(prefix), n_q, seed=8600 + n_q, in_dtype=in_dtype)
