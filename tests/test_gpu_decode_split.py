"""GPU parity of decode's automatic work split at the edges of its rule (one
chunk per sequence, one workgroup per CU with and without the output-dim
split, short chunks where that would leave one long chunk), against the oracle
(src/engine.cpp:3528-3564): max |diff| <= 2e-2 and relative RMS <= 3e-3; of its
weight offset under scores that move by hundreds of bits from group to group or
by one key in any block of a group, with the same bars; and of
the one-token Gated-DeltaNet step on either side of its workgroup sizes, bit
for bit."""
import numpy as np
import pytest

import _oracle as O
import kvc
from gpu_util import D, NKV, NQ, Mirror, fill_seq, say

pytestmark = pytest.mark.gpu

CASES = {
    "one_chunk": [1, 31, 96],                 # every sequence in one chunk of 3 blocks
    "four_blocks": [97],                      # first length in several chunks, of one block
    "one_block_chunks": [1024],               # 32 chunks of one block
    "past_32_chunks": [1025],                 # 33 blocks: chunks of two
    "short_launch": [1000, 1024],             # 64 blocks: 32 chunks, two parts
    "four_blocks_many": [97 + 2 * i for i in range(13)],  # a chunk per sequence again
    "past_short_launch": [1000, 1056],        # 65 blocks: 22 chunks, two parts
    "past_short_launch_one_part": [700] * 3,  # 66 blocks: 33 chunks, one part
    "ragged_one_round": [777, 2001, 65, 1500],
    "very_ragged": [9000] + [33] * 40,        # 64 chunks of up to 12 blocks
    "full_batch": [40 + 7 * i for i in range(64)],  # a chunk per sequence
    "full_batch_ragged": [4000] + [33] * 63,  # short chunks (4 blocks), in rounds
}


@pytest.mark.parametrize("flags", [0, kvc.FLAG_DECODE_SPLIT_D, kvc.FLAG_DECODE_NO_SPLIT_D])
@pytest.mark.parametrize("name", CASES)
def test_decode_automatic_split(name, flags):
    lengths = CASES[name]
    say(f"decode split {name}, flags {flags}")
    h = kvc.hip()
    n = len(lengths)
    with kvc.Context(n_attn_layers=1, n_ssm_layers=0, max_seqs=n, max_seq_len=max(lengths) + 32,
                     pool_blocks=sum(x // 32 + 1 for x in lengths) + 8, snapshot_slots=0, alloc_seed=77,
                     flags=flags) as ctx:
        m = Mirror(1)
        seqs = [ctx.seq_create() for _ in lengths]
        for s, x in zip(seqs, lengths):
            fill_seq(ctx, m, [s], x, seed=500 + x)
        q = O.normal_bf16(n * NQ * D, 42).reshape(n, NQ * D)
        qb, ob = kvc.to_device(q), h.malloc(n * NQ * D * 4)
        ctx.decode_attn(0, seqs, qb, ob)
        ctx.sync()
        out = ob.download(np.float32, (n, NQ, D))
        qb.free()
        ob.free()
    for i, x in enumerate(lengths):
        kk, vv = m.get(seqs[i], 0)
        O.assert_attn_close(out[i], O.decode_attn(q[i], kk, vv, x), rel_rms=3e-3, what=f"{name}: length {x}")


# mean score of each group of 4 blocks, in units of 23 bits of the weights: the
# walk moves its weight offset at each group's first block, downwards by 16
# bits of the largest score at most
LEVELS = {
    "falling": [-2.0 * i for i in range(12)],   # 500 bits in all: an unbounded offset overflows
    "falling_slowly": [-0.3 * i for i in range(12)],
    "rising": [2.0 * i for i in range(12)],
    "alternating": [0.0, -0.5, 0.1, -3.0, 0.2, -0.6] * 2,
    "late_peak": [-4.0] * 11 + [0.0],
}


@pytest.mark.parametrize("flags", [kvc.FLAG_DECODE_SPLIT_D, kvc.FLAG_DECODE_NO_SPLIT_D])
@pytest.mark.parametrize("name", LEVELS)
def test_decode_weight_offset(name, flags):
    say(f"decode weight offset {name}, flags {flags}")
    h = kvc.hip()
    L = 12 * 128 - 27
    rng = np.random.default_rng(9)
    lev = np.repeat(np.asarray(LEVELS[name], np.float32), 128)[:L, None]
    k = O.f32_to_bf16(lev + 0.1 * rng.standard_normal((L, NKV * D)).astype(np.float32))
    v = O.normal_bf16(L * NKV * D, 91).reshape(L, NKV * D)
    q = O.f32_to_bf16(np.ones(NQ * D, np.float32))
    with kvc.Context(n_attn_layers=1, n_ssm_layers=0, max_seqs=1, max_seq_len=L + 32, pool_blocks=L // 32 + 8,
                     snapshot_slots=0, alloc_seed=78, decode_chunk_blocks=48, flags=flags) as ctx:
        s = ctx.seq_create()
        ctx.reserve([s], L)
        bufs = [kvc.to_device(x) for x in (k, v, q)]
        ob = h.malloc(NQ * D * 4)
        ctx.append(0, [s], L, bufs[0], bufs[1])
        ctx.commit([s], L)
        ctx.decode_attn(0, [s], bufs[2], ob)
        ctx.sync()
        out = ob.download(np.float32, (NQ, D))
        for b in bufs + [ob]:
            b.free()
    O.assert_attn_close(out, O.decode_attn(q, k, v, L), rel_rms=3e-3, what=name)


@pytest.mark.parametrize("flags", [kvc.FLAG_DECODE_SPLIT_D, kvc.FLAG_DECODE_NO_SPLIT_D])
@pytest.mark.parametrize("bits", [100, 150, 500])
@pytest.mark.parametrize("block", range(8))
def test_decode_weight_offset_single_peak(block, bits, flags):
    """One key `bits` bits above all others, in each block of a group of 4 (the
    offset moves down only at a group's first), followed by lower groups and a
    tail of 3 blocks, and in each wave's 8 tokens of the block: the largest
    score met has to bound the offset wherever it stood."""
    say(f"decode weight offset, peak of {bits} bits in block {block}, flags {flags}")
    h = kvc.hip()
    L = 11 * 32 - 5
    rng = np.random.default_rng(10 + block)
    lev = np.zeros((L, 1), np.float32)
    wave = (block + bits // 50) % 4
    lev[32 * block + 8 * wave + block % 8] = bits / 23.08
    k = O.f32_to_bf16(lev + 0.1 * rng.standard_normal((L, NKV * D)).astype(np.float32))
    v = O.normal_bf16(L * NKV * D, 92 + block).reshape(L, NKV * D)
    q = O.f32_to_bf16(np.ones(NQ * D, np.float32))
    with kvc.Context(n_attn_layers=1, n_ssm_layers=0, max_seqs=1, max_seq_len=L + 32, pool_blocks=L // 32 + 8,
                     snapshot_slots=0, alloc_seed=79, decode_chunk_blocks=16, flags=flags) as ctx:
        s = ctx.seq_create()
        ctx.reserve([s], L)
        bufs = [kvc.to_device(x) for x in (k, v, q)]
        ob = h.malloc(NQ * D * 4)
        ctx.append(0, [s], L, bufs[0], bufs[1])
        ctx.commit([s], L)
        ctx.decode_attn(0, [s], bufs[2], ob)
        ctx.sync()
        out = ob.download(np.float32, (NQ, D))
        for b in bufs + [ob]:
            b.free()
    assert np.isfinite(out).all()
    O.assert_attn_close(out, O.decode_attn(q, k, v, L), rel_rms=3e-3, what=f"peak in block {block}")


def test_deltanet_one_token_workgroup_sizes():
    """16 sequences take 1024-thread workgroups, 17 take 512: same bits."""
    say("deltanet, one token, 16 and 17 sequences")
    h = kvc.hip()
    rng = np.random.default_rng(5)
    C, PROJ, OUT = O.SSM_C, O.SSM_PROJ, O.SSM_NV * O.SSM_DV
    n = 17
    w = [(0.5 * rng.standard_normal((4, C))), rng.standard_normal(O.SSM_NV),
         -rng.uniform(0.05, 1.0, O.SSM_NV), rng.uniform(0.5, 1.5, O.SSM_DV)]
    proj = O.f32_to_bf16(rng.standard_normal((3, n, PROJ)).astype(np.float32))
    with kvc.Context(n_attn_layers=1, n_ssm_layers=1, max_seqs=2 * n, max_seq_len=64, pool_blocks=8,
                     snapshot_slots=0) as ctx:
        bufs = [kvc.to_device(x.astype(np.float32)) for x in w]
        sets = [[ctx.seq_create() for _ in range(n)] for _ in range(2)]
        got = []
        for group, parts in zip(sets, ((n,), (16, 1))):
            outs = []
            for step in range(3):
                pb, ob = kvc.to_device(proj[step]), h.malloc(n * OUT * 4)
                i0 = 0
                for k in parts:
                    ctx.deltanet_step(0, group[i0:i0 + k], 1, pb.ptr + i0 * PROJ * 2, *bufs, ob.ptr + i0 * OUT * 4)
                    i0 += k
                ctx.sync()
                outs.append(ob.download(np.float32, (n, OUT)))
                pb.free()
                ob.free()
            state = []
            for s in group:
                r, c = ctx.state_ptrs(s, 0)
                state.append(kvc.DeviceBuffer(h, r, OUT * O.SSM_DK * 4).download(np.uint32, (OUT * O.SSM_DK,)))
                state.append(kvc.DeviceBuffer(h, c, 3 * C * 4).download(np.uint32, (3 * C,)))
            got.append((outs, state))
        for b in bufs:
            b.free()
    for a, b in zip(got[0][0] + got[0][1], got[1][0] + got[1][1]):
        assert np.array_equal(a.view(np.uint32), b.view(np.uint32))
