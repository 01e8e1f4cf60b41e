"""The softmax normaliser of long items against 64 bits, in both attention kernels.

A lane adds the 16 probabilities of a tile first and the tile's sum once to its running row sum, so a row sum has
one rounding per tile against the whole sum, not one per key.  Scores that all round the same way show the
difference, random ones do not: here one dominant key in the first tile of each KV part has probability 1 and every
other key the same p, chosen so that adding p alone to a sum in [1, 2) loses 0.45 of its last place each time.

With u = 2^-24, an fp32 addition of positive terms is off by at most u times its result, so a lane's row sum over n
tiles of a part is off by a relative (n + 16 + P) u at most: n tile sums, the 16 terms of a tile, the parts' merge.
At one rounding per key the lane would lose 16 x 0.45 x 2 u per tile of a sum below 2, several times that bound.
"""

from __future__ import annotations

import ctypes
import math

import numpy as np
import pytest
import torch

from trianglemix import cabi, native
from trianglemix.workload import make_cache

U = 2.0 ** -24
EXP = 2.0 ** -22  # of p: the hardware's exp2 is within 1 ulp (at most 2^-23)


def _is_wide(tq, qs, seq, prompt):
    f = ctypes.CDLL(str(native.HIP_LIBRARY)).tmi_chunk_is_wide
    f.argtypes = [ctypes.c_int] + [ctypes.c_int64] * 4
    return f(int(prompt is None), tq, qs, seq, prompt if prompt is not None else seq)


def _inputs(seq, tq, parts, tiles, dominant_value):
    """Q = e0 and K = e0 on the first key of tiles 0 .. parts - 1, 0 elsewhere; V is dominant_value on those keys.
    tiles: of one part.  Returns the inputs, the scale and p in 64 bits."""
    ulp = 2 * U  # of a sum in [1, 2)
    p = (math.floor(0.9 / (16 * tiles) / ulp) + 0.45) * ulp
    scale = np.float32(-math.log2(p) / 1.4426950408889634)
    c2 = np.float32(scale * np.float32(1.4426950408889634))  # the library's, in fp32
    k, v, bt = make_cache(seq, 1, std=0.0)
    for key in range(0, 32 * parts, 32):
        k[int(bt[0, key // 128]), key % 128, :, 0] = 1.0
        v[int(bt[0, key // 128]), key % 128] = dominant_value
    q = torch.zeros(tq, 32, 128, dtype=torch.bfloat16)
    q[:, :, 0] = 1.0
    return q, k, v, bt, float(scale), 2.0 ** -float(c2)


# (query_start, query_tokens, prompt_len or None for the dense companion, KV parts, 64-row kernel)
SPLIT = [
    (8192, 96, 8288, 4, 1),         # 13 iterations
    (15360, 1024, 16384, 2, 1),     # 32 iterations
    (40960, 1024, None, 1, 1),      # 656 iterations
    (129024, 2048, 131072, 1, 1),   # 256 iterations
    (2357, 512, 2869, 4, 0),        # the eight-wave kernel: 11 iterations
    (30720, 2048, 32768, 1, 0),     # 64 iterations
]


@pytest.mark.gpu
@pytest.mark.parametrize("qs,tq,prompt,parts,wide", SPLIT, ids=[f"{q}+{t}{'' if p else '_dense'}" for q, t, p, _, _ in SPLIT])
def test_row_sum_of_a_long_piece_matches_64_bits(gpu, qs, tq, prompt, parts, wide):
    """The fp32 row sums of the first piece of the last row block, read from the partial records that a split launch
    leaves in its workspace."""
    seq = qs + tq
    plan_parts, per_item, _ = cabi.chunk_plan(tq, qs, seq, prompt)
    all_tiles = (seq + 31) // 32  # the last row block is dense
    pieces = -(-all_tiles // per_item)
    assert plan_parts == parts and pieces > 1 and _is_wide(tq, qs, seq, prompt) == wide
    tiles = -(-all_tiles // pieces)  # the first piece's
    longest_part = -(-tiles // parts)
    print(f"row sum qs={qs} tq={tq} prompt={prompt}: {pieces} pieces, {tiles} tiles, {parts} parts", flush=True)
    q, k, v, bt, scale, p = _inputs(seq, tq, parts, longest_part, 0.0)
    qd, kd, vd, btd = q.to(gpu), k.to(gpu), v.to(gpu), bt.to(gpu)
    out = torch.full_like(qd, float("nan"))
    need = cabi.workspace_size(tq, qs, seq, prompt)
    workspace = torch.zeros(need, dtype=torch.uint8, device=gpu)
    if prompt is None:
        cabi.dense_paged_causal_attention(qd, kd, vd, btd, out, query_start=qs, seq_len=seq, scale=scale,
                                          workspace=workspace)
    else:
        cabi.triangle_paged_sparse_attention(qd, kd, vd, btd, out, query_start=qs, seq_len=seq, prompt_len=prompt,
                                             scale=scale, workspace=workspace)
    torch.cuda.synchronize()
    # records [KV head][item][O 4 x 64 x 64, row max 4 x 64, row sum 4 x 64]; item 0 is the last row block's first piece
    records = workspace[cabi.WORKSPACE_COUNTER_BYTES:].view(torch.float32).view(8, -1, 4 * 64 * 66)
    got = records[:, 0, 4 * 64 * 65:].view(8, 4, 2, 32).double().cpu()  # [KV head][head][half of the keys][row]
    first_half = parts + (16 * tiles - parts) * p
    want = torch.tensor([first_half, 16 * tiles * p], dtype=torch.float64).view(1, 1, 2, 1)
    error = ((got - want).abs() / want).amax(dim=(0, 1, 3))
    bound = (longest_part + 16 + parts) * U + EXP
    print(f"relative error, keys with and without the dominant one: {error.tolist()}, bound {bound:.2e}", flush=True)
    assert (error <= bound).all()


@pytest.mark.gpu
def test_output_of_unsplit_long_items_is_unbiased(gpu):
    """The dense companion's 2048 rows at 32768 keys (KV whole, 961 to 1024 iterations, nothing split): with V
    nonzero on the dominant key alone an output is v / l, and its mean relative error over 2048 rows and the 128
    significands v shows l's error below bf16's rounding (uniform within 2^-8 at most: 2^-8 / sqrt(3) each)."""
    qs, tq = 30720, 2048
    seq = qs + tq
    assert cabi.chunk_plan(tq, qs, seq, None) == (1, 1024, 64) and _is_wide(tq, qs, seq, None) == 1
    values = 1.0 + torch.arange(128, dtype=torch.float32) / 128
    q, k, v, bt, scale, p = _inputs(seq, tq, 1, 1024, values.to(torch.bfloat16))
    qd, kd, vd, btd = q.to(gpu), k.to(gpu), v.to(gpu), bt.to(gpu)
    out = torch.full_like(qd, float("nan"))
    cabi.dense_paged_causal_attention(qd, kd, vd, btd, out, query_start=qs, seq_len=seq, scale=scale)
    torch.cuda.synchronize()
    row_sum = 1.0 + torch.arange(qs, seq, dtype=torch.float64) * p
    want = values.double().view(1, 1, -1) / row_sum.view(-1, 1, 1)
    bias = abs((out.double().cpu() / want - 1.0).mean().item())
    bound = (1024 + 16) * U + EXP + 4 * 2.0 ** -8 / math.sqrt(3 * tq * 128)
    print(f"mean relative error of the outputs {bias:.2e}, bound {bound:.2e}", flush=True)
    assert bias <= bound
