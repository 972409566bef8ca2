"""The sparse input linear at the edges of its work split (64 rows a
workgroup, an eighth of the active slots a wave, 8 slots a batch) against
float64 sums.  Bar: |y - exact| <= 2^-11 |exact| + (n + 2) 2^-23 sum |w x|, the
fp16 rounding of the result and fp32 sums of n products (two roundings each)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("out,in_f,kk,bs,qbs,rows", [
    (1, 32, 1, 32, 32, 1),        # one row, one slot: seven idle waves
    (64, 256, 8, 32, 32, 2),      # one slot a wave
    (65, 2080, 65, 32, 32, 3),    # a workgroup of one row, a second batch of one slot
    (193, 4096, 70, 32, 64, 5),   # entries left out, one repeated
    (130, 2048, 5, 256, 64, 4),   # blocks of 8 slots, a wave's range cutting them
])
def test_input_linear_splits(gpu, orc, out, in_f, kk, bs, qbs, rows):
    from next_step_ai_amd.sparse_mlp import triton_sparse_input_linear_4bit

    print(f"input linear out={out} in={in_f} kk={kk} bs={bs}", flush=True)
    rng = np.random.default_rng(out + in_f)
    w = (rng.standard_normal((out, in_f)) * 0.02).astype(np.float32)
    packed, absmax = orc.nf4_quantize(w, qbs)
    wd = orc.nf4_dequant(packed, absmax, out * in_f, qbs).reshape(out, in_f).astype(np.float64)
    x = rng.standard_normal((rows, in_f)).astype(np.float16)
    blocks = in_f // bs
    idx = np.stack([rng.permutation(np.arange(max(blocks, kk)))[:kk] for _ in range(rows)]).astype(np.int32)
    if kk > 3:
        idx[0, 1], idx[0, 2] = -1, idx[0, 0]  # left out; counted twice
    bias = rng.standard_normal(out).astype(np.float16)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)  # noqa: E731
    y = triton_sparse_input_linear_4bit(
        t(x), t(idx), packed_weight=t(packed), absmax=t(absmax), code=torch.tensor(orc.nf4_code(), device=gpu),
        out_features=out, in_features=in_f, quant_block_size=qbs, bias=t(bias), block_size=bs).cpu().numpy()
    for r in range(rows):
        cnt = np.zeros(in_f)
        for b in idx[r]:
            if 0 <= b < blocks:
                cnt[b * bs:(b + 1) * bs] += 1
        prod = wd * (x[r].astype(np.float64) * cnt)
        exact = prod.sum(axis=1) + bias.astype(np.float64)
        mag = np.abs(prod).sum(axis=1) + np.abs(bias.astype(np.float64))
        bar = 2.0 ** -11 * np.abs(exact) + (kk * bs + 2) * 2.0 ** -23 * mag + 2.0 ** -24
        assert np.all(np.abs(y[r].astype(np.float64) - exact) <= bar), r
