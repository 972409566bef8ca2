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


@pytest.mark.parametrize("H,A,kk,rows,out,dtype", [
    (256, 1, 1, 2, 32, torch.float16),
    (512, 37, 9, 20, 512, torch.float16),   # entries left out, repeated and out of range
    (1280, 20, 20, 3, 1280, torch.float16),
    (2048, 16, 5, 4, 2048, torch.bfloat16),
])
def test_fused_rows_equal_composition(gpu, orc, H, A, kk, rows, out, dtype):
    """The several-row fused call against its parts (output linears, silu
    product, input linear), fp16 inputs bit for bit: masks that are not 0 or 1,
    biases, entries of active_idx left out, repeated and out of range."""
    from next_step_ai_amd import sparse_mlp as sm

    print(f"fused rows H={H} A={A} kk={kk} rows={rows}", flush=True)
    rng = np.random.default_rng(H + A)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)  # noqa: E731
    half = lambda *s: t(rng.standard_normal(s).astype(np.float16))  # noqa: E731

    def nf4(o, i, q):
        p, a = orc.nf4_quantize((rng.standard_normal((o, i)) * 0.02).astype(np.float32), q)
        return t(p), t(a)

    (gp, ga), (up, ua), (dp, da) = nf4(A * 32, H, 64), nf4(A * 32, H, 64), nf4(out, A * 32, 32)
    gb, ub, db = half(A * 32), half(A * 32), half(out)
    code = torch.tensor(orc.nf4_code(), device=gpu)
    idx = np.stack([rng.permutation(A)[:kk] for _ in range(rows)]).astype(np.int32)
    if kk > 3:
        idx[1, :3] = idx[1, 3], -1, A + 5
    idx = t(idx)
    mask = t((rng.integers(0, 4, (rows, A * 32)) / 2).astype(np.float16))
    x = half(rows, H).to(dtype)
    lin = dict(input_dim=H, quant_block_size=64, block_size=32, code=code)
    g = sm.triton_sparse_output_linear_4bit(x.half(), idx, mask, packed_weight=gp, absmax=ga, bias=gb, **lin)
    u = sm.triton_sparse_output_linear_4bit(x.half(), idx, mask, packed_weight=up, absmax=ua, bias=ub, **lin)
    act = torch.empty_like(g)
    from next_step_ai_amd import _lib
    from next_step_ai_amd._runtime import ptr, stream_handle
    _lib.call("nsmlp_silu_mul_f16", ptr(g), ptr(u), ptr(act), g.numel(), stream_handle(gpu))
    ref = sm.triton_sparse_input_linear_4bit(act, idx, packed_weight=dp, absmax=da, code=code, out_features=out,
                                             in_features=A * 32, quant_block_size=32, bias=db, block_size=32)
    y = sm.triton_fused_sparse_mlp_decode_4bit(
        x, idx, mask, gate_packed_weight=gp, gate_absmax=ga, gate_code=code, gate_input_dim=H,
        gate_quant_block_size=64, gate_bias=gb, up_packed_weight=up, up_absmax=ua, up_code=code, up_input_dim=H,
        up_quant_block_size=64, up_bias=ub, down_packed_weight=dp, down_absmax=da, down_code=code,
        down_out_features=out, down_in_features=A * 32, down_quant_block_size=32, down_bias=db, block_size=32)
    assert y.dtype == dtype and torch.equal(y, ref.to(dtype))


@pytest.mark.parametrize("rows", [1, 3])
def test_converted_arguments_keep_their_values(gpu, orc, rows):
    """Arguments of other types (bfloat16 masks and biases, float64 absmax and
    codes) give what the same values of the kernels' types give: every converted
    copy lives until the call is enqueued."""
    from next_step_ai_amd import sparse_mlp as sm

    print(f"converted arguments rows={rows}", flush=True)
    H, A, kk = 512, 16, 6
    rng = np.random.default_rng(rows)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)  # noqa: E731

    def nf4(o, i, q):
        p, a = orc.nf4_quantize((rng.standard_normal((o, i)) * 0.02).astype(np.float32), q)
        return t(p), t(a)

    (gp, ga), (up, ua), (dp, da) = nf4(A * 32, H, 64), nf4(A * 32, H, 64), nf4(H, A * 32, 32)
    biases = [t(rng.standard_normal(n).astype(np.float32)).bfloat16() for n in (A * 32, A * 32, H)]
    code = torch.tensor(orc.nf4_code(), device=gpu)
    idx = t(np.stack([rng.permutation(A)[:kk] for _ in range(rows)]).astype(np.int32))
    mask = t(rng.integers(0, 3, (rows, A * 32)).astype(np.float32) / 2).bfloat16()
    x = t(rng.standard_normal((rows, H)).astype(np.float16))

    def fused(half, wide):
        return sm.triton_fused_sparse_mlp_decode_4bit(
            x, idx, half(mask), gate_packed_weight=gp, gate_absmax=wide(ga), gate_code=wide(code), gate_input_dim=H,
            gate_quant_block_size=64, gate_bias=half(biases[0]), up_packed_weight=up, up_absmax=wide(ua),
            up_code=wide(code), up_input_dim=H, up_quant_block_size=64, up_bias=half(biases[1]),
            down_packed_weight=dp, down_absmax=wide(da), down_code=wide(code), down_out_features=H,
            down_in_features=A * 32, down_quant_block_size=32, down_bias=half(biases[2]), block_size=32)

    def linears(half, wide):
        g = sm.triton_sparse_output_linear_4bit(x, idx, half(mask), packed_weight=gp, absmax=wide(ga), code=wide(code),
                                                input_dim=H, quant_block_size=64, bias=half(biases[0]), block_size=32)
        y = sm.triton_sparse_input_linear_4bit(g, idx, packed_weight=dp, absmax=wide(da), code=wide(code),
                                               out_features=H, in_features=A * 32, quant_block_size=32,
                                               bias=half(biases[2]), block_size=32)
        return torch.cat((g, y), dim=1)

    for call in (fused, linears):
        ref = call(lambda v: v.half(), lambda v: v)
        assert torch.isfinite(ref.float()).all()
        assert torch.equal(call(lambda v: v, lambda v: v.double()), ref), call.__name__


def test_fused_rows_bf16_tokens(gpu, orc):
    """bf16 tokens through the several-row call against float64: fp16 gate, up
    and act (2^-11 each, 2 in the product) and a bf16 result, whose rounding has
    an rms of 2^-9 / sqrt(3) of a value at most: relL2 <= 2e-3, and no further
    off than the three calls it replaces, which hand over bf16."""
    from next_step_ai_amd import sparse_mlp as sm

    H, A, kk, rows = 2048, 16, 5, 4
    rng = np.random.default_rng(77)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)  # noqa: E731

    def nf4(o, i, q):
        p, a = orc.nf4_quantize((rng.standard_normal((o, i)) * 0.02).astype(np.float32), q)
        return t(p), t(a), orc.nf4_dequant(p, a, o * i, q).reshape(o, i).astype(np.float64)

    (gp, ga, wg), (up, ua, wu), (dp, da, wd) = nf4(A * 32, H, 64), nf4(A * 32, H, 64), nf4(H, A * 32, 32)
    code = torch.tensor(orc.nf4_code(), device=gpu)
    idx = np.stack([rng.permutation(A)[:kk] for _ in range(rows)]).astype(np.int32)
    mask = torch.ones((rows, A * 32), dtype=torch.float16, device=gpu)
    x = t(rng.standard_normal((rows, H)).astype(np.float32)).bfloat16()
    lin = dict(input_dim=H, quant_block_size=64, block_size=32, code=code, bias=None)
    g = sm.triton_sparse_output_linear_4bit(x, t(idx), mask, packed_weight=gp, absmax=ga, **lin)
    u = sm.triton_sparse_output_linear_4bit(x, t(idx), mask, packed_weight=up, absmax=ua, **lin)
    assert g.dtype == torch.bfloat16
    act = (torch.nn.functional.silu(g.float()) * u.float()).half().bfloat16()
    parts = sm.triton_sparse_input_linear_4bit(act, t(idx), packed_weight=dp, absmax=da, code=code, out_features=H,
                                               in_features=A * 32, quant_block_size=32, bias=None, block_size=32)
    y = sm.triton_fused_sparse_mlp_decode_4bit(
        x, t(idx), mask, gate_packed_weight=gp, gate_absmax=ga, gate_code=code, gate_input_dim=H,
        gate_quant_block_size=64, gate_bias=None, up_packed_weight=up, up_absmax=ua, up_code=code, up_input_dim=H,
        up_quant_block_size=64, up_bias=None, down_packed_weight=dp, down_absmax=da, down_code=code,
        down_out_features=H, down_in_features=A * 32, down_quant_block_size=32, down_bias=None, block_size=32)
    xd = x.float().cpu().numpy().astype(np.float64)
    gd, ud = xd @ wg.T, xd @ wu.T
    live = np.zeros((rows, A * 32))
    for r in range(rows):
        for b in idx[r]:
            live[r, b * 32:(b + 1) * 32] = 1.0
    ref = (gd / (1.0 + np.exp(-gd)) * ud * live) @ wd.T
    err = [orc.rel_l2(v.float().cpu().numpy().astype(np.float64), ref) for v in (y, parts)]
    print(f"bf16 rows: fused {err[0]:.2e}, parts {err[1]:.2e}", flush=True)
    assert y.dtype == torch.bfloat16 and err[0] <= 2e-3 and err[0] <= err[1]
