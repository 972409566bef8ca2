"""Decode over hidden sizes that do not fill 2048-column splits, and over
row-major gathered down weights, at the edges of their tiling.  Bars as in the
decode tests: relL2(gpu, exact) <= max(1e-3, e_ref), e_ref the error of the
oracle's fp16 fallback restatement; equalities are exact."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _u16(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def _np(t):
    return t.detach().cpu().contiguous().numpy()


def _gather(orc, L, blocks):
    gp, ga = orc.gather_rows_blocks(_np(L.gate_packed), _np(L.gate_absmax), blocks, L.H, L.qbs)
    upk, ua = orc.gather_rows_blocks(_np(L.up_packed), _np(L.up_absmax), blocks, L.H, L.qbs)
    dp, da = orc.gather_down_columns(_np(L.down_packed), _np(L.down_absmax), blocks, L.H, L.I, L.qbs)
    return gp, ga, upk, ua, dp, da


@pytest.mark.parametrize("H,I,k,qbs", [
    (256, 512, 1, 64),       # 8 lanes of one split
    (1280, 2048, 7, 32),     # 40 lanes; absmax2 blocks straddled
    (2304, 4096, 61, 128),   # two splits, the second of 8 lanes
    (5120, 1024, 32, 64),    # three splits: two waves idle
    (6144, 2048, 33, 64),    # three whole splits
    (9472, 1024, 9, 256),    # five splits, one item a round
    (14336, 1024, 32, 64),   # seven whole splits, every block
    (16128, 512, 5, 64),     # eight splits, the last 1792 columns
    (1280, 67200, 9, 64),    # 2100 blocks: the selection takes eight scores a thread
    (10240, 67584, 3, 128),  # the same over five splits
])
def test_decode_hidden_sizes_match_oracle(gpu, orc, H, I, k, qbs):
    from next_step_ai_amd.synth import make_synthetic_layer

    print(f"decode H={H} I={I} k={k} qbs={qbs}", flush=True)
    L = make_synthetic_layer(H=H, I=I, R=16, seed=H + k, device=gpu, qbs=qbs, double_quant=True)
    out, sel = L.layer(k, absmax="dq").forward(L.x)
    out_f, sel_f = L.layer(k, absmax="f32").forward(L.x)
    assert torch.equal(sel, sel_f) and torch.equal(out, out_f)
    _, _, sel_o = orc.route(_u16(L.x), _u16(L.enc_w), _u16(L.enc_b), _u16(L.score_w), _u16(L.score_b), k)
    blocks = np.sort(sel_o).astype(np.int64)
    assert np.array_equal(_np(sel).astype(np.int64), blocks)
    ye, yf = orc.sparse_mlp(_u16(L.x).reshape(1, H), np.arange(k, dtype=np.int32).reshape(1, k),
                            *_gather(orc, L, blocks), qbs=qbs)
    e_ref = orc.rel_l2(orc.f16_bits_to_f32(yf[0]).astype(np.float64), ye[0])
    assert orc.rel_l2(_np(out).astype(np.float64), ye[0]) <= max(1e-3, e_ref)
    # an unavailable block adds nothing, host copies give the same bits
    half = L.slot_table(resident_blocks=torch.arange(0, L.NB, 2, dtype=torch.int32), host_copy=True, absmax="dq")
    assert torch.equal(half.decode(L.x, sel), out)


@pytest.mark.parametrize("H,A,kk", [
    (256, 2, 1),
    (256, 37, 37),      # four rows of 64, one wave's blocks cut over block groups
    (2048, 48, 48),
    (1280, 130, 97),
    (4096, 300, 300),   # tiles of a wave ending in 1 to 3 blocks
    (8192, 300, 290),   # two block groups
    (16384, 208, 203),  # one block group: the workgroup writes the output, a wave's last tile is short
    (16384, 512, 512),  # the most blocks that one group's activations hold
    (16384, 520, 515),  # more: the two-launch kernels, which read the row-major weight directly
])
def test_gathered_down_equals_slot_path(gpu, orc, H, A, kk):
    """Row-major gathered blocks in any order, with entries left out (-1):
    the bits of the slot-table decode over the same blocks in that order."""
    from next_step_ai_amd.sparse_mlp import triton_fused_sparse_mlp_decode_4bit
    from next_step_ai_amd.synth import make_synthetic_layer

    print(f"gathered H={H} A={A} kk={kk}", flush=True)
    I = 32 * ((A + 3) // 4 * 4)
    L = make_synthetic_layer(H=H, I=I, R=16, seed=A + kk, device=gpu)
    gp, ga, upk, ua, dp, da = _gather(orc, L, np.arange(A, dtype=np.int64))
    rng = np.random.default_rng(kk)
    idx = rng.permutation(A)[:kk].astype(np.int32)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu).reshape(-1)  # noqa: E731
    code = torch.tensor(orc.nf4_code(), device=gpu)

    def fused(ids):
        return triton_fused_sparse_mlp_decode_4bit(
            L.x.reshape(1, H), t(ids).reshape(1, -1), torch.ones((1, A * 32), dtype=torch.float16, device=gpu),
            gate_packed_weight=t(gp), gate_absmax=t(ga), gate_code=code, gate_input_dim=H, gate_quant_block_size=64,
            gate_bias=None, up_packed_weight=t(upk), up_absmax=t(ua), up_code=code, up_input_dim=H,
            up_quant_block_size=64, up_bias=None, down_packed_weight=t(dp), down_absmax=t(da), down_code=code,
            down_out_features=H, down_in_features=A * 32, down_quant_block_size=32, down_bias=None,
            block_size=32).reshape(-1)

    assert torch.equal(fused(idx), L.slot_table().decode(L.x, t(idx)))
    if kk > 2:
        holes = idx.copy()
        holes[1::3] = -1
        kept = L.slot_table(resident_blocks=t(idx[[i for i in range(kk) if i % 3 != 1]]))
        assert torch.equal(fused(holes), kept.decode(L.x, t(idx)))


@pytest.mark.parametrize("H,A,kk", [(256, 3, 2), (1280, 40, 33), (5120, 24, 17), (6144, 9, 9), (16384, 20, 13)])
def test_gathered_biases_and_masks(gpu, orc, H, A, kk):
    """Gate, up and down biases and a mask that is not 0 or 1 in the one-row
    fused call, hidden sizes that fill their splits and that do not, against
    float64: relL2 <= 1e-3 (fp16 activations and result)."""
    from next_step_ai_amd.sparse_mlp import triton_fused_sparse_mlp_decode_4bit

    print(f"biases and masks H={H} A={A} kk={kk}", flush=True)
    rng = np.random.default_rng(H + A)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)  # noqa: E731

    def nf4(o, i, q):
        p, a = orc.nf4_quantize((rng.standard_normal((o, i)) * 0.02).astype(np.float32), q)
        return t(p), t(a), orc.nf4_dequant(p, a, o * i, q).reshape(o, i).astype(np.float64)

    (gp, ga, wg), (up, ua, wu), (dp, da, wd) = nf4(A * 32, H, 64), nf4(A * 32, H, 64), nf4(H, A * 32, 32)
    gb, ub, db = (rng.standard_normal(n).astype(np.float16) for n in (A * 32, A * 32, H))
    mask = (rng.integers(0, 4, (1, A * 32)) / 2).astype(np.float16)
    x = rng.standard_normal((1, H)).astype(np.float16)
    idx = np.sort(rng.permutation(A)[:kk]).astype(np.int32)
    code = torch.tensor(orc.nf4_code(), device=gpu)
    y = triton_fused_sparse_mlp_decode_4bit(
        t(x), t(idx).reshape(1, -1), t(mask), gate_packed_weight=gp, gate_absmax=ga, gate_code=code, gate_input_dim=H,
        gate_quant_block_size=64, gate_bias=t(gb), up_packed_weight=up, up_absmax=ua, up_code=code, up_input_dim=H,
        up_quant_block_size=64, up_bias=t(ub), down_packed_weight=dp, down_absmax=da, down_code=code,
        down_out_features=H, down_in_features=A * 32, down_quant_block_size=32, down_bias=t(db), block_size=32)
    m = mask[0].astype(np.float64)
    xd = x[0].astype(np.float64)
    g, u = (wg @ xd + gb) * m, (wu @ xd + ub) * m
    act = g / (1.0 + np.exp(-g)) * u
    live = np.zeros(A * 32)
    for b in idx:
        live[b * 32:(b + 1) * 32] = 1.0
    ref = wd @ (act * live) + db
    assert orc.rel_l2(_np(y).reshape(-1).astype(np.float64), ref) <= 1e-3
