"""Prefill calls of at most 32 tokens (the few-token kernels) against the
oracle, over the edges of their tiling: one token, a full and an overfull
16-token tile, hidden sizes whose 128-column chunks fill the column waves
exactly, partly and over two column groups, unions smaller than a chunk of
four blocks and larger than one batch of tile sums, host copies, duplicates
and invalid ids.  Bars as in the prefill tests: relL2(gpu, exact) <=
max(1e-3, e_ref) per token row, e_ref the fallback restatement's own error."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _u16(t):
    return t.detach().cpu().contiguous().view(torch.int16).numpy().view(np.uint16)


def _np(t):
    return t.detach().cpu().contiguous().numpy()


def _check(orc, L, x, sel, out, what):
    """Every row of out against the oracle over the row's distinct blocks."""
    y = _np(out).astype(np.float64)
    for r in range(x.shape[0]):
        blocks = np.unique(sel[r][(sel[r] >= 0) & (sel[r] < L.NB)])
        gp, ga = orc.gather_rows_blocks(_np(L.gate_packed), _np(L.gate_absmax), blocks, L.H, L.qbs)
        upk, ua = orc.gather_rows_blocks(_np(L.up_packed), _np(L.up_absmax), blocks, L.H, L.qbs)
        dp, da = orc.gather_down_columns(_np(L.down_packed), _np(L.down_absmax), blocks, L.H, L.I, L.qbs)
        local = np.arange(len(blocks), dtype=np.int32).reshape(1, -1)
        ye, yf = orc.sparse_mlp(_u16(x[r:r + 1]), local, gp, ga, upk, ua, dp, da, qbs=L.qbs)
        e_ref = orc.rel_l2(orc.f16_bits_to_f32(yf[0]).astype(np.float64), ye[0])
        e_gpu = orc.rel_l2(y[r], ye[0])
        assert e_gpu <= max(1e-3, e_ref), (what, r, e_gpu, e_ref)


@pytest.mark.parametrize("H,I,M,k,qbs,dq", [
    (256, 256, 1, 1, 64, False),       # 2 chunks of one wave, one block
    (256, 1024, 16, 3, 128, True),
    (1280, 2048, 17, 5, 64, True),     # 10 chunks over 2 column waves, second token tile
    (2304, 2176, 5, 9, 64, False),     # 18 chunks over 4 column waves, 68 blocks
    (5120, 1024, 12, 20, 64, True),    # 40 chunks over 8 column waves
    (9216, 512, 16, 9, 64, True),      # 72 chunks: two column groups
    (16384, 1024, 32, 11, 256, False),  # two token tiles over four column groups
    (512, 32768, 32, 200, 64, True),   # 1024 blocks: several batches of tile sums a workgroup
    (256, 131072, 32, 200, 64, False),  # 4096 blocks, the most: a union of about 3200
    (256, 66560, 9, 700, 64, True),    # 2080 blocks: three a thread of the list, the last threads none
])
def test_few_tokens_match_oracle(gpu, orc, H, I, M, k, qbs, dq):
    from next_step_ai_amd.synth import make_synthetic_layer, synth_normal_f16

    print(f"few tokens H={H} I={I} M={M} k={k} qbs={qbs} dq={dq}", flush=True)
    L = make_synthetic_layer(H=H, I=I, R=16, seed=H + M, device=gpu, qbs=qbs, double_quant=dq)
    x = synth_normal_f16(900 + M, (M, H), 1.0, gpu)
    t = L.slot_table()
    sel = L.router().route(x, k)
    out = t.prefill(x, sel, check=True)
    assert torch.equal(out, t.prefill(x, sel)), "not deterministic"
    if dq:
        assert torch.equal(out, L.slot_table(absmax="f32").prefill(x, sel))
    _check(orc, L, x, _np(sel).astype(np.int64), out, f"H={H} M={M}")


def test_few_tokens_host_copies_duplicates_and_invalid_ids(gpu, orc):
    """Half of the blocks in host copies: the same bits as all resident; a
    repeated id counts once; an id out of range is reported and adds nothing."""
    from next_step_ai_amd.synth import make_synthetic_layer, synth_normal_f16

    H, I, M, k = 1024, 2048, 20, 6
    L = make_synthetic_layer(H=H, I=I, R=16, seed=5, device=gpu, double_quant=True)
    x = synth_normal_f16(6, (M, H), 1.0, gpu)
    sel = _np(L.router().route(x, k)).copy()
    sel[3, 2] = sel[3, 1]
    for absmax in ("dq", "f32"):
        full = L.slot_table(absmax=absmax)
        out = full.prefill(x, torch.from_numpy(sel).to(gpu), check=True)
        resident = torch.arange(0, L.NB, 2, dtype=torch.int32)
        part = L.slot_table(resident_blocks=resident, host_copy=True, absmax=absmax)
        assert torch.equal(part.prefill(x, torch.from_numpy(sel).to(gpu), check=True), out)
    _check(orc, L, x, sel.astype(np.int64), out, "duplicates")
    bad = sel.copy()
    bad[7, 0], bad[8, 5] = -1, L.NB + 3
    with pytest.raises(RuntimeError, match="out of range"):
        full.prefill(x, torch.from_numpy(bad).to(gpu), check=True)
    out_bad = full.prefill(x, torch.from_numpy(bad).to(gpu))
    _check(orc, L, x, bad.astype(np.int64), out_bad, "invalid ids")


def test_few_tokens_do_not_mix(gpu):
    """A token with an infinity leaves every other token's output as it is,
    also where they share blocks."""
    from next_step_ai_amd.synth import make_synthetic_layer, synth_normal_f16

    H, I, M = 1024, 1024, 9
    L = make_synthetic_layer(H=H, I=I, R=16, seed=8, device=gpu)
    t = L.slot_table()
    x = synth_normal_f16(9, (M, H), 1.0, gpu)
    sel = torch.arange(8, dtype=torch.int32, device=gpu).repeat(M, 1)
    sel[4] += 4
    out = t.prefill(x, sel)
    x2 = x.clone()
    x2[4, 100] = float("inf")
    out2 = t.prefill(x2, sel)
    others = [r for r in range(M) if r != 4]
    assert torch.equal(out2[others], out[others])
    assert not torch.isfinite(out2[4].float()).all()


def _swap_selections(rng, NB, M, k, first):
    """M ascending selections of k blocks, row 0 = first."""
    sel = np.stack([np.sort(rng.permutation(NB)[:k]) for _ in range(M)]).astype(np.int32)
    sel[0] = first
    return sel


@pytest.mark.parametrize("H,NB,k,Ms", [
    (1024, 128, 6, (1, 5, 16)),        # M k < 2 NB: one and several groups of blocks
    (4096, 448, 64, (1, 2, 13, 16)),   # on both sides of 2 NB
    (2048, 96, 20, (17, 32)),          # two token tiles
])
def test_few_tokens_independent_of_other_selections(gpu, H, NB, k, Ms):
    """A token's output bits do not depend on what the other tokens select,
    nor (within a token tile) on how many there are: the down sums are exact,
    so a block's place in the union does not matter."""
    from next_step_ai_amd.synth import make_synthetic_layer, synth_normal_f16

    print(f"few tokens, selections H={H} NB={NB} k={k}", flush=True)
    L = make_synthetic_layer(H=H, I=32 * NB, R=16, seed=H + k, device=gpu, double_quant=True)
    t = L.slot_table()
    x = synth_normal_f16(31, (max(Ms), H), 1.0, gpu)
    rng = np.random.default_rng(k)
    first = np.sort(rng.permutation(NB)[:k]).astype(np.int32)
    seen = []
    for M in Ms:
        for _ in range(3):
            sel = torch.from_numpy(_swap_selections(rng, NB, M, k, first)).to(gpu)
            seen.append(t.prefill(x[:M], sel, check=True)[0])
    assert all(torch.equal(s, seen[0]) for s in seen), [int((s != seen[0]).sum()) for s in seen]


@pytest.mark.parametrize("M,k", [(3, 10), (20, 10)])
def test_few_tokens_down_sums_are_exact(gpu, M, k):
    """Two blocks whose contributions cancel (the same weights, the down absmax
    of one negated, about 2^15 each) leave the bits of the call without them:
    the sums hold 2^-31 below 2^20, where fp32 sums would hold 2^-9."""
    from next_step_ai_amd.synth import make_synthetic_layer, synth_normal_f16

    H, NB = 1024, 64
    L = make_synthetic_layer(H=H, I=32 * NB, R=16, seed=77, device=gpu)
    t = L.slot_table(absmax="f32")
    t.down_absmax[11] *= 65536.0
    for name in ("gate_packed", "gate_absmax", "up_packed", "up_absmax", "down_packed"):
        w = getattr(t, name)
        w[40] = w[11]
    t.down_absmax[40] = -t.down_absmax[11]
    x = synth_normal_f16(78, (M, H), 1.0, gpu)
    rng = np.random.default_rng(M)
    others = np.setdiff1d(np.arange(NB), [11, 40])
    pick = np.stack([rng.permutation(others)[: k - 2] for _ in range(M)])
    without = np.sort(np.concatenate([pick, pick[:, :2]], axis=1), axis=1).astype(np.int32)  # repeats count once
    both = np.sort(np.concatenate([pick, np.tile([11, 40], (M, 1))], axis=1), axis=1).astype(np.int32)
    a = t.prefill(x, torch.from_numpy(without).to(gpu), check=True)
    b = t.prefill(x, torch.from_numpy(both).to(gpu), check=True)
    only = both.copy()
    only[:, :] = 11
    big = t.prefill(x, torch.from_numpy(only).to(gpu), check=True).float().abs().amax()
    assert 2.0 ** 10 < float(big) < 2.0 ** 16, float(big)
    assert torch.equal(a, b), int((a != b).sum())


@pytest.mark.parametrize("bad", [float("nan"), float("inf")])
@pytest.mark.parametrize("M", [5, 20])
def test_few_tokens_absmax_not_finite(gpu, M, bad):
    """A down absmax that is NaN or infinite (its zero codes are then NaN
    weights) makes the outputs of the tokens that selected its block NaN, and
    leaves the others."""
    from next_step_ai_amd.synth import make_synthetic_layer, synth_normal_f16

    H, NB, k = 1024, 64, 8
    L = make_synthetic_layer(H=H, I=32 * NB, R=16, seed=79, device=gpu)
    t = L.slot_table(absmax="f32")
    x = synth_normal_f16(80, (M, H), 1.0, gpu)
    rng = np.random.default_rng(M)
    sel = np.stack([np.sort(rng.permutation(NB - 1)[:k]) for _ in range(M)]).astype(np.int32)
    sel[1::2, -1] = NB - 1
    ids = torch.from_numpy(sel).to(gpu)
    out = t.prefill(x, ids)
    t.down_absmax[NB - 1, 3:] = bad
    got = t.prefill(x, ids)
    assert torch.equal(got[0::2], out[0::2]) and torch.equal(got[:, :3], out[:, :3])
    hit = got[1::2, 3:].float()
    assert torch.isnan(hit).all()


def test_few_tokens_no_valid_block(gpu):
    """A call whose every id is out of range: reported, zero outputs."""
    from next_step_ai_amd.synth import make_synthetic_layer, synth_normal_f16

    H, M, k = 512, 3, 2
    L = make_synthetic_layer(H=H, I=1024, R=16, seed=12, device=gpu)
    t = L.slot_table()
    x = synth_normal_f16(13, (M, H), 1.0, gpu)
    sel = torch.tensor([[-1, L.NB]] * M, dtype=torch.int32, device=gpu)
    with pytest.raises(RuntimeError, match="out of range"):
        t.prefill(x, sel, check=True)
    assert not t.prefill(x, sel).any()
