"""Activations with outliers through the batched layer on the GPU (run with -m gpu).

A block of 32 activations shares its scales (csrc/q6.h), so one value far above
the others may not cost them their bits. One to three columns of every second
block of the normalised input are `ratio` times the others, and every expert's
gate and up weights are zero there; some rows of gate and up make SwiGLU values
about `ratio` times the others, and down is zero there. What comes out then is made
by the outliers' neighbours alone. All tokens go to the same experts, so passes of
one to four row blocks run; the shared expert is MXFP4 with the same plants. Every
call is made twice, the second time with outliers in the odd tokens alone.

Tolerance: against 64 bits an output is two f32 dot products one after another, of
640 and 384 terms. Each rounds by at most 2^-24 of a partial sum, n = 640 or 384
times; independent and uniform they add up to 2^-24 sqrt(n / 3) of the final sum,
8.7e-7 and 6.7e-7, 1.1e-6 together (bf16 pieces, which keep every bit of a value,
gave 1.8e-7 to 8.4e-7 in this test). With five pieces and no further ones the
neighbours of a value 100 times as large were off by 1.7e-6 to 3.6e-6, of 30000 times
by 4e-4 to 1.2e-3."""
import numpy as np
import pytest

from oracle import moe_oracle as O
from oracle import synth
from windlass_amd import hip as H_
from windlass_amd import moe, synthdata

pytestmark = pytest.mark.gpu
H, I, E, K = 640, 384, 16, 2
CFG = dict(hidden=H, moe_inter=I, n_routed_experts=E, n_experts_per_tok=K, n_layers=1, routed_scaling=2.5, rms_eps=1e-5)
SEED = 41
IN_COLS = [c for b in range(0, H // 32, 2) for c in [32 * b + 5, 32 * b + 17, 32 * b + 30][:1 + b % 3]]
MID_COLS = [32 * b + 11 for b in range(0, I // 32, 2)]
BAR = 1.1e-6


def _zero_columns(nib, cols):
    for c in cols:
        nib[:, c // 2] &= np.uint8(0xF0 if c % 2 == 0 else 0x0F)


def _block(e, ratio):
    gw, gs, uw, us, dw, ds = [a.copy() for a in synth.expert_block(H, I, SEED, 0, e)]
    for w in (gw, uw):
        _zero_columns(w, IN_COLS)
    _zero_columns(dw, MID_COLS)
    up = int(round(np.log2(ratio) / 2))  # the product of gate and up
    gs[MID_COLS] += np.uint8(up + 3)     # (silu is g / 2 near zero)
    us[MID_COLS] += np.uint8(up)
    return [gw, gs, uw, us, dw, ds]


def _wide(b):
    return [O.dequant(b[2 * i], b[2 * i + 1]).astype(np.float64) for i in range(3)]


def _ffn(x, w):
    g = x @ w[0].T  # (exp may overflow: the value is 0 then)
    with np.errstate(over="ignore"):
        return (g / (1.0 + np.exp(-g)) * (x @ w[1].T)) @ w[2].T


@pytest.mark.parametrize("ratio", [1, 100, 2000, 30000])
def test_neighbours_of_outliers_keep_their_bits(gpu, ratio):
    ctx = moe.Context(moe.make_config(**CFG))
    ctx.slot_pool_create(E)
    lay = moe.expert_layout(ctx.cfg)
    staging = H_.DeviceBuffer(lay.total)
    blocks = [_block(e, ratio) for e in range(E)]
    for e in range(E):
        staging.upload(np.concatenate([p.reshape(-1) for p in blocks[e]]))
        moe.expert_to_native(ctx.cfg, staging.ptr, ctx.slot_pool_ptr(e))
        H_.synchronize()
        ctx.slot_bind(0, e, ctx.slot_pool_ptr(e))
    shared = _block(0xFFFF, ratio)
    dense = synthdata.dense_layer(H, E, I, SEED, 0)
    bias = dense["bias"].copy()
    bias[[3, 7]] += 10.0
    bufs = [H_.DeviceBuffer.from_array(a) for a in
            (dense["router_w"], bias, np.concatenate([p.reshape(-1) for p in shared]))]
    ctx.set_layer(0, bufs[0].ptr, bufs[1].ptr, None, bufs[2].ptr, moe.SHARED_MXFP4)
    worst = {}
    for T in (3, 16, 20, 40, 64, 70, 150):
        for step in (1, 2):
            hs = np.stack([synth.hidden_state(H, 4100 + T, t) for t in range(T)]).astype(np.float32)
            hs[step - 1::step, IN_COLS] *= np.float32(ratio)
            x, o = H_.DeviceBuffer.from_array(hs), H_.DeviceBuffer(4 * T * H)
            ctx.run_moe_batched(0, T, x.ptr, None, o.ptr)
            ctx.check_error()
            got = o.download(np.float32).reshape(T, H)
            _, ids, wts = ctx.batched_routing(T)
            assert all(sorted(i.tolist()) == [3, 7] for i in ids)
            h64 = hs.astype(np.float64)
            xn = h64 / np.sqrt((h64 * h64).mean(-1, keepdims=True) + CFG["rms_eps"])
            ref = _ffn(xn, _wide(shared))
            for e in (3, 7):
                ref += _ffn(xn, _wide(blocks[e])) * np.where(ids == e, wts, 0).sum(1)[:, None]
            worst[T, step] = max(O.rel_to_scale(ref[t], got[t]) for t in range(T))
    print(f"ratio {ratio}: " + ", ".join(f"T={T}/{n} {w:.1e}" for (T, n), w in worst.items()), flush=True)
    assert max(worst.values()) < BAR, worst
    ctx.close()
