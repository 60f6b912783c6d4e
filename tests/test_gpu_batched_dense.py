"""The dense MLP over many positions on the GPU (run with -m gpu): both batched
entry points against the oracle and the one-position path.

Sizes: positions at the edges of row blocks and passes and past a chunk; hidden of
an odd number of 128-column steps; inter that ends inside a step, a weight
row block and a 16-byte group's neighbour. The residual is added in place and
absent.

Tolerance: an output sums inter products; both sides hold each to three bf16 pieces
or f32 and sum in f32, so their difference stays below 2 * 2^-24 * sqrt(inter)
of the row's scale for independent roundings, 4e-6 at 1096 (twice, for the two
projections): the 1e-5 bar of the one-position tests."""
import numpy as np
import pytest

from oracle import attention as A
from oracle import moe_oracle as O
from oracle import synth
from windlass_amd import hip as H_, moe, synthdata
from windlass_amd.model import DeviceModel

pytestmark = pytest.mark.gpu
TOL = 1e-5


@pytest.mark.parametrize("shape", [(384, 264), (640, 1096)])
@pytest.mark.parametrize("T", [2, 15, 17, 33, 49, 64, 65, 100, 513])
def test_dense_batched(gpu, T, shape):
    H, DI = shape
    ctx = moe.Context(moe.make_config(hidden=H, moe_inter=256, n_routed_experts=16, n_experts_per_tok=1, rms_eps=1e-5))
    w = synthdata.dense_mlp(H, DI, 31, 0)
    dev = {k: H_.DeviceBuffer.from_array(v) for k, v in w.items()}
    ctx.set_layer_dense(0, dev["post_ln"].ptr, dev["gate"].ptr, dev["up"].ptr, dev["down"].ptr, DI)
    hs = np.stack([synth.hidden_state(H, 3100, t) for t in range(T)]).astype(np.float32)
    wf = synthdata.as_f32(w)
    ref = A.dense_mlp(hs, wf, dict(rms_eps=1e-5))
    one = H_.DeviceBuffer(4 * H)
    for run in (ctx.run_moe_batched, ctx.run_moe_batched_noalloc):
        d = H_.DeviceBuffer.from_array(hs)
        run(0, T, d.ptr, d.ptr, d.ptr)  # in place, the residual the input
        got = d.download(np.float32).reshape(T, H)
        for t in range(T):
            assert O.rel_to_scale(ref[t] - hs[t], got[t] - hs[t]) < TOL, t
        d = H_.DeviceBuffer.from_array(hs)
        o = H_.DeviceBuffer(4 * T * H)
        run(0, T, d.ptr, None, o.ptr)
        got = o.download(np.float32).reshape(T, H)
        for t in (0, T // 2, T - 1):
            ctx.run_moe_batched(0, 1, d.ptr + 4 * H * t, None, one.ptr)
            assert O.rel_to_scale(one.download(np.float32), got[t]) < TOL, t
    ctx.close()


def _dense(ctx, layer, H, DI, seed, ln=True):
    """Binds synthetic dense weights; the buffers, to be kept."""
    w = synthdata.dense_mlp(H, DI, seed, layer)
    dev = {k: H_.DeviceBuffer.from_array(v) for k, v in w.items()}
    ctx.set_layer_dense(layer, dev["post_ln"].ptr if ln else None, dev["gate"].ptr, dev["up"].ptr, dev["down"].ptr, DI)
    return dev


def _rows(H, T, seed):
    return np.stack([synth.hidden_state(H, seed, t) for t in range(T)]).astype(np.float32)


def test_dense_calls_keep_the_batched_routing_and_allocate_nothing(gpu):
    """A dense call through either entry point leaves what the last MoE call of
    that entry point can still be asked for (its counts, ids, weights and logits),
    and takes no device memory: its scratch comes with the layer. A larger layer
    bound later, a smaller one and a layer without a norm weight run the same way."""
    c = dict(hidden=384, moe_inter=256, n_routed_experts=48, n_experts_per_tok=6, n_shared=1, routed_scaling=2.5,
             rms_eps=1e-5)
    H, T = c["hidden"], 70
    dm = DeviceModel(c, seed=24, n_layers=4)  # layers 1 to 3 bound again below
    keep = [_dense(dm.ctx, 1, H, 1096, 33), _dense(dm.ctx, 2, H, 264, 34), _dense(dm.ctx, 3, H, 2200, 35, ln=False)]
    x = H_.DeviceBuffer.from_array(_rows(H, T, 3300))
    o = H_.DeviceBuffer(4 * T * H)
    for run in (dm.ctx.run_moe_batched, dm.ctx.run_moe_batched_noalloc):
        run(0, T, x.ptr, None, o.ptr)
        dm.ctx.check_error()
        before = (dm.ctx.batched_counts(), *dm.ctx.batched_routing(T))
        free0, _ = H_.mem_info()
        for layer in (1, 2, 3):
            run(layer, T, x.ptr, None, o.ptr)
            H_.synchronize()
        assert H_.mem_info()[0] == free0
        after = (dm.ctx.batched_counts(), *dm.ctx.batched_routing(T))
        assert before[0].sum() == T * c["n_experts_per_tok"]
        for a, b in zip(before, after):
            assert np.array_equal(a, b)
    w = {k: synthdata.as_f32(synthdata.dense_mlp(H, 2200, 35, 3))[k] for k in ("gate", "up", "down")}
    ref = A.dense_mlp(_rows(H, T, 3300), dict(w, post_ln=np.ones(H, np.float32)), dict(rms_eps=1e-5))
    got, hs = o.download(np.float32).reshape(T, H), _rows(H, T, 3300)
    for t in range(T):
        assert O.rel_to_scale(ref[t] - hs[t], got[t]) < TOL, t
    del keep
    dm.close()


def test_both_entry_points_and_graphs_give_the_same_bits(gpu):
    """One call of 513 positions (a chunk of 512 and one more) through either entry
    point, and captured into a graph through either and replayed three times with
    eager work of the program between the replays: the same bits."""
    H, DI, T = 3072, 1024, 513
    ctx = moe.Context(moe.make_config(hidden=H, moe_inter=256, n_routed_experts=16, n_experts_per_tok=1, rms_eps=1e-5))
    keep = _dense(ctx, 0, H, DI, 36)
    x = H_.DeviceBuffer.from_array(_rows(H, T, 3600))
    o = H_.DeviceBuffer(4 * T * H)
    other = H_.DeviceBuffer(4 * 9 * H)
    ctx.run_moe_batched(0, T, x.ptr, x.ptr, o.ptr)
    eager = o.download(np.uint32)
    st = H_.Stream()
    for run in (ctx.run_moe_batched, ctx.run_moe_batched_noalloc):
        o.zero()
        run(0, T, x.ptr, x.ptr, o.ptr)
        assert np.array_equal(o.download(np.uint32), eager)
        g = H_.Graph(st)
        g.begin()
        run(0, T, x.ptr, x.ptr, o.ptr, st.handle)
        g.end()
        for rep in range(3):
            o.zero()
            H_.synchronize()
            g.launch()
            st.synchronize()
            assert np.array_equal(o.download(np.uint32), eager), rep
            run(0, 9, x.ptr, None, other.ptr, st.handle)
            st.synchronize()
        g.destroy()
    del keep
    ctx.close()


def test_values_past_bf16_range(gpu):
    """SwiGLU values that leave the f32 range, or lie between bf16's largest value
    and f32's: the same infinities, NaNs and finite values as one position at a
    time. Planted inner rows: 5 the product of 2^65 and 2^65 (infinite; 0 for a
    negative input), 70 the product 2^127 * 1.998. Down weighs the first with 0 in
    some rows (NaN) and the second with 2^-20."""
    H, DI, T = 384, 264, 20
    ctx = moe.Context(moe.make_config(hidden=H, moe_inter=256, n_routed_experts=16, n_experts_per_tok=1, rms_eps=1e-5))
    w = synthdata.dense_mlp(H, DI, 37, 0)

    def bits(x):
        return (np.asarray(x, np.float32).view(np.uint32) >> 16).astype(np.uint16)

    for m in ("gate", "up"):
        w[m][[5, 70]] = 0
    w["gate"][5, 7] = w["up"][5, 7] = bits(2.0**65)
    w["gate"][70, 9] = bits(2.0**64)
    w["up"][70, 9], w["up"][70, 11] = bits(2.0**63 * 1.9921875), bits(2.0**63 * 1.5 / 256)
    w["down"][:, 5] = bits(1.0)
    w["down"][::3, 5] = 0
    w["down"][1::7, 5] = bits(-1.0)
    w["down"][:, 70] = bits(2.0**-20)
    w["post_ln"][:] = bits(1.0)
    dev = {k: H_.DeviceBuffer.from_array(v) for k, v in w.items()}
    ctx.set_layer_dense(0, dev["post_ln"].ptr, dev["gate"].ptr, dev["up"].ptr, dev["down"].ptr, DI)
    hs = np.ones((T, H), np.float32)  # normalised: 1 - 5e-6
    hs[1::2, 7] = -1.0  # these rows stay finite
    x = H_.DeviceBuffer.from_array(hs)
    o, one = H_.DeviceBuffer(4 * T * H), H_.DeviceBuffer(4 * H)
    ctx.run_moe_batched(0, T, x.ptr, None, o.ptr)
    got = o.download(np.float32).reshape(T, H)
    for t in range(T):
        ctx.run_moe_batched(0, 1, x.ptr + 4 * H * t, None, one.ptr)
        ref = one.download(np.float32)
        fin = np.isfinite(ref)
        assert np.array_equal(np.isnan(ref), np.isnan(got[t])), t
        assert np.array_equal(ref[np.isinf(ref)], got[t][np.isinf(ref)]), t
        assert fin.all() if t % 2 else (not fin.any() and np.isinf(ref).any() and np.isnan(ref).any())
        if fin.any():
            assert np.abs(ref[fin]).min() > 2.0**106
            assert O.rel_to_scale(ref[fin], got[t][fin]) < TOL, t
    ctx.close()
