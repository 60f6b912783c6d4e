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
