"""The batched layer's passes at their edges on the GPU (run with -m gpu).

An expert's tokens are cut into row blocks of 16 and those into passes of at
most four; calls of at most 2048 entries group them by expert inside
the gate/up kernel, larger ones in kernels of their own. A bias gives three
experts every token, so their passes end at, before and after a block and a
pass; the other three choices spread thinly over the rest. Every token is
compared with the single-token decode path, which computes from f32 rows, and
the first and last with the oracle.

Tolerance: an output is a sum of K + 1 = 7 rows of f32 dot products over at most
640 columns; both sides round each product's sum within 2^-24 sqrt(640) of the
row's scale, 7 rows in two projections stay below 14 * 26 * 6e-8 = 2.2e-5 in the
worst case and, the errors being independent, below 1e-5 in practice: the bar of
the other batched tests."""
import numpy as np
import pytest

from oracle import moe_oracle as O
from .test_gpu_batched import SMALL, TOL, _batched, _decode, _tokens
from windlass_amd.model import DeviceModel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [dict(hidden=384, moe_inter=256), dict(hidden=640, moe_inter=384)],
                         ids=["odd-k-tiles", "ragged-units"])
@pytest.mark.parametrize("T", [15, 16, 17, 32, 33, 49, 64, 65, 80, 81, 85, 86, 161])
def test_passes_at_block_edges(gpu, T, shape):
    c = dict(SMALL, **shape)
    H, E = c["hidden"], c["n_routed_experts"]
    off = np.zeros(E, np.float32)
    off[[3, 7, 11]] = 5.0
    dm = DeviceModel(c, seed=21, n_layers=1, bias_offset=off)
    hs = _tokens(H, T, 2100 + T)
    out = _batched(dm, hs)
    assert np.array_equal(out, _batched(dm, hs))
    counts = dm.ctx.batched_counts()
    assert all(counts[e] == T for e in (3, 7, 11)) and counts.sum() == T * c["n_experts_per_tok"]
    src = O.ExpertSource(H, c["moe_inter"], 21)
    for t in range(T):
        assert O.rel_to_scale(_decode(dm, hs[t]), out[t]) < TOL, t
        if t in (0, T - 1):
            assert O.rel_to_scale(O.moe_layer(hs[t], dm.dense[0], src, 0, c)["out"], out[t]) < TOL, t
    dm.close()


@pytest.mark.parametrize("E,K,T", [(48, 1, 512), (48, 1, 513), (48, 1, 2048), (48, 1, 2049), (192, 1, 2048), (208, 1, 2048),
                                   (624, 1, 512), (640, 1, 512), (48, 8, 64), (48, 8, 256), (16, 16, 32), (624, 2, 31)])
def test_entries_grouped_by_expert(gpu, E, K, T):
    """Up to 2048 entries are grouped inside the gate/up kernel (one to four a thread;
    a bit per token and expert, 48 KB of them), more of them, more bits, or more
    experts than leave room for the tokens, by kernels of their own. Hidden 256 and inter 128: a unit is one step. Counts equal the ids'; every
    seventh token and the last agree with the decode path."""
    c = dict(SMALL, hidden=256, moe_inter=128, n_routed_experts=E, n_experts_per_tok=K)
    dm = DeviceModel(c, seed=22, n_layers=1)
    hs = _tokens(256, T, 2200 + T)
    out = _batched(dm, hs)
    _, ids, _ = dm.ctx.batched_routing(T)
    assert np.array_equal(dm.ctx.batched_counts(), np.bincount(ids.reshape(-1), minlength=E))
    for t in [*range(0, T, 7), T - 1]:
        assert O.rel_to_scale(_decode(dm, hs[t]), out[t]) < TOL, t
    dm.close()
