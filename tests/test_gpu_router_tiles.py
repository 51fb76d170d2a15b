"""The router for more than 64 tokens (MFMA tiles; rows of more than 5120 inputs with few experts and
tokens a wave each) ranks every expert as the oracle does, whatever the widths:
partial token and expert tiles, rows that end inside a 512-wide block of lane chains, bf16 and fp32
router weights, a shared gate beside them. top_k is the expert count (at most 64), so the
indices are the order of all logits: any logit off by a bit that changes the order of two shows."""
import numpy as np
import pytest

import oracle
from bigrig_amd import formats as F
from bigrig_amd import layer as ops
from bigrig_amd.spec import E256_SHARED, OLMOE_1B_7B
from tests.gpu_util import to_dev_bits
from tests.helpers import make_x, small

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f32", [False, True], ids=["bf16", "f32"])
@pytest.mark.parametrize("T,H,E", [(65, 64, 16), (80, 512, 15), (81, 576, 17), (129, 1024, 64), (300, 2880, 33),
                                   (97, 8192, 40), (2051, 192, 1), (300, 8192, 64), (129, 5184, 128),
                                  (513, 5184, 9), (512, 5184, 16),
                                   (2100, 576, 64), (1050, 1088, 257)])
def test_full_ranking_matches_oracle(gpu, T, H, E, f32):
    base = E256_SHARED if E == 33 else OLMOE_1B_7B
    spec = small(base, hidden=H, n_experts=E, top_k=min(E, 64), route="topk_softmax", n_group=0, topk_group=0,
                 router_dtype="float32" if f32 else "bfloat16")
    rng = np.random.default_rng(T + H + E)
    wr = rng.standard_normal((E, H), dtype=np.float32) * np.float32(0.02)
    wr[:: 3] *= np.exp2(rng.integers(-8, 8, (wr[::3].shape[0], H))).astype(np.float32)   # uneven terms
    w = wr if f32 else F.f32_to_bf16_bits(wr)
    sgw = F.f32_to_bf16_bits(rng.standard_normal(H, dtype=np.float32) * 0.02) if spec.shared_inter else None
    x = make_x(T, H, seed=T)
    print(f"[router] T={T} H={H} E={E} f32={f32}", flush=True)
    idx, wt, sg = ops.router_topk(spec, to_dev_bits(x, gpu), to_dev_bits(w, gpu), None,
                                  None if sgw is None else to_dev_bits(sgw, gpu))
    _, oidx, ow, osg = oracle.router(x, w, f32, None, spec.top_k, spec.route_mode, sgw)
    assert np.array_equal(idx.cpu().numpy(), oidx)
    np.testing.assert_allclose(wt.cpu().numpy(), ow, rtol=1e-5, atol=1e-7)
    if sgw is not None:
        np.testing.assert_allclose(sg.cpu().numpy(), osg, rtol=1e-5, atol=1e-7)
