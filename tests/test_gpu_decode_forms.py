"""A decode step of several tokens gives the same bits whichever of its two forms runs it.

A step of few entries and narrow experts runs as one gate/up and one down launch, a larger one as a
plan and one block per (entry, rows): the same pairs, once as the rows of one call of many pairs
and once as calls of a few pairs each, take the two forms."""
import numpy as np
import pytest

from bigrig_amd import formats as F
from bigrig_amd import layer as ops
from bigrig_amd import lib as L
from bigrig_amd.spec import QWEN3_30B_A3B
from tests.gpu_util import bits, build_gpu_layer, to_dev_bits
from tests.helpers import make_layer, make_x, small

pytestmark = pytest.mark.gpu
Q = F.QuantSpec


@pytest.mark.parametrize("quant", [Q(4, 64, "affine"), Q(3, 64, "affine"), Q(8, 64, "affine", "float16"),
                                   Q(4, 32, "mxfp4"), Q(16, 0, "none")],
                         ids=["4bit", "3bit", "8bit", "mxfp4", "bf16"])
@pytest.mark.parametrize("T,k", [(2, 8), (8, 4), (5, 6), (8, 8)])   # 16, 32, 30 and 64 pairs
def test_forms_agree(gpu, quant, T, k):
    import torch
    spec = small(QWEN3_30B_A3B, hidden=448, inter=320, n_experts=12, top_k=k, quant=quant)
    lay = make_layer(spec, seed=13)
    _, _, pool, _ = build_gpu_layer(lay, gpu)
    pool.g2s_device(torch.cuda.current_stream().cuda_stream)
    pool.device.sync()
    x = to_dev_bits(make_x(T, spec.hidden, seed=14), gpu)
    rng = np.random.default_rng(T * 100 + k)
    pexp = rng.integers(0, 12, T * k).astype(np.int32)          # repeats, within a token too
    ptok = np.repeat(np.arange(T, dtype=np.int32), k)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)   # noqa: E731
    print(f"[forms] T={T} k={k} {quant.mode} {quant.bits}-bit", flush=True)

    def run(step):
        y = torch.full((T * k, spec.hidden), float("nan"), dtype=torch.bfloat16, device=gpu)
        for p in range(0, T * k, step):
            sel = np.arange(p, min(p + step, T * k), dtype=np.int32)
            ops.forward_pairs(spec, pool, x, dev(ptok[sel]), dev(pexp[sel]), dev(sel), y, L.FWD_FORCE_DECODE)
        torch.cuda.synchronize()
        return bits(y)

    whole = run(T * k)
    for step in (7, 31):
        part = run(step)
        assert np.array_equal(whole, part), f"{int((whole != part).any(-1).sum())} rows differ at {step} pairs a call"
    pool.close()
