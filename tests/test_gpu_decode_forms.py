"""A decode step of several tokens gives the same bits whichever of its two forms runs it.

A step of few entries and narrow experts runs as one gate/up and one down launch, a larger one as a
plan and one block per (entry, rows), then the combine. The same pairs, once as the rows of one call
of many pairs and once as calls of a few pairs each, take the two forms; so do the tokens of a whole
block (ranking, the shared expert's group, the weighted combine), once all together and once fewer at
a time. Every call is far enough from the line between the forms (32 entries, or 20 M weights of a
projection over the entries from 18 of them on, in every format) to be on the side it states."""
import numpy as np
import pytest

import oracle
from bigrig_amd import formats as F
from bigrig_amd import layer as ops
from bigrig_amd import lib as L
from bigrig_amd.spec import E256_SHARED, QWEN3_30B_A3B
from tests.gpu_util import bits, build_gpu_layer, to_dev_bits
from tests.helpers import make_layer, make_x, small

pytestmark = pytest.mark.gpu
Q = F.QuantSpec
QUANTS = pytest.mark.parametrize("quant", [Q(4, 64, "affine"), Q(3, 64, "affine"), Q(8, 64, "affine", "float16"),
                                           Q(4, 32, "mxfp4"), Q(16, 0, "none")],
                                 ids=["4bit", "3bit", "8bit", "mxfp4", "bf16"])


def _per_entry(spec, entries):
    """Whether a step of several tokens with this many entries runs per entry; None near the line."""
    weights = entries * spec.hidden * max(spec.inter, spec.shared_inter)
    if entries >= 32 or (entries >= 18 and weights >= 20e6):
        return True
    return False if weights < 20e6 else None


@QUANTS
@pytest.mark.parametrize("T,k,H,I", [(8, 4, 448, 320), (8, 8, 448, 320),       # 32 and 64 entries
                                     (3, 6, 2048, 768)])                       # 18, 28 M weights
def test_forms_agree(gpu, quant, T, k, H, I):
    import torch
    spec = small(QWEN3_30B_A3B, hidden=H, inter=I, n_experts=12, top_k=k, quant=quant)
    lay = make_layer(spec, seed=13, bank=5)
    _, _, pool, _ = build_gpu_layer(lay, gpu)
    pool.g2s_device(torch.cuda.current_stream().cuda_stream)
    pool.device.sync()
    xb = make_x(T, spec.hidden, seed=14)
    x = to_dev_bits(xb, gpu)
    rng = np.random.default_rng(T * 100 + k)
    pexp = rng.integers(0, 12, T * k).astype(np.int32)          # repeats, within a token too
    ptok = np.repeat(np.arange(T, dtype=np.int32), k)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)   # noqa: E731
    print(f"[forms] T={T} k={k} {quant.mode} {quant.bits}-bit", flush=True)

    def run(step):
        y = torch.full((T * k, spec.hidden), float("nan"), dtype=torch.bfloat16, device=gpu)
        for p in range(0, T * k, step):
            sel = np.arange(p, min(p + step, T * k), dtype=np.int32)
            assert _per_entry(spec, sel.size) is (step == T * k)
            ops.forward_pairs(spec, pool, x, dev(ptok[sel]), dev(pexp[sel]), dev(sel), y, L.FWD_FORCE_DECODE)
        torch.cuda.synchronize()
        return bits(y)

    whole = run(T * k)
    for step in (7, 12 if T == 3 else 31):
        part = run(step)
        assert np.array_equal(whole, part), f"{int((whole != part).any(-1).sum())} rows differ at {step} pairs a call"
    w = np.full((T, k), 1.0 / k, np.float32)
    _, yref = oracle.moe_forward(spec, lay.experts, xb, pexp.reshape(T, k), w, want_unreduced=True)
    got, want = F.bf16_bits_to_f32(whole), F.bf16_bits_to_f32(yref.reshape(T * k, -1))
    # bf16 activations and rows: unit roundoff 2^-9 each, as in the other layer tests
    assert oracle.rel_l2(got, want) < 1e-2
    pool.close()


@QUANTS
@pytest.mark.parametrize("T,part,k,H,I,sh", [(8, 7, 4, 448, 320, 192), (8, 2, 4, 448, 320, 384),   # 33 against 29 and 9
                                             (3, 2, 6, 2048, 640, 0), (4, 2, 6, 1280, 640, 704)])
def test_blocks_agree(gpu, quant, T, part, k, H, I, sh):
    """The tokens of a block: T at once per entry, `part` at a time in one launch each."""
    import torch
    spec = small(E256_SHARED, hidden=H, inter=I, n_experts=24, top_k=k, quant=quant, shared_inter=sh)
    lay = make_layer(spec, seed=15, bank=5, zipf=0.8)
    _, sw, pool, _ = build_gpu_layer(lay, gpu)
    pool.g2s_device(torch.cuda.current_stream().cuda_stream)
    pool.device.sync()
    xb = make_x(T, H, seed=16)
    router, bias = to_dev_bits(lay.router, gpu), to_dev_bits(lay.bias, gpu)
    sgw = to_dev_bits(lay.sgate_w, gpu) if sh else None
    print(f"[forms] block T={T} {part} at a time k={k} {quant.mode} {quant.bits}-bit", flush=True)

    def run(n):
        res = []
        for t in list(range(0, T - n, n)) + [T - n]:
            assert _per_entry(spec, n * k + (1 if sh else 0)) is (n == T)
            gi = torch.full((n, k), -1, dtype=torch.int32, device=gpu)
            gw = torch.zeros((n, k), dtype=torch.float32, device=gpu)
            out = ops.moe_block(spec, pool, to_dev_bits(xb[t:t + n], gpu), router, bias, sgw, sw.shared,
                                out_idx=gi, out_w=gw, flags=L.FWD_FORCE_DECODE)
            torch.cuda.synchronize()
            res.append((t, bits(out), gi.cpu().numpy(), gw.cpu().numpy().view(np.uint32)))
        return res

    (_, out, idx, w), = run(T)
    for t, o, i, wt in run(part):
        assert np.array_equal(i, idx[t:t + part]) and np.array_equal(wt, w[t:t + part])
        assert np.array_equal(o, out[t:t + part]), f"{int((o != out[t:t + part]).any(-1).sum())} tokens differ from {t}"
    _, oidx, ow, sg = oracle.router(xb, lay.router, False, lay.bias, k, spec.route_mode, lay.sgate_w)
    assert np.array_equal(idx, oidx)
    ref, _ = oracle.moe_forward(spec, lay.experts, xb, oidx, ow, lay.shared, sg)
    assert oracle.rel_l2(F.bf16_bits_to_f32(out), F.bf16_bits_to_f32(ref)) < 1e-2
    pool.close()
