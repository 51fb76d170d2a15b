"""Rows of the thin-tile GEMM equal the general grouped GEMM's, bit for bit.

A call of at most 40 pairs an expert goes to the thin-tile kernel (M tiles of 16, 32 or 64 rows;
blocks of 64 weight rows up to 4 pairs an expert, of 128 above), a larger one to the general kernel
(bf16: to its own), with the same operands in the same order: a row must have the same bits from
both. The experts hold run lengths at the edges of the thin tiles; the same pairs repeated sixteen
times take the general kernel. Widths give odd and
single 64-wide stages and last column blocks that are half empty.
"""
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

RUNS = [1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 100, 0, 2, 7, 0, 3]   # pairs of expert 0, 1, ...
FEW64 = [40, 1, 0, 2, 16, 0, 0, 3, 0, 0, 0, 0, 0, 0, 0, 1]
FEW32 = [1, 2, 0, 15, 16, 17, 0, 3, 0, 0, 4, 0, 2, 0, 0, 1]
FEW16 = [1, 2, 0, 8, 16, 7, 0, 3, 0, 0, 4, 0, 2, 0, 0, 1]
Q = F.QuantSpec


def _spec(H, I, quant, **kw):
    return small(QWEN3_30B_A3B, hidden=H, inter=I, n_experts=len(RUNS), top_k=2, quant=quant, **kw)


# (runs, weight rows of a block without and with the shared expert's pairs)
@pytest.mark.parametrize("runs,block,block_shared", [
    (RUNS, 128, 128), ([min(r, 32) for r in RUNS], 128, 128), ([min(r, 16) for r in RUNS], 128, 128),
    (FEW64, 64, 128), (FEW32, 64, 128), (FEW16, 64, 64)],
    ids=["rows64", "rows32", "rows16", "few64", "few32", "few16"])
@pytest.mark.parametrize("spec", [
    _spec(512, 256, Q(4, 64, "affine")),
    _spec(576, 320, Q(4, 64, "affine", "float16")),
    _spec(64, 64, Q(4, 64, "affine")),
    _spec(512, 384, Q(4, 128, "affine")),
    _spec(320, 192, Q(3, 64, "affine")),
    _spec(192, 320, Q(2, 64, "affine")),
    _spec(512, 128, Q(2, 128, "affine", "float16")),
    _spec(448, 192, Q(6, 64, "affine")),
    _spec(192, 448, Q(8, 64, "affine")),
    _spec(576, 320, Q(4, 32, "mxfp4"), has_bias=True, act="swiglu_clamped", route="topk_softmax"),
    _spec(320, 192, Q(16, 0, "none")),
    _spec(320, 192, Q(4, 64, "affine"), act="silu_mlp"),
    small(E256_SHARED, hidden=512, inter=192, n_experts=len(RUNS), top_k=4, shared_inter=320),
], ids=["4bit", "4bit-f16-odd", "4bit-one-stage", "4bit-g128", "3bit-odd", "2bit-odd", "2bit-g128", "6bit-odd",
        "8bit-odd", "mxfp4-odd", "bf16-odd", "silu-mlp", "shared"])
def test_thin_rows_equal_general_rows(gpu, spec, runs, block, block_shared):
    import torch
    T = max(runs)        # 16, 32 or more tokens: the thin tile heights
    lay = make_layer(spec, seed=41)
    _, _, pool, _ = build_gpu_layer(lay, gpu)
    pool.g2s_device(torch.cuda.current_stream().cuda_stream)
    pool.device.sync()
    x = make_x(T, spec.hidden, seed=42)
    xd = to_dev_bits(x, gpu)
    pexp = np.repeat(np.arange(len(runs), dtype=np.int32), runs)
    ptok = np.concatenate([(np.arange(r) * 3 + e) % T for e, r in enumerate(runs)]).astype(np.int32)
    shared = None
    if spec.shared_inter:
        shared = torch.from_numpy(np.frombuffer(lay.shared, np.uint8).copy()).to(gpu)
        pexp = np.concatenate([pexp, np.full(T, spec.n_experts, np.int32)])
        ptok = np.concatenate([ptok, np.arange(T, dtype=np.int32)])
    n = pexp.size
    print(f"[thin] H={spec.hidden} I={spec.inter} {spec.quant.mode} {spec.quant.bits}-bit pairs={n}", flush=True)

    def run(copies):
        rows = np.arange(n * copies, dtype=np.int32)
        y = torch.full((n * copies, spec.hidden), float("nan"), dtype=torch.bfloat16, device=gpu)
        dev = lambda a: torch.from_numpy(np.ascontiguousarray(np.tile(a, copies))).to(gpu)  # noqa: E731
        ops.forward_pairs(spec, pool, xd, dev(ptok), dev(pexp), torch.from_numpy(rows).to(gpu), y,
                          L.FWD_FORCE_PREFILL, shared=shared)
        torch.cuda.synchronize()
        return bits(y)

    E_ext = spec.n_experts + (1 if shared is not None else 0)
    assert n <= 40 * E_ext < 16 * n
    assert (n <= 4 * E_ext) == ((block_shared if spec.shared_inter else block) == 64)
    thin, general = run(1), run(16)
    for c in range(16):
        part = general[c * n:(c + 1) * n]
        assert np.array_equal(thin, part), f"{int((thin != part).any(-1).sum())} rows differ"
    # the oracle, one routed pair a token: pairs p and p + 1 of equal weight are not needed, the
    # unreduced rows are compared
    routed = np.flatnonzero(pexp < spec.n_experts)
    idx = np.stack([pexp[routed], (pexp[routed] + 1) % spec.n_experts], 1)
    if spec.top_k != 2:
        idx = np.stack([(pexp[routed] + j) % spec.n_experts for j in range(spec.top_k)], 1)
    w = np.full(idx.shape, 1.0 / spec.top_k, np.float32)
    _, yref = oracle.moe_forward(spec, lay.experts, x[ptok[routed]], idx.astype(np.int32), w, want_unreduced=True)
    got = F.bf16_bits_to_f32(thin[routed])
    ref = F.bf16_bits_to_f32(np.ascontiguousarray(yref.reshape(len(routed), spec.top_k, -1)[:, 0]))
    # bf16 weights, activations and rows: unit roundoff 2^-9 each, as in the other layer tests
    assert oracle.rel_l2(got, ref) < 1e-2
    pool.close()
