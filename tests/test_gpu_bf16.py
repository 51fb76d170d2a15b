"""Unquantized bf16 experts (the mx.gather_mm branch of StreamingSwitchGLU._proj,
bigrig_engine/stream.py:1626-1628; layers whose tensors carry no scales, direct.py:110-142) on
the GPU: the dequant hook returns the weights bit for bit; decode and prefill layers against the
oracle and the float64 truth (a shared expert, biases, a two-layer expert, a partial feature
tile); the whole block with its routing bit-exact and the same bits as router + operator; a
bounded pool bit-identical to full residency; a bf16 checkpoint served through a bounded pool.
The full-size Qwen3-30B-A3B-bf16 layer runs in test_gpu_full_size.py."""
from dataclasses import replace

import numpy as np
import pytest

import oracle
from bigrig_amd import formats as F
from bigrig_amd import layer as ops
from bigrig_amd import lib as L
from bigrig_amd.spec import E256_SHARED, QWEN3_30B_A3B
from tests.gpu_util import bits, build_gpu_layer, bytes_dev, to_dev_bits
from tests.helpers import make_layer, make_x, small

pytestmark = pytest.mark.gpu

TOL = 1e-2
QN = F.QuantSpec(16, 0, "none")
SPECS = {
    "qwen3": small(QWEN3_30B_A3B, hidden=512, inter=320, n_experts=16, top_k=4, quant=QN),
    "shared-bias": small(E256_SHARED, hidden=576, inter=256, n_experts=16, top_k=4, shared_inter=384,
                         quant=QN, has_bias=True),
    "mlp": small(QWEN3_30B_A3B, hidden=512, inter=320, n_experts=16, top_k=4, quant=QN, act="silu_mlp"),
}


@pytest.mark.parametrize("name", list(SPECS))
def test_bf16_dequant_is_the_weights(gpu, name):
    spec = SPECS[name]
    lay = make_layer(spec, seed=850)
    for e in (0, spec.n_experts - 1):
        dev = bytes_dev(lay.experts[e], gpu)
        for p in (0, 2) if spec.act == "silu_mlp" else (0, 1, 2):
            got = ops.dequant(spec, dev, p).cpu().numpy()
            want = oracle.dequant(spec, lay.experts[e], p)
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (e, p)


def _check(lay, moe, T, seed, f64=True):
    import torch
    spec = lay.spec
    x = make_x(T, spec.hidden, seed=seed)
    out = moe(to_dev_bits(x, moe.router_w.device))
    torch.cuda.synchronize()
    _, idx, w, sg = oracle.router(x, lay.router, spec.router_dtype == "float32", lay.bias,
                                  spec.top_k, spec.route_mode, lay.sgate_w)
    ref, _ = oracle.moe_forward(spec, lay.experts, x, idx, w, lay.shared, sg)
    got = F.bf16_bits_to_f32(bits(out))
    r = oracle.rel_l2(got, F.bf16_bits_to_f32(ref))
    assert r < TOL, f"rel L2 vs C oracle {r:.3e}"
    if f64:
        truth, _ = oracle.moe_forward_f64(spec, lay.experts, x, idx, w, lay.shared, sg)
        assert oracle.rel_l2(got, truth) < TOL
    return bits(out)


@pytest.mark.parametrize("name", list(SPECS))
@pytest.mark.parametrize("T", [1, 3, 8, 9, 64, 300])
def test_bf16_layer(gpu, name, T):
    spec = SPECS[name]
    lay = make_layer(spec, seed=860, zipf=0.9)
    moe, _, pool, _ = build_gpu_layer(lay, gpu)
    print(f"[bf16] layer {name} T={T}", flush=True)
    _check(lay, moe, T, seed=8600 + T, f64=T <= 64)
    pool.close()


@pytest.mark.parametrize("T", [1, 8, 40])
def test_bf16_block(gpu, T):
    """The whole block (routing ranked in the decode kernel): routing bit-exact, output within
    tolerance, and the same bits as router + operator through the separate entry points."""
    import torch
    spec = SPECS["shared-bias"]
    lay = make_layer(spec, seed=870, zipf=0.9)
    _, sw, pool, _ = build_gpu_layer(lay, gpu)
    pool.g2s_device(torch.cuda.current_stream().cuda_stream)
    x = make_x(T, spec.hidden, seed=8700 + T)
    xd = to_dev_bits(x, gpu)
    router = to_dev_bits(lay.router, gpu)
    bias = None if lay.bias is None else to_dev_bits(lay.bias, gpu)
    sgw = to_dev_bits(lay.sgate_w, gpu)
    print(f"[bf16] block T={T}", flush=True)
    gi = torch.full((T, spec.top_k), -1, dtype=torch.int32, device=gpu)
    out = ops.moe_block(spec, pool, xd, router, bias, sgw, sw.shared, out_idx=gi,
                        flags=ops.path_flag(T, spec.top_k))
    torch.cuda.synchronize()
    _, idx, w, sg = oracle.router(x, lay.router, False, lay.bias, spec.top_k, spec.route_mode,
                                  lay.sgate_w)
    assert np.array_equal(gi.cpu().numpy(), idx)
    ref, _ = oracle.moe_forward(spec, lay.experts, x, idx, w, lay.shared, sg)
    assert oracle.rel_l2(F.bf16_bits_to_f32(bits(out)), F.bf16_bits_to_f32(ref)) < TOL
    moe = ops.MoELayer(spec, router, sw, router_bias=bias, shared_gate_w=sgw)
    sw._sync_free = False
    out2 = moe(xd)
    torch.cuda.synchronize()
    assert np.array_equal(bits(out2), bits(out))
    pool.close()


@pytest.mark.parametrize("T,C,steps", [(1, 6, 16), (40, 8, 3)], ids=["decode-C6", "spans-C8"])
def test_bf16_bounded_pool_bit_identical(gpu, T, C, steps):
    import torch
    spec = SPECS["qwen3"]
    lay = make_layer(spec, seed=880, zipf=0.8)
    xs = [make_x(T, spec.hidden, seed=8800 + i) for i in range(steps)]
    res = {}
    for cap in (spec.n_experts, C):
        moe, sw, pool, _ = build_gpu_layer(lay, gpu, capacity=cap)
        print(f"[bf16] bounded pool C={cap} T={T}", flush=True)
        outs = [moe(to_dev_bits(x, gpu)) for x in xs]
        torch.cuda.synchronize()
        res[cap] = [bits(o) for o in outs]
        if cap == C:
            assert pool.evicts > 0
        pool.close()
    for a, b in zip(res[spec.n_experts], res[C]):
        assert np.array_equal(a, b)


def test_bf16_checkpoint_bounded_pool(gpu, tmp_path):
    """A bf16 MLX checkpoint (weights without scales) read into the pinned host store and
    served by a 6-slot pool: routing bit-exact and outputs within 1e-2 of the oracle on the
    experts read back from the shards."""
    from bigrig_amd import checkpoint as CK
    from bigrig_amd.layer import MoELayer, StreamingSwitchGLU
    from bigrig_amd.pool import ExpertPool, HostStore, PinnedFetcher
    from tests.ckpt_util import make_checkpoint
    H, I, E, C = 512, 256, 16, 6
    cfg = {"model_type": "qwen3_moe", "num_experts_per_tok": 4, "norm_topk_prob": True}
    d = str(tmp_path / "ckpt_bf16")
    make_checkpoint(d, {0: (H, I, E, QN, False)}, config=cfg, shards=2, seed=9)
    man = CK.expert_manifest(d)
    spec = CK.layer_spec(man, 0)
    assert spec.quant == QN and spec.bytes_per_expert == 3 * H * I * 2
    store = HostStore.from_checkpoint(man)
    experts = [CK.read_expert(man, 0, e) for e in range(E)]
    rng = np.random.default_rng(19)
    router = F.f32_to_bf16_bits(rng.standard_normal((E, H), dtype=np.float32) * 0.02)
    pool = ExpertPool(0, spec, C).build()
    moe = MoELayer(spec, to_dev_bits(router, gpu), StreamingSwitchGLU(pool, PinnedFetcher(store)))
    for T in (1, 7, 40):
        print(f"[bf16 checkpoint] H={H} I={I} E={E} C={C} T={T}", flush=True)
        x = make_x(T, H, seed=410 + T)
        _, idx, w, _ = oracle.router(x, router, False, None, spec.top_k, spec.route_mode)
        out = moe(to_dev_bits(x, gpu))
        ref, _ = oracle.moe_forward(spec, experts, x, idx, w)
        r = oracle.rel_l2(F.bf16_bits_to_f32(bits(out)), F.bf16_bits_to_f32(ref))
        assert r < TOL, f"T={T}: rel L2 {r:.3e}"
    assert pool.admits > C
    pool.close()


def _bf16_copy(lay):
    """The layer with its MXFP4 experts' weights, which bf16 holds exactly, unquantized."""
    spec = lay.spec
    wide = replace(spec, quant=QN)
    def conv(blob):
        sp = spec.expert_spec()
        arr = F.split_expert(blob, sp)
        out = b""
        for p in sp:
            w = F.dequantize_projection(arr, p, spec.quant)
            b = F.f32_to_bf16_bits(w)
            assert np.array_equal(F.bf16_bits_to_f32(b), w)
            out += b.tobytes()
            if (p, "bias") in arr:
                out += np.ascontiguousarray(arr[(p, "bias")]).tobytes()
        assert len(out) == wide.bytes_per_expert
        return out
    return replace(lay, spec=wide, experts=[conv(e) for e in lay.experts])


TALL_RUNS = [700, 513, 512, 511, 300, 257, 256, 255, 129, 128, 127, 65, 64, 33, 0, 1] + 112 * [25]   # to 256 rows
DENSE_RUNS = [300, 256, 257, 129, 128, 127, 65, 64, 33, 32, 31, 1, 0, 7, 100, 200]                  # to 128 rows
THIN_RUNS = [1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 100, 0, 2, 7, 0, 3]               # 64-row tiles, 128-row blocks
FEW_RUNS = [1, 15, 16, 17, 2, 0, 3, 0, 1, 0, 0, 2, 0, 0, 0, 1]                        # 64-row blocks


@pytest.mark.parametrize("runs", [TALL_RUNS, DENSE_RUNS, THIN_RUNS, FEW_RUNS, [min(r, 16) for r in FEW_RUNS]],
                         ids=["tall", "dense", "thin", "thin-few", "thin-few16"])
@pytest.mark.parametrize("kw", [dict(hidden=1536, inter=768), dict(hidden=576, inter=192, has_bias=True,
                                                                 act="swiglu_clamped"),
                                dict(hidden=64, inter=64), dict(hidden=320, inter=448, act="silu_mlp")],
                         ids=["1536x768", "576x192-clamped", "64x64", "320x448-mlp"])
def test_bf16_rows_are_the_exactly_quantized_rows(gpu, kw, runs):
    """MXFP4 weights are exact in bf16, and every grouped GEMM sums a row over K in one order: the
    bf16 kernels give the bits the 4-bit kernels give for the same weights, in tiles of every height."""
    import torch
    E = len(runs)
    spec = small(QWEN3_30B_A3B, n_experts=E, top_k=2, quant=F.QuantSpec(4, 32, "mxfp4"), **kw)
    lay = make_layer(spec, seed=890, bank=16)
    T = min(max(runs), 64)
    xd = to_dev_bits(make_x(T, spec.hidden, seed=891), gpu)
    pexp = np.repeat(np.arange(E, dtype=np.int32), runs)
    ptok = np.concatenate([(np.arange(r) * 3 + e) % T for e, r in enumerate(runs)]).astype(np.int32)
    n = pexp.size
    # which kernel: the bf16 one above 40 pairs an expert, with 256-row tiles once those of 128 rows
    # may be more than one block a CU; below it the thin one, whose blocks halve at 4 pairs an expert
    assert (n > 40 * E) == (max(runs) > 100) and (n <= 4 * E) == (max(runs) <= 17)
    if n > 40 * E and spec.hidden > 64:
        fpb = 256 if spec.act == "silu_mlp" else 128
        blocks = (-(-n // 128) + E) * max(-(-spec.inter // fpb), -(-spec.hidden // 256))
        assert (blocks > 256) == (runs is TALL_RUNS)
    res = []
    for layer in (lay, _bf16_copy(lay)):
        print(f"[bf16 order] {layer.spec.quant.mode} H={spec.hidden} I={spec.inter} pairs={n}", flush=True)
        _, _, pool, _ = build_gpu_layer(layer, gpu)
        pool.g2s_device(torch.cuda.current_stream().cuda_stream)
        pool.device.sync()
        y = torch.full((n, spec.hidden), float("nan"), dtype=torch.bfloat16, device=gpu)
        dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(gpu)   # noqa: E731
        ops.forward_pairs(layer.spec, pool, xd, dev(ptok), dev(pexp), dev(np.arange(n, dtype=np.int32)), y,
                          L.FWD_FORCE_PREFILL)
        torch.cuda.synchronize()
        res.append(bits(y))
        pool.close()
    assert not np.isnan(F.bf16_bits_to_f32(res[0])).any()
    assert np.array_equal(*res), f"{int((res[0] != res[1]).any(-1).sum())} of {n} rows differ"
