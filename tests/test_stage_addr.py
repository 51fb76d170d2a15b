"""Every staged load of the thin-tile and bf16 GEMMs reads inside its buffer or nothing at all.

A host program walks the loads of whole tiles through the address functions the kernels use
(csrc/stage_addr.h). A load is safe if it is inside the buffer with both its offsets added, or if the
range check refuses it whether or not that check counts the scalar offset. Walked: the last rows of
an activation buffer that ends with them, odd and even stage counts, the steps a ring requests past
the last, and the last weight row of an expert, whose bytes end with the down projection's arrays.
"""
import ctypes
import os
import shutil
import subprocess

import pytest

from bigrig_amd import formats as F

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SRC = r"""
#include <initializer_list>
#include "stage_addr.h"
using namespace brx;

static long bad;
static long reads;
// a load of `n` bytes; `must`: its bytes are used
static void load(uint32_t records, uint32_t lane, uint32_t scalar, uint32_t n, uint64_t bytes, bool must) {
    if ((uint64_t)lane + scalar + n <= bytes && records == bytes) { ++reads; return; }
    const bool counted = lane >= records - scalar;     // unsigned, as a wrapped difference would be
    const bool uncounted = lane >= records;
    if (must || !counted || !uncounted) ++bad;
}

template <int SG, int MQ>
static void thin_a(int NR, int nst, int rows, uint32_t pitch, uint32_t m0) {
    const uint32_t bytes = (m0 + rows) * pitch;
    const int nsteps = (nst + SG - 1) / SG;
    for (int wv = 0; wv < kTWaves; ++wv)
        for (int p = 0; p < (nsteps + NR - 1) / NR * NR + NR - 1; ++p) {
            const int q = p * SG + thin_a_stage<SG, MQ>(wv);
            const StageSrc src = stage_src(q, nst, bytes, (uint32_t)q * 128u);
            for (int i = 0; i < kTAWave<SG, MQ>; ++i) {
                if (thin_a_copy<SG, MQ>(wv, i) / (2 * MQ) != thin_a_stage<SG, MQ>(wv)) ++bad;
                for (int lane = 0; lane < 64; ++lane) {
                    const int r = thin_a_row<SG, MQ>(wv, i, lane);
                    for (int c = 0; c < 8; ++c)
                        load(src.records, a_lane_offset(r, rows, (m0 + (r < rows ? r : rows - 1)) * pitch, c, bytes),
                             src.soffset, 16, bytes, r < rows && q < nst);
                }
            }
        }
}

extern "C" {
long walk_reads() { return reads; }

long walk_thin_a(int SG, int MQ, int NR, int K, int rows, unsigned pitch, unsigned m0) {
    bad = reads = 0;
#define CASE(S, M) if (SG == S && MQ == M) thin_a<S, M>(NR, K / 64, rows, pitch, m0)
    CASE(1, 1); CASE(1, 2); CASE(1, 4); CASE(2, 1); CASE(2, 2); CASE(2, 4);
    return bad;
}

// the matrix at byte `w` of an expert of `bytes` bytes: n_out rows of K inputs
long walk_thin_b(int bits, int SG, int NR, int K, int n_out, unsigned w, unsigned bytes) {
    bad = reads = 0;
    const int nst = K / 64, nsteps = (nst + SG - 1) / SG;
    const int nl = bits == 16 ? 2 : bits < 4 ? 1 : (bits + 3) / 4;    // loads of a lane
    for (int row : {0, n_out - 1})
        for (int p = 0; p < (nsteps + NR - 1) / NR * NR + NR - 1; ++p)
            for (int g = 0; g < 4; ++g)
                for (int l = 0; l < nl; ++l) {
                    const StageSrc src = stage_src(p, nsteps, bytes, w + thin_b_step(bits, SG, p));
                    const uint32_t n = bits == 16 ? 16 : bits < 4 ? 4 * bits : (bits == 6 && l) ? 8 : 16;
                    load(src.records, thin_b_lane(bits, K, row, g) + (bits == 16 ? 64 : 16) * l, src.soffset, n, bytes,
                         p < nsteps);
                }
    return bad;
}

// the bf16 GEMM: 8 rows a copy of both operands, stages requested NS - 1 ahead
long walk_dense(int NS, int K, int rows, int tile, unsigned pitch, unsigned w, int n_out, unsigned bytes) {
    bad = reads = 0;
    const int nst = K / 64;
    for (int s = 0; s < nst + NS - 1; ++s)
        for (int c = 0; c < 8; ++c) {
            const StageSrc sa = stage_src(s, nst, rows * pitch, (uint32_t)s * 128u);
            for (int r = 0; r < tile; ++r)
                load(sa.records, a_lane_offset(r, rows, (r < rows ? r : rows - 1) * pitch, c, rows * pitch),
                     sa.soffset, 16, rows * pitch, r < rows && s < nst);
            const StageSrc sb = stage_src(s, nst, bytes, (uint32_t)s * 128u);
            load(sb.records, w + (n_out - 1) * (unsigned)(K * 2) + c * 16, sb.soffset, 16, bytes, s < nst);
        }
    return bad;
}
}
"""


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    d = tmp_path_factory.mktemp("stage_addr")
    (d / "walk.cpp").write_text(SRC)
    so = str(d / "walk.so")
    r = subprocess.run([shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-I",
                        os.path.join(ROOT, "bigrig_amd", "csrc"), str(d / "walk.cpp"), "-o", so],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    lib = ctypes.CDLL(so)
    for f in ("walk_reads", "walk_thin_a", "walk_thin_b", "walk_dense"):
        getattr(lib, f).restype = ctypes.c_long
    return lib


WIDTHS = [64, 128, 192, 576, 768, 2048, 2880]    # 1, 2, 3, 9, 12, 32 and 45 stages


@pytest.mark.parametrize("K", WIDTHS)
@pytest.mark.parametrize("SG,MQ,NR", [(1, 1, 4), (1, 2, 4), (1, 4, 3), (2, 1, 2), (2, 2, 2), (2, 4, 2),
                                      (2, 1, 4), (2, 2, 4), (2, 4, 3)])
def test_thin_activations(walk, K, SG, MQ, NR):
    for rows in (1, 16 * MQ - 1, 16 * MQ):
        for pitch, m0 in ((2 * K, 0), (2 * K, 7), (2 * K + 128, 3)):     # x, h rows, h rows of a wider layer
            assert walk.walk_thin_a(SG, MQ, NR, K, rows, pitch, m0) == 0, (rows, pitch, m0)
            assert walk.walk_reads() > 0


def _down(H, I, q):
    """(offset of the down projection, bytes of the expert)"""
    spec = F.expert_spec(H, I, q)
    return F.spec_offsets(spec)[("down_proj", "weight")], F.spec_bytes(spec)


@pytest.mark.parametrize("K", WIDTHS)
@pytest.mark.parametrize("bits,group", [(2, 64), (3, 64), (4, 64), (6, 64), (8, 64), (2, 128), (4, 128), (8, 128),
                                        (4, 32), (16, 0)])
def test_thin_weights(walk, K, bits, group):
    if group == 128 and K % 128:
        pytest.skip("not a whole number of groups")
    mode = {0: "none", 32: "mxfp4"}.get(group, "affine")
    for H in (64, 2048) if group != 128 else (128, 2048):
        w, total = _down(H, K, F.QuantSpec(bits, group, mode))
        for NR in (2, 3, 4):
            assert walk.walk_thin_b(bits, 1 if bits == 16 else 2, NR, K, H, w, total) == 0, (H, NR)


@pytest.mark.parametrize("K", WIDTHS)
@pytest.mark.parametrize("NS,tile", [(3, 32), (3, 64), (3, 128), (2, 256)])
def test_dense(walk, K, NS, tile):
    w, total = _down(192, K, F.QuantSpec(16, 0, "none"))
    for rows in (1, tile - 1, tile):
        assert walk.walk_dense(NS, K, rows, tile, 2 * K, w, 192, total) == 0, rows
