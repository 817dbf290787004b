"""Every workgroup shape of the wide kernel, in the formats it takes, at ragged
rows, columns and RHS counts, against the FP64 oracle and, bit for bit, between
qmr_encode and qmr_encode_static."""
import os

import numpy as np
import pytest

import oracle
import qmr.synth as synth
from helpers import assert_gate, upload_matrix

pytestmark = pytest.mark.gpu
THREADS = min(16, os.cpu_count() or 1)
NAME = {"bf16": "_bf16", "f32": ""}
# (row tiles, RHS tiles, waves) of 16, each with the K splits it is run with.
SHAPES = [(0, 0, 0, 0), (2, 1, 8, 1), (4, 1, 4, 2), (4, 1, 8, 1), (5, 1, 8, 1), (8, 1, 8, 2), (8, 1, 4, 3),
          (4, 2, 4, 2), (4, 2, 8, 1), (5, 2, 8, 2), (6, 2, 4, 1), (6, 2, 8, 2), (7, 2, 4, 1), (8, 2, 4, 2)]


# One row more than whole tiles; a last unit of 32, 64 or 128 columns; odd group
# counts (a BF16 row that starts inside a word); one RHS more than a tile or an
# image; a matrix of fewer groups than a metadata window's; enough units for
# several metadata chunks of eight waves in each of two K splits.
@pytest.mark.parametrize("rows,cols,bits,group,meta,batch",
                         [(129, 1056, 4, 32, "bf16", 33), (65, 864, 8, 32, "f32", 17), (81, 1088, 4, 64, "bf16", 5),
                          (257, 1024, 4, 64, "f32", 70), (113, 1984, 8, 64, "bf16", 256), (145, 1408, 4, 128, "bf16", 16),
                          (33, 640, 8, 128, "f32", 34), (17, 64, 4, 64, "bf16", 6), (8, 128, 8, 128, "f32", 18),
                          (33, 4288, 4, 64, "bf16", 20), (40, 4480, 8, 128, "f32", 40)])
def test_wide_shapes_and_formats(gpu, rows, cols, bits, group, meta, batch):
    rng = np.random.default_rng(rows * cols + batch)
    top = 2**bits
    w = rng.integers(0, 2**32, rows * cols * bits // 32, dtype=np.uint32)
    sf = rng.uniform(0.002, 0.02, rows * cols // group).astype(np.float32)
    bf = (-top / 2 * sf + rng.normal(0, 1e-3, sf.size)).astype(np.float32)
    s, b = (synth.f32_to_bf16_bits(sf), synth.f32_to_bf16_bits(bf)) if meta == "bf16" else (sf, bf)
    x = (rng.standard_normal((batch, cols)) * np.exp2(rng.integers(-12, 13, (batch, 1)))).astype(np.float32)
    want = oracle.matmul_f64(w, s, b, meta, x, rows, cols, bits, group, batch, THREADS).reshape(batch, rows)
    # x in two halves is good to 2^-22, and no sum passes A = sum |x| (|s| top
    # + |b|); a group makes at most 2 * group / 32 products, the scaling and
    # the bias, each rounded to 2^-24 of A, and 32 more join classes and splits.
    per = (np.repeat(np.abs(sf), group) * top + np.repeat(np.abs(bf), group)).reshape(rows, cols) * 1.01
    roundings = cols / group * (group / 16 + 3) + 32
    bound = (2.0**-21 + roundings * 2.0**-24) * (np.abs(x).astype(np.float64) @ per.T)
    # Over an RHS's rows the roundings are independent, so that they add as
    # their root, here four times over (x without its lo half: 2e-4).
    typical = 2.0**-21 + 4 * roundings**0.5 * 2.0**-24
    buffers = [*upload_matrix(gpu, w, s, b), gpu.upload_f32(x.ravel()), gpu.alloc_f32(batch * rows)]
    name, params = "matmul_affine_wide" + NAME[meta], [rows, cols, bits, group, batch]
    try:
        for rt, ct, nw, ns in SHAPES:
            print(f"shape {rt} {ct} {nw} splits {ns}", flush=True)
            gpu.set_gemv_plan(-6, nw * 100000 + ns * 1000 + ct * 100 + rt)
            gpu.dispatch(name, buffers, params)
            assert gpu.last_hip_kernel().startswith("wide_mfma_kernel")
            got = gpu.read_f32(buffers[4], batch * rows)
            excess = np.abs(got.reshape(batch, rows) - want) / bound
            assert excess.max() <= 1, f"shape {rt} {ct} {nw} splits {ns}: {excess.max():.2f} of the bound"
            rel = np.linalg.norm(got.reshape(batch, rows) - want, axis=1) / np.linalg.norm(want, axis=1)
            assert rel.max() <= typical, f"shape {rt} {ct} {nw} splits {ns}: RHS {rel.argmax()} off by {rel.max():.1e}"
            command = gpu.begin()
            command.encode(name, buffers, params, rows * 32, 64, static_scratch=True)
            command.finish()
            assert np.array_equal(gpu.read_f32(buffers[4], batch * rows), got), "encode_static differs"
    finally:
        gpu.set_gemv_plan(0, 0)


# On both sides of the lines in rows, in columns and in RHS count; odd group
# counts in 16-bit metadata (4128 and 9248 columns).
@pytest.mark.parametrize("rows,cols,bits,meta,batch,wide", [(7001, 4096, 4, "f32", 4, True), (6999, 4096, 4, "f32", 4, False),
                                                            (7000, 4064, 4, "bf16", 4, False), (7000, 5120, 8, "f32", 4, True),
                                                            (7000, 5088, 8, "f16", 4, False), (17, 12320, 4, "f16", 3, True),
                                                            (17, 12288, 8, "f32", 3, False), (40, 9248, 8, "bf16", 4, True),
                                                            (7003, 4128, 4, "f16", 4, True), (7000, 20480, 4, "bf16", 2, False)])
def test_group_32_blocks_on_either_kernel(gpu, rows, cols, bits, meta, batch, wide):
    """The default route of a group 32 block, against the FP64 oracle and, bit
    for bit, through qmr_encode_static."""
    rng = np.random.default_rng(rows + cols)
    w = rng.integers(0, 2**32, rows * cols * bits // 32, dtype=np.uint32)
    store = {"f32": lambda v: v, "bf16": synth.f32_to_bf16_bits, "f16": lambda v: v.astype(np.float16).view(np.uint16)}[meta]
    sf = rng.uniform(0.002, 0.02, rows * cols // 32).astype(np.float32)
    s, b = store(sf), store((-(2.0 ** (bits - 1)) * sf + rng.normal(0, 1e-3, sf.size)).astype(np.float32))
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    want = oracle.matmul_f64(w, s, b, meta, x, rows, cols, bits, 32, batch, THREADS)
    name = "matmul_affine" + {"f32": "", "bf16": "_bf16", "f16": "_f16meta"}[meta]
    got = []
    for static in (False, True):
        buffers = [*upload_matrix(gpu, w, s, b), gpu.upload_f32(x.ravel()), gpu.alloc_f32(batch * rows)]
        command = gpu.begin()
        command.encode(name, buffers, [rows, cols, bits, 32, batch], rows * 32, 64, static_scratch=static)
        command.finish()
        assert (gpu.last_hip_kernel() == "wide_mfma_kernel") == wide
        got.append(gpu.read_f32(buffers[4], batch * rows))
        assert_gate(got[-1], want)
    assert np.array_equal(got[0], got[1])


# A wide block whose columns fill units, quarters and two RHS tiles, blocks of
# three and four over the lines that send them to the wide kernel, and the
# three metadata types.
@pytest.mark.parametrize("name,rows,cols,bits,batch", [("matmul_affine_wide", 65, 1056, 4, 33),
                                                       ("matmul_affine_wide_bf16", 40, 4128, 8, 7),
                                                       ("matmul_affine_bf16", 33, 9248, 4, 4),
                                                       ("matmul_affine_f16meta", 33, 12320, 8, 3)])
def test_group_32_keeps_every_bit_of_x(gpu, name, rows, cols, bits, batch):
    """x as the vector-ALU kernel multiplies it: FP32 values of any size. A
    token's columns spread over 2^60, one is 2^118 where the weights are zero,
    and then one is Inf and one NaN."""
    rng = np.random.default_rng(rows + cols)
    meta = {"wide": "f32", "bf16": "bf16", "f16meta": "f16"}[name.split("_")[-1]]
    store = {"f32": lambda v: v, "bf16": synth.f32_to_bf16_bits, "f16": lambda v: v.astype(np.float16).view(np.uint16)}[meta]
    load = {"f32": lambda v: v, "bf16": synth.bf16_bits_to_f32, "f16": synth.f16_bits_to_f32}[meta]
    middle = 2 ** (bits - 1)
    codes = rng.integers(0, 2**bits, (rows, cols), dtype=np.uint32)
    s = store(rng.uniform(0.002, 0.02, (rows, cols // 32)).astype(np.float32))
    b = store(rng.uniform(0.001, 0.01, (rows, cols // 32)).astype(np.float32))
    x = (rng.standard_normal((batch, cols)) * np.exp2(rng.integers(-40, 21, (batch, cols)))).astype(np.float32)
    big = cols - 5
    codes[:, big], x[:, big] = middle, np.float32(2.0**118)
    b[:, big // 32] = store(-middle * load(s)[:, big // 32])
    codes[:, 37] |= 1
    pack = 32 // bits
    w = (codes.reshape(rows, -1, pack) << (np.arange(pack, dtype=np.uint32) * bits)).sum(axis=2, dtype=np.uint32)
    want = oracle.matmul_f64(w.ravel(), s.ravel(), b.ravel(), meta, x, rows, cols, bits, 32, batch, THREADS).reshape(batch, rows)
    # A group's three products, its scaling and its bias are each rounded to
    # 2^-24 of the sum of magnitudes at the very most, and 32 more join
    # classes and splits.
    weight = np.repeat(load(s), 32, axis=1) * np.abs(codes.astype(np.float64) - middle) + \
        np.repeat(np.abs(load(b).astype(np.float64) + middle * load(s)), 32, axis=1)
    bound = 1.01 * (cols / 32 * 5 + 32) * 2.0**-24 * (np.abs(x).astype(np.float64) @ weight.T)
    params = [rows, cols, bits, 32, batch]
    buffers = [*upload_matrix(gpu, w, s, b), gpu.upload_f32(x.ravel()), gpu.alloc_f32(batch * rows)]
    gpu.dispatch(name, buffers, params)
    assert gpu.last_hip_kernel() == "wide_mfma_kernel"
    assert (np.abs(gpu.read_f32(buffers[4], batch * rows).reshape(batch, rows) - want) <= bound).all()
    x[1, 37], x[2, 40] = np.inf, np.nan
    buffers[3] = gpu.upload_f32(x.ravel())
    got = []
    try:
        for plan in ((0, 0), (-1, 0)):
            gpu.set_gemv_plan(*plan)
            gpu.dispatch(name, buffers, params)
            got.append(gpu.read_f32(buffers[4], batch * rows).reshape(batch, rows))
    finally:
        gpu.set_gemv_plan(0, 0)
    assert np.isposinf(got[0][1]).all() and np.isnan(got[0][2]).all() and np.isfinite(np.delete(got[0], (1, 2), axis=0)).all()
    for kind in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(kind(got[0]), kind(got[1]))


@pytest.mark.parametrize("rows,cols,bits,group,meta,batch", [(65, 1056, 4, 32, "f32", 18), (40, 2080, 8, 32, "bf16", 5),
                                                             (65, 1088, 4, 64, "bf16", 18), (40, 1152, 8, 128, "f32", 6)])
@pytest.mark.parametrize("static", [False, True])
def test_wide_views_at_four_byte_offsets(gpu, rows, cols, bits, group, meta, batch, static):
    """Codes that are not 16-byte aligned keep FP32 products: group 32 on the
    wide kernel, the others as blocks on the vector ALU."""
    rng = np.random.default_rng(rows + cols)
    top = 2**bits
    w = rng.integers(0, 2**32, rows * cols * bits // 32, dtype=np.uint32)
    sf = rng.uniform(0.002, 0.02, rows * cols // group).astype(np.float32)
    bf = (-top / 2 * sf + rng.normal(0, 1e-3, sf.size)).astype(np.float32)
    s, b = (synth.f32_to_bf16_bits(sf), synth.f32_to_bf16_bits(bf)) if meta == "bf16" else (sf, bf)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    want = oracle.matmul_f64(w, s, b, meta, x, rows, cols, bits, group, batch, THREADS)
    pad = lambda a: np.concatenate([np.full(4, 0xA5, np.uint8), np.ascontiguousarray(a).view(np.uint8).ravel()])
    buffers = [gpu.upload_bytes(pad(a)) for a in (w, s, b, x, np.zeros(batch * rows + 4, np.float32))]
    name, params = "matmul_affine_wide" + NAME[meta], [rows, cols, bits, group, batch]
    command = gpu.begin()
    command.encode(name, buffers, params, rows * 32, 64, [4] * 5, static_scratch=static)
    command.finish()
    assert gpu.last_hip_kernel() == ("wide_mfma_kernel" if group == 32 else "affine_gemv_kernel")
    assert_gate(gpu.read_f32(buffers[4], batch * rows, 4), want)
    assert not gpu.read_f32(buffers[4], 4, 4 + 4 * batch * rows).any()


@pytest.mark.parametrize("rows,cols,bits,group,meta,batch", [(65, 2048, 4, 64, "bf16", 40), (65, 2112, 4, 64, "f32", 6),
                                                             (40, 1984, 8, 64, "bf16", 33), (33, 1920, 4, 128, "f32", 20),
                                                             (33, 2176, 8, 128, "bf16", 5)])
def test_large_columns_do_not_cost_the_others_bits(gpu, rows, cols, bits, group, meta, batch):
    """Every third group's x is 2^40 times larger under weights of zero, and
    every RHS has a size of its own: the other groups keep their precision."""
    rng = np.random.default_rng(rows * cols)
    top = 2**bits
    w = rng.integers(0, 2**32, rows * cols * bits // 32, dtype=np.uint32)
    sf = rng.uniform(0.002, 0.02, (rows, cols // group)).astype(np.float32)
    bf = (-top / 2 * sf + rng.normal(0, 1e-3, sf.shape)).astype(np.float32)
    sf[:, 1::3] = bf[:, 1::3] = 0
    s, b = (synth.f32_to_bf16_bits(sf), synth.f32_to_bf16_bits(bf)) if meta == "bf16" else (sf, bf)
    x = (rng.standard_normal((batch, cols)) * np.exp2(rng.integers(-12, 13, (batch, 1)))).astype(np.float32)
    x *= np.where(np.arange(cols) // group % 3 == 1, np.float32(2.0**40), np.float32(1))
    want = oracle.matmul_f64(w, s.ravel(), b.ravel(), meta, x, rows, cols, bits, group, batch, THREADS).reshape(batch, rows)
    # As in test_wide_shapes_and_formats.
    per = np.repeat(np.abs(sf) * top + np.abs(bf), group, axis=1) * 1.01
    bound = (2.0**-21 + (cols / group * (group / 16 + 3) + 32) * 2.0**-24) * (np.abs(x).astype(np.float64) @ per.T)
    buffers = [*upload_matrix(gpu, w, s, b), gpu.upload_f32(x.ravel()), gpu.alloc_f32(batch * rows)]
    gpu.dispatch("matmul_affine_wide" + NAME[meta], buffers, [rows, cols, bits, group, batch])
    assert gpu.last_hip_kernel() == "wide_mfma_kernel"
    assert (np.abs(gpu.read_f32(buffers[4], batch * rows).reshape(batch, rows) - want) <= bound).all()


@pytest.mark.parametrize("bits,group", [(4, 64), (4, 128), (8, 64)])
def test_columns_of_zeros_change_no_bit(gpu, bits, group):
    """The arithmetic does not depend on whether the rows are whole 256
    columns: a matrix and the same one with a group of zeros at its end give
    the same bits under the same plan."""
    rows, cols, batch = 70, 512, 40
    rng = np.random.default_rng(bits * group)
    w = rng.integers(0, 2**32, (rows, cols * bits // 32), dtype=np.uint32)
    s = rng.uniform(0.002, 0.02, (rows, cols // group)).astype(np.float32)
    b = (-(2.0 ** (bits - 1)) * s + rng.normal(0, 1e-3, s.shape)).astype(np.float32)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    got = []
    gpu.set_gemv_plan(-6, 401208)
    try:
        for extra in (0, group):
            pad = lambda a, n: np.pad(a, ((0, 0), (0, n))).ravel()
            buffers = [*upload_matrix(gpu, pad(w, extra * bits // 32), pad(s, extra // group), pad(b, extra // group)),
                       gpu.upload_f32(pad(x, extra)), gpu.alloc_f32(batch * rows)]
            gpu.dispatch("matmul_affine_wide", buffers, [rows, cols + extra, bits, group, batch])
            assert gpu.last_hip_kernel().startswith("wide_mfma_kernel")
            got.append(gpu.read_f32(buffers[4], batch * rows))
    finally:
        gpu.set_gemv_plan(0, 0)
    assert np.array_equal(got[0], got[1])


# Images of 32 RHS: 2.3 MB (Q8), 3.4 MB (group 32), 2.3 MB (ragged columns);
# the scratch has 8 MiB.
@pytest.mark.parametrize("rows,cols,bits,group,batch", [(33, 17408, 8, 64, 97), (40, 17408, 4, 32, 130),
                                                        (17, 17472, 4, 64, 256), (17, 8192, 8, 128, 256)])
def test_static_entry_runs_the_same_passes(gpu, rows, cols, bits, group, batch):
    """A wide block whose images pass the static scratch takes several passes
    over fewer RHS in both entries, with the same bits."""
    rng = np.random.default_rng(rows + cols + batch)
    w = rng.integers(0, 2**32, rows * cols * bits // 32, dtype=np.uint32)
    s = rng.uniform(0.002, 0.02, rows * cols // group).astype(np.float32)
    b = (-(2.0 ** (bits - 1)) * s + rng.normal(0, 1e-3, s.size)).astype(np.float32)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    want = oracle.matmul_f64(w, s, b, "f32", x, rows, cols, bits, group, batch, THREADS)
    got = []
    for static in (False, True):
        buffers = [*upload_matrix(gpu, w, s, b), gpu.upload_f32(x.ravel()), gpu.upload_f32(np.full(batch * rows, np.nan))]
        command = gpu.begin()
        command.encode("matmul_affine_wide", buffers, [rows, cols, bits, group, batch], rows * 32, 64, static_scratch=static)
        command.finish()
        assert gpu.last_hip_kernel() == "wide_mfma_kernel"
        got.append(gpu.read_f32(buffers[4], batch * rows))
        assert_gate(got[-1], want)
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("rows,cols,bits,batch,wide", [(64, 1024, 4, 5, False), (65, 1056, 8, 8, False),
                                                       (65, 1056, 4, 9, True), (1024, 4096, 4, 8, False),
                                                       (1025, 4096, 4, 8, True), (1000, 4128, 4, 5, True),
                                                       (2000, 2080, 8, 5, True), (2048, 2048, 8, 6, False)])
def test_small_group_32_blocks_run_as_blocks(gpu, rows, cols, bits, batch, wide):
    """On both sides of the lines in size, in columns and in RHS count."""
    rng = np.random.default_rng(rows + cols)
    w = rng.integers(0, 2**32, rows * cols * bits // 32, dtype=np.uint32)
    s = rng.uniform(0.002, 0.02, rows * cols // 32).astype(np.float32)
    b = (-(2.0 ** (bits - 1)) * s + rng.normal(0, 1e-3, s.size)).astype(np.float32)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    buffers = [*upload_matrix(gpu, w, s, b), gpu.upload_f32(x.ravel()), gpu.alloc_f32(batch * rows)]
    gpu.dispatch("matmul_affine_wide", buffers, [rows, cols, bits, 32, batch])
    assert (gpu.last_hip_kernel() == "wide_mfma_kernel") == wide
    assert_gate(gpu.read_f32(buffers[4], batch * rows), oracle.matmul_f64(w, s, b, "f32", x, rows, cols, bits, 32, batch, THREADS))
