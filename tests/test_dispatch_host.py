"""Dry runs of the fused aggregation entry points on the CPU: which kernel a shape is sent to and
with what launch geometry (no device, no launch).  Every lane-group count a kernel's loops step
by must be at least one, for every shape the eligibility checks let through."""
import ctypes

import pytest

from f2cgt_amd import capi

A16 = ctypes.c_void_p(1 << 20)   # a 16-byte aligned stand-in for every buffer (never dereferenced)


def plan_log_sq(bits, feat_dim, rows=1000, fanout=10, n_cb=1, idx=capi.DT_I64):
    per = max(1, 8 // bits)
    src_dim = (feat_dim + per - 1) // per
    column_slice = (feat_dim + n_cb - 1) // n_cb
    dt = capi.DT_I16 if bits == 16 else (capi.DT_I8 if bits == 8 else capi.DT_U8)
    return capi.dry_run("f2cgt_sq_decompress_spmm_csr", A16, dt, A16, A16, A16, idx, A16, rows, rows * fanout,
                        5000, src_dim, feat_dim, n_cb, bits, column_slice, None)


def plan_affine(bits, feat_dim, rows=1000, fanout=10, idx=capi.DT_I64):
    per = 8 // bits
    src_dim = (feat_dim + per - 1) // per
    return capi.dry_run("f2cgt_sq_affine_decompress_spmm_csr", A16, A16, feat_dim, A16, A16, idx, A16, rows,
                        rows * fanout, 5000, src_dim, feat_dim, bits, None)


def check_geometry(plan):
    name = plan.kernel.decode()
    assert plan.grid >= 1 and plan.block in (64, 128, 256, 512, 1024), (name, plan.grid, plan.block)
    assert plan.lds_bytes <= 160 * 1024
    if name == "sq_block_kernel":
        assert plan.aux[0] >= 1 and plan.aux[1] >= 1 and plan.rows_per_block >= 1      # row slots, edge capacity
    elif name == "sq_rows_kernel":
        assert plan.aux[0] >= 1 and plan.aux[1] >= 1 and plan.aux[2] >= 8 and plan.rows_per_block >= 8
    elif name == "sq_affine_acc_kernel":
        assert plan.aux[0] >= 1 and plan.aux[1] >= 1 and plan.aux[2] >= 8 and plan.rows_per_block >= plan.aux[2]
    elif name == "hybrid_acc_kernel":
        assert plan.aux[0] >= 1 and plan.rows_per_block >= 8
    elif name == "agg_kernel":
        assert plan.aux[0] >= 1
    else:
        assert name in ("vq_wave_kernel", "vq_pipe_kernel", "vq_strip_kernel"), name
    return name


WIDE = [2040, 2044, 2048, 2052, 3000, 4080, 4088, 4092, 4096]


@pytest.mark.parametrize("bits", [1, 2, 4, 8])
def test_fused_sq_geometry_over_feature_widths(bits):
    per = 8 // bits
    dims = sorted(set([4, 8, 12, 16, 24, 36, 64, 100, 128, 256, 300, 512, 768, 1000, 1024, 2000] + WIDE +
                      [6, 10, 18, 30, 66, 102, 130, 602, 1022, 2042, 2046, 4090, 4094]))   # 4 k + 2 columns
    seen = set()
    for d in dims:
        for fanout in (1, 10, 60):
            if d % per == 0 or bits == 8:
                rc, plan = plan_log_sq(bits, d, fanout=fanout)
                assert rc == 0 and plan is not None, (bits, d, capi.lib().f2cgt_last_error())
                seen.add(check_geometry(plan))
            rc, plan = plan_affine(bits, d, fanout=fanout)
            assert rc == 0 and plan is not None, (bits, d, capi.lib().f2cgt_last_error())
            seen.add(check_geometry(plan))
    assert "sq_rows_kernel" in seen and (bits < 4 or "agg_kernel" in seen)


def test_even_widths_that_are_no_multiple_of_four_take_the_row_block_kernels():
    for d in (18, 66, 102, 602):
        for bits in (4, 8):
            assert plan_affine(bits, d)[1].kernel.decode() == "sq_affine_acc_kernel", (bits, d)
            assert plan_log_sq(bits, d)[1].kernel.decode() == "sq_rows_kernel", (bits, d)
    for bits in (1, 2):
        assert plan_log_sq(bits, 602)[1].kernel.decode() == "sq_rows_kernel"
        assert plan_affine(bits, 602)[1].kernel.decode() == "sq_rows_kernel"
    for d in (17, 101, 601):   # odd widths: one column per lane
        assert plan_affine(4, d)[1].kernel.decode() == "agg_kernel"
    vq = capi.dry_run("f2cgt_vq_decompress_spmm_csr", A16, capi.DT_U8, A16, A16, A16, capi.DT_I64, A16, 200_000,
                      2_000_000, 1_000_000, 602, 19, 256, 32, None)
    assert vq[0] == 0 and vq[1].kernel.decode() == "vq_wave_kernel" and vq[1].aux[0] == 1


def test_wide_rows_leave_the_row_block_kernels():
    # staged pitch above 2 KB: 8-bit codes from 2044 columns, 4-bit codes from 4088
    for bits, d in ((8, 2044), (8, 2048), (8, 4096), (4, 4088), (4, 4092), (4, 4096)):
        for planner in (plan_log_sq, plan_affine):
            rc, plan = planner(bits, d)
            assert rc == 0
            assert plan.kernel.decode() == "agg_kernel", (bits, d, plan.kernel)
    # just below the bound the staged-rows kernel still takes them
    assert plan_log_sq(8, 2040)[1].kernel.decode() == "sq_rows_kernel"
    assert plan_log_sq(4, 4080)[1].kernel.decode() == "sq_rows_kernel"


def test_headline_shapes_take_the_fast_kernels():
    rc, plan = plan_affine(4, 100, rows=250_000, fanout=2)
    assert rc == 0 and plan.kernel.decode() == "sq_affine_acc_kernel"
    rc, plan = plan_affine(8, 128, rows=10_000, fanout=10)
    assert rc == 0 and plan.kernel.decode() == "sq_affine_acc_kernel"
    rc, plan = plan_log_sq(4, 100, rows=250_000, fanout=2)
    assert rc == 0 and plan.kernel.decode() == "sq_rows_kernel"
    vq = lambda rows, fanout, d, n_cb, w: capi.dry_run(
        "f2cgt_vq_decompress_spmm_csr", A16, capi.DT_U8, A16, A16, A16, capi.DT_I64, A16, rows, rows * fanout,
        1_000_000, d, n_cb, 256, w, None)
    for rows, fanout, d, n_cb, w in ((500_000, 15, 128, 16, 8), (600_000, 10, 768, 24, 32), (4096, 15, 128, 16, 8)):
        rc, plan = vq(rows, fanout, d, n_cb, w)
        assert rc == 0 and plan.kernel.decode().startswith("vq_"), plan.kernel
        assert plan.lds_bytes <= 160 * 1024
    hyb = capi.dry_run("f2cgt_hybrid_decompress_spmm_csr", A16, A16, A16, 128, A16, A16, A16, A16, capi.DT_I64, A16,
                       1_000_000, 12_000_000, 100_000_000, 5_000_000, 95_000_000, 128, 8, 256, 16, None)
    assert hyb[0] == 0 and hyb[1].kernel.decode() == "hybrid_acc_kernel"
    # four columns: one chunk per row, outside the row-block form (its reciprocal does not fit 32 bits)
    hyb4 = capi.dry_run("f2cgt_hybrid_decompress_spmm_csr", A16, A16, A16, 4, A16, A16, A16, A16, capi.DT_I64, A16,
                        100, 1000, 1000, 500, 500, 4, 1, 256, 4, None)
    assert hyb4[0] == 0 and hyb4[1].kernel.decode() == "agg_kernel"


def test_unsigned_eight_bit_log_codes_are_refused():
    lib = capi.lib()
    rc = lib.f2cgt_sq_decompress(A16, capi.DT_U8, A16, A16, 4, 16, 16, 1, 8, 16, None)
    assert rc == -2 and b"int8" in lib.f2cgt_last_error()
    rc, _ = capi.dry_run("f2cgt_sq_decompress_spmm_csr", A16, capi.DT_U8, A16, A16, A16, capi.DT_I64, A16, 4, 8, 10,
                         16, 16, 1, 8, 16, None)
    assert rc == -2 and b"int8" in lib.f2cgt_last_error()
    rc, plan = capi.dry_run("f2cgt_sq_decompress_spmm_csr", A16, capi.DT_I8, A16, A16, A16, capi.DT_I64, A16, 4, 8,
                            10, 16, 16, 1, 8, 16, None)
    assert rc == 0 and plan is not None


def test_rows_per_block_follow_the_launch_size():
    # integer-accumulating kernel: the degree decides from 2.5e5 rows on, smaller launches get smaller
    # blocks (at least 8 rows) so that a CU still overlaps several of them
    want = {(250_000, 2): 64, (65_536, 2): 32, (16_384, 2): 8, (1024, 2): 8, (10_000, 10): 8}
    for (rows, fanout), rb in want.items():
        bits, d = (8, 128) if fanout == 10 else (4, 100)
        rc, plan = plan_affine(bits, d, rows=rows, fanout=fanout)
        assert rc == 0 and plan.kernel.decode() == "sq_affine_acc_kernel"
        assert plan.rows_per_block == rb, (rows, fanout, plan.rows_per_block)
        assert plan.rows_per_block % plan.aux[2] == 0 and plan.grid == -(-rows // rb)
    # staged-rows kernel: at least 16 rows, about a thousand workgroups
    for rows, rb in ((250_000, 64), (65_536, 64), (16_384, 16), (4096, 16), (20_000, 16)):
        rc, plan = plan_log_sq(4, 100, rows=rows, fanout=2)
        assert rc == 0 and plan.kernel.decode() == "sq_rows_kernel"
        assert plan.rows_per_block == rb, (rows, plan.rows_per_block)
    # long rows keep their small degree-based blocks
    rc, plan = plan_log_sq(4, 100, rows=4096, fanout=60)
    assert rc == 0 and plan.rows_per_block == 8


def plan_vq(rows, fanout, d, n_cb, w, n_src, edges=None, codes=A16):
    rc, plan = capi.dry_run("f2cgt_vq_decompress_spmm_csr", codes, capi.DT_U8, A16, A16, A16, capi.DT_I64, A16, rows,
                            rows * fanout if edges is None else edges, n_src, d, n_cb, 256, w, None)
    assert rc == 0
    return plan


def test_fused_vq_lane_layout_by_shape():
    """aux of a vq_wave_kernel plan: float4 per lane and edge (2: a row has sixteen lanes of eight columns, 1: 32 of four),
    rows of a mini-block, columns that are no multiple of four, codes read byte by byte.  The output is written in one way
    per layout, whatever the table, the output's size and the store mode."""
    def layout(*args, **kw):
        plan = plan_vq(*args, **kw)
        assert plan.kernel.decode() == "vq_wave_kernel"
        return tuple(plan.aux)
    eight = (2, 4, 0, 0)
    shapes = [(300_000, 5, 128, 16, 8, 1_000_000), (300_000, 10, 128, 16, 8, 1_000_000), (300_000, 5, 128, 4, 32, 1_000_000),
              (300_000, 14, 256, 16, 16, 10_000_000), (100_000, 14, 512, 16, 32, 1_000_000), (500_000, 15, 128, 16, 8, 10_000_000),
              (600_000, 10, 768, 24, 32, 240_000_000), (122_880, 15, 128, 16, 8, 16_777_217), (49_152, 11, 512, 16, 32, 20_000_000)]
    for mode in (capi.STORE_AUTO, capi.STORE_STREAM, capi.STORE_CACHED):
        was = capi.set_store_mode(mode)
        try:
            for shape in shapes:
                assert layout(*shape) == eight, shape
        finally:
            capi.set_store_mode(was)
    # rows of a mini-block: rows of one length up to 16 / 32 edges, ragged ones up to 0.9 of that
    assert [layout(100_000, f, 128, 16, 8, 1_000_000)[1] for f in (16, 17, 32, 33, 200)] == [4, 2, 2, 1, 1]
    assert [layout(100_000, 0, 128, 16, 8, 1_000_000, edges=e)[1] for e in (1_439_999, 1_440_001, 2_879_999, 2_880_001)] == [4, 2, 2, 1]
    # widths that are no multiple of eight: one float4 per lane; of two columns over; the block kernel for long rows of
    # whole code words
    assert layout(300_000, 10, 100, 25, 8, 1_000_000) == (1, 4, 0, 1) and layout(300_000, 10, 124, 16, 8, 1_000_000) == (1, 4, 0, 0)
    assert layout(300_000, 10, 602, 19, 32, 1_000_000) == (1, 4, 1, 1) and layout(300_000, 40, 602, 19, 32, 1_000_000)[:2] == (1, 4)
    assert plan_vq(300_000, 16, 124, 16, 8, 1_000_000).kernel.decode() == "vq_pipe_kernel"
    # codes read byte by byte: rows of codes that are no whole words, or not aligned to them
    assert layout(300_000, 10, 192, 24, 8, 1_000_000) == (2, 4, 0, 1)
    assert layout(300_000, 10, 128, 16, 8, 1_000_000, codes=ctypes.c_void_p((1 << 20) + 8)) == (2, 4, 0, 1)
    # odd multiples of eight columns in several tiles, few edges: one float4 per lane
    lanes = lambda *args: layout(*args)[0]
    assert lanes(1_000_000, 3, 200, 25, 8, 1_000_000) == 1 and lanes(300_000, 10, 200, 25, 8, 1_000_000) == 2
    assert lanes(1_000_000, 3, 192, 24, 8, 1_000_000) == 2 and lanes(1_000_000, 3, 64, 8, 8, 1_000_000) == 2
    assert lanes(1_000_000, 3, 224, 7, 32, 1_000_000) == 2 and lanes(1_000_000, 3, 600, 19, 32, 1_000_000) == 1


def test_fused_vq_rows_of_split_pieces():
    lanes = lambda *args: plan_vq(*args).aux[0]
    for dim in (160, 192, 224, 304, 320, 384, 416, 448, 480, 544, 768):
        assert lanes(300_000, 10, dim, dim // 8, 8, 20_000_000) == 2
    # odd multiples of eight columns: one float4 per lane
    assert lanes(41_667, 12, 600, 19, 32, 1_000_000) == 1
    assert lanes(41_666, 12, 600, 19, 32, 1_000_000) == 2
    assert lanes(41_667, 13, 600, 19, 32, 1_000_000) == 2
    assert lanes(41_667, 16, 600, 19, 32, 15_000_000) == 1
    # a last tile of few columns leaves the lanes of its workgroups idle
    for dim, up_to in ((136, 8), (152, 8), (168, 12), (200, 12), (216, 16), (264, 8), (280, 8), (296, 12), (328, 12), (360, 16),
                       (392, 12), (456, 16), (504, 16), (520, 12), (568, 16), (648, 12), (712, 16), (760, 16)):
        forms = [lanes(300_000, fanout, dim, -(-dim // 8), 8, 30_000_000) for fanout in (8, 9, 12, 13, 16, 17)]
        assert forms == [1 if fanout <= up_to else 2 for fanout in (8, 9, 12, 13, 16, 17)], dim
    assert lanes(335_545, 12, 200, 25, 8, 1_000_000) == 1 and lanes(335_544, 12, 200, 25, 8, 1_000_000) == 2
    assert lanes(125_000, 12, 200, 25, 8, 12_000_000) == 1
    assert lanes(700_000, 9, 104, 13, 8, 1_000_000) == 2          # one column tile
    assert lanes(400_000, 12, 208, 26, 8, 1_000_000) == 2         # whole 64-byte pieces


def test_dealt_items_and_column_form_of_one_codebook():
    """1-bit rows: items take 256 threads per workgroup, the column form 128."""
    def block(rows, dim, fanout, n_cb=1, bits=1):
        rc, plan = plan_log_sq(bits, dim, rows, fanout, n_cb)
        assert rc == 0 and check_geometry(plan) == "sq_rows_kernel"
        return plan.block
    assert block(200000, 128, 10) == 256 and block(200000, 128, 10, n_cb=2) == 128
    # few edges per row: the column form in large cached launches of narrow rows only
    for bits in (1, 2):
        assert block(200000, 128, 1, bits=bits) == 128 and block(200000, 128, 2, bits=bits) == 128
        assert block(200000, 128, 3, bits=bits) == 256           # more edges per row
        assert block(99999, 128, 1, bits=bits) == 256            # fewer rows
        assert block(120000, 300, 1, bits=bits) == 256           # wider rows
        assert block(480000, 128, 1, bits=bits) == 256           # streamed output (246 MB)
    assert block(100000, 32, 1, bits=2) == 256                   # fewer values


def test_decode_through_a_row_list_counts_its_row_table():
    """The looked-up rows (8.2 KB) lie in LDS beside the decode table: past 64 KB together the shape is left to fetch and
    decode, refused before a launch.  (The admitted side, one codebook less, runs in the GPU tests.)"""
    lib = capi.lib()
    for feat_dim, n_cb in ((540, 54), (610, 61), (620, 62)):
        assert lib.f2cgt_sq_decompress_rows(A16, capi.DT_I8, A16, capi.DT_I64, None, 0, None, A16, A16, 4, 100, feat_dim, feat_dim,
                                            n_cb, 8, 10, None) == -2


def test_plain_rows_of_few_edges_stay_with_the_skeleton():
    def kernel(rows, edges, dim, dtype=capi.DT_F32):
        rc, plan = capi.dry_run("f2cgt_spmm_csr", A16, dtype, A16, A16, A16, capi.DT_I64, rows, edges, 100_000, dim, None)
        assert rc == 0
        return plan.kernel.decode()
    for dtype, dim in ((capi.DT_F32, 128), (capi.DT_F32, 602), (capi.DT_F32, 33), (capi.DT_F16, 64), (capi.DT_F64, 64)):
        assert kernel(1000, 2250, dim, dtype) == "agg_kernel" and kernel(1000, 2251, dim, dtype) == "agg_plain_kernel"
        assert kernel(1000, 0, dim, dtype) == "agg_kernel"
    # 39 of 64 lanes of four columns: up to three
    assert kernel(1000, 3000, 154) == "agg_kernel" and kernel(1000, 3001, 154) == "agg_plain_kernel"
    assert kernel(1000, 9000, 24) == "agg_plain_kernel" and kernel(1000, 9000, 16) == "agg_kernel"


def test_which_of_the_dense_layers_kernels_a_size_takes():
    """Bits: 1 the forward kernel without gradients, 2 with them, 4 the backward kernel."""
    take = lambda m, n, k0, k1=None: capi.lib().f2cgt_sage_linear_ahead(m, n, k0, k0 if k1 is None else k1)
    assert take(1024, 256, 128) == take(257, 17, 4) == take(4096, 128, 128) == take(4096, 47, 100) == 7
    # where the library splits the columns: few rows, few outputs, large products but for outputs in whole tiles
    assert take(256, 256, 128) == take(1024, 16, 128) == take(4096, 129, 128) == take(1024, 600, 64) == 4
    assert take(4096, 256, 128) == 6 and take(4096, 256, 64) == 7 and take(4096, 224, 128) == 6 and take(4096, 288, 64) == 4
    # more columns than one order covers
    assert take(1024, 256, 132, 4) == take(1024, 256, 4, 132) == 4
    # many rows: no gradients, and without them up to 2^27 multiply-adds in 2^19 outputs
    assert take(4097, 127, 128) == 3 and take(4097, 128, 128) == 0 and take(30840, 17, 128) == 3 and take(30841, 17, 128) == 0
    assert take(60000, 256, 128) == take(60000, 256, 1000) == 0
    # wide gradients
    assert take(4096, 512, 128) == 4 and take(1024, 512, 512) == 4 and take(1025, 512, 512) == 0
    assert take(0, 1, 4) == take(1, 0, 4) == take(1, 1 << 20, 4) == take(1 << 31, 1, 4) == 0
