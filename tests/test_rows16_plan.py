"""What the plan picks for 16-bit x beyond one 16-row chunk per group, at both sides of its lines; 256 CUs, no device needed."""
import re

import pytest

from ms_custom_ops_amd import cabi


def _plan(m, k, n, e, layout="kn", bits=8, override=0):
    op = cabi.GmmOp(x_dtype=cabi.DT_BF16, out_dtype=cabi.DT_BF16, antiquant_dtype=cabi.DT_BF16, weight_dtype=cabi.DT_I4 if bits == 4 else cabi.DT_I8,
                    group_list_dtype=cabi.DT_I64, weight_layout=cabi.WL_PACKED if layout == "packed" else cabi.WL_ROW_MAJOR, kernel_override=override)
    try:
        op.plan(m, k, n, e)
    except cabi.BackendError:
        pass   # (a split plan allocates counters on the device; the plan itself stands)
    info = op.plan_info()
    op.close()
    return info.split("kernel=")[1].split()[0], int(re.search(r"split_k=(\d+)", info)[1]), int(re.search(r"workspace=(\d+)", info)[1])


@pytest.mark.parametrize("m,k,n,e,layout,bits,kernel,split", [
    # the model of the time plans from 8 groups and K = 512 on
    (800, 4096, 2048, 8, "kn", 8, "a16w8_rows128x256_2", 2), (700, 4096, 2048, 7, "kn", 8, "a16w8_skinny_rows", 1),
    (800, 512, 2048, 8, "kn", 8, "a16w8_rows128x256", 1), (800, 496, 2048, 8, "kn", 8, "a16w8_skinny_rows", 1),
    # 4-bit weights: beyond 30 rows a group the 128-row kernel reads the nibbles
    (240, 2048, 4096, 8, "kn", 4, "a16w4_skinny_regt", 2), (600, 2048, 4096, 8, "kn", 4, "a16w4_rows128x256_2", 1),
    # ... but up to 43 rows the register-transpose kernels stay where its workgroups fill no more than half of the chip (128 and 136 of them)
    (330, 4416, 4096, 8, "kn", 4, "a16w4_skinny_regt", 1), (330, 4416, 4352, 8, "kn", 4, "a16w4_rows128x256_2", 1), (352, 4416, 4096, 8, "kn", 4, "a16w4_rows128x256_2", 1),
    # strips of 512 columns where they fill the chip, of 256 where they do not, two sets of waves with a K split where those do not either
    (4096, 4096, 14336, 8, "packed", 8, "a16w8_rows128", 1), (131072, 1024, 1024, 128, "packed", 8, "a16w8_rows128x256", 1),
    (816, 6336, 544, 16, "kn", 8, "a16w8_rows128x256_2", 3),
    # two sets of waves in one round (256 workgroups), one set beyond
    (1600, 4096, 4096, 8, "kn", 8, "a16w8_rows128x256_2", 1), (1600, 4096, 4112, 8, "kn", 8, "a16w8_rows128x256", 1),
    (1600, 4096, 4096, 8, "kn", 4, "a16w4_rows128x256_2", 1), (1600, 4096, 4112, 8, "kn", 4, "a16w4_rows128x256", 1),
    # packed weights, two sets: 256 workgroups are a round, 288 are two
    (210, 5472, 8176, 8, "packed", 8, "a16w8_rows128x256_2", 1), (210, 5472, 8816, 8, "packed", 8, "a16w8_rows128", 1),
    # strips of 512 where N fills them to four fifths, one row block a group not on more than two 256-column workgroups per CU
    (11501, 3328, 832, 128, "kn", 8, "a16w8_rows128", 1), (11501, 3328, 816, 128, "kn", 8, "a16w8_rows128x256", 1),
    (11501, 3328, 832, 128, "kn", 4, "a16w4_rows128", 1), (11501, 3328, 816, 128, "kn", 4, "a16w4_rows128x256", 1),
    (103, 1856, 2912, 8, "packed", 8, "a16w8_rows128x256", 1), (179, 1760, 8640, 16, "packed", 8, "a16w8_stream_rows", 1),
    # more than 65535 pairs of expert and chunk: beyond the grids of the kernels with smaller chunks
    (200000, 1024, 512, 1024, "kn", 8, "a16w8_rows128", 1), (200000, 1024, 512, 1024, "kn", 4, "a16w4_rows128x256", 1)])
def test_picks(m, k, n, e, layout, bits, kernel, split):
    assert _plan(m, k, n, e, layout, bits)[:2] == (kernel, split)


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("layout", ["kn", "packed"])
def test_a_split_that_the_plan_picks_fits_a_launch_without_an_allocation(layout, bits):
    if layout == "packed" and bits == 4:
        pytest.skip("4-bit weights are not packed")
    seen = 0
    for e in (8, 16, 32, 64):
        for rows in (20, 40, 100, 200, 400):
            for k, n in ((8192, 512), (8192, 1024), (6144, 2048), (4096, 768), (2048, 4096)):
                kernel, split, size = _plan(rows * e, k, n, e, layout, bits)
                if "rows128" in kernel and split > 1:
                    seen += 1
                    assert size <= cabi.STATIC_WORKSPACE_BYTES, (rows, k, n, e, kernel, split, size)
    assert seen > 5
