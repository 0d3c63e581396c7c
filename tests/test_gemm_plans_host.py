"""The dense GEMM plans that the library makes without a GPU: which kernel takes a call."""
import pytest


def _plan(M, N, K, fmt=0, block=0, **fields):
    from vllm_mach_amd import _lib
    return _lib.plan_name("mxl_gemm_plan_name", M, N, K, fmt, block, options=_lib.GemmOptions(**fields))


# every tile, split and wave field by itself, and some together
FIELDS = [dict(splits=2), dict(splits=1, hybrid=1), dict(tile_n=2), dict(tile_n=4, splits=1), dict(tile_m=4),
          dict(tile_m=8, tile_n=1), dict(waves=4), dict(waves=8), dict(waves=8, tile_n=2, splits=3)]


@pytest.mark.parametrize("fields", FIELDS)
@pytest.mark.parametrize("M,N,K", [(40, 17408, 5248), (40, 17408, 5120), (333, 5120, 2688), (17, 512, 128),
                                   (63, 18432, 2560), (2048, 2048, 1152)])
def test_tile_fields_outside_the_four_wave_kernel(pkg, fields, M, N, K):
    """Fewer than 64 rows, or K an odd number of 128-blocks: the four-wave tiles do not run these
    shapes, so a call that sets a field of theirs takes the generic kernel."""
    assert _plan(M, N, K, 2, **fields).startswith("gemm_kernel<2,")
    assert _plan(M, N, K, 0, 1, **fields).startswith("gemm_kernel<0,")


def test_tile_fields_keep_the_kernels_of_short_k(pkg):
    """Fields of the wide kernel leave the automatic choice of kernel as it is without its 2 x 2-wave
    tiles: the chunked kernel and the generic one at a short K."""
    assert _plan(96, 4608, 2048, 2, splits=2) == "gemm_chunk_kernel<2,4,1>"
    assert _plan(200, 2048, 2048, 0, splits=2).startswith("gemm_kernel<0,4,1")
    assert _plan(200, 4096, 2048, 0, splits=2).startswith("gemm_wide_kernel<0,8,")


@pytest.mark.parametrize("kernel", [-1, 1])
def test_a_tile_that_is_not_built_is_refused(pkg, kernel):
    from vllm_mach_amd import _lib
    with pytest.raises(_lib.MxlError):
        _plan(128, 17408, 5120, 2, kernel=kernel, tile_n=1, tile_m=4, splits=1)
    assert _plan(128, 17408, 5120, 2, kernel=kernel, tile_n=1, tile_m=8, splits=1).startswith("gemm_wide_kernel<2,8,1")


GENERIC, WIDE = "gemm_kernel<", "gemm_wide_kernel<"


@pytest.mark.parametrize("M,N,K,block,mxfp8,mxfp6", [
    # up to 32 rows: a workgroup of 16 columns per CU (two at a short K)
    (17, 2672, 3072, 0, GENERIC, GENERIC), (32, 4096, 8192, 0, GENERIC, GENERIC), (32, 4097, 8192, 0, WIDE, WIDE),
    (32, 4096, 9088, 0, WIDE, GENERIC), (32, 4096, 9216, 0, WIDE, WIDE), (32, 1040, 8192, 0, GENERIC, GENERIC),
    (32, 1040, 8320, 0, WIDE, WIDE), (32, 1024, 8320, 0, WIDE, GENERIC), (17, 512, 896, 0, GENERIC, GENERIC),
    (17, 512, 768, 0, WIDE, WIDE), (31, 8192, 2048, 0, GENERIC, GENERIC), (31, 8193, 2048, 0, WIDE, WIDE),
    # 33 to 64 rows: 32 rows by 32 columns; past K = 4096 only where its workgroups do not split K, past
    # 4608 only where the row groups share an XCD (a multiple of eight column groups)
    (33, 4096, 4096, 0, GENERIC, GENERIC), (33, 4097, 4096, 0, WIDE, WIDE), (64, 2048, 4608, 0, GENERIC, GENERIC),
    (64, 2016, 4608, 0, WIDE, WIDE), (64, 2080, 4608, 0, GENERIC, GENERIC), (64, 2080, 4736, 0, WIDE, WIDE),
    (64, 2304, 6144, 0, GENERIC, GENERIC), (64, 2304, 6272, 0, WIDE, GENERIC), (64, 2304, 7424, 0, WIDE, GENERIC),
    (64, 2304, 7552, 0, WIDE, WIDE),
    # more: 64 rows by 16 columns
    (65, 2048, 4096, 0, GENERIC, GENERIC), (65, 2049, 4096, 0, WIDE, WIDE), (65, 2048, 4352, 0, GENERIC, GENERIC),
    (65, 2032, 4352, 0, WIDE, WIDE), (65, 2048, 5376, 0, GENERIC, GENERIC), (65, 2048, 5504, 0, WIDE, WIDE),
    (65, 1536, 5376, 0, GENERIC, GENERIC), (65, 1408, 4480, 0, WIDE, WIDE), (512, 512, 5376, 0, GENERIC, GENERIC),
    (513, 384, 5376, 0, WIDE, WIDE), (513, 384, 4352, 0, GENERIC, GENERIC), (640, 400, 2176, 0, GENERIC, GENERIC),
    (641, 256, 3200, 0, WIDE, WIDE), (1024, 192, 3072, 0, GENERIC, GENERIC), (1025, 192, 2688, 0, WIDE, WIDE),
    (1280, 192, 2560, 0, GENERIC, GENERIC), (1281, 128, 2176, 0, WIDE, WIDE),
    # block-FP8
    (32, 4096, 4608, 1, GENERIC, None), (32, 4096, 4736, 1, WIDE, None), (64, 4096, 4352, 1, GENERIC, None),
    (64, 4064, 4352, 1, WIDE, None), (64, 4064, 2176, 1, GENERIC, None), (65, 128, 2176, 1, WIDE, None),
    (17, 8192, 2048, 1, WIDE, None),
])
def test_one_round_of_the_generic_kernel(pkg, M, N, K, block, mxfp8, mxfp6):
    assert _plan(M, N, K, 0, block).startswith(mxfp8)
    if mxfp8 == GENERIC:
        assert not _plan(M, N, K, 0, block).endswith("reduce8_kernel") or K > 4096
    if not block:
        assert _plan(M, N, K, 2).startswith(mxfp6) and _plan(M, N, K, 3).startswith(mxfp6)


def test_kept_plans_are_the_plans_of_their_sizes(pkg):
    """More shapes than a thread keeps plans for, from one thread and from several, and around a registered
    entry: a kept plan answers for its own sizes, format and mode only."""
    from concurrent.futures import ThreadPoolExecutor

    from vllm_mach_amd import _lib
    shapes = [(M, N, K, fmt, block) for M in (24, 96, 333, 2048) for N in (512, 2560, 17408) for K in (1024, 2688, 9216)
              for fmt, block in ((0, 0), (2, 0), (3, 0), (0, 1))]

    def plans(order):
        return {s: (_plan(*s), _lib.query("mxl_gemm_workspace_bytes_ex", *s, None)) for s in order}

    one_by_one = {}
    for s in shapes:  # a new thread has kept nothing
        with ThreadPoolExecutor(1) as pool:
            one_by_one[s] = pool.submit(plans, [s]).result()[s]
    with ThreadPoolExecutor(4) as pool:
        for got in pool.map(plans, [shapes, shapes[::-1], shapes * 2, shapes[::3] + shapes]):
            assert all(one_by_one[s] == p for s, p in got.items())
    s = (333, 2560, 2688, 2, 0)
    _lib.call("mxl_set_gemm_config", *s, _lib.options_ptr(_lib.GemmOptions(kernel=2)))
    assert _plan(*s).startswith("gemm_kernel<2,") != one_by_one[s][0].startswith("gemm_kernel<2,")
    _lib.call("mxl_clear_gemm_configs")
    assert plans([s])[s] == one_by_one[s]


@pytest.mark.parametrize("M,N,K,block", [(749, 6400, 1024, 0), (1002, 4688, 1024, 0), (637, 8152, 1536, 0),
                                         (256, 18432, 1024, 0), (793, 5504, 2432, 1), (197, 17920, 3584, 1),
                                         (2048, 2560, 9216, 0)])
def test_a_part_round_of_tiles_runs_in_one_launch(pkg, M, N, K, block):
    """Up to 64 tiles of 128 x 128 past one round of the CUs: their quarters beside the whole tiles, not a K
    split and its reduce (2 to 5 us slower at each of these)."""
    assert _plan(M, N, K, 0, block) == f"gemm_wide_kernel<0,8,2,{'true' if block else 'false'},false,2>"


@pytest.mark.parametrize("M", [65, 112, 113, 120, 127, 129])
@pytest.mark.parametrize("N,K,fmt", [(4608, 2048, 2), (8192, 1920, 3), (17408, 1536, 0)])
def test_tiles_take_the_rows_on_either_side_of_the_chunked_plan(pkg, M, N, K, fmt):
    assert _plan(M, N, K, fmt).startswith(f"gemm_wide_kernel<{fmt},")
