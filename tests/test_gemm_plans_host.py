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
