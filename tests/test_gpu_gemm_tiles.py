"""GPU parity of the wide GEMM's 2 x 2-wave tiles where they can go wrong: the first and last
rows and columns of every tile size, a K of one, odd and half super-tiles, K splits, the
output formats and alignments that leave the accumulators another way, swizzled activation
scales.  The four-wave and generic kernels, themselves checked against the oracle, are the
reference: whole-K sums are the same chain of MFMAs (equal bits); others meet the GEMM bar."""
import pytest
import torch

from test_gpu_gemm import _act, _check, _weights

pytestmark = pytest.mark.gpu


def _options(ops, **fields):
    from vllm_mach_amd import _lib
    return _lib.GemmOptions(**fields)


def _plan(M, N, K, fmt, block=0):
    from vllm_mach_amd import _lib
    return _lib.plan_name("mxl_gemm_plan_name", M, N, K, fmt, block)


def _mx(pkg, oracle_mod, dev, M, N, K, fmt):
    ops = pkg.ops
    _, ws, stored = _weights(oracle_mod, N, K, fmt, 0.02, 5 + N + K)
    tiled, tiled_s = ops.pack_weight(torch.from_numpy(stored).to(dev), torch.from_numpy(ws).to(dev), fmt)
    a, sa = torch.ops.mach_amd.quantize_mxfp8(_act(M, K, 9 + M).to(dev), 0)
    return a, sa, tiled, tiled_s


def _block(pkg, dev, M, N, K):
    g = torch.Generator().manual_seed(31 + M + K)
    w = torch.randn(N, K, generator=g) * 0.02
    wb = w.reshape(N // 128, 128, K // 128, 128)
    sb = (wb.abs().amax(dim=(1, 3)) / 448.0).float()
    wq = (wb / sb[:, None, :, None]).reshape(N, K).to(torch.float8_e4m3fn)
    tiled, _ = pkg.ops.pack_weight(wq.to(dev), None, 0)
    q, s = torch.ops.mach_amd.quantize_block_fp8(torch.randn(M, K, generator=g).bfloat16().to(dev))
    return q, s, tiled, sb.to(dev)


# M, N, K, fmt, tile (rows / 16, columns / 64) the planner takes, K splits
TILES = [
    (17, 12296, 1152, 0, "4,1", False),    # the fewest rows; N % 64 = 8; nine slices (2.25 super-tiles)
    (20, 2560, 9216, 0, "4,1", True),
    (600, 4100, 128, 2, "4,1", False),     # one slice; N % 16 = 4
    (63, 18440, 768, 3, "4,2", False),     # N % 128 = 8, one and a half super-tiles
    (257, 4104, 896, 3, "4,2", False),     # one row in the last row of tiles
    (160, 6000, 2048, 0, "8,1", False),
    (200, 1152, 14336, 3, "8,1", True),
    (200, 9000, 1024, 0, "8,2", False),
    (129, 17408, 5120, 2, "8,2", True),    # whole-K tiles and split remainder in one launch
    (900, 10000, 384, 0, "8,4", False),    # less than a super-tile
    (1090, 8200, 640, 0, "8,4", False),    # quarters of 41 tiles past a full round: 2 rows, 8 columns of the last
    (1500, 18432, 512, 0, "16,4", False),  # one super-tile; quarters
    (700, 18400, 2560, 2, "16,4", False),  # N % 256 = 224
    (2000, 9000, 1280, 3, "16,4", False),  # quarters of 32 tiles: 80 rows, 40 columns of the last
    (749, 6408, 1024, 0, "8,2", False),    # quarters of 50 tiles beside the one round of whole ones
    (1290, 3208, 1664, 3, "8,2", False),   # of 30, an odd count of slices: 10 rows, 8 columns of the last
]


@pytest.mark.parametrize("M,N,K,fmt,tile,split", TILES)
def test_mx_tiles(pkg, oracle_mod, dev, monkeypatch, M, N, K, fmt, tile, split):
    ops = pkg.ops
    plan = _plan(M, N, K, fmt)
    assert plan.startswith(f"gemm_wide_kernel<{fmt},{tile},false,false,2>")
    assert plan.endswith("wide_tile_reduce_kernel") == split
    a, sa, w, sw = _mx(pkg, oracle_mod, dev, M, N, K, fmt)
    monkeypatch.setattr(ops, "_tuning", None)
    y = torch.ops.mach_amd.mx_gemm(a, sa, w, sw, N, K, fmt, None)
    four = M >= 64 and K % 256 == 0
    monkeypatch.setattr(ops, "_tuning", _options(ops, tile_n=2, splits=1, waves=4) if four else _options(ops, kernel=2))
    ref = torch.ops.mach_amd.mx_gemm(a, sa, w, sw, N, K, fmt, None)
    if four and not split:
        assert torch.equal(y, ref)
    _check(y.float().cpu().numpy(), ref.float().cpu().numpy())


@pytest.mark.parametrize("M,N,K,tile,split", [
    (17, 18432, 1024, "4,2", False),
    (40, 2560, 9344, "4,1", True),      # 73 slices: the last stage is past K
    (130, 18432, 640, "4,2", False),
    (300, 18432, 2560, "8,2", False),
    (1090, 7552, 1280, "8,2", False),   # quarters of 19 tiles, 2 rows of the last
    (793, 5504, 1152, "8,2", False),    # of 45 tiles beside the one round
])
def test_block_fp8_tiles(pkg, dev, monkeypatch, M, N, K, tile, split):
    ops = pkg.ops
    plan = _plan(M, N, K, 0, 1)
    assert plan.startswith(f"gemm_wide_kernel<0,{tile},true,false,2>")
    assert plan.endswith("wide_tile_reduce_kernel") == split
    q, s, w, sb = _block(pkg, dev, M, N, K)
    monkeypatch.setattr(ops, "_tuning", None)
    y = torch.ops.mach_amd.block_fp8_gemm(q, s, w, sb, N, K, None)
    four = M >= 64 and K % 256 == 0
    monkeypatch.setattr(ops, "_tuning", _options(ops, tile_n=2, splits=1, waves=4) if four else _options(ops, kernel=2))
    ref = torch.ops.mach_amd.block_fp8_gemm(q, s, w, sb, N, K, None)
    if four and not split:
        assert torch.equal(y, ref)
    _check(y.float().cpu().numpy(), ref.float().cpu().numpy())


@pytest.mark.parametrize("N", [640, 642, 641])       # columns of 16-, 4- and 2-byte alignment
@pytest.mark.parametrize("out_dtype,alpha,bias,pad", [(0, 1.0, False, 0), (0, 1.0, True, 8), (1, 0.5, False, 3),
                                                      (0, 1.0, False, 1)])
@pytest.mark.parametrize("splits", [1, 3])
def test_tile_outputs(pkg, oracle_mod, dev, N, out_dtype, alpha, bias, pad, splits):
    """The output forms of a 128 x 128 tile and of its split reduce: element format, scale,
    bias, row stride and odd widths, against the four-wave kernel (equal bits)."""
    from vllm_mach_amd import _lib
    M, K, fmt = 200, 2304, 0
    a, sa, w, sw = _mx(pkg, oracle_mod, dev, M, N, K, fmt)
    b = (torch.randn(N, generator=torch.Generator().manual_seed(2)) * 0.5).bfloat16().to(dev) if bias else None
    got = []
    for waves in (4, 8):
        o = _options(pkg.ops, tile_n=2, splits=splits, waves=waves, out_dtype=out_dtype, alpha=alpha)
        nbytes = _lib.query("mxl_gemm_workspace_bytes_ex", M, N, K, fmt, 0, _lib.options_ptr(o))
        ws = torch.empty(max(nbytes, 16), dtype=torch.uint8, device=dev)
        out = torch.full((M, N + pad), 7.0, dtype=torch.float16 if out_dtype else torch.bfloat16, device=dev)
        _lib.call("mxl_mx_gemm_ex", a.data_ptr(), sa.data_ptr(), M, w.data_ptr(), sw.data_ptr(), N, K, fmt,
                  None if b is None else b.data_ptr(), out.data_ptr(), N + pad, ws.data_ptr(), nbytes,
                  _lib.options_ptr(o), torch.cuda.current_stream(dev).cuda_stream)
        got.append(out)
    assert torch.equal(got[0], got[1])
    assert bool((got[1][:, N:] == 7.0).all())  # nothing past the row


@pytest.mark.parametrize("M,N,K", [(300, 1024, 2560), (200, 1024, 2304), (70, 512, 256)])
def test_tiles_read_swizzled_scales(pkg, oracle_mod, dev, M, N, K):
    from vllm_mach_amd import _lib
    a, sa, w, sw = _mx(pkg, oracle_mod, dev, M, N, K, 2)
    swz = torch.empty(_lib.query("mxl_swizzled_scale_bytes", M, K), dtype=torch.uint8, device=dev)
    stream = torch.cuda.current_stream(dev).cuda_stream
    _lib.call("mxl_swizzle_scales", sa.data_ptr(), M, K, swz.data_ptr(), stream)
    got = []
    for layout, scales in ((0, sa), (1, swz)):
        o = _options(pkg.ops, sa_layout=layout, tile_n=2, splits=1, waves=8)
        out = torch.empty((M, N), dtype=torch.bfloat16, device=dev)
        _lib.call("mxl_mx_gemm_ex", a.data_ptr(), scales.data_ptr(), M, w.data_ptr(), sw.data_ptr(), N, K, 2, None,
                  out.data_ptr(), N, None, 0, _lib.options_ptr(o), stream)
        got.append(out)
    assert torch.equal(got[0], got[1])


@pytest.mark.parametrize("M,N,K,fmt,bias", [
    (200, 9216, 32768, 0, False), (768, 4096, 17408, 0, False), (1500, 2040, 17408, 2, True),  # parts of the columns
    (30000, 250, 17408, 3, True),                                                              # one n-block: of the rows
])
def test_noalloc_takes_a_plan_past_its_scratch(pkg, dev, M, N, K, fmt, bias):
    """Shapes whose plan splits K past the no-allocation scratch, though the plan without the 2 x 2-wave
    tiles fits it (so the entry point takes them): the bits of mxl_mx_gemm with a workspace."""
    from vllm_mach_amd import _lib
    assert _lib.query("mxl_gemm_workspace_bytes_ex", M, N, K, fmt, 0, None) > _lib.query("mxl_noalloc_scratch_bytes")
    g = torch.Generator(device=dev).manual_seed(M)
    width = K if fmt == 0 else K * 3 // 4
    codes = torch.randint(0, 0x70 if fmt == 0 else 256, (N, width), generator=g, dtype=torch.uint8, device=dev)
    scales = torch.randint(118, 122, (N, K // 32), generator=g, dtype=torch.uint8, device=dev)
    w, sw = pkg.ops.pack_weight(codes.view(torch.float8_e4m3fn) if fmt == 0 else codes, scales, fmt)
    a, sa = torch.ops.mach_amd.quantize_mxfp8(torch.randn(M, K, generator=g, device=dev).bfloat16(), 0)
    b = torch.randn(N, generator=g, device=dev).bfloat16() if bias else None
    out = torch.empty((M, N), dtype=torch.bfloat16, device=dev)
    _lib.call("mxl_mx_gemm_noalloc", a.data_ptr(), sa.data_ptr(), M, w.data_ptr(), sw.data_ptr(), N, K, fmt,
              None if b is None else b.data_ptr(), out.data_ptr(), N, torch.cuda.current_stream(dev).cuda_stream)
    assert torch.equal(out, torch.ops.mach_amd.mx_gemm(a, sa, w, sw, N, K, fmt, b))


@pytest.mark.parametrize("N,K,fmt,gathered", [(200, 128, 2, False), (384, 1152, 3, True), (264, 2048, 0, True)])
def test_grouped_tiles(pkg, dev, monkeypatch, N, K, fmt, gathered):
    """Experts without rows, of one row, and either side of a 64- and a 128-row block, against the
    per-expert kernel; ragged N, one slice and an odd count of them."""
    ops = pkg.ops
    counts = [0, 1, 64, 65, 0, 128, 129, 200, 63, 3]
    E, R = len(counts), sum(counts)
    g = torch.Generator().manual_seed(N + K)
    width = K if fmt == 0 else K * 3 // 4
    codes = torch.randint(0, 0x70 if fmt == 0 else 256, (E, N, width), generator=g, dtype=torch.uint8).to(dev)
    scales = torch.randint(118, 122, (E, N, K // 32), generator=g, dtype=torch.uint8).to(dev)
    w, sw = ops.pack_weight(codes.view(torch.float8_e4m3fn) if fmt == 0 else codes, scales, fmt)
    offsets = torch.tensor([0] + counts).cumsum(0).to(dev)
    index = torch.randperm(R, generator=g).to(torch.int32).to(dev) if gathered else None
    a, sa = torch.ops.mach_amd.quantize_mxfp8(_act((R + 1) // 2 if gathered else R, K, 4).to(dev), 0)
    args = (a, sa, index, 2 if gathered else 1, offsets, R, w, sw, N, K, fmt)
    got = []
    for fields in (dict(kernel=ops.KERNEL_WIDE), dict(kernel=ops.KERNEL_WIDE, tile_m=4), dict(kernel=ops.KERNEL_GENERIC)):
        monkeypatch.setattr(ops, "_tuning", _options(ops, **fields))
        got.append(torch.ops.mach_amd.grouped_gemm(*args).float().cpu().numpy())
    assert (got[0] == got[1]).all()  # whole-K sums are the same chain of MFMAs
    _check(got[0], got[2])


def _byte_past(t):
    """The same bytes one past a dword boundary."""
    flat = torch.empty(t.numel() + 4, dtype=torch.uint8, device=t.device)
    flat[1:1 + t.numel()] = t.reshape(-1).view(torch.uint8)
    return flat[1:1 + t.numel()].view(t.shape)


@pytest.mark.parametrize("M,N,K", [(40, 4352, 5248), (333, 2048, 2688), (700, 4096, 2560)])
def test_scales_at_any_byte(pkg, oracle_mod, dev, M, N, K):
    """The tiles copy activation scales by the dword: scales that are not dword-aligned run on the
    generic kernel (the same bits), dense and grouped."""
    from vllm_mach_amd import _lib
    ops = pkg.ops
    a, sa, w, sw = _mx(pkg, oracle_mod, dev, M, N, K, 2)
    assert _lib.plan_name("mxl_gemm_plan_name", M, N, K, 2, 0).startswith("gemm_wide_kernel<")
    with ops.tuning(kernel=ops.KERNEL_GENERIC):
        ref = torch.ops.mach_amd.mx_gemm(a, sa, w, sw, N, K, 2, None)
    assert torch.equal(torch.ops.mach_amd.mx_gemm(a, _byte_past(sa), w, sw, N, K, 2, None), ref)
    offsets = torch.tensor([0, M], device=dev)
    with ops.tuning(kernel=ops.KERNEL_GENERIC):
        ref = torch.ops.mach_amd.grouped_gemm(a, sa, None, 1, offsets, M, w, sw, N, K, 2)
    assert _lib.plan_name("mxl_grouped_plan_name", M, 1, K, 2, 0, 0).startswith("gemm_wide_kernel<")
    assert torch.equal(torch.ops.mach_amd.grouped_gemm(a, _byte_past(sa), None, 1, offsets, M, w, sw, N, K, 2), ref)
