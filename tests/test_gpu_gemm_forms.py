"""GPU parity of the plain GEMM's automatic choice at the edges of its tiles: m and n around
multiples of 16, 32, 64 and 128, one column piece to many column tiles, fewer k steps than a
workgroup has waves and more than their rings hold, and enough tiles for every form (16 x 16 tiles
to 128 x 128 ones with one and two workgroups per CU). int32 against the register-staged 128 x 128
kernel (UWC_FLAG_TILE128) and, where it is cheap, the CPU oracle; the dequant epilogues (fp32, bf16,
fp32 beside the int32 sums, fp32 with a residual) bit for bit with the oracle's roundings; nothing is written past the rows."""
import numpy as np
import pytest
import torch

import oracle as O

pytestmark = pytest.mark.gpu


def _rand(dev, seed, *shape):
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    return torch.randint(-128, 128, shape, dtype=torch.int8, device=dev, generator=g)


def _gemm(A, B, out_mode, out, flags=0, sx=None, sw=None):
    from uwc_amd import _lib
    m, k = A.shape
    _lib.call("uwc_noisy_gemm", A.data_ptr(), B.data_ptr(), m, B.shape[0], k, 0, None, None, None, 0, None, None, None,
              0, None if sx is None else sx.data_ptr(), None if sw is None else sw.data_ptr(), out.data_ptr(), out_mode,
              flags, None, torch.cuda.current_stream().cuda_stream)
    return out


SHAPES = [(m, n, k) for m in (1, 15, 16, 17, 33, 64, 65, 127, 129) for n, k in ((4, 128), (36, 384), (132, 1152))] + [
    (31, 4100, 640), (63, 8196, 256), (96, 2052, 2176), (200, 4096, 2048), (257, 1028, 6144), (333, 2052, 1152),
    (333, 12288, 256), (640, 4100, 384), (777, 2048, 640), (777, 12292, 256), (1000, 4100, 384), (2049, 1540, 384),
    (2050, 12292, 128), (4100, 4100, 256), (16, 12292, 640), (250, 12292, 2176)]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_edges(dev, m, n, k):
    from uwc_amd import _lib, ops
    A, B = _rand(dev, m + k, m, k), _rand(dev, n + 3 * k, n, k)
    # rows 0 .. m - 1 of a taller buffer: the rows behind keep their values
    full = torch.full((m + 40, n), -77, dtype=torch.int32, device=dev)
    C = _gemm(A, B, ops.OUT_I32, full[:m])
    ref = _gemm(A, B, ops.OUT_I32, torch.empty((m, n), dtype=torch.int32, device=dev), flags=ops.FLAG_TILE128)
    assert torch.equal(C, ref)
    assert bool((full[m:] == -77).all())
    if m * n * k <= 1 << 25:
        assert np.array_equal(C.cpu().numpy(), O.igemm(A.cpu().numpy(), B.cpu().numpy()))
    acc = ref.cpu().numpy()
    rng = np.random.default_rng(m * n + k)
    sx = (rng.random(m, dtype=np.float32) * 1e-2 + 1e-4).astype(np.float32)
    sw = (rng.random(n, dtype=np.float32) * 1e-3 + 1e-5).astype(np.float32)
    x = rng.standard_normal((m, n)).astype(np.float32)
    sxt, swt, xt = (torch.from_numpy(t).to(dev) for t in (sx, sw, x))
    want = O.dequant(acc, sx, sw)
    Y = _gemm(A, B, ops.OUT_F32, torch.empty((m, n), device=dev), sx=sxt, sw=swt)
    assert np.array_equal(Y.cpu().numpy().view(np.uint32), want.view(np.uint32))
    Yb = _gemm(A, B, ops.OUT_BF16, torch.empty((m, n), dtype=torch.bfloat16, device=dev), sx=sxt, sw=swt)
    assert np.array_equal(Yb.cpu().view(torch.int16).numpy().view(np.uint16), O.scale_bf16(acc, sx, sw))
    C2, Y2 = torch.empty((m, n), dtype=torch.int32, device=dev), torch.empty((m, n), device=dev)
    _lib.call("uwc_igemm_i32_dequant_f32", A.data_ptr(), B.data_ptr(), m, n, k, sxt.data_ptr(), swt.data_ptr(),
              C2.data_ptr(), Y2.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert torch.equal(C2, ref) and torch.equal(Y2.view(torch.int32), Y.view(torch.int32))
    R = torch.full((m + 40, n), 7.0, device=dev)
    _lib.call("uwc_igemm_dequant_residual_f32", A.data_ptr(), B.data_ptr(), m, n, k, sxt.data_ptr(), swt.data_ptr(),
              xt.data_ptr(), R.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert np.array_equal(R[:m].cpu().numpy().view(np.uint32), (x + want).view(np.uint32))
    assert bool((R[m:] == 7.0).all())


@pytest.mark.parametrize("m,n,k", [(5, 6, 128), (40, 132, 192), (70, 132, 192), (300, 130, 128)])
def test_shapes_left_to_the_other_kernels(dev, m, n, k):
    """n % 4 != 0, k % 128 != 0 and unaligned outputs keep their kernels, with the same results."""
    from uwc_amd import ops
    A, B = _rand(dev, m, m, k), _rand(dev, n, n, k)
    want = O.igemm(A.cpu().numpy(), B.cpu().numpy())
    buf = torch.empty(m * n + 1, dtype=torch.int32, device=dev)
    for out in (buf[:-1].view(m, n), buf[1:].view(m, n)):
        assert np.array_equal(_gemm(A, B, ops.OUT_I32, out).cpu().numpy(), want)


# tiles of the forms by number (uwc_plain_gemm_route); forms 0 .. 2 have a kernel for whole tiles and one
# for ragged ones, 3 .. 8 one for a single row of tiles (weights read once, not kept in the caches) and one
# for more
TILES = [(128, 128), (128, 128), (64, 128), (64, 64), (64, 64), (64, 32), (32, 32), (16, 32), (16, 16)]
EPILOGUES = {"i32": (1, 0), "bf16": (2, 0), "f32": (3, 0), "residual": (3, 1), "both": (1, 2)}


def _shape_for(form, first, out, second):
    """The smallest of a grid of shapes that the rule puts on this form and kernel, on this device."""
    from uwc_amd import _lib
    route, (bm, bn) = _lib.lib().uwc_plain_gemm_route, TILES[form]
    best = None
    for m in (1, 16, 17, 31, 32, 33, 48, 63, 64, 65, 96, 127, 128, 129, 200, 256, 300, 384, 512, 640, 777, 1024, 1100, 1536, 2048):
        if ((m <= bm) != first) if form > 2 else (first and m % bm):
            continue
        for n in (4, 36, 132, 1028, 2048, 2052, 3072, 4096, 4100, 6144, 8196, 12288, 16384, 20480, 28672):
            if form <= 2 and (m % bm == 0 and n % bn == 0) != first:
                continue
            for k in (128, 256, 384, 640, 1152, 2048, 4096, 6144):
                if (best is None or m * n * k < best[0]) and route(m, n, k, out, second, 0) == form:
                    best = (m * n * k, m, n, k)
    return best and best[1:]


@pytest.mark.parametrize("epilogue", list(EPILOGUES))
@pytest.mark.parametrize("first", [True, False])
@pytest.mark.parametrize("form", range(9))
def test_every_form_and_epilogue(dev, form, first, epilogue):
    """Each instantiation the rule can take, whatever its constants: against the staged kernel's int32
    sums and the oracle's roundings."""
    from uwc_amd import _lib, ops
    out, second = EPILOGUES[epilogue]
    shape = _shape_for(form, first, out, second)
    assert shape or epilogue != "f32", "a form that the rule never takes"
    if shape is None:
        pytest.skip("the rule does not take this kernel with this epilogue")
    m, n, k = shape
    A, B = _rand(dev, m + k, m, k), _rand(dev, n + 3 * k, n, k)
    ref = _gemm(A, B, ops.OUT_I32, torch.empty((m, n), dtype=torch.int32, device=dev), flags=ops.FLAG_TILE128)
    rng = np.random.default_rng(form)
    sx = (rng.random(m, dtype=np.float32) * 1e-2 + 1e-4).astype(np.float32)
    sw = (rng.random(n, dtype=np.float32) * 1e-3 + 1e-5).astype(np.float32)
    sxt, swt = torch.from_numpy(sx).to(dev), torch.from_numpy(sw).to(dev)
    acc = ref.cpu().numpy()
    st = torch.cuda.current_stream().cuda_stream
    if epilogue == "residual":
        x = rng.standard_normal((m, n)).astype(np.float32)
        Y = torch.empty((m, n), device=dev)
        xt = torch.from_numpy(x).to(dev)
        _lib.call("uwc_igemm_dequant_residual_f32", A.data_ptr(), B.data_ptr(), m, n, k, sxt.data_ptr(), swt.data_ptr(),
                  xt.data_ptr(), Y.data_ptr(), st)
        assert np.array_equal(Y.cpu().numpy().view(np.uint32), (x + O.dequant(acc, sx, sw)).view(np.uint32))
    elif epilogue == "both":
        C, Y = torch.empty((m, n), dtype=torch.int32, device=dev), torch.empty((m, n), device=dev)
        _lib.call("uwc_igemm_i32_dequant_f32", A.data_ptr(), B.data_ptr(), m, n, k, sxt.data_ptr(), swt.data_ptr(),
                  C.data_ptr(), Y.data_ptr(), st)
        assert torch.equal(C, ref)
        assert np.array_equal(Y.cpu().numpy().view(np.uint32), O.dequant(acc, sx, sw).view(np.uint32))
    else:
        dt = {"i32": torch.int32, "bf16": torch.bfloat16, "f32": torch.float32}[epilogue]
        Y = _gemm(A, B, out, torch.empty((m, n), dtype=dt, device=dev), sx=sxt, sw=swt)
        if epilogue == "i32":
            assert torch.equal(Y, ref)
        elif epilogue == "f32":
            assert np.array_equal(Y.cpu().numpy().view(np.uint32), O.dequant(acc, sx, sw).view(np.uint32))
        else:
            assert np.array_equal(Y.cpu().view(torch.int16).numpy().view(np.uint16), O.scale_bf16(acc, sx, sw))
