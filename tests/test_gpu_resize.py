"""GPU parity of cvcudaResize[VarShape]Submit against the CPU oracle.

Rows are the reference's own table (tests/cvcuda/system/TestOpResize.cpp:49-91)
with seeded random inputs, plus the two benchmark configurations at full size.
Bars: NEAREST bit-exact vs the golden; LINEAR/CUBIC on integer types <= 1 LSB vs the golden (the
reference's own tolerance) and bit-exact vs the restatement of the shipped arithmetic (the float32 device
formula; for 8-bit LINEAR the 15-bit fixed-point blend, oracle variant 4); f32 cubic within 1e-4 of it.
"""
import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
NEAREST, LINEAR, CUBIC = 0, 1, 2


def make_input(orc, shape, dtype, seed):
    if np.dtype(dtype) == np.float32:
        return orc.fill_f32(shape, seed)
    raw = orc.fill_u8(tuple(shape) + (np.dtype(dtype).itemsize,), seed)
    return raw.view(dtype).reshape(shape)


def check(res, src, out_hw, interp, orc, varshape=False):
    golden = orc.resize(src, out_hw, interp, variant=0)
    device = orc.resize_shipped(src, out_hw, interp, varshape)
    if interp == NEAREST:
        np.testing.assert_array_equal(res, golden)
    elif res.dtype == np.float32:
        assert np.abs(res - device).max() <= 1e-4
    else:
        # The reference golden takes |.| of the bilinear sum as well (ResizeUtils.cpp:241-247) although
        # its device kernel does not (OpResize.cu:225-228); they only differ for negative signed
        # inputs, which the reference never tests. Follow the device there.
        if not (interp == LINEAR and np.issubdtype(res.dtype, np.signedinteger)):
            # 1 LSB is the reference's bound, which it only exercises on uint8. The device computes
            # source coordinates in float32, the golden in double: for 16-bit samples the coordinate
            # rounding (width * 2^-24 pixels) times the sample range exceeds 1 LSB on wide sources.
            lsb = 1 if res.dtype.itemsize == 1 else 1 + int(np.ceil(max(src.shape[1:3]) * 2.0 ** -24 * 65536 * 2))
            assert np.abs(res.astype(np.int64) - golden.astype(np.int64)).max() <= lsb
        # no FMA contraction on either side (integers for 8-bit LINEAR): the restatement is reproduced exactly
        np.testing.assert_array_equal(res, device)


TABLE = [
    (42, 48, 23, 24, NEAREST, 1, np.uint8, 4), (113, 12, 12, 36, NEAREST, 1, np.uint8, 4),
    (421, 148, 223, 124, NEAREST, 2, np.uint8, 4), (313, 212, 412, 336, NEAREST, 3, np.uint8, 4),
    (42, 40, 21, 20, LINEAR, 1, np.uint8, 4), (21, 21, 42, 42, LINEAR, 1, np.uint8, 4),
    (420, 420, 210, 210, LINEAR, 4, np.uint8, 4), (210, 210, 420, 420, LINEAR, 5, np.uint8, 4),
    (42, 40, 21, 20, CUBIC, 1, np.uint8, 4), (21, 21, 42, 42, CUBIC, 6, np.uint8, 4),
    (420, 420, 420, 420, CUBIC, 2, np.uint8, 4), (420, 420, 40, 42, CUBIC, 1, np.uint8, 4),
    (1920, 1080, 640, 320, CUBIC, 2, np.uint8, 4), (1080, 1920, 720, 1280, LINEAR, 1, np.uint8, 4),
    (720, 1280, 480, 854, CUBIC, 1, np.uint8, 4), (2160, 3840, 1080, 1920, LINEAR, 1, np.uint8, 4),
    (1080, 1920, 360, 640, CUBIC, 1, np.uint8, 4),
] + [(42, 48, 23, 24, interp, 1, dt, c) for dt in (np.uint8, np.uint16, np.int16, np.float32) for c in (1, 3, 4)
     for interp in (NEAREST, LINEAR, CUBIC)]


@pytest.mark.parametrize("row", TABLE, ids=lambda r: "%dx%d-%dx%d-i%d-n%d-%s%d" % (r[:6] + (np.dtype(r[6]).name, r[7])))
def test_tensor_table(cv, orc, gpu, row):
    sw, sh, dw, dh, interp, n, dt, c = row
    src = make_input(orc, (n, sh, sw, c), dt, 0xC0FFEE01 + sw + 31 * sh + c)
    tin = cv.Tensor.from_numpy(src, "NHWC")
    tout = cv.Tensor.alloc([n, dh, dw, c], dt, "NHWC")
    cv.Resize()(None, tin, tout, interp)
    torch.cuda.synchronize()
    check(tout.numpy(), src, (dh, dw), interp, orc)


# bicubic reductions by 2x or more take the tap-major kernel (pixels of whole dwords only): ragged
# tiles, sources narrower than the 4-tap window, every staged pixel size
STAGED = [(sw, sh, dw, dh, CUBIC, n, dt, c)
          for (sw, sh, dw, dh, n) in [(131, 37, 65, 9, 2), (640, 50, 67, 13, 1), (3, 9, 1, 2, 1), (7, 5, 3, 6, 3),
                                      (1000, 20, 130, 10, 1)]
          for dt, c in [(np.uint8, 4), (np.uint16, 4), (np.int16, 4), (np.float32, 1), (np.float32, 3),
                        (np.float32, 4)]]


@pytest.mark.parametrize("row", STAGED, ids=lambda r: "%dx%d-%dx%d-i%d-n%d-%s%d" % (r[:6] + (np.dtype(r[6]).name, r[7])))
def test_tensor_cubic_reduction(cv, orc, gpu, row):
    test_tensor_table(cv, orc, gpu, row)


# 8-bit bicubic at vertical scales up to 4 walks the source rows, here 4 and 8 output rows per wave: the benchmark's images, ragged
# widths and heights, scale 2 exactly (every window advances by 2), 1.25, an enlargement beyond 2, horizontal enlargement with
# vertical reduction
STRIPS = [(sw, sh, dw, dh, CUBIC, n, np.uint8, c)
          for c in (3, 4, 1)
          for (sw, sh, dw, dh, n) in [(1920, 1080, 1280, 720, 3), (1917, 1083, 1283, 719, 3), (1024, 1408, 512, 704, 8),
                                      (1600, 900, 1280, 720, 3), (640, 360, 1000, 1100, 2), (300, 1080, 700, 720, 6),
                                      # enlargements: by 1.5, by 2 exactly (the limit of the enlarging strips), by 1.2 with
                                      # ragged sizes, and equal heights (every window advances by 1)
                                      (1280, 720, 1920, 1080, 2), (640, 360, 1280, 720, 3), (1003, 601, 1201, 721, 3),
                                      (1920, 720, 1280, 720, 3)]]


@pytest.mark.parametrize("row", STRIPS, ids=lambda r: "%dx%d-%dx%d-i%d-n%d-%s%d" % (r[:6] + (np.dtype(r[6]).name, r[7])))
def test_tensor_cubic_u8_strips(cv, orc, gpu, row):
    test_tensor_table(cv, orc, gpu, row)


# The same at its limits: outputs one column short of a wave, a wave and one more (the last tile overlaps its neighbour); rows of
# 16 bytes and of 8; four source rows; vertical scale 4 and a little more (three and four channels; one channel, which walks from
# 128 columns on, and launches that pass every line: the test after this one)
@pytest.mark.parametrize("c", [1, 3, 4])
@pytest.mark.parametrize("shape", [(40, 30, 63, 67, 64), (40, 30, 64, 67, 64), (40, 30, 65, 67, 32), (200, 31, 257, 61, 64), (254, 64, 255, 64, 64),
                                   (9, 4, 71, 64, 64), (6, 9, 66, 33, 128), (90, 256, 68, 64, 64), (90, 260, 68, 64, 64), (129, 70, 99, 66, 64),
                                   (260, 70, 66, 66, 64), (270, 70, 66, 66, 64), (4, 40, 4, 71, 256), (333, 5, 999, 640, 2), (600, 70, 154, 66, 64), (610, 70, 154, 66, 64),
                                   (9, 40, 128, 64, 64), (165, 40, 127, 64, 64)],
                         ids=lambda sh: "%dx%d-%dx%d-n%d" % sh)
def test_tensor_cubic_u8_walks(cv, orc, gpu, shape, c):
    sw, sh, dw, dh, n = shape
    src = make_input(orc, (n, sh, sw, c), np.uint8, 0x11 + sw + dw + c)
    out = torch.full((n, dh, dw, c), 7, dtype=torch.uint8, device="cuda")
    cv.Resize()(None, cv.Tensor.from_torch(torch.from_numpy(src).cuda(), "NHWC"), cv.Tensor.from_torch(out, "NHWC"), CUBIC)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(out.cpu().numpy(), orc.resize_shipped(src, (dh, dw), CUBIC, threads=8))


# The same in launches on both sides of each line that decides it: (channels, source, output, images, columns between output rows).
# Strips of 4, 8, 16 and 32 rows, the last of an image one row or cut off; 32 only under a row pitch of whole lines of 64 bytes;
# reductions by more than 2 (one channel: 1.75), also with a quarter of the lanes idle. One channel: horizontal scales on both sides of
# 1.3 (one 8-byte load or two) and of 3.9, rows of 8 bytes, four source rows, vertical scale 4
WALKS = [(1, 169, 70, 130, 66, 64, 0), (1, 170, 70, 130, 66, 64, 0), (1, 507, 70, 130, 66, 64, 0), (1, 508, 70, 130, 66, 64, 0),
         (1, 8, 40, 128, 64, 64, 0), (1, 7, 40, 128, 64, 64, 0), (1, 260, 4, 255, 66, 61, 0), (1, 300, 264, 200, 66, 90, 0),
         (1, 300, 264, 200, 66, 91, 0), (1, 300, 264, 191, 66, 91, 3), (1, 300, 265, 200, 66, 91, 0),
         (1, 250, 9, 256, 9, 767, 0), (1, 250, 9, 256, 9, 768, 0), (1, 250, 20, 256, 17, 2047, 0), (1, 250, 20, 256, 17, 2048, 0),
         (1, 200, 25, 256, 33, 8191, 0), (1, 200, 25, 256, 33, 8192, 0), (1, 200, 25, 256, 33, 8192, 1),
         (3, 40, 20, 64, 9, 1400, 0), (3, 64, 264, 64, 66, 481, 0), (3, 64, 264, 64, 66, 482, 0), (3, 70, 264, 70, 66, 300, 5),
         (3, 60, 8, 66, 9, 639, 0), (3, 60, 8, 66, 9, 640, 0), (3, 60, 12, 66, 9, 1023, 0), (3, 60, 12, 66, 9, 1024, 2),
         (3, 50, 20, 64, 17, 2559, 0), (3, 50, 20, 64, 17, 2560, 0), (3, 41, 30, 64, 33, 8191, 0), (3, 41, 30, 64, 33, 8192, 0),
         (3, 41, 30, 64, 47, 8192, 1), (4, 64, 264, 64, 66, 240, 0), (4, 64, 264, 64, 66, 241, 0), (4, 40, 20, 60, 9, 1023, 0),
         (4, 40, 20, 60, 9, 1024, 0), (4, 50, 20, 60, 17, 2048, 3), (4, 41, 30, 64, 33, 8192, 0), (4, 41, 30, 64, 33, 8192, 1)]


@pytest.mark.parametrize("row", WALKS, ids=lambda r: "x%d-%dx%d-%dx%d-n%d-gap%d" % r)
def test_tensor_cubic_u8_walks_by_launch(cv, orc, gpu, row):
    c, sw, sh, dw, dh, n, gap = row
    some = make_input(orc, (3, sh, sw, c), np.uint8, 0x31 + sw + dw + c)
    which = torch.arange(n, device="cuda") % 3  # (images next to each other differ)
    src = torch.from_numpy(some).cuda()[which]
    out = torch.full((n, dh, dw + gap, c), 7, dtype=torch.uint8, device="cuda")
    cv.Resize()(None, cv.Tensor.from_torch(src, "NHWC"), cv.Tensor.from_torch(out[:, :, :dw], "NHWC"), CUBIC)
    torch.cuda.synchronize()
    want = torch.from_numpy(orc.resize_shipped(some, (dh, dw), CUBIC, threads=8)).cuda()
    assert torch.equal(out[:, :, :dw], want[which])
    assert bool((out[:, :, dw:] == 7).all())


# 8-bit bilinear in launches of few waves, whose strips are 2 rows (two columns per lane; four, up to 768 strips of 8) and 4 (four
# columns, up to 3072): one row, heights one off a strip's, widths one off a wave's and of one column, vertical reductions by 2 (all
# of a strip's windows), a little more and 5 (steps), and the launches on both sides of each line
@pytest.mark.parametrize("c", [1, 3, 4])
@pytest.mark.parametrize("shape", [(40, 30, 61, 1, 1), (40, 30, 1, 31, 2), (40, 30, 257, 33, 1), (100, 33, 255, 34, 3), (5, 3, 77, 19, 9),
                                   (400, 60, 127, 30, 3), (250, 70, 129, 35, 2), (130, 70, 126, 33, 2), (130, 70, 128, 14, 2),
                                   (90, 80, 256, 40, 7), (64, 16, 256, 24, 256), (64, 16, 256, 25, 256), (64, 16, 257, 24, 512),
                                   (64, 16, 256, 25, 768), (64, 16, 256, 25, 769), (120, 17, 128, 16, 1024), (120, 17, 128, 17, 1024)],
                         ids=lambda sh: "%dx%d-%dx%d-n%d" % sh)
def test_tensor_linear_u8_small_launches(cv, orc, gpu, shape, c):
    sw, sh, dw, dh, n = shape
    src = make_input(orc, (n, sh, sw, c), np.uint8, 0x51 + sw + dw + c)
    out = torch.full((n, dh, dw + 3, c), 7, dtype=torch.uint8, device="cuda")
    cv.Resize()(None, cv.Tensor.from_torch(torch.from_numpy(src).cuda(), "NHWC"), cv.Tensor.from_torch(out[:, :, :dw], "NHWC"), LINEAR)
    torch.cuda.synchronize()
    got = out.cpu().numpy()
    np.testing.assert_array_equal(got[:, :, :dw], orc.resize_shipped(src, (dh, dw), LINEAR, threads=8))
    assert (got[:, :, dw:] == 7).all()


# 8-bit nearest neighbour enlarging by 1.5 or more horizontally (and not reducing vertically) runs as strips once the
# launch has 2048 of them: 1.5, 2 and 3 times, ragged sizes, mixed scales (2.5 across, 1 down: every source row once),
# and a vertical reduction with the same widths (wave patches)
NN_STRIPS = [(sw, sh, dw, dh, NEAREST, n, np.uint8, c)
             for c in (3, 1, 4)
             for (sw, sh, dw, dh, n) in [(1280, 720, 1920, 1080, 2), (640, 360, 1280, 720, 6), (427, 241, 1283, 725, 6),
                                         (512, 720, 1280, 720, 6), (512, 720, 1280, 700, 6), (9, 2000, 30, 2100, 8)]]


@pytest.mark.parametrize("row", NN_STRIPS, ids=lambda r: "%dx%d-%dx%d-i%d-n%d-%s%d" % (r[:6] + (np.dtype(r[6]).name, r[7])))
def test_tensor_nearest_u8_strips(cv, orc, gpu, row):
    test_tensor_table(cv, orc, gpu, row)


# Nearest neighbour of 1 and 3 channels in rows of 256: at their limits (one channel's windows of 2 dwords up to a scale of 4 / 3, of
# 4 up to 4; three channels up to 1; 2560 strips of 8 rows, 2 of 5 of the last tile's columns, 24 source columns), each side of
# them, over packed rows of odd widths and pitched ones, where the image's last row is used and where it is not
@pytest.mark.parametrize("c", [1, 3])
@pytest.mark.parametrize("row_align", [0, 1])
@pytest.mark.parametrize("size", [(300, 9, 256, 9, 1280), (341, 13, 256, 9, 1280), (342, 13, 256, 9, 1280), (1024, 20, 256, 9, 1280),
                                  (1025, 20, 256, 9, 1280), (399, 40, 397, 17, 427), (24, 30, 103, 9, 1280), (23, 30, 103, 9, 1280),
                                  (99, 30, 102, 9, 1280), (255, 12, 256, 9, 1280), (255, 9, 256, 11, 1280), (257, 9, 257, 9, 640),
                                  (513, 33, 514, 7, 853), (511, 36, 509, 12, 640), (100, 9, 1021, 6, 640), (100, 9, 1021, 6, 639)])
def test_tensor_nearest_u8_rows(cv, orc, gpu, size, row_align, c):
    sw, sh, dw, dh, n = size
    src = orc.fill_u8((n, sh, sw, c), 77 + sw)
    tin  = cv.Tensor.from_numpy(src, "NHWC", row_align=row_align)
    tout = cv.Tensor.alloc([n, dh, dw, c], np.uint8, "NHWC", row_align=row_align)
    tout.torch_view().fill_(7)
    cv.Resize()(None, tin, tout, NEAREST)
    np.testing.assert_array_equal(tout.numpy(), orc.resize(src, (dh, dw), NEAREST, variant=0))


# the strip kernels on views that start at an odd byte and have an odd row pitch (their window loads take the aligned
# dwords around a pixel: nothing may be assumed of where a row starts), output bytes outside the rows untouched
@pytest.mark.parametrize("c", [3, 1, 4])
@pytest.mark.parametrize("shape", [(1531, 700, 1021, 467, LINEAR), (701, 500, 1283, 915, LINEAR), (1531, 700, 1021, 467, CUBIC),
                                   (701, 500, 1283, 915, CUBIC), (701, 500, 1283, 915, NEAREST)],
                         ids=lambda sh: "%dx%d-%dx%d-i%d" % sh)
def test_strips_on_odd_bases_and_pitches(cv, orc, gpu, shape, c):
    sw, sh, dw, dh, interp = shape
    n = 6
    src = make_input(orc, (n, sh, sw, c), np.uint8, 0xBEEF + sw + c)

    def view(w, h, fill):
        pitch, plane = w * c + 3, (w * c + 3) * h + 7
        buf = torch.full((n * plane + 64,), fill, dtype=torch.uint8, device="cuda")
        t = cv.Tensor.wrap(buf.data_ptr() + 1, [n, h, w, c], [plane, pitch, c, 1], np.uint8, "NHWC", keep=buf)
        return buf, t, torch.as_strided(buf[1:], (n, h, w, c), (plane, pitch, c, 1)), (plane, pitch)

    big_in, tin, in_view, _ = view(sw, sh, 0)
    in_view.copy_(torch.from_numpy(src).cuda())
    big_out, tout, out_view, (plane, pitch) = view(dw, dh, 0xCD)
    cv.Resize()(None, tin, tout, interp)
    torch.cuda.synchronize()
    check(out_view.cpu().numpy(), src, (dh, dw), interp, orc)
    mask = torch.ones_like(big_out, dtype=torch.bool)
    torch.as_strided(mask[1:], (n, dh, dw * c), (plane, pitch, 1)).fill_(False)
    assert bool((big_out[mask] == 0xCD).all())


# 8-bit bilinear at horizontal scales up to 2 takes the kernel in which a lane owns two columns: both
# directions, the scale limit itself, ragged widths (1 - 3 columns left over), odd heights, tiny outputs
PAIRS = [(sw, sh, dw, dh, LINEAR, n, np.uint8, c)
         for c in (3, 1, 4)
         for (sw, sh, dw, dh, n) in [(131, 37, 66, 19, 2), (100, 40, 50, 20, 1), (64, 48, 97, 71, 2), (640, 360, 431, 243, 1),
                                     (33, 9, 130, 30, 1), (5, 4, 7, 3, 3), (4, 4, 2, 2, 1), (257, 33, 129, 17, 1),
                                     (1280, 720, 1920, 1080, 1), (1920, 1080, 1280, 720, 1),
                                     # enlargements by 1.5 or more: four columns per lane; ragged widths, odd heights,
                                     # the limit itself (3 * src == 2 * dst), one wave's worth and less
                                     (100, 40, 151, 61, 2), (257, 33, 771, 99, 1), (40, 30, 61, 46, 1), (4, 4, 7, 9, 2),
                                     (640, 360, 1921, 1079, 1), (86, 20, 129, 30, 1), (171, 7, 257, 11, 1),
                                     (6, 5, 9, 8, 1), (341, 50, 1023, 75, 1)]]


@pytest.mark.parametrize("row", PAIRS, ids=lambda r: "%dx%d-%dx%d-i%d-n%d-%s%d" % (r[:6] + (np.dtype(r[6]).name, r[7])))
def test_tensor_linear_u8_pair_columns(cv, orc, gpu, row):
    test_tensor_table(cv, orc, gpu, row)


def test_output_padding_is_untouched_and_hwc_layout(cv, orc, gpu):
    src = make_input(orc, (1, 33, 47, 3), np.uint8, 5)
    tin = cv.Tensor.from_numpy(src[0], "HWC")
    tout = cv.Tensor.alloc([20, 30, 3], np.uint8, "HWC")
    d = tout.export()
    pitch = d.buffer.strides[0]
    assert pitch > 30 * 3
    raw = cv._bytes_view(d.buffer.basePtr, pitch * 20, tout)
    raw.fill_(0xAB)
    cv.Resize()(None, tin, tout, LINEAR)
    torch.cuda.synchronize()
    check(tout.numpy()[None], src, (20, 30), LINEAR, orc)
    pad = raw.view(20, pitch)[:, 30 * 3:].cpu().numpy()
    assert (pad == 0xAB).all()


def test_config1_full_size_and_knife_edge_columns(cv, orc, gpu):
    # batch 8, u8 NHWC 3ch 1920x1080 -> 224x224; nearest bit-exact, linear <= 1 LSB.
    src = orc.fill_u8((8, 1080, 1920, 3), 0xC0FFEE01)
    tin = cv.Tensor.from_numpy(src, "NHWC")
    for interp in (NEAREST, LINEAR):
        tout = cv.Tensor.alloc([8, 224, 224, 3], np.uint8, "NHWC")
        cv.Resize()(None, tin, tout, interp)
        torch.cuda.synchronize()
        check(tout.numpy(), src, (224, 224), interp, orc)
    # a ramp image (value = column index) exposes any deviation of the nearest index on the 32
    # columns dx = 3 (mod 7) where (dx+.5)*1920/224 is an exact integer
    ramp = np.tile(np.arange(1920, dtype=np.uint16).reshape(1, 1, 1920, 1), (1, 4, 1, 1))
    tout = cv.Tensor.alloc([1, 4, 224, 1], np.uint16, "NHWC")
    cv.Resize()(None, cv.Tensor.from_numpy(ramp, "NHWC"), tout, NEAREST)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(tout.numpy(), orc.resize(ramp, (4, 224), NEAREST))


def test_config5_bicubic_f32_full_size(cv, orc, gpu):
    # batch 16 f32 NHWC 4ch 3840x2160 -> 640x360, values in [0,1), 1e-4 abs. Every image
    # is different (one random image rolled by 5 * n columns and 3 * n rows) and all 16 go through the oracle.
    N = 16
    one = orc.fill_f32((2160, 3840, 4), 0xC0FFEE05)
    tin = cv.Tensor.alloc([N, 2160, 3840, 4], np.float32, "NHWC")
    view = tin.torch_view()
    refs = []
    for n in range(N):
        img = np.roll(one, (3 * n, 5 * n), axis=(0, 1))
        view[n].copy_(torch.from_numpy(img))
        refs.append(orc.resize(img[None], (360, 640), CUBIC, variant=1, threads=8)[0])
    tout = cv.Tensor.alloc([N, 360, 640, 4], np.float32, "NHWC")
    cv.Resize()(None, tin, tout, CUBIC)
    torch.cuda.synchronize()
    res = tout.numpy()
    for n in range(N):
        assert np.abs(res[n] - refs[n]).max() <= 1e-4, n
    assert not (res[1] == res[0]).all()


def _format_for(cv, K, dt, c):
    import cvcuda_amd._capi as capi
    kind = {np.uint8: K.DATA_KIND_UNSIGNED, np.uint16: K.DATA_KIND_UNSIGNED, np.int16: K.DATA_KIND_SIGNED,
            np.float32: K.DATA_KIND_FLOAT}[dt]
    bits = np.dtype(dt).itemsize * 8
    pack = getattr(K, "PACKING_" + "_".join("%s%d" % (n, bits) for n in "XYZW"[:c]))
    swz = [K.SWIZZLE_X000, None, K.SWIZZLE_XYZ1, K.SWIZZLE_XYZW][c - 1]
    f = C.c_uint64()
    cv.check(capi.nvcv.nvcvMakeNonColorImageFormat(C.byref(f), K.MEM_LAYOUT_PL, kind, swz, pack, 0, 0, 0,
                                                   K.ALPHA_ASSOCIATED, None))
    return f.value


@pytest.mark.parametrize("interp", [NEAREST, LINEAR, CUBIC])
@pytest.mark.parametrize("dt,c", [(np.uint8, 3), (np.uint8, 4), (np.uint8, 1), (np.uint16, 3), (np.int16, 4),
                                  (np.float32, 1), (np.float32, 4)])
def test_varshape(cv, K, orc, gpu, interp, dt, c):
    rng = np.random.default_rng(17)
    fmt = _format_for(cv, K, dt, c)
    n = 7
    bin_, bout, hosts, outs = cv.ImageBatchVarShape(n), cv.ImageBatchVarShape(n), [], []
    for i in range(n):
        sw, sh = int(rng.integers(20, 300)), int(rng.integers(20, 200))
        dw, dh = int(rng.integers(10, 350)), int(rng.integers(10, 250))
        a = make_input(orc, (sh, sw, c), dt, 100 + i)
        hosts.append(a)
        bin_.push_back(cv.Image.from_numpy(a, fmt))
        o = cv.Image.alloc((dw, dh), fmt)
        outs.append(o)
        bout.push_back(o)
    cv.Resize()(None, bin_, bout, interp)
    torch.cuda.synchronize()
    for a, o in zip(hosts, outs):
        w, h = o.size
        res = o.plane_view(0, dt, c).cpu().numpy()[None]
        check(res, a[None], (h, w), interp, orc, varshape=True)


# large image batches of 8-bit bilinear resizes run in the tensor kernels' strips: mostly enlarged by 1.5 or more (wide
# tiles, with a reduced and a strongly reduced image among them), mostly reduced or slightly enlarged (narrow tiles)
@pytest.mark.parametrize("c", [3, 1, 4])
@pytest.mark.parametrize("mix", ["enlarging", "reducing"])
def test_varshape_linear_u8_strips(cv, K, orc, gpu, mix, c):
    rng = np.random.default_rng(23 + c)
    fmt = _format_for(cv, K, np.uint8, c)
    n = 16  # (2048 tiles and more of 256 x 32, respectively 128 x 16)
    bin_, bout, hosts, outs = cv.ImageBatchVarShape(n), cv.ImageBatchVarShape(n), [], []
    for i in range(n):
        if mix == "enlarging":
            sw, sh = int(rng.integers(700, 900)), int(rng.integers(500, 650))
            f = [1.5, 1.9, 2.0, 3.1][i % 4] if i < n - 2 else [0.7, 0.3][i - (n - 2)]
        else:
            sw, sh = int(rng.integers(900, 1300)), int(rng.integers(500, 800))
            f = [1 / 1.5, 0.5, 0.9, 1.2, 1 / 1.51][i % 5] if i < n - 2 else [0.31, 1.6][i - (n - 2)]
        dw, dh = max(1, int(sw * f) + int(rng.integers(0, 3))), max(1, int(sh * f) + int(rng.integers(0, 3)))
        a = make_input(orc, (sh, sw, c), np.uint8, 500 + i)
        hosts.append(a)
        bin_.push_back(cv.Image.from_numpy(a, fmt))
        o = cv.Image.alloc((dw, dh), fmt)
        outs.append(o)
        bout.push_back(o)
    cv.Resize()(None, bin_, bout, LINEAR)
    torch.cuda.synchronize()
    for a, o in zip(hosts, outs):
        w, h = o.size
        res = o.plane_view(0, np.uint8, c).cpu().numpy()[None]
        check(res, a[None], (h, w), LINEAR, orc, varshape=True)


# large image batches of 8-bit nearest-neighbour enlargements of 1 and 3 channels run in the tensor kernel's strips
# (256 x 32 tiles, 2048 and more), images of other scales among them as patches
@pytest.mark.parametrize("c", [3, 1])
def test_varshape_nearest_u8_strips(cv, K, orc, gpu, c):
    rng = np.random.default_rng(61 + c)
    fmt = _format_for(cv, K, np.uint8, c)
    n = 16
    bin_, bout, hosts, outs = cv.ImageBatchVarShape(n), cv.ImageBatchVarShape(n), [], []
    for i in range(n):
        sw, sh = int(rng.integers(700, 900)), int(rng.integers(500, 650))
        f = [1.5, 1.9, 2.0, 3.1][i % 4] if i < n - 2 else [0.7, 1.2][i - (n - 2)]
        dw, dh = max(1, int(sw * f) + int(rng.integers(0, 3))), max(1, int(sh * f) + int(rng.integers(0, 3)))
        a = make_input(orc, (sh, sw, c), np.uint8, 900 + i)
        hosts.append(a)
        bin_.push_back(cv.Image.from_numpy(a, fmt))
        o = cv.Image.alloc((dw, dh), fmt)
        outs.append(o)
        bout.push_back(o)
    cv.Resize()(None, bin_, bout, NEAREST)
    torch.cuda.synchronize()
    for a, o in zip(hosts, outs):
        w, h = o.size
        res = o.plane_view(0, np.uint8, c).cpu().numpy()[None]
        check(res, a[None], (h, w), NEAREST, orc, varshape=True)


# large image batches of 8-bit bicubic resizes of 3 and 4 channels walk the source rows like the tensor kernels (64 x 64
# tiles, 2048 and more): reductions up to 2, enlargements up to 2, and a few images beyond among them
@pytest.mark.parametrize("c", [3, 4])
def test_varshape_cubic_u8_strips(cv, K, orc, gpu, c):
    rng = np.random.default_rng(41 + c)
    fmt = _format_for(cv, K, np.uint8, c)
    n = 16
    bin_, bout, hosts, outs = cv.ImageBatchVarShape(n), cv.ImageBatchVarShape(n), [], []
    for i in range(n):
        sw, sh = int(rng.integers(600, 900)), int(rng.integers(400, 650))
        f = [1 / 1.5, 1.5, 2.0, 0.5, 1.0, 1.25][i % 6] if i < n - 2 else [0.3, 2.6][i - (n - 2)]
        dw, dh = max(1, int(sw * f) + int(rng.integers(0, 3))), max(1, int(sh * f) + int(rng.integers(0, 3)))
        a = make_input(orc, (sh, sw, c), np.uint8, 700 + i)
        hosts.append(a)
        bin_.push_back(cv.Image.from_numpy(a, fmt))
        o = cv.Image.alloc((dw, dh), fmt)
        outs.append(o)
        bout.push_back(o)
    cv.Resize()(None, bin_, bout, CUBIC)
    torch.cuda.synchronize()
    for a, o in zip(hosts, outs):
        w, h = o.size
        res = o.plane_view(0, np.uint8, c).cpu().numpy()[None]
        check(res, a[None], (h, w), CUBIC, orc, varshape=True)


AREA = 3
AREA_ROWS = [(44, 40, 22, 20, 2, np.uint8, 4), (30, 30, 20, 20, 2, np.uint8, 4), (30, 30, 60, 60, 4, np.uint8, 4),
             (1440, 2560, 1080, 1920, 1, np.uint8, 4), (720, 1280, 360, 640, 1, np.uint8, 4),
             (1440, 2560, 720, 1280, 1, np.uint8, 4), (1920, 1080, 224, 224, 2, np.uint8, 3),
             (97, 61, 13, 9, 2, np.uint16, 1), (97, 61, 13, 9, 2, np.int16, 3), (97, 61, 40, 33, 2, np.float32, 4),
             # u8x3 at horizontal scales up to 2 (one 12-byte load per source row): 1.5, fractional, exactly 2 and 1,
             # an enlargement, a mixed pair of scales, sources barely wider than the load
             (1920, 1080, 1280, 720, 1, np.uint8, 3), (97, 61, 61, 40, 2, np.uint8, 3), (64, 48, 32, 24, 2, np.uint8, 3),
             (33, 21, 33, 21, 1, np.uint8, 3), (50, 40, 75, 60, 2, np.uint8, 3), (40, 90, 31, 20, 2, np.uint8, 3),
             (4, 4, 3, 3, 1, np.uint8, 3), (5, 9, 3, 2, 2, np.uint8, 3), (640, 3, 427, 2, 1, np.uint8, 3),
             # the same form for 1- and 4-byte pixels
             (97, 61, 61, 40, 2, np.uint8, 1), (64, 48, 32, 24, 2, np.uint8, 1), (50, 40, 75, 60, 2, np.uint8, 1),
             (5, 9, 3, 2, 2, np.uint8, 1), (97, 61, 61, 40, 2, np.uint8, 4), (50, 40, 75, 60, 2, np.uint8, 4),
             (5, 9, 3, 2, 2, np.uint8, 4), (1920, 1080, 1280, 720, 1, np.uint8, 4)]


@pytest.mark.parametrize("row", AREA_ROWS, ids=lambda r: "%dx%d-%dx%d-n%d-%s%d" % (r[:5] + (np.dtype(r[5]).name, r[6])))
def test_area_tensor(cv, orc, gpu, row):
    # box-filter resize, tensors (reference rows TestOpResize.cpp:67-78 plus other types and the
    # 1080p -> 224 case): <= 1 LSB against the float64 golden, and against the restatement of the shipped
    # arithmetic (8-bit pixels at reductions of up to 3: the fixed-point form; otherwise the reference's device
    # order in float32) exactly for integers, within float rounding of the long sums for float32
    sw, sh, dw, dh, n, dt, c = row
    src = make_input(orc, (n, sh, sw, c), dt, 0xA0EA + sw + dh)
    tout = cv.Tensor.alloc([n, dh, dw, c], dt, "NHWC")
    cv.Resize()(None, cv.Tensor.from_numpy(src, "NHWC"), tout, AREA)
    torch.cuda.synchronize()
    res = tout.numpy()
    golden = orc.resize(src, (dh, dw), AREA, variant=0, threads=8)
    device = orc.resize_shipped(src, (dh, dw), AREA, threads=8)
    if dt == np.float32:
        assert np.abs(res - device).max() <= 1e-5 and np.abs(res - golden).max() <= 1e-4
    else:
        np.testing.assert_array_equal(res, device)
        # the golden's box filter and the device expression part ways on fractional enlargements (there the device
        # weights do not sum to 1); the reference's own rows hold reductions and the exact 2x enlargement
        if (sw >= dw and sh >= dh) or (dw == 2 * sw and dh == 2 * sh):
            assert np.abs(res.astype(np.int64) - golden.astype(np.int64)).max() <= 1


# the window form of larger reductions: whole scales of every window size, scales just below and above them, the widest,
# axes that differ (one of them within the fixed-point form's 3), boxes at the right and lower edge, output columns that
# leave most of a wave idle; dense odd rows and views whose rows start anywhere
@pytest.mark.parametrize("sw,sh,dw,dh", [(256, 64, 64, 16), (390, 66, 65, 11), (512, 40, 64, 5), (780, 60, 65, 5), (257, 65, 64, 16),
                                         (391, 67, 79, 11), (511, 41, 86, 5), (600, 50, 76, 9), (779, 61, 65, 5), (100, 90, 33, 8),
                                         (133, 99, 129, 9), (67, 31, 20, 30), (64, 200, 16, 20), (90, 13, 8, 4), (1201, 45, 101, 4)])
@pytest.mark.parametrize("c", [1, 3, 4])
@pytest.mark.parametrize("kind", ["dense", "view"])
def test_area_larger_reductions(cv, orc, gpu, sw, sh, dw, dh, c, kind):
    src = make_input(orc, (2, sh, sw, c), np.uint8, 0xA3EA + sw + dh)
    lead, pitch = (0, sw * c) if kind == "dense" else (3, sw * c + 5)
    # exactly the rows and nothing behind the last one
    buf = torch.zeros(lead + (2 * sh - 1) * pitch + sw * c, dtype=torch.uint8, device="cuda")
    torch.as_strided(buf, (2, sh, sw, c), (sh * pitch, pitch, c, 1), lead).copy_(torch.from_numpy(src).cuda())
    tin = cv.Tensor.wrap(buf.data_ptr() + lead, [2, sh, sw, c], [sh * pitch, pitch, c, 1], np.uint8, "NHWC", keep=buf)
    out = torch.zeros((2, dh, dw, c), dtype=torch.uint8, device="cuda")
    cv.Resize()(None, tin, cv.Tensor.from_torch(out, "NHWC"), AREA)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(out.cpu().numpy(), orc.resize_shipped(src, (dh, dw), AREA, threads=8))


# every width of the window, at whole scales and just above and below them (the widest boxes of a width)
@pytest.mark.parametrize("sw,dw", [(300, 75), (299, 75), (301, 75), (375, 75), (374, 75), (376, 75), (449, 75), (451, 75),
                                   (599, 75), (601, 75), (675, 75), (749, 75), (751, 75), (899, 75), (900, 75)])
@pytest.mark.parametrize("c", [1, 3, 4])
def test_area_window_widths(cv, orc, gpu, sw, dw, c):
    src = make_input(orc, (2, 47, sw, c), np.uint8, 0xA0 + sw)
    tout = cv.Tensor.alloc([2, 11, dw, c], np.uint8, "NHWC")
    cv.Resize()(None, cv.Tensor.from_numpy(src, "NHWC"), tout, AREA)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(tout.numpy(), orc.resize_shipped(src, (11, dw), AREA, threads=8))


# the last tile's lanes without columns: all of them work up to 1024 blocks, beyond that those below 16
@pytest.mark.parametrize("c", [1, 3, 4])
@pytest.mark.parametrize("dw", [8, 15, 16, 17, 65, 79, 80, 127])
@pytest.mark.parametrize("blocks", [1024, 1040])
def test_area_window_idle_lanes(cv, orc, gpu, blocks, dw, c):
    test_tensor_table(cv, orc, gpu, (dw * 7 // 2 + 60 // c, 83, dw, 32, AREA, blocks // 8 // -(-dw // 64), np.uint8, c))


# boxes of 4 to 11 rows: whole batches of the window form's rows, and one and two rows behind them, with partial rows and not
@pytest.mark.parametrize("sh", [44, 55, 66, 77, 88, 99, 110, 121, 43, 56, 87, 100])
@pytest.mark.parametrize("c,dw", [(1, 45), (3, 45), (3, 62), (4, 45), (4, 78)])
def test_area_window_rows(cv, orc, gpu, sh, c, dw):
    src = make_input(orc, (2, sh, 315, c), np.uint8, 0xA7 + sh)
    tout = cv.Tensor.alloc([2, 11, dw, c], np.uint8, "NHWC")
    cv.Resize()(None, cv.Tensor.from_numpy(src, "NHWC"), tout, AREA)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(tout.numpy(), orc.resize_shipped(src, (11, dw), AREA, threads=8))


# boxes that are walked one lane per pixel in launches of many blocks and by windows in smaller ones: just below and at the
# numbers of blocks where that changes (an image of 8 rows is two blocks)
@pytest.mark.parametrize("n,sw,sh,dw,dh,c", [(255, 80, 32, 20, 8, 3), (256, 80, 32, 20, 8, 3), (680, 80, 48, 20, 8, 3),
                                             (128, 160, 16, 20, 8, 3), (128, 240, 16, 20, 8, 3), (127, 160, 16, 20, 8, 3),
                                             (63, 30, 832, 20, 256, 3), (64, 30, 832, 20, 256, 3), (511, 30, 40, 20, 8, 4),
                                             (512, 30, 40, 20, 8, 4), (512, 40, 33, 20, 8, 4), (127, 160, 16, 20, 8, 4),
                                             (128, 160, 16, 20, 8, 4), (512, 160, 16, 20, 8, 4)])
def test_area_small_boxes_in_large_launches(cv, orc, gpu, n, sw, sh, dw, dh, c):
    src = make_input(orc, (n, sh, sw, c), np.uint8, 0xA9 + n)
    tout = cv.Tensor.alloc([n, dh, dw, c], np.uint8, "NHWC")
    cv.Resize()(None, cv.Tensor.from_numpy(src, "NHWC"), tout, AREA)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(tout.numpy(), orc.resize_shipped(src, (dh, dw), AREA, threads=8))


# the row windows of the bicubic strips, the bicubic patches and the box filter, on dense images whose rows start at every
# byte of a dword in turn, from every start of the first: the buffer ends with the image, whose last rows are read
@pytest.mark.parametrize("c", [3, 1])
@pytest.mark.parametrize("lead", [0, 1, 2, 3])
@pytest.mark.parametrize("shape", [(1535, 703, 1021, 467, CUBIC, 6), (701, 101, 1285, 151, CUBIC, 1), (703, 90, 401, 57, AREA, 2),
                                   (131, 37, 67, 19, AREA, 1), (67, 19, 66, 18, CUBIC, 2), (701, 501, 1003, 751, CUBIC, 5)],
                         ids=lambda sh: "%dx%d-%dx%d-i%d-n%d" % sh)
def test_rows_from_every_byte_of_a_dword(cv, orc, gpu, shape, lead, c):
    sw, sh, dw, dh, interp, n = shape
    src = make_input(orc, (n, sh, sw, c), np.uint8, 0xD0D + sw + lead)
    buf = torch.zeros(lead + src.size, dtype=torch.uint8, device="cuda")
    buf[lead:].copy_(torch.from_numpy(src.reshape(-1)))
    tin = cv.Tensor.wrap(buf.data_ptr() + lead, [n, sh, sw, c], [sh * sw * c, sw * c, c, 1], np.uint8, "NHWC", keep=buf)
    tout = cv.Tensor.alloc([n, dh, dw, c], np.uint8, "NHWC")
    cv.Resize()(None, tin, tout, interp)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(tout.numpy(), orc.resize_shipped(src, (dh, dw), interp, threads=8))


def test_area_sources_one_and_two_pixels_wide(cv, orc, gpu):
    # u8x3 rows shorter than the 4- and 8-byte tap loads: 1 x 1, 1 x H, 2 x 1 and W x 1 sources, every
    # interpolation (the tap loads of the last row must not be moved in front of the row)
    for (sw, sh) in ((1, 1), (1, 7), (2, 1), (2, 5), (9, 1)):
        src = make_input(orc, (2, sh, sw, 3), np.uint8, 31 * sw + sh)
        for interp in (NEAREST, LINEAR, CUBIC, AREA):
            for (dw, dh) in ((1, 1), (3, 2), (5, 9)):
                tout = cv.Tensor.alloc([2, dh, dw, 3], np.uint8, "NHWC")
                cv.Resize()(None, cv.Tensor.from_numpy(src, "NHWC"), tout, interp)
                torch.cuda.synchronize()
                device = orc.resize_shipped(src, (dh, dw), interp)
                np.testing.assert_array_equal(tout.numpy(), device, err_msg=str((sw, sh, dw, dh, interp)))


@pytest.mark.parametrize("dt,c", [(np.uint8, 4), (np.uint8, 3), (np.uint8, 1), (np.uint16, 1), (np.int16, 3), (np.float32, 4)])
def test_area_varshape(cv, K, orc, gpu, dt, c):
    # image batches run the reference's separate AREA kernel (reductions: same sums, corners last;
    # enlargements: a bilinear variant). Sizes: the reference's rows (TestOpResize.cpp:67-69) plus
    # fractional factors in both directions and mixed reduce/enlarge.
    fmt = _format_for(cv, K, dt, c)
    sizes = [(44, 40, 22, 20), (30, 30, 20, 20), (30, 30, 60, 60), (97, 61, 13, 9), (50, 70, 75, 90), (64, 48, 32, 96),
             (33, 21, 33, 21), (120, 90, 47, 31)]
    n = len(sizes)
    bin_, bout, hosts, outs = cv.ImageBatchVarShape(n), cv.ImageBatchVarShape(n), [], []
    for i, (sw, sh, dw, dh) in enumerate(sizes):
        a = make_input(orc, (sh, sw, c), dt, 0xA0EA + i)
        hosts.append(a)
        bin_.push_back(cv.Image.from_numpy(a, fmt))
        o = cv.Image.alloc((dw, dh), fmt)
        outs.append(o)
        bout.push_back(o)
    cv.Resize()(None, bin_, bout, AREA)
    torch.cuda.synchronize()
    for a, o, (sw, sh, dw, dh) in zip(hosts, outs, sizes):
        res = o.plane_view(0, dt, c).cpu().numpy()[None]
        golden = orc.resize(a[None], (dh, dw), AREA, variant=3)
        device = orc.resize_shipped(a[None], (dh, dw), AREA, varshape=True)
        if dt == np.float32:
            assert np.abs(res - device).max() <= 1e-5 and np.abs(res - golden).max() <= 1e-4
        else:
            np.testing.assert_array_equal(res, device)
            # float32 source coordinates against the golden's double: a pixel whose box edge lands on an
            # integer can take a different tap, so the 1-LSB bar is required of all but a few pixels
            # (the reference's own rows have none)
            bad = np.abs(res.astype(np.int64) - golden.astype(np.int64)) > 1
            assert bad.mean() <= (0.0 if (sw, sh, dw, dh) in sizes[:3] else 0.02), (sw, sh, dw, dh, bad.mean())


# one-channel float maps whose rows are not reduced, in launches that take the whole-rows form and some that do not (too few
# blocks, too narrow): 1, 2, 3 and 12 pieces of 256 columns (4, 2 and 1 groups of 4 rows per block) with remainders, 3, 4 and 5
# source rows per group, the smallest source and the narrowest rows, equal heights; dense odd rows, the library's padded rows, and views whose rows start 4 bytes off
@pytest.mark.parametrize("n,sw,sh,dw,dh", [(512, 2, 2, 5, 7), (300, 40, 9, 257, 21), (256, 30, 20, 256, 33), (130, 100, 13, 700, 61),
                                           (50, 1301, 41, 1025, 41), (90, 5, 50, 513, 73), (520, 9, 5, 13, 6),
                                           (704, 2, 2, 145, 7), (70, 1301, 41, 1025, 41), (704, 40, 5, 97, 64), (150, 1500, 20, 3001, 41)])
@pytest.mark.parametrize("kind", ["dense", "padded", "view"])
def test_linear_float_maps_by_whole_rows(cv, orc, gpu, n, sw, sh, dw, dh, kind):
    src = make_input(orc, (n, sh, sw, 1), np.float32, 0xF10A + sw + dw)
    want = orc.resize(src, (dh, dw), LINEAR, variant=1, threads=8)
    tin = cv.Tensor.from_torch(torch.from_numpy(src).cuda(), "NHWC")
    if kind == "padded":
        tout = cv.Tensor.alloc([n, dh, dw, 1], np.float32, "NHWC")
        view, spare = tout.torch_view(), None
    else:
        lead, pitch = (0, dw) if kind == "dense" else (1, dw + 3)
        spare = torch.full((n * dh * pitch + 8,), -7.0, device="cuda")
        view = torch.as_strided(spare, (n, dh, dw, 1), (dh * pitch, pitch, 1, 1), lead)
        tout = cv.Tensor.from_torch(view, "NHWC")
    cv.Resize()(None, tin, tout, LINEAR)
    torch.cuda.synchronize()
    # four products of values below 1 and three sums, each rounded once or twice: under 12 roundings of 2^-24
    assert np.abs(view.cpu().numpy() - want).max() <= 12 * 2.0 ** -24 * max(1.0, float(np.abs(src).max()))
    if spare is not None:
        view.fill_(-7.0)
        assert bool((spare == -7.0).all()), "floats outside the rows written"


# the same at the widths that leave room for one block less in a CU's LDS, each with all it may have of it
@pytest.mark.parametrize("dw", [2528, 2529, 2552, 2553, 3325, 3328, 3329, 3352, 3353])
@pytest.mark.parametrize("kind", ["dense", "padded", "view"])
def test_linear_float_maps_by_whole_rows_at_the_lds_limits(cv, orc, gpu, dw, kind):
    test_linear_float_maps_by_whole_rows(cv, orc, gpu, 512, 40, 4, dw, 9, kind)


# seeded random cases: 8-bit pixels of 1, 3 and 4 channels, every interpolation, scales of 0.42 to 2.4 per axis (now
# and then equal, or exactly 1/2, 2/3, 1, 1.5, 2), small and 1080p-sized images, batches below and above the sizes
# at which the strip kernels take over, as packed tensors, as views with odd leads and pitches (bytes outside the
# rows must stay untouched) and as image batches of mixed sizes
@pytest.mark.parametrize("seed", [11, 12, 13])
def test_random_shapes_scales_and_pitches(cv, K, orc, gpu, seed):
    rng = np.random.default_rng(seed)
    for it in range(36):
        c = int(rng.choice([3, 3, 4, 1]))
        interp = int(rng.choice([NEAREST, LINEAR, LINEAR, CUBIC, CUBIC, AREA]))
        kind = str(rng.choice(["tensor", "view", "varshape"]))
        fx, fy = (float(np.exp(rng.uniform(np.log(0.42), np.log(2.4)))) for _ in range(2))
        if rng.random() < 0.2:
            fy = fx
        if rng.random() < 0.1:
            fx = float(rng.choice([0.5, 1.0, 1.5, 2.0, 2 / 3]))
        if rng.random() < 0.4:
            sw, sh = int(rng.integers(600, 2300)), int(rng.integers(400, 1300))
        else:
            sw, sh = int(rng.integers(4, 700)), int(rng.integers(4, 500))
        dw, dh = max(1, int(round(sw * fx))), max(1, int(round(sh * fy)))
        n = int(np.clip(rng.choice([1, 2, 2048 * 64 * 16 // (dw * dh) + 1, 2048 * 256 * 8 // (dw * dh) + 1]), 1, 16))
        n = min(n, max(1, int(60e6 / ((sw * sh + dw * dh) * c))))
        case = "seed %d case %d: %s u8x%d interp %d %dx%d -> %dx%d n %d" % (seed, it, kind, c, interp, sw, sh, dw, dh, n)

        def compare(res, src, out_hw, varshape):
            if interp == AREA:  # (the golden's box filter parts ways with the device expression on enlargements)
                np.testing.assert_array_equal(res, orc.resize_shipped(src, out_hw, AREA, varshape), err_msg=case)
            else:
                check(res, src, out_hw, interp, orc, varshape)

        try:
            if kind == "varshape":
                fmt = _format_for(cv, K, np.uint8, c)
                bin_, bout, hosts, outs = cv.ImageBatchVarShape(n), cv.ImageBatchVarShape(n), [], []
                for i in range(n):
                    w, h = max(8, sw + int(rng.integers(-30, 30))), max(8, sh + int(rng.integers(-30, 30)))
                    gx, gy = (fx, fy) if rng.random() < 0.8 else (float(rng.uniform(0.3, 3)), float(rng.uniform(0.3, 3)))
                    hosts.append(make_input(orc, (h, w, c), np.uint8, 1000 * it + i + seed))
                    bin_.push_back(cv.Image.from_numpy(hosts[-1], fmt))
                    outs.append(cv.Image.alloc((max(1, int(w * gx)), max(1, int(h * gy))), fmt))
                    bout.push_back(outs[-1])
                cv.Resize()(None, bin_, bout, interp)
                torch.cuda.synchronize()
                for a, o in zip(hosts, outs):
                    w, h = o.size
                    compare(o.plane_view(0, np.uint8, c).cpu().numpy()[None], a[None], (h, w), True)
                continue
            src = make_input(orc, (n, sh, sw, c), np.uint8, 77 * it + seed)
            if kind == "tensor":
                tout = cv.Tensor.alloc([n, dh, dw, c], np.uint8, "NHWC")
                cv.Resize()(None, cv.Tensor.from_numpy(src, "NHWC"), tout, interp)
                torch.cuda.synchronize()
                compare(tout.numpy(), src, (dh, dw), False)
                continue

            def view(w, h, fill):
                pad, lead = int(rng.integers(0, 9)), int(rng.integers(0, 5))
                pitch = w * c + pad
                plane = pitch * h + int(rng.integers(0, 9))
                buf = torch.full((n * plane + 64,), fill, dtype=torch.uint8, device="cuda")
                t = cv.Tensor.wrap(buf.data_ptr() + lead, [n, h, w, c], [plane, pitch, c, 1], np.uint8, "NHWC", keep=buf)
                return buf, t, lead, plane, pitch

            _, tin, lead, plane, pitch = view(sw, sh, 0)
            torch.as_strided(_[lead:], (n, sh, sw, c), (plane, pitch, c, 1)).copy_(torch.from_numpy(src).cuda())
            big_out, tout, lead, plane, pitch = view(dw, dh, 0xCD)
            cv.Resize()(None, tin, tout, interp)
            torch.cuda.synchronize()
            compare(torch.as_strided(big_out[lead:], (n, dh, dw, c), (plane, pitch, c, 1)).cpu().numpy(), src, (dh, dw), False)
            mask = torch.ones_like(big_out, dtype=torch.bool)
            torch.as_strided(mask[lead:], (n, dh, dw * c), (plane, pitch, 1)).fill_(False)
            assert bool((big_out[mask] == 0xCD).all()), "bytes outside the rows written"
        except AssertionError as e:
            raise AssertionError(case + ": " + str(e)) from e


def test_negative_cases(cv, gpu):
    a = cv.Tensor.alloc([2, 8, 8, 3], np.uint8, "NHWC")
    op = cv.Resize()
    cases = [
        (cv.Tensor.alloc([2, 4, 4, 3], np.float32, "NHWC"), LINEAR),   # dtype differs
        (cv.Tensor.alloc([3, 4, 4, 3], np.uint8, "NHWC"), LINEAR),     # batch differs
        (cv.Tensor.alloc([2, 4, 4, 4], np.uint8, "NHWC"), LINEAR),     # channels differ
        (cv.Tensor.alloc([2, 3, 4, 4], np.uint8, "NCHW"), LINEAR),     # layout differs
        (cv.Tensor.alloc([2, 4, 4, 3], np.uint8, "NHWC"), 4),          # LANCZOS unsupported
    ]
    for out, interp in cases:
        with pytest.raises(cv.Error) as e:
            op(None, a, out, interp)
        assert e.value.status == 2
    with pytest.raises(cv.Error) as e:
        cv.ResizeCropConvertReformat()(None, a, a, LINEAR) if False else cv.check(
            __import__("cvcuda_amd")._capi.cvcuda.cvcudaResizeSubmit(cv.ResizeCropConvertReformat().handle, None,
                                                                     a.handle, a.handle, LINEAR))
    assert e.value.status == 9  # handle of another operator -> NOT_COMPATIBLE


# float boxes, their rows summed by column first: every number of pieces per lane, reductions that are whole along one axis,
# both or none, the last rows and columns, rows that end inside a lane's 16 bytes; an infinity outside a box does not reach
# it. Against the box filter in 64 bits over the same float32 edges: a result is a sum of ny products, then of nx, times a
# scale of 4 roundings, each off by at most 2^-24 of itself, all of them positive.
@pytest.mark.parametrize("sw,sh,dw,dh", [(67, 41, 61, 37), (128, 66, 64, 33), (131, 50, 66, 25), (197, 47, 66, 30), (198, 47, 66, 30), (263, 83, 66, 21),
                                         (264, 84, 66, 21), (397, 61, 66, 9), (527, 33, 66, 4), (791, 40, 66, 3), (792, 36, 66, 3),
                                         (20, 19, 13, 7), (16, 64, 2, 5), (601, 40, 151, 9), (1537, 30, 128, 3),
                                         (329, 31, 66, 8), (330, 36, 66, 9), (461, 40, 66, 6), (462, 50, 66, 7), (594, 30, 66, 4),
                                         (659, 33, 66, 5), (660, 30, 66, 3), (725, 45, 66, 4), (726, 44, 66, 4)])
@pytest.mark.parametrize("c", [1, 3, 4])
def test_area_of_floats(cv, orc, gpu, sw, sh, dw, dh, c):
    src = orc.fill_f32((2, sh, sw, c), 0xF0 + sw)
    src = np.abs(src)
    src[1, 0, 0, 0] = np.inf
    buf = torch.zeros(src.size, dtype=torch.float32, device="cuda")
    buf.copy_(torch.from_numpy(src.reshape(-1)))
    tin = cv.Tensor.wrap(buf.data_ptr(), [2, sh, sw, c], [sh * sw * c * 4, sw * c * 4, c * 4, 4], np.float32, "NHWC", keep=buf)
    tout = cv.Tensor.alloc([2, dh, dw, c], np.float32, "NHWC")
    cv.Resize()(None, tin, tout, AREA)
    torch.cuda.synchronize()
    res = tout.numpy()

    def shares(size, new):  # [new, size] of each source pixel in each box, from float32 edges, over the box's nominal size
        scale = np.float32(size) / np.float32(new)
        lo = np.arange(new, dtype=np.float32) * scale
        hi = np.minimum(lo + scale, np.float32(size))
        i = np.arange(size, dtype=np.float64)
        covered = np.clip(np.minimum(i + 1, hi[:, None]) - np.maximum(i, lo[:, None]), 0, None)
        return covered / np.minimum(scale, np.float32(size) - lo)[:, None].astype(np.float64)

    wy, wx = shares(sh, dh), shares(sw, dw)
    clean = np.where(np.isinf(src), 0, src).astype(np.float64)
    ref = np.einsum("yh,nhwc,xw->nyxc", wy, clean, wx)
    assert np.isinf(res[1, 0, 0, 0])
    res[1, 0, 0, 0] = ref[1, 0, 0, 0]
    bound = 2.0 ** -24 * (2 * (np.ceil(sh / dh) + np.ceil(sw / dw)) + 12)
    assert (np.abs(res - ref) <= bound * np.abs(ref)).all(), np.max(np.abs(res - ref) / np.abs(ref)) / bound


# bicubic floats in strips of 16 rows (launches of 2048 strips and more): enlarged, the same size, reduced by almost 2, strips
# cut off by the lower edge, sources of 4 pixels along an axis. Against the formula in 64 bits over the float32 weights: two
# sums of 4 products each.
@pytest.mark.parametrize("sw,sh,dw,dh,n", [(131, 97, 197, 145, 60), (130, 33, 131, 33, 230), (200, 63, 101, 32, 512), (4, 4, 65, 17, 512),
                                           (67, 50, 64, 49, 512), (301, 7, 151, 250, 48)])
@pytest.mark.parametrize("c", [1, 3, 4])
def test_bicubic_float_strips(cv, orc, gpu, sw, sh, dw, dh, n, c):
    assert ((dw + 63) // 64) * ((dh + 15) // 16) * n >= 2048
    one = orc.fill_f32((3, sh, sw, c), 0xCC + sw)
    src = torch.from_numpy(one).cuda().repeat((n + 2) // 3, 1, 1, 1)[:n].contiguous()
    tin = cv.Tensor.wrap(src.data_ptr(), [n, sh, sw, c], [sh * sw * c * 4, sw * c * 4, c * 4, 4], np.float32, "NHWC", keep=src)
    tout = cv.Tensor.alloc([n, dh, dw, c], np.float32, "NHWC")
    cv.Resize()(None, tin, tout, CUBIC)
    torch.cuda.synchronize()
    res = tout.numpy()

    def axis(size, new, horizontal):
        f = np.float32
        at = (np.arange(new, dtype=f) + f(.5)) * (f(size) / f(new)) - f(.5)
        s = np.floor(at).astype(np.int64)
        d = at - s.astype(f)
        if horizontal:
            d = np.where((s < 1) | (s >= size - 3), f(0), d)
        s = np.clip(s, 1, size - 3)
        a, d, one, e = f(-.75), d.astype(f), f(1), f(1) - d.astype(f)
        w = [((a * (d + one) - 5 * a) * (d + one) + 8 * a) * (d + one) - 4 * a, ((a + f(2)) * d - (a + f(3))) * d * d + one,
             ((a + f(2)) * e - (a + f(3))) * e * e + one]
        assert all(x.dtype == f for x in w)
        m = np.zeros((new, size))
        for i, wi in enumerate(w + [one - w[0] - w[1] - w[2]]):
            m[np.arange(new), s - 1 + i] += wi.astype(np.float64)
        return m

    ref = np.abs(np.einsum("yh,nhwc,xw->nyxc", axis(sh, dh, False), one.astype(np.float64), axis(sw, dw, True)))
    ref = np.concatenate([ref] * ((n + 2) // 3))[:n]
    # the weights of an axis add up to at most 1.375 in magnitude; 4 products and 3 additions, twice
    assert np.abs(res - ref).max() <= 2 * 7 * 2.0 ** -24 * 1.375 ** 2 * np.abs(one).max()


# rows of zeros between rows of the type's lowest value: the horizontal sums of the latter pass the type's range, the rows
# between must not see it (vertical weights of exactly 0 there)
@pytest.mark.parametrize("c", [1, 3, 4])
def test_bicubic_float_strips_next_to_extreme_values(cv, gpu, c):
    n, sw, sh, dw = 230, 43, 33, 129
    src = torch.zeros((n, sh, sw, c), dtype=torch.float32, device="cuda")
    src[:, 1::2] = torch.finfo(torch.float32).min
    tin = cv.Tensor.from_torch(src, "NHWC")
    out = torch.full((n, sh, dw, c), -7.0, device="cuda")
    cv.Resize()(None, tin, cv.Tensor.from_torch(out, "NHWC"), CUBIC)
    torch.cuda.synchronize()
    # (the last rows' taps are moved into the image, but their fraction stays 0, so every row is one source row)
    rows = out.cpu().numpy()
    assert not np.isnan(rows).any()
    assert (rows[:, 2:sh - 3:2] == 0).all()


# the forms of float tensors on sources and results that are views (rows 4 bytes off a 16-byte boundary in another pitch): the
# dense result, bit for bit, and nothing outside the rows
@pytest.mark.parametrize("c", [1, 3, 4])
@pytest.mark.parametrize("n,sw,sh,dw,dh,interp", [(2, 131, 50, 66, 25, AREA), (2, 263, 83, 66, 21, AREA), (2, 20, 19, 13, 7, AREA),
                                                  (2, 791, 40, 66, 3, AREA), (60, 131, 97, 197, 145, CUBIC), (512, 67, 50, 64, 49, CUBIC),
                                                  (512, 4, 4, 65, 17, CUBIC)])
def test_floats_in_views(cv, orc, gpu, n, sw, sh, dw, dh, interp, c):
    src = torch.from_numpy(orc.fill_f32((2, sh, sw, c), 0xF1 + sw)).cuda().repeat(n // 2, 1, 1, 1)
    results = []
    for lead, extra in ((0, 0), (1, 3), (3, 5)):
        def view(h, w, fill):
            pitch = w * c + extra
            # (the source's buffer ends with its last row)
            buf = torch.full((lead + n * h * pitch - extra,), fill, device="cuda")
            t = torch.as_strided(buf, (n, h, w, c), (h * pitch, pitch, c, 1), lead)
            return buf, t, cv.Tensor.wrap(buf.data_ptr() + 4 * lead, [n, h, w, c], [4 * h * pitch, 4 * pitch, 4 * c, 4], np.float32,
                                          "NHWC", keep=buf)
        _, s, tin = view(sh, sw, 99.0)
        s.copy_(src)
        buf, d, tout = view(dh, dw, -7.0)
        cv.Resize()(None, tin, tout, interp)
        torch.cuda.synchronize()
        results.append(d.clone())
        d.fill_(-7.0)
        assert bool((buf == -7.0).all()), "floats outside the rows written"
    assert torch.equal(results[0], results[1]) and torch.equal(results[0], results[2])
    assert not torch.isnan(results[0]).any()


# Bicubic strips of 4, 8 and 16 rows of three and four channels whose furthest request, the fourth row behind an output row's upper middle one, is the
# row before the image's last or that row itself: on both sides of what takes the loop without a test for the last row
@pytest.mark.parametrize("c", [3, 4])
@pytest.mark.parametrize("rows,n", [(4, 16), (8, 80), (16, 320)])
@pytest.mark.parametrize("sh", [20, 21, 27, 28, 33, 34, 41, 50, 63])
def test_cubic_strips_at_the_last_row(cv, orc, gpu, sh, rows, n, c):
    dw, dh, sw = 256, 64, 201
    places = np.floor((np.arange(dh, dtype=np.float32) + np.float32(.5)) * (np.float32(sh) / np.float32(dh)) - np.float32(.5))
    behind = np.clip(places, 1, sh - 3)[rows - 1::rows] + 4 - (sh - 1)  # of each strip; below 0: clear of the last row
    assert behind.min() < 0 <= behind.max()
    src = orc.fill_u8((2, sh, sw, c), 40 + sh)
    out = torch.full((n, dh, dw, c), 7, dtype=torch.uint8, device="cuda")
    cv.Resize()(None, cv.Tensor.from_torch(torch.from_numpy(src[np.arange(n) % 2]).cuda(), "NHWC"), cv.Tensor.from_torch(out, "NHWC"), CUBIC)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(out.cpu().numpy(), orc.resize_shipped(src, (dh, dw), CUBIC, threads=8)[np.arange(n) % 2])


# Images whose waves, counted along the rows, fill a multiple of 16 blocks, which get one more: in the forms that are counted so
@pytest.mark.parametrize("row", [(300, 20, 1021, 64, NEAREST, 48, np.uint8, 3), (300, 20, 1021, 64, NEAREST, 48, np.uint8, 1),
                                 (1100, 80, 1021, 64, NEAREST, 80, np.uint8, 1), (200, 50, 256, 64, CUBIC, 16, np.uint8, 3),
                                 (200, 50, 256, 64, CUBIC, 16, np.uint8, 4), (600, 160, 256, 64, AREA, 3, np.uint8, 3),
                                 (900, 200, 256, 64, LINEAR, 128, np.uint8, 1), (200, 20, 256, 16, NEAREST, 3, np.float32, 3),
                                 (200, 100, 256, 128, CUBIC, 64, np.float32, 1), (700, 40, 256, 16, LINEAR, 3, np.float32, 4)],
                         ids=lambda r: "%dx%d-%dx%d-i%d-n%d-%s-c%d" % (r[:6] + (np.dtype(r[6]).name, r[7])))
def test_tensors_of_16_blocks(cv, orc, gpu, row):
    test_tensor_table(cv, orc, gpu, row)


# Nearest neighbour of larger pixels on both sides of what keeps the block of 64 x 4: enlarged down by 4/3, rows that end with a sector
# (pitches of their own and packed), waves filled to 80 %
@pytest.mark.parametrize("c", [3, 4])
@pytest.mark.parametrize("row_align", [0, 1])
@pytest.mark.parametrize("size", [(50, 30, 208, 40), (50, 31, 208, 41), (50, 30, 205, 40), (50, 30, 204, 43), (33, 9, 103, 45), (33, 9, 102, 45), (7, 3, 64, 5),
                                  (300, 20, 1280, 37), (300, 20, 1281, 37)])
def test_tensor_nearest_of_larger_pixels(cv, orc, gpu, size, row_align, c):
    sw, sh, dw, dh = size
    src = np.ascontiguousarray(orc.fill_u8((3, sh, sw, c), 5 + dw), np.float32)
    tin = cv.Tensor.from_numpy(src, "NHWC", row_align=row_align)
    tout = cv.Tensor.alloc([3, dh, dw, c], np.float32, "NHWC", row_align=row_align)
    tout.torch_view().fill_(-7)
    cv.Resize()(None, tin, tout, NEAREST)
    np.testing.assert_array_equal(tout.numpy(), orc.resize(src, (dh, dw), NEAREST, variant=0))


# Rows that share what they read, on both sides of what keeps a block's waves below one another: as much as they write of it, waves filled to
# 70 or 80 %, blocks to 3/4, and sources of no less than a tenth, an eighth or a fourth of what is written; and rows of 8 blocks and
# of others
@pytest.mark.parametrize("row", [(sw, sh, dw, 64, interp, 2 * n // -(-dw // 64), dtype, c)
                                 for (interp, n, dtype, c, least, w, full, small) in [(NEAREST, 3, np.float32, 3, 140, 140, 135, (224, 4)), (NEAREST, 3, np.float32, 4, 140, 140, 135, (224, 4)),
                                                                                      (CUBIC, 384, np.float32, 1, 342, 128, 154, (256, 4)),
                                                                                      (CUBIC, 243, np.float32, 3, 205, 128, 154, (205, 10)),
                                                                                      (LINEAR, 384, np.uint8, 4, 427, 128, 154, (256, 8))]
                                 for (sw, sh, dw) in [(least - 1, 32, w), (least, 32, w), (least, 32, 130), (least * full // w + 2, 32, full),
                                                      (least * full // w + 2, 32, full - 1), (small[0] - 1, small[1], w), (small[0], small[1], w)]]
                                + [(sw, 8, 128, dh, interp, 512, dtype, c) for (sw, interp, dtype, c) in [(300, CUBIC, np.float32, 1), (400, LINEAR, np.uint8, 4)]
                                   for dh in (23, 24)]
                                + [(300, 2, 140, dh, NEAREST, 3, np.float32, c) for c in (3, 4) for dh in (5, 6)]
                                + [(sw, 4, dw, 9, NEAREST, 2, np.float32, 3) for (sw, dw) in [(2000, 1800), (2000, 1793), (2000, 1791), (2400, 2100)]],
                         ids=lambda r: "%dx%d-%dx%d-i%d-n%d-%s-c%d" % (r[:6] + (np.dtype(r[6]).name, r[7])))
def test_tensors_whose_rows_share_sources(cv, orc, gpu, row):
    test_tensor_table(cv, orc, gpu, row)


# One column of more rows than one dimension of a launch has waves for
def test_nearest_of_a_tall_image(cv, orc, gpu):
    h   = 2 ** 26
    src = np.ascontiguousarray(orc.fill_u8((1, 997, 1, 3), 17), np.float32)
    tin, tout = cv.Tensor.from_numpy(src, "NHWC", row_align=1), cv.Tensor.alloc([1, h, 1, 3], np.float32, "NHWC", row_align=1)
    cv.Resize()(None, tin, tout, NEAREST)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(tout.numpy(), orc.resize(src, (h, 1), NEAREST, variant=0))


# Float bicubic reductions by 4 and more down, whose waves are counted along the rows: tiles of 64 columns that do not fill blocks of
# four or rows, one wave in the last block, and each side of the scale of 4
@pytest.mark.parametrize("row", [(sw, sh, dw, dh, CUBIC, n, np.float32, c)
                                 for c in (3, 4)
                                 for (sw, sh, dw, dh, n) in [(200, 33, 63, 8, 2), (200, 32, 64, 8, 1), (261, 31, 65, 8, 2), (700, 21, 130, 5, 3),
                                                             (1300, 9, 257, 1, 2), (517, 40, 129, 3, 1), (640, 101, 320, 25, 2)]],
                         ids=lambda r: "%dx%d-%dx%d-i%d-n%d-%s-c%d" % (r[:6] + (np.dtype(r[6]).name, r[7])))
def test_tensor_cubic_waves_along_rows(cv, orc, gpu, row):
    test_tensor_table(cv, orc, gpu, row)


# Rows per wave by the size of the launch: the box filter at scales of 1 to 3 (4 rows to a wave up to 2048 waves of 16, 8 up to 8192, then 16), for nearest
# neighbour enlarging by 1.5 or more (strips of 4 rows from 1024 strips of 8 on, 1536 with three channels; 8 rows for one channel
# from 15360 on, 6144 where a source row is 2.2 output rows and more) and for float bicubic (4 rows, 8, 16; from 128 waves of 4 rows on,
# 512 with three and four channels, with four reducing 1024, by more than 1.5 2048)
@pytest.mark.parametrize("row", [(sw, sh, dw, dh, AREA, n, np.uint8, c)
                                 for c in (1, 3, 4)
                                 for (sw, sh, dw, dh, n) in [(97, 23, 61, 9, 1), (64, 40, 65, 39, 2), (130, 30, 64, 15, 3), (190, 50, 63, 17, 4),
                                                             (70, 18, 64, 16, 2048), (70, 19, 64, 17, 1025), (70, 19, 65, 16, 4096),
                                                             (70, 18, 64, 16, 8193)]]
                         + [(sw, sh, dw, dh, NEAREST, n, np.uint8, c)
                            for c in (1, 3, 4)
                            for (sw, sh, dw, dh, n) in [(100, 6, 256, 7, 1024), (100, 6, 253, 9, 513), (100, 6, 257, 8, 768), (100, 8, 255, 3, 1535),
                                                        (100, 8, 256, 8, 1536), (170, 5, 256, 5, 1600)]]
                         + [(100, 6, 256, 8, NEAREST, 15360, np.uint8, 1), (100, 6, 256, 7, NEAREST, 15360, np.uint8, 1), (100, 6, 253, 8, NEAREST, 15360, np.uint8, 1)]
                         + [(sw, sh, dw, dh, CUBIC, n, np.float32, c)
                            for c in (1, 3, 4)
                            for (sw, sh, dw, dh, n) in [(40, 8, 64, 4, 127), (40, 8, 64, 4, 128), (40, 8, 64, 5, 256), (40, 8, 64, 3, 512),
                                                        (60, 9, 65, 6, 256), (60, 9, 63, 7, 3840), (60, 9, 63, 7, 4500), (60, 9, 64, 9, 2560),
                                                        (60, 9, 64, 9, 2305)]]
                         + [(100, 5, 256, 11, NEAREST, 3071, np.uint8, 1), (100, 5, 256, 11, NEAREST, 3072, np.uint8, 1), (90, 5, 253, 12, NEAREST, 3073, np.uint8, 1),
                            (60, 9, 61, 7, CUBIC, 511, np.float32, 4), (60, 9, 61, 7, CUBIC, 512, np.float32, 4), (60, 9, 64, 5, CUBIC, 1023, np.float32, 4),
                            (60, 9, 64, 5, CUBIC, 1024, np.float32, 4), (60, 9, 63, 12, CUBIC, 2600, np.float32, 3), (60, 10, 63, 12, CUBIC, 2600, np.float32, 3)],
                         ids=lambda r: "%dx%d-%dx%d-i%d-n%d-%s-c%d" % (r[:6] + (np.dtype(r[6]).name, r[7])))
def test_tensor_rows_per_wave(cv, orc, gpu, row):
    if row[4] == AREA:
        test_area_tensor(cv, orc, gpu, row[:4] + row[5:])
    else:
        test_tensor_table(cv, orc, gpu, row)
