"""GPU parity of cvcudaWarpAffine / cvcudaWarpPerspective [VarShape] Submit.

Exact-equality rows: the reference's table on tiny RGBA8 images with small integer and quarter-step
matrices, all five borders, three interpolations, forward and inverse maps
(tests/cvcuda/system/TestOpWarpAffine.cpp:232-319). Random rotations/scales: <= 1 LSB against the
reference's golden (oracle variant 0) and bit-exact against the restatement of this build's device
arithmetic: oracle variant 1 for NEAREST and CUBIC; on 8-bit pixels LINEAR is the 15-bit fixed-point blend
and CUBIC the 14-bit one (oracle variant 2); the bilinear one equals the golden wherever the weights are
dyadic (every row of the reference's table); LINEAR on the other types evaluates the bilinear sum in the
golden's own association, so variant 0 IS the device arithmetic there. BASELINE configuration 4 at full size."""
import itertools

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
NEAREST, LINEAR, CUBIC = 0, 1, 2
INVERSE_MAP = 16


def device_variant(interp, dtype=np.uint8):
    if interp != NEAREST and np.dtype(dtype) == np.uint8:
        return 2
    return 0 if interp == LINEAR else 1


def dyadic(values, bits=7):
    return all(float(v * (1 << bits)).is_integer() for v in values)

SIZES = [(5, 4, 5, 4), (5, 4, 6, 8), (7, 8, 4, 5)]
MATS = [(1, 0, 0, 0, 1, 0), (1, 0, 1, 0, 1, 2), (1, 2, 1, 2, 1, 2), (2, 2, 1, 3, 1, 2), (1, 2, 0, 1, 1, 0),
        (2, 2, 0, 3, 1, 1), (1, 0, 0, 0, 1, 1), (1, 2, 0, 2, 1, 1), (2, 2, 0, 3, 1, 0), (0.5, 2, 1, 0.75, 1, 2)]


def to_inverse(orc, m, inverse_given):
    return np.asarray(m, np.float32) if inverse_given else orc.invert_affine(m)


@pytest.mark.parametrize("interp", [NEAREST, LINEAR, CUBIC])
@pytest.mark.parametrize("border", [0, 1, 2, 3, 4])
def test_reference_table_exact(cv, orc, gpu, interp, border):
    op = cv.WarpAffine(0)
    for (sw, sh, dw, dh), m, inv in itertools.product(SIZES, MATS, (True, False)):
        src = orc.fill_u8((4, sh, sw, 4), sw * 100 + dh + int(m[1]))
        tin = cv.Tensor.from_numpy(src, "NHWC")
        tout = cv.Tensor.alloc([4, dh, dw, 4], np.uint8, "NHWC")
        op(None, tin, tout, m, interp | (INVERSE_MAP if inv else 0), border, (1, 2, 3, 4))
        torch.cuda.synchronize()
        res = tout.numpy()
        minv = to_inverse(orc, m, inv)
        dev = orc.warp(src, (dh, dw), minv, interp, border, (1, 2, 3, 4), variant=device_variant(interp))
        np.testing.assert_array_equal(res, dev, err_msg=str((sw, sh, dw, dh, m, inv)))
        gold = orc.warp(src, (dh, dw), minv, interp, border, (1, 2, 3, 4), variant=0)
        # LINEAR weights that are multiples of 2^-7 per axis are exact in the fixed-point blend as in float32
        exact = interp != CUBIC and dyadic(minv)
        tol = 0 if exact else 1
        assert np.abs(res.astype(np.int16) - gold.astype(np.int16)).max() <= tol, (sw, sh, dw, dh, m, inv)



@pytest.mark.parametrize("c", [1, 3, 4])
def test_tiny_sources_at_the_border_forms_limits(cv, orc, gpu, c):
    # 8-bit samples next to the image's edge take straight-line forms that fetch a pixel with one 4-byte load, moved
    # back where it would pass the image's last byte; images of under 4 bytes keep the generic loop. Sources of 1 to
    # 5 pixels (the mirroring and repeating borders' single folds do not reach that far: generic loop), every
    # interpolation and border mode: exact against the restatement.
    op = cv.WarpAffine(0)
    m = [0.8, 0.3, -0.4, -0.2, 0.9, 0.6]
    for (sw, sh) in [(1, 1), (2, 1), (1, 2), (3, 1), (1, 4), (2, 2), (5, 1), (1, 5)]:
        src = orc.fill_u8((2, sh, sw, c), 40 + sw * 7 + sh)
        for interp, border in itertools.product((NEAREST, LINEAR, CUBIC), (0, 1, 2, 3, 4)):
            tout = cv.Tensor.alloc([2, 6, 9, c], np.uint8, "NHWC")
            op(None, cv.Tensor.from_numpy(src, "NHWC"), tout, m, interp | INVERSE_MAP, border, (9, 200, 31, 77))
            torch.cuda.synchronize()
            dev = orc.warp(src, (6, 9), np.asarray(m, np.float32), interp, border, (9, 200, 31, 77), variant=device_variant(interp))
            np.testing.assert_array_equal(tout.numpy(), dev, err_msg=str((sw, sh, c, interp, border)))



@pytest.mark.parametrize("c", [1, 3, 4])
def test_mirroring_and_repeating_borders_near_and_far(cv, orc, gpu, c):
    # Under REFLECT, WRAP and REFLECT101 samples whose taps lie within one image size of the image take straight-line
    # forms with a single fold of the index; farther out the generic loop with its modulo. A destination 5 times the
    # source's size around it, shifted and slightly rotated, has both kinds in every interpolation: exact.
    op = cv.WarpAffine(0)
    sw, sh = 23, 17
    src = orc.fill_u8((2, sh, sw, c), 77 + c)
    m = [0.93, 0.11, -2.3 * sw, -0.07, 1.04, -1.9 * sh]  # destination (0, 0) maps about two image sizes in front
    for interp, border in itertools.product((NEAREST, LINEAR, CUBIC), (2, 3, 4)):
        tout = cv.Tensor.alloc([2, 5 * sh, 5 * sw, c], np.uint8, "NHWC")
        op(None, cv.Tensor.from_numpy(src, "NHWC"), tout, m, interp | INVERSE_MAP, border, (0, 0, 0, 0))
        torch.cuda.synchronize()
        dev = orc.warp(src, (5 * sh, 5 * sw), np.asarray(m, np.float32), interp, border, (0, 0, 0, 0), variant=device_variant(interp))
        np.testing.assert_array_equal(tout.numpy(), dev, err_msg=str((c, interp, border)))


# The same of elements that list their samples at the edge: a wave's list has samples of both kinds, few and more than 64 of each.
@pytest.mark.parametrize("dt,c", [(np.int16, 3), (np.uint16, 1), (np.float32, 1), (np.float32, 4)])
@pytest.mark.parametrize("scale", [0.3, 1.0, 2.5])
def test_listed_samples_near_and_far(cv, orc, gpu, dt, c, scale):
    sw, sh = 23, 17
    src = (orc.fill_u8((2, sh, sw, c), 77 + c).astype(np.float64) - (100 if dt == np.int16 else 0)).astype(dt)
    m = [0.93 * scale, 0.11, -2.3 * sw * scale, -0.07, 1.04 * scale, -1.9 * sh * scale]
    for interp, border in itertools.product((NEAREST, LINEAR, CUBIC), (2, 3, 4)):
        tout = cv.Tensor.alloc([2, 5 * sh, 5 * sw, c], dt, "NHWC")
        cv.WarpAffine(0)(None, cv.Tensor.from_numpy(src, "NHWC"), tout, m, interp | INVERSE_MAP, border, (0, 0, 0, 0))
        torch.cuda.synchronize()
        dev = orc.warp(src, (5 * sh, 5 * sw), np.asarray(m, np.float32), interp, border, (0, 0, 0, 0), variant=device_variant(interp, dt))
        if dt == np.float32:
            # 16 products of up to 255 * 1.6 each rounded in another order: 16 * 408 * 2^-24 = 3.9e-4
            assert np.abs(tout.numpy() - dev).max() <= 4e-4, (interp, border)
        else:
            np.testing.assert_array_equal(tout.numpy(), dev, err_msg=str((interp, border)))


# row windows of dense images whose rows start at every byte of a dword in turn, from every start of the first; widths about
# the tap blocks' and the windows' own (samples whose window would pass the row's end take the border's forms). The buffer
# ends with the last image.
@pytest.mark.parametrize("c", [1, 3, 4])
@pytest.mark.parametrize("lead", [0, 1, 2, 3])
@pytest.mark.parametrize("size", [(1, 9), (4, 4), (7, 5), (11, 6), (61, 40), (70, 41)], ids=lambda s: "%dx%d" % s)
def test_rows_from_every_byte_of_a_dword(cv, orc, gpu, size, lead, c):
    w, h = size
    src = orc.fill_u8((2, h, w, c), 0xD0D + w + lead)
    buf = torch.zeros(lead + src.size, dtype=torch.uint8, device="cuda")
    buf[lead:].copy_(torch.from_numpy(src.reshape(-1)))
    tin = cv.Tensor.wrap(buf.data_ptr() + lead, [2, h, w, c], [h * w * c, w * c, c, 1], np.uint8, "NHWC", keep=buf)
    for interp, border in itertools.product((NEAREST, LINEAR, CUBIC), (0, 1, 2, 3, 4)):
        for m in (rotation(w, h, 4.0, 1.02), [1.0, 0.0, 0.3, 0.0, 1.0, -0.6], rotation(w, h, 21.0, 0.7)):
            tout = cv.Tensor.alloc([2, h + 3, w + 5, c], np.uint8, "NHWC")
            cv.WarpAffine(0)(None, tin, tout, m, interp, border, (9, 200, 31, 77))
            torch.cuda.synchronize()
            dev = orc.warp(src, (h + 3, w + 5), orc.invert_affine(m), interp, border, (9, 200, 31, 77), variant=device_variant(interp))
            np.testing.assert_array_equal(tout.numpy(), dev, err_msg=str((size, lead, c, interp, border, m)))


# single-channel taps read alone where the map turns by more than 45 degrees (bicubic: 56), in windows below that, from rows that
# start at every byte of a dword and up to the last bytes of the smallest sources
@pytest.mark.parametrize("lead", [0, 1, 2, 3])
@pytest.mark.parametrize("size", [(2, 2), (4, 4), (5, 9), (7, 5), (64, 40), (71, 43)], ids=lambda s: "%dx%d" % s)
def test_single_channel_quarter_turns(cv, orc, gpu, size, lead):
    w, h = size
    src = orc.fill_u8((2, h, w, 1), 0x90 + w + lead)
    buf = torch.zeros(lead + src.size, dtype=torch.uint8, device="cuda")
    buf[lead:].copy_(torch.from_numpy(src.reshape(-1)))
    tin = cv.Tensor.wrap(buf.data_ptr() + lead, [2, h, w, 1], [h * w, w, 1, 1], np.uint8, "NHWC", keep=buf)
    for deg in (44.0, 46.0, 55.0, 58.0, 90.0, 133.0, 270.0):
        for scale in (0.9, 1.7):
            m = rotation(w, h, deg, scale)
            for interp in (LINEAR, CUBIC):
                tout = cv.Tensor.alloc([2, h + 3, w + 5, 1], np.uint8, "NHWC")
                cv.WarpAffine(0)(None, tin, tout, m, interp, 1, (0, 0, 0, 0))
                torch.cuda.synchronize()
                dev = orc.warp(src, (h + 3, w + 5), orc.invert_affine(m), interp, 1, (0, 0, 0, 0), variant=device_variant(interp))
                np.testing.assert_array_equal(tout.numpy(), dev, err_msg=str((deg, scale, interp)))


# the windows next to the edge, three channels, in launches of two patches a wave (one image) and of four: the smallest sources that
# have room for a window, dense rows that start at every byte of a dword
@pytest.mark.parametrize("n", [1, 205])
@pytest.mark.parametrize("lead", [0, 1, 2, 3])
@pytest.mark.parametrize("size", [(4, 4), (5, 2), (7, 5), (37, 21), (70, 41)], ids=lambda s: "%dx%d" % s)
def test_bicubic_windows_of_large_launches(cv, orc, gpu, size, lead, n):
    (w, h), c = size, 3
    dw, dh = 66, 66  # 2 x 5 tiles
    src = orc.fill_u8((n, h, w, c), 0xB1C + w + lead)
    buf = torch.zeros(lead + src.size, dtype=torch.uint8, device="cuda")
    buf[lead:].copy_(torch.from_numpy(src.reshape(-1)))
    tin = cv.Tensor.wrap(buf.data_ptr() + lead, [n, h, w, c], [h * w * c, w * c, c, 1], np.uint8, "NHWC", keep=buf)
    for m in (rotation(w, h, 4.0, 1.02), [dw / w, 0.0, 0.3, 0.0, dh / h, -0.6], rotation(w, h, 21.0, 2.7)):
        for border, color in ((0, (9, 200, 77, 0)), (1, (0, 0, 0, 0))):
            tout = cv.Tensor.alloc([n, dh, dw, c], np.uint8, "NHWC")
            cv.WarpAffine(0)(None, tin, tout, m, CUBIC, border, color)
            torch.cuda.synchronize()
            dev = orc.warp(src, (dh, dw), orc.invert_affine(m), CUBIC, border, color, variant=device_variant(CUBIC), threads=8)
            np.testing.assert_array_equal(tout.numpy(), dev, err_msg=str((border, m)))


def rotation(w, h, deg, s):
    t = np.deg2rad(deg)
    c, sn = s * np.cos(t), s * np.sin(t)
    cx, cy = (w - 1) / 2.0, (h - 1) / 2.0
    return [c, -sn, cx - c * cx + sn * cy, sn, c, cy - sn * cx - c * cy]


# waves that the image's edge passes through list their samples there and share them out: images smaller than a wave's part
# and a little larger, all borders, with many, few and no samples inside
@pytest.mark.parametrize("size", [(1, 1), (3, 2), (9, 8), (33, 9), (40, 70), (65, 17)], ids=lambda s: "%dx%d" % s)
@pytest.mark.parametrize("c", [1, 3, 4])
@pytest.mark.parametrize("dt", [np.uint8, np.uint16, np.int16, np.float32])
def test_samples_at_the_edge(cv, orc, gpu, dt, c, size):
    w, h = size
    src = (orc.fill_u8((2, h, w, c), 5 + w + c).astype(np.float64) * (200 if dt in (np.uint16, np.int16) else 1)
           - (20000 if dt == np.int16 else 0)).astype(dt)
    tin = cv.Tensor.from_numpy(src, "NHWC")
    dh, dw = h + 11, w + 14
    tout = cv.Tensor.alloc([2, dh, dw, c], dt, "NHWC")
    for m in ([0.9, -0.5, 6.3, 0.5, 0.9, -2.7], [1.0, 0.0, -0.5, 0.0, 1.0, 3.0], [0.3, 0.1, 700.0, 0.0, 0.4, -300.0]):
        for interp in (NEAREST, LINEAR, CUBIC):
            for border in range(5):
                cv.WarpAffine(0)(None, tin, tout, m, interp | INVERSE_MAP, border, (9, 200, 31, 77))
                torch.cuda.synchronize()
                dev = orc.warp(src, (dh, dw), np.asarray(m, np.float32), interp, border, (9, 200, 31, 77), variant=device_variant(interp, dt))
                if dt == np.float32:
                    assert np.abs(tout.numpy() - dev).max() <= 1e-3, (m, interp, border)  # (as above)
                else:
                    np.testing.assert_array_equal(tout.numpy(), dev, err_msg=str((m, interp, border)))


@pytest.mark.parametrize("dt,c", [(np.uint8, 3), (np.uint8, 1), (np.uint8, 4), (np.uint16, 3), (np.int16, 4),
                                  (np.float32, 1), (np.float32, 3)])
@pytest.mark.parametrize("interp", [NEAREST, LINEAR, CUBIC])
def test_random_rotations_tensor(cv, orc, gpu, dt, c, interp):
    n, h, w = 2, 97, 131
    if dt == np.float32:
        src = orc.fill_f32((n, h, w, c), 7) * 255
    else:
        src = orc.fill_u8((n, h, w, c, np.dtype(dt).itemsize), 7).view(dt).reshape(n, h, w, c)
    op = cv.WarpAffine(0)
    for deg, s, border in [(17.0, 1.1, 0), (-29.0, 0.85, 1), (5.5, 1.0, 4), (30.0, 1.2, 3), (-11.0, 0.9, 2)]:
        m = rotation(w, h, deg, s)
        tout = cv.Tensor.alloc([n, 80, 150, c], dt, "NHWC")
        op(None, cv.Tensor.from_numpy(src, "NHWC"), tout, m, interp, border, (9, 8, 7, 6))
        torch.cuda.synchronize()
        res = tout.numpy()
        minv = orc.invert_affine(m)
        dev = orc.warp(src, (80, 150), minv, interp, border, (9, 8, 7, 6), variant=device_variant(interp, dt))
        if dt == np.float32:
            assert np.abs(res - dev).max() <= 1e-3
        else:
            np.testing.assert_array_equal(res, dev)
            if dt == np.uint8 and interp != NEAREST:
                gold = orc.warp(src, (80, 150), minv, interp, border, (9, 8, 7, 6), variant=0)
                assert np.abs(res.astype(np.int16) - gold.astype(np.int16)).max() <= 1


# 12- and 16-byte pixels leave the wave 16 bytes per lane: widths about a wave's 32 columns, rows that end in 1 to 3 dwords
@pytest.mark.parametrize("c", [3, 4])
@pytest.mark.parametrize("dw,dh", [(1, 1), (3, 9), (31, 8), (33, 17), (62, 5), (64, 16), (67, 23)])
def test_wide_pixels_at_the_tile_edges(cv, orc, gpu, dw, dh, c):
    src = orc.fill_f32((2, 21, 37, c), 5 + dw)
    m = rotation(37, 21, 12.0, 0.9)
    buf = torch.full((2 * dh * dw * c + 8,), -7.0, device="cuda")
    tout = cv.Tensor.wrap(buf.data_ptr() + 16, [2, dh, dw, c], [dh * dw * c * 4, dw * c * 4, c * 4, 4], np.float32, "NHWC", keep=buf)
    cv.WarpAffine(0)(None, cv.Tensor.from_numpy(src, "NHWC"), tout, m, NEAREST, 1, (0, 0, 0, 0))
    torch.cuda.synchronize()
    res = buf.cpu().numpy()
    dev = orc.warp(src, (dh, dw), orc.invert_affine(m), NEAREST, 1, (0, 0, 0, 0), variant=1)
    np.testing.assert_array_equal(res[4:-4].reshape(dev.shape), dev)
    assert (res[:4] == -7).all() and (res[-4:] == -7).all()


# launches of up to 3072 waves of four patches give each wave two: results about both tiles' edges, in the largest launch of the one
# form and the smallest of the other, each image of a batch as the oracle has it and nothing written beside them
@pytest.mark.parametrize("dt,c", [(np.uint8, 1), (np.uint8, 3), (np.uint8, 4), (np.float32, 1), (np.float32, 3), (np.float32, 4)])
@pytest.mark.parametrize("dw,dh", [(1, 1), (15, 7), (17, 9), (31, 8), (33, 17), (62, 5), (64, 16), (67, 23)])
def test_patches_per_wave(cv, orc, gpu, dw, dh, dt, c):
    src = (orc.fill_f32((2, 21, 37, c), 5 + dw) * 255).astype(dt)
    tiles, size = -(-dw // 64) * -(-dh // 16), np.dtype(dt).itemsize
    for n in (768 // tiles, 768 // tiles + 1):
        tin = cv.Tensor.from_numpy(src[np.arange(n) % 2], "NHWC")
        buf = torch.empty((n * dh * dw * c * size + 32,), dtype=torch.uint8, device="cuda")
        tout = cv.Tensor.wrap(buf.data_ptr() + 16, [n, dh, dw, c], [dh * dw * c * size, dw * c * size, c * size, size], dt, "NHWC", keep=buf)
        for interp, border in itertools.product((NEAREST, LINEAR, CUBIC), (0, 1, 4)):
            m = rotation(37, 21, 12.0 + border, 0.9)
            buf.fill_(0xA5)
            cv.WarpAffine(0)(None, tin, tout, m, interp, border, (9, 8, 7, 6))
            torch.cuda.synchronize()
            res = buf.cpu().numpy()
            assert (res[:16] == 0xA5).all() and (res[-16:] == 0xA5).all()
            got = res[16:-16].view(dt).reshape(n, dh, dw, c)
            np.testing.assert_array_equal(got, got[np.arange(n) % 2])
            dev = orc.warp(src, (dh, dw), orc.invert_affine(m), interp, border, (9, 8, 7, 6), variant=device_variant(interp, dt))
            if dt == np.float32:
                assert np.abs(got[:2] - dev).max() <= 1e-3, (interp, border)  # (as above)
            else:
                np.testing.assert_array_equal(got[:2], dev, err_msg=str((interp, border)))


@pytest.mark.parametrize("n", [2, 3])  # of 300 tiles of 64 x 16 each, and what is left over at their edges
def test_patches_per_wave_of_image_batches(cv, K, orc, gpu, n):
    bi, bo, hosts, outs, mats = cv.ImageBatchVarShape(n), cv.ImageBatchVarShape(n), [], [], []
    for i in range(n):
        w, h = 639 - 17 * i, 475 + i
        hosts.append(orc.fill_u8((h, w, 3), 70 + i))
        bi.push_back(cv.Image.from_numpy(hosts[i], K.IMAGE_FORMAT_RGB8))
        outs.append(cv.Image.alloc((w, h), K.IMAGE_FORMAT_RGB8))
        bo.push_back(outs[i])
        mats.append(rotation(w, h, 11.0 - 9 * i, 1.1))
    mats = np.asarray(mats, np.float32)
    for interp, border in itertools.product((NEAREST, LINEAR, CUBIC), (0, 1)):
        cv.WarpAffine(n)(None, bi, bo, cv.Tensor.from_numpy(mats, "NW"), interp, border, (10, 20, 30, 40))
        torch.cuda.synchronize()
        for i in range(n):
            w, h = outs[i].size
            dev = orc.warp(hosts[i][None], (h, w), orc.invert_affine(mats[i]), interp, border, (10, 20, 30, 40),
                           variant=device_variant(interp))[0]
            np.testing.assert_array_equal(outs[i].plane_view(0, np.uint8, 3).cpu().numpy(), dev, err_msg=str((interp, border, i)))


# Bicubic of three 8-bit channels on both sides of what its waves stand alone for: blocks of four with no wave outside the images, up to and
# past 32 768 waves; a tenth, a fiftieth outside
@pytest.mark.parametrize("size", [(161, 192, 32), (148, 172, 68), (148, 173, 73), (342, 192, 128), (341, 190, 125), (205, 223, 41), (93, 641, 41), (21, 97, 480)])
@pytest.mark.parametrize("batch", [False, True])
def test_bicubic_waves_in_blocks(cv, K, orc, gpu, size, batch):
    n, w, h = size
    src, m = orc.fill_u8((2, h, w, 3), 80 + w), rotation(w, h, 7.0, 1.05)
    dev = orc.warp(src, (h, w), orc.invert_affine(m), CUBIC, 1, (0, 0, 0, 0), variant=device_variant(CUBIC))
    if not batch:
        tin = cv.Tensor.from_numpy(src[np.arange(n) % 2], "NHWC")
        tout = cv.Tensor.alloc([n, h, w, 3], np.uint8, "NHWC")
        cv.WarpAffine(0)(None, tin, tout, m, CUBIC, 1, (0, 0, 0, 0))
        torch.cuda.synchronize()
        np.testing.assert_array_equal(tout.numpy(), dev[np.arange(n) % 2])
        return
    two = [cv.Image.from_numpy(s, K.IMAGE_FORMAT_RGB8) for s in src]
    bi, bo = cv.ImageBatchVarShape(n), cv.ImageBatchVarShape(n)
    outs = [cv.Image.alloc((w, h), K.IMAGE_FORMAT_RGB8) for _ in range(n)]
    for i in range(n):
        bi.push_back(two[i % 2])
        bo.push_back(outs[i])
    mats = cv.Tensor.from_numpy(np.asarray([m] * n, np.float32), "NW")
    cv.WarpAffine(n)(None, bi, bo, mats, CUBIC, 1, (0, 0, 0, 0))
    torch.cuda.synchronize()
    for i in range(n):
        np.testing.assert_array_equal(outs[i].plane_view(0, np.uint8, 3).cpu().numpy(), dev[i % 2], err_msg=str(i))


# 75 000 rows of tiles of the form whose blocks are one wave; at whole places a bicubic sum is the pixel itself
def test_bicubic_of_a_tall_image(cv, orc, gpu):
    src = orc.fill_u8((1, 600000, 16, 3), 91)
    tin, tout = cv.Tensor.from_numpy(src, "NHWC"), cv.Tensor.alloc([1, 600000, 16, 3], np.uint8, "NHWC")
    cv.WarpAffine(0)(None, tin, tout, [1.0, 0.0, 0.0, 0.0, 1.0, 0.0], CUBIC, 1, (0, 0, 0, 0))
    torch.cuda.synchronize()
    np.testing.assert_array_equal(tout.numpy(), src)


# the same for the other interpolations and borders, and for sources and results that are views: rows 4 bytes off a 16-byte
# boundary in another pitch. A view's result is the dense one's, bit for bit
@pytest.mark.parametrize("c", [3, 4])
@pytest.mark.parametrize("interp", [NEAREST, LINEAR, CUBIC])
@pytest.mark.parametrize("border", [0, 1, 2, 3, 4])
def test_wide_pixels_in_views(cv, orc, gpu, c, interp, border):
    for sw, sh, dw, dh, deg, scale in ((37, 21, 33, 17, 12.0, 0.9), (90, 70, 131, 41, -31.0, 1.4)):
        src = orc.fill_f32((2, sh, sw, c), 5 + dw + border)
        m, colour = rotation(sw, sh, deg, scale), (0.25, -3.0, 7.5, 0.125)
        results = []
        for lead, extra in ((0, 0), (1, 3)):
            def view(h, w, fill):
                buf = torch.full((2 * h * (w * c + extra) + 2 * lead + 8,), fill, device="cuda")
                t = torch.as_strided(buf, (2, h, w, c), (h * (w * c + extra), w * c + extra, c, 1), lead)
                return buf, t, cv.Tensor.wrap(buf.data_ptr() + 4 * lead, [2, h, w, c],
                                              [4 * h * (w * c + extra), 4 * (w * c + extra), 4 * c, 4], np.float32, "NHWC", keep=buf)
            _, s, tin = view(sh, sw, 99.0)
            s.copy_(torch.from_numpy(src))
            buf, d, tout = view(dh, dw, -7.0)
            cv.WarpAffine(0)(None, tin, tout, m, interp, border, colour)
            torch.cuda.synchronize()
            results.append(d.cpu().numpy().copy())
            d.fill_(-7.0)
            assert bool((buf == -7.0).all()), "floats outside the rows written"
        np.testing.assert_array_equal(results[0], results[1])
        dev = orc.warp(src, (dh, dw), orc.invert_affine(m), interp, border, colour, variant=1)
        assert np.abs(results[0] - dev).max() <= 1e-3


def make_c4_batch(cv, K, orc, n, seed):
    rng = np.random.default_rng(seed)
    bi, bo, hosts, outs, mats = cv.ImageBatchVarShape(n), cv.ImageBatchVarShape(n), [], [], []
    for i in range(n):
        w, h = int(rng.integers(640, 1921)), int(rng.integers(480, 1081))
        a = orc.fill_u8((h, w, 3), 0xC0FFEE04 + i)
        hosts.append(a)
        bi.push_back(cv.Image.from_numpy(a, K.IMAGE_FORMAT_RGB8))
        o = cv.Image.alloc((w, h), K.IMAGE_FORMAT_RGB8)
        outs.append(o)
        bo.push_back(o)
        mats.append(rotation(w, h, float(rng.uniform(-30, 30)), float(rng.uniform(0.8, 1.2))))
    return bi, bo, hosts, outs, np.asarray(mats, np.float32)


def test_config4_varshape_full_size(cv, K, orc, gpu):
    # 32 u8 RGB images, sizes in [640,1920]x[480,1080], rotation +-30deg / scale
    # 0.8-1.2 about the centre as forward maps, bilinear, constant border 0; <= 1 LSB vs golden
    n = 32
    bi, bo, hosts, outs, mats = make_c4_batch(cv, K, orc, n, 4)
    txf = cv.Tensor.from_numpy(mats, "NW")
    cv.WarpAffine(n)(None, bi, bo, txf, LINEAR, 0, (0, 0, 0, 0))
    torch.cuda.synchronize()
    for i in range(n):
        a, o = hosts[i], outs[i]
        res = o.plane_view(0, np.uint8, 3).cpu().numpy()
        minv = orc.invert_affine(mats[i])
        gold = orc.warp(a[None], a.shape[:2], minv, LINEAR, 0, (0, 0, 0, 0), variant=0, threads=1)[0]
        assert np.abs(res.astype(np.int16) - gold.astype(np.int16)).max() <= 1
        assert (res != gold).mean() < 0.02  # the fixed-point blend rounds differently on about 1 % of the bytes
        if i < 4:
            dev = orc.warp(a[None], a.shape[:2], minv, LINEAR, 0, (0, 0, 0, 0), variant=2)[0]
            np.testing.assert_array_equal(res, dev)


def test_varshape_small_all_modes_and_inverse_flag(cv, K, orc, gpu):
    rng = np.random.default_rng(11)
    n = 5
    bi, bo, hosts, outs, mats = cv.ImageBatchVarShape(n), cv.ImageBatchVarShape(n), [], [], []
    for i in range(n):
        w, h = int(rng.integers(20, 120)), int(rng.integers(20, 90))
        dw, dh = int(rng.integers(20, 140)), int(rng.integers(20, 100))
        a = orc.fill_u8((h, w, 4), 200 + i)
        hosts.append(a)
        bi.push_back(cv.Image.from_numpy(a, K.IMAGE_FORMAT_RGBA8))
        o = cv.Image.alloc((dw, dh), K.IMAGE_FORMAT_RGBA8)
        outs.append(o)
        bo.push_back(o)
        mats.append(rotation(w, h, float(rng.uniform(-40, 40)), float(rng.uniform(0.7, 1.4))))
    mats = np.asarray(mats, np.float32)
    op = cv.WarpAffine(8)
    for interp, border, inv in itertools.product((NEAREST, LINEAR, CUBIC), range(5), (False, True)):
        op(None, bi, bo, cv.Tensor.from_numpy(mats, "NW"), interp | (INVERSE_MAP if inv else 0), border,
           (10, 20, 30, 40))
        torch.cuda.synchronize()
        for i in range(n):
            w, h = outs[i].size
            res = outs[i].plane_view(0, np.uint8, 4).cpu().numpy()
            minv = mats[i] if inv else orc.invert_affine(mats[i])
            dev = orc.warp(hosts[i][None], (h, w), minv, interp, border, (10, 20, 30, 40), variant=device_variant(interp))[0]
            np.testing.assert_array_equal(res, dev, err_msg=str((interp, border, inv, i)))
    with pytest.raises(cv.Error) as e:
        cv.WarpAffine(4)(None, bi, bo, cv.Tensor.from_numpy(mats, "NW"), LINEAR)  # batch 5 > max 4
    assert e.value.status == 2
    with pytest.raises(cv.Error) as e:
        cv.WarpAffine(0)(None, bi, bo, cv.Tensor.from_numpy(mats, "NW"), LINEAR)
    assert e.value.status == 2


def homography_inverse(m):
    f = np.asarray(m, np.float32)
    d = f[0] * (f[4] * f[8] - f[5] * f[7]) + f[1] * (f[5] * f[6] - f[3] * f[8]) + f[2] * (f[3] * f[7] - f[4] * f[6])
    return np.array([(f[4] * f[8] - f[5] * f[7]) / d, -(f[1] * f[8] - f[2] * f[7]) / d, (f[1] * f[5] - f[2] * f[4]) / d,
                     -(f[3] * f[8] - f[5] * f[6]) / d, (f[0] * f[8] - f[2] * f[6]) / d, -(f[0] * f[5] - f[2] * f[3]) / d,
                     (f[3] * f[7] - f[4] * f[6]) / d, -(f[0] * f[7] - f[1] * f[6]) / d, (f[0] * f[4] - f[1] * f[3]) / d],
                    np.float32)


def test_warp_perspective(cv, K, orc, gpu):
    src = orc.fill_u8((2, 60, 80, 3), 21)
    H = [1.05, 0.08, -3.0, -0.04, 0.97, 2.0, 2e-4, -1e-4, 1.0]
    op = cv.WarpPerspective(4)
    for interp, border in itertools.product((NEAREST, LINEAR, CUBIC), (0, 1, 4)):
        for inv in (True, False):
            tout = cv.Tensor.alloc([2, 50, 90, 3], np.uint8, "NHWC")
            op(None, cv.Tensor.from_numpy(src, "NHWC"), tout, H, interp | (INVERSE_MAP if inv else 0), border,
               (5, 6, 7, 0))
            torch.cuda.synchronize()
            minv = np.asarray(H, np.float32) if inv else homography_inverse(H)
            ref = orc.warp(src, (50, 90), minv, interp, border, (5, 6, 7, 0), perspective=True, variant=device_variant(interp))
            d = np.abs(tout.numpy().astype(np.int16) - ref.astype(np.int16))
            # 1/x on the device is correctly rounded like the host's; allow 1 LSB for the inverse path whose
            # matrix entries come from float divisions evaluated on host in this test
            assert d.max() <= (0 if inv else 1)
    # var-shape: two images, matrices in a [N,9] tensor
    bi, bo = cv.ImageBatchVarShape(2), cv.ImageBatchVarShape(2)
    outs = []
    for i in range(2):
        bi.push_back(cv.Image.from_numpy(src[i], K.IMAGE_FORMAT_RGB8))
        o = cv.Image.alloc((90, 50), K.IMAGE_FORMAT_RGB8)
        outs.append(o)
        bo.push_back(o)
    mats = np.asarray([H, H], np.float32)
    op(None, bi, bo, cv.Tensor.from_numpy(mats, "NW"), LINEAR | INVERSE_MAP, 1, (0, 0, 0, 0))
    torch.cuda.synchronize()
    ref = orc.warp(src, (50, 90), H, LINEAR, 1, perspective=True, variant=2)
    for i in range(2):
        np.testing.assert_array_equal(outs[i].plane_view(0, np.uint8, 3).cpu().numpy(), ref[i])


# a perspective's quotients against the correctly rounded ones, for every mantissa of the third row and both signs: 1 / x is
# carried into the result by a bilinear sample of a row of 0, 1, 2, ... at (2^n / x, 0), which float32 holds exactly
# (24 bits in all: the products of the integer part and the fraction are exact, and so is their sum). In the range of
# exponents that takes the shorter form, its ends, and outside it
@pytest.mark.parametrize("sign", [1, -1])
@pytest.mark.parametrize("e", [-126, -124, -123, -64, 0, 1, 77, 121, 122, 123, 126])
def test_perspective_quotients(cv, gpu, e, sign):
    n = min(20, 127 - e)  # (2^(n + e) is a float32)
    ramp = torch.arange((1 << n) + 8, dtype=torch.float32, device="cuda").repeat(3, 1)[None, :, :, None].contiguous()
    w, h = 4096, 2048
    out = torch.zeros((1, h, w, 1), device="cuda")
    x0 = sign * 2.0 ** e
    # (a quotient below 0 times -0 is 0, and 0 is inside the image)
    m = [0.0, 0.0, sign * 2.0 ** (n + e)] + [sign * 0.0] * 3 + [x0 * 2.0 ** -23, x0 * 2.0 ** -11, x0]
    cv.WarpPerspective(0)(None, cv.Tensor.from_torch(ramp, "NHWC"), cv.Tensor.from_torch(out, "NHWC"), m, LINEAR | INVERSE_MAP, 1,
                          (0, 0, 0, 0))
    torch.cuda.synchronize()
    x = (np.float32(x0) * (1 + np.arange(w * h, dtype=np.float64) * 2.0 ** -23)).astype(np.float32)
    want = np.float64(np.float32(1) / x) * (sign * 2.0 ** (n + e))
    np.testing.assert_array_equal(out.cpu().numpy().reshape(-1), want)


def test_perspective_quotients_in_and_out_of_range_in_one_wave(cv, gpu):
    # third rows on both sides of 2^123, and of 2^-123, within the samples of one lane
    ramp = torch.arange(40, dtype=torch.float32, device="cuda").repeat(3, 1)[None, :, :, None].contiguous()
    for e, num in ((118, 123), (-125, -120)):
        out = torch.zeros((1, 8, 64, 1), device="cuda")
        m = [0.0, 0.0, 2.0 ** num, 0.0, 0.0, 0.0, 2.0 ** e, 0.0, 2.0 ** e]
        cv.WarpPerspective(0)(None, cv.Tensor.from_torch(ramp, "NHWC"), cv.Tensor.from_torch(out, "NHWC"), m, LINEAR | INVERSE_MAP, 1,
                              (0, 0, 0, 0))
        torch.cuda.synchronize()
        x = (2.0 ** e * np.arange(1, 65)).astype(np.float32)
        want = np.float64(np.float32(1) / x) * 2.0 ** num
        np.testing.assert_array_equal(out.cpu().numpy().reshape(8, 64), np.tile(want, (8, 1)))


# seeded random cases: every element type and channel count, interpolation and border mode; sources and outputs from 1
# pixel to 1400 x 900; rotations by any angle with independent axis scales of 0.4 to 2.5 and a shear, mapped near the
# source's centre or far outside it; affine and perspective; tensors and image batches of mixed sizes. Inverse maps
# are given, so device and oracle start from the same float32 matrix: exact for integers, 1e-3 for float32.
@pytest.mark.parametrize("seed", [31, 32])
def test_random_cases(cv, K, orc, gpu, seed):
    rng = np.random.default_rng(seed)
    fmts = {(np.uint8, 1): "U8", (np.uint8, 3): "RGB8", (np.uint8, 4): "RGBA8", (np.float32, 1): "F32", (np.float32, 3): "RGBf32"}
    types = [(np.uint8, 3), (np.uint8, 3), (np.uint8, 1), (np.uint8, 4), (np.uint16, 3), (np.int16, 1), (np.float32, 3),
             (np.float32, 4), (np.float32, 1)]
    for it in range(150):
        dt, c = types[int(rng.integers(0, len(types)))]
        interp, border, n = int(rng.integers(0, 3)), int(rng.integers(0, 5)), int(rng.integers(1, 4))
        persp = rng.random() < 0.3
        varshape = (dt, c) in fmts and rng.random() < 0.5
        big = rng.random() < 0.2
        bval = tuple(float(v) for v in rng.integers(0, 255, 4))

        def size():
            if big:
                return int(rng.integers(300, 1400)), int(rng.integers(200, 900))
            return int(rng.integers(1, 200)), int(rng.integers(1, 150))

        def matrix(sw, sh, dw, dh):
            t = np.deg2rad(float(rng.uniform(-180, 180)) if rng.random() < 0.8 else float(rng.choice([0, 90, 180, 45])))
            sx, sy = float(np.exp(rng.uniform(-0.9, 0.9))), float(np.exp(rng.uniform(-0.9, 0.9)))
            a, b, d, e = sx * np.cos(t), -sy * np.sin(t) + float(rng.uniform(-0.2, 0.2)), sx * np.sin(t), sy * np.cos(t)
            off = float(rng.uniform(-0.3, 0.3)) if rng.random() < 0.85 else float(rng.uniform(-3, 3))
            cx, cy = (sw - 1) / 2 + off * sw, (sh - 1) / 2 + off * sh
            m = [a, b, cx - a * (dw - 1) / 2 - b * (dh - 1) / 2, d, e, cy - d * (dw - 1) / 2 - e * (dh - 1) / 2]
            if persp:
                m += [float(rng.uniform(-2e-4, 2e-4)), float(rng.uniform(-2e-4, 2e-4)), 1.0]
            return np.asarray(m, np.float32)

        def image(h, w, s):
            if dt == np.float32:
                return orc.fill_f32((h, w, c), s) * 255
            return orc.fill_u8((h, w, c, np.dtype(dt).itemsize), s).view(dt).reshape(h, w, c)

        def compare(res, src, hw, m, what):
            dev = orc.warp(src, hw, m, interp, border, bval, perspective=persp, variant=device_variant(interp, dt))
            case = "seed %d case %d %s: %s x%d interp %d border %d persp %d %s -> %s m %s" % (
                seed, it, what, np.dtype(dt).name, c, interp, border, persp, src.shape, hw, m.tolist())
            if dt == np.float32:
                assert np.abs(res - dev).max() <= 1e-3, case
            else:
                np.testing.assert_array_equal(res, dev, err_msg=case)

        op = (cv.WarpPerspective if persp else cv.WarpAffine)(8)
        if varshape:
            fmt = getattr(K, "IMAGE_FORMAT_" + fmts[(dt, c)])
            bi, bo, hosts, outs, mats = cv.ImageBatchVarShape(n), cv.ImageBatchVarShape(n), [], [], []
            for i in range(n):
                (sw, sh), (dw, dh) = size(), size()
                hosts.append(image(sh, sw, 100 * it + i + seed))
                bi.push_back(cv.Image.from_numpy(hosts[-1], fmt))
                outs.append(cv.Image.alloc((dw, dh), fmt))
                bo.push_back(outs[-1])
                mats.append(matrix(sw, sh, dw, dh))
            mats = np.asarray(mats, np.float32)
            op(None, bi, bo, cv.Tensor.from_numpy(mats, "NW"), interp | INVERSE_MAP, border, bval)
            torch.cuda.synchronize()
            for i in range(n):
                w, h = outs[i].size
                compare(outs[i].plane_view(0, dt, c).cpu().numpy()[None], hosts[i][None], (h, w), mats[i], "image %d" % i)
        else:
            (sw, sh), (dw, dh) = size(), size()
            src = np.stack([image(sh, sw, 100 * it + i + seed) for i in range(n)])
            m = matrix(sw, sh, dw, dh)
            tout = cv.Tensor.alloc([n, dh, dw, c], dt, "NHWC")
            op(None, cv.Tensor.from_numpy(src, "NHWC"), tout, m.tolist(), interp | INVERSE_MAP, border, bval)
            torch.cuda.synchronize()
            compare(tout.numpy(), src, (dh, dw), m, "tensor")


def test_tensor_negative(cv, gpu):
    op = cv.WarpAffine(0)
    a = cv.Tensor.alloc([2, 8, 8, 3], np.uint8, "NHWC")
    ident = [1, 0, 0, 0, 1, 0]
    for out, flags, border in [(cv.Tensor.alloc([2, 8, 8, 3], np.float32, "NHWC"), LINEAR, 0),
                               (cv.Tensor.alloc([3, 8, 8, 3], np.uint8, "NHWC"), LINEAR, 0),
                               (cv.Tensor.alloc([2, 8, 8, 4], np.uint8, "NHWC"), LINEAR, 0),
                               (cv.Tensor.alloc([2, 3, 8, 8], np.uint8, "NCHW"), LINEAR, 0),
                               (cv.Tensor.alloc([2, 8, 8, 3], np.uint8, "NHWC"), 3, 0),     # AREA
                               (cv.Tensor.alloc([2, 8, 8, 3], np.uint8, "NHWC"), LINEAR, 9)]:
        with pytest.raises(cv.Error) as e:
            op(None, a, out, ident, flags, border)
        assert e.value.status == 2
