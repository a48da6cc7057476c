"""ReadChannels / WriteChannels of small pixels (four pixels a lane) and their transfer tables on the GPU, at the sizes
where the split of a row into groups, the alignment of the user image or the tables' bounds matter."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BPC = {1: 1, 2: 2, 3: 2, 4: 4, 5: 4}
SMALL_PIXELS = [(fmt, channels) for fmt in BPC for channels in range(1, 9) if channels * BPC[fmt] <= 8]


def halves(rng, count):
    return rng.integers(0, 0x3C01, count, dtype=np.uint16)                # [0, 1]


def read(ntc, device, d_planar, w, h, set_channels, first, count, fmt, stride, offset, dither=0, spaces=(0, 0), pitch=None):
    pitch = pitch or w * stride + BPC[fmt]
    d_dst = device.alloc(offset + h * pitch)
    d_dst.fill(0xEE)
    rc = ntc.abi.ReadChannels()
    rc.planarPairs, rc.planarBytes = d_planar.ptr, d_planar.nbytes
    rc.width, rc.height, rc.setChannels, rc.firstChannel, rc.numChannels = w, h, set_channels, first, count
    rc.dst, rc.dstBytes, rc.format, rc.pixelStride, rc.rowPitch, rc.useDithering = d_dst.ptr + offset, d_dst.nbytes - offset, fmt, stride, pitch, dither
    for i in range(count):
        rc.srcColorSpaces[i], rc.dstColorSpaces[i] = spaces
    device.call("read_channels", rc)
    device.synchronize()
    return d_dst.download()[offset:], pitch


@pytest.mark.parametrize("fmt,channels", SMALL_PIXELS)
def test_read_groups_at_their_edges(ntc, device, oracle, fmt, channels):
    rng = np.random.default_rng(10 * fmt + channels)
    zeros = np.zeros(16, dtype=np.uint8)
    for w, h, first, dither in ((1, 3, 0, 0), (3, 1, 1, 1), (4, 2, 1, 0), (5, 9, 0, 1), (31, 3, 2, 0), (33, 35, 1, 1), (130, 5, 3, 0), (257, 18, 0, 1), (259, 4, 4, 0)):
        count = min(channels, 12 - first) if w != 130 else max(1, channels - 2)          # (130: default-valued channels behind the copied ones)
        planar = halves(rng, w * h * 12)
        d_planar = device.upload(planar)
        got, pitch = read(ntc, device, d_planar, w, h, 12, first, count, fmt, channels * BPC[fmt], (w % 3) * BPC[fmt], dither)
        want = np.full(got.size, 0xEE, dtype=np.uint8)
        assert oracle.ntc_oracle_read_channels_ex(planar.ctypes.data, w, h, 12, first, count, want.ctypes.data, fmt, channels * BPC[fmt], pitch, dither,
                                                  zeros.ctypes.data, zeros.ctypes.data) == 0
        assert np.array_equal(got, want), (w, h, first)


@pytest.mark.parametrize("fmt,channels", SMALL_PIXELS)
def test_write_groups_at_their_edges(ntc, device, oracle, fmt, channels):
    rng = np.random.default_rng(100 + 10 * fmt + channels)
    for w, h, first, flip in ((1, 3, 0, 0), (3, 1, 1, 1), (4, 2, 1, 0), (5, 9, 0, 1), (31, 3, 2, 0), (33, 35, 1, 1), (130, 5, 3, 0), (257, 18, 0, 1), (259, 4, 4, 0)):
        count = min(channels, 12 - first) if w != 130 else max(1, channels - 2)
        stride, offset = channels * BPC[fmt], (w % 3) * BPC[fmt]
        pitch = w * stride + BPC[fmt]
        if fmt == 3:
            image = halves(rng, (offset + h * pitch) // 2).view(np.uint8)
        elif fmt == 4:
            image = rng.uniform(-2, 70000, (offset + h * pitch) // 4).astype(np.float32).view(np.uint8)
        else:
            image = rng.integers(0, 256, offset + h * pitch, dtype=np.uint8)
        start = np.full(w * h * 12, 0x1234, dtype=np.uint16)
        d_image, d_planar = device.upload(image), device.upload(start)
        wc = ntc.abi.WriteChannels()
        wc.src, wc.srcBytes, wc.format, wc.verticalFlip, wc.pixelStride, wc.rowPitch = d_image.ptr + offset, d_image.nbytes - offset, fmt, flip, stride, pitch
        wc.planarPairs, wc.planarBytes = d_planar.ptr, d_planar.nbytes
        wc.width, wc.height, wc.setChannels, wc.firstChannel, wc.numChannels = w, h, 12, first, count
        device.call("write_channels", wc)
        device.synchronize()
        want, user = start.copy(), np.ascontiguousarray(image[offset:])
        assert oracle.ntc_oracle_write_channels(user.ctypes.data, fmt, flip, stride, pitch, want.ctypes.data, w, h, 12, first, count) == 0
        assert np.array_equal(d_planar.download().view(np.uint16), want), (w, h, first, flip)


@pytest.mark.parametrize("spaces", [(1, 1), (1, 0), (0, 1), (2, 0), (0, 2), (2, 1), (1, 2), (2, 2)])
def test_tables_in_lds_and_in_memory_give_the_same(ntc, device, spaces):
    """Every half, through the launch that stages a table (an image of two million pixels) and through one that does
    not (65536 pixels); one pixel a lane (a stride of 16 bytes) as well."""
    w, h = 2048, 1028
    every = np.arange(65536, dtype=np.uint16)
    planar = np.zeros(w * h * 2, dtype=np.uint16).reshape(h, w, 2)
    planar[:, :, 0] = np.resize(every, w * h).reshape(h, w)
    d_big = device.upload(planar.reshape(-1))
    big, pitch = read(ntc, device, d_big, w, h, 2, 0, 1, 4, 4, 0, spaces=spaces, pitch=4 * w)
    small_planar = np.zeros(65536 * 2, dtype=np.uint16)
    small_planar[0::2] = every
    d_small = device.upload(small_planar)
    small, _ = read(ntc, device, d_small, 256, 256, 2, 0, 1, 4, 4, 0, spaces=spaces, pitch=4 * 256)
    wide, _ = read(ntc, device, d_small, 256, 256, 2, 0, 1, 4, 16, 0, spaces=spaces, pitch=16 * 256)
    assert np.array_equal(big.view(np.uint32), np.resize(small.view(np.uint32), w * h))
    assert np.array_equal(wide.view(np.uint32).reshape(-1, 4)[:, 0], small.view(np.uint32))


@pytest.mark.parametrize("space", [1, 2])
@pytest.mark.parametrize("w,h", [(64, 16), (2048, 1024)])
def test_resized_colour_channels_equal_their_parts(ntc, device, space, w, h):
    """A 2 : 1 reduction of a channel stored in sRGB / HLG against decoding (read as FLOAT32), averaging (numpy) and
    encoding (write from FLOAT32, by the math library): halves of every magnitude, with and without tables in LDS."""
    rng = np.random.default_rng(w + space)
    planar = np.zeros((h, 2, w, 2), dtype=np.uint16)                      # four channels: pairs (0, 1) and (2, 3)
    planar[:, 0] = halves(rng, h * w * 2).reshape(h, w, 2)
    planar[:, 1] = rng.integers(0x3000, 0x3E00, h * w * 2, dtype=np.uint16).reshape(h, w, 2)      # up to 1.5
    d_src = device.upload(planar.reshape(-1))
    spaces = (ntc.abi.C.c_uint8 * 16)(*([space, 0, space, space] + [0] * 12))
    d_dst = device.alloc(w * h * 2)
    device.call("resize_planar", d_src.ptr, d_src.nbytes, w, h, d_dst.ptr, d_dst.nbytes, w // 2, h // 2, 4, spaces)
    device.synchronize()
    got = d_dst.download().view(np.uint16).reshape(h // 2, 2, w // 2, 2)
    for channel in range(4):
        linear, _ = read(ntc, device, d_src, w, h, 4, channel, 1, 4, 4, 0, spaces=(spaces[channel], 0), pitch=4 * w)
        v = linear.view(np.float32).reshape(h, w)
        mean = ((v[0::2, 0::2] + v[0::2, 1::2]) + v[1::2, 0::2]) + v[1::2, 1::2]
        mean = np.ascontiguousarray(mean * np.float32(0.25))
        d_mean, d_out = device.upload(mean), device.alloc(w * h)
        wc = ntc.abi.WriteChannels()
        wc.src, wc.srcBytes, wc.format, wc.pixelStride, wc.rowPitch = d_mean.ptr, d_mean.nbytes, 4, 4, 2 * w
        wc.planarPairs, wc.planarBytes = d_out.ptr, d_out.nbytes
        wc.width, wc.height, wc.setChannels, wc.firstChannel, wc.numChannels = w // 2, h // 2, 2, 0, 1
        wc.dstColorSpaces[0] = spaces[channel]
        device.call("write_channels", wc)
        device.synchronize()
        want = d_out.download().view(np.uint16).reshape(h // 2, w // 2, 2)[:, :, 0]
        assert np.array_equal(got[:, channel // 2, :, channel % 2], want), channel


@pytest.mark.parametrize("w,h", [(1, 1), (128, 4), (128, 8), (129, 5), (256, 127), (1024, 1028), (4100, 33)])
def test_loss_sums_of_one_group_and_of_many(ntc, device, oracle, w, h):
    """One workgroup, one group of workgroups, several groups, one row a wave and more: twice, so that the arrival
    counters are found as they were left."""
    rng = np.random.default_rng(w + h)
    a, b = halves(rng, w * h * 6), halves(rng, w * h * 6)
    d_a, d_b = device.upload(a), device.upload(b)
    want = np.zeros(16, dtype=np.float64)
    oracle.ntc_oracle_image_loss(a.ctypes.data, b.ctypes.data, w, h, 6, 0x37, want.ctypes.data)
    results = []
    for _ in range(2):
        got = (ntc.abi.C.c_float * 16)()
        device.call("image_loss", d_a.ptr, d_b.ptr, d_a.nbytes, w, h, 6, 0x37, -1, 0, got)
        results.append(np.array(got[:]))
    assert np.allclose(results[0], want, rtol=2e-7, atol=0) and np.array_equal(results[0], results[1])


@pytest.mark.parametrize("w,h,channels", [(3, 50000, 2), (4, 40001, 16), (7, 20777, 2), (255, 530, 14), (1023, 137, 10), (1029, 1030, 6), (2050, 601, 4),
                                          (361, 363, 8), (4099, 1100, 2), (65536, 3, 2), (2100, 403, 16), (3841, 402, 12), (5000, 301, 16), (7170, 3000, 2)])
def test_loss_sums_of_whole_rows(ntc, device, oracle, w, h, channels):
    """Rows of one, two and more steps of the workgroup's lanes with what is left of them, several rows a workgroup's lanes
    take together, fewer pairs than are loaded together, shares that begin and end inside a row, more workgroups than have a
    share, and images that fall to the other kernel."""
    rng = np.random.default_rng(w * h)
    a, b = halves(rng, w * h * channels), halves(rng, w * h * channels)
    d_a, d_b = device.upload(a), device.upload(b)
    want, got = np.zeros(16, dtype=np.float64), (ntc.abi.C.c_float * 16)()
    mask = 0x5FF7 & ((1 << channels) - 1)
    oracle.ntc_oracle_image_loss(a.ctypes.data, b.ctypes.data, w, h, channels, mask, want.ctypes.data)
    device.call("image_loss", d_a.ptr, d_b.ptr, d_a.nbytes, w, h, channels, mask, -1, 0, got)
    # (two texels' squares are added in float, the rest in double; rounded to float once)
    assert np.allclose(got[:], want, rtol=2e-7, atol=0)


@pytest.mark.parametrize("w,h", [(75, 64), (255, 530), (1023, 137), (1029, 1030), (2051, 601), (4099, 1100)])
def test_loss_of_odd_widths_adds_every_square_in_double(ntc, device, w, h):
    """Every other square is less than half a unit in the last place of the one before it: a sum of the two in float would
    drop it, and the mean comes out a unit lower."""
    faint = np.float16(0.995 * 2.0 ** -12)
    image = np.zeros((h, 2, w, 2), dtype=np.float16)
    image[:, :, 0:w - 1:2] = 1
    image[:, :, 1:w - 1:2] = faint
    flat, ones = image.reshape(-1).view(np.uint16), (w - 1) // 2 * h
    d_a, d_b = device.upload(flat), device.upload(np.zeros_like(flat))
    want = np.float32(ones * (1 + float(faint) ** 2) / (w * h))
    assert want != np.float32(ones / (w * h))
    got = (ntc.abi.C.c_float * 16)()
    device.call("image_loss", d_a.ptr, d_b.ptr, d_a.nbytes, w, h, 4, 0xF, -1, 0, got)
    assert list(got[:4]) == [want] * 4


@pytest.mark.parametrize("mask_channel", [-1, 5])
def test_loss_behind_queued_work(ntc, device, mask_channel):
    """Work of several milliseconds in front of the call, the last of which writes the image: the host's look for early sums
    gives up, and the sums are those of the written image."""
    big, w, h = device.alloc(1 << 30), 64, 64
    d_a, d_b = device.upload(np.zeros(w * h * 6, dtype=np.uint16)), device.upload(np.zeros(w * h * 6, dtype=np.uint16))
    got = (ntc.abi.C.c_float * 16)()
    for _ in range(30):                                                   # 30 GB written: 4 ms at least
        device.call("memset", big.ptr, 0, big.nbytes)
    device.call("memset", d_a.ptr, 0x38, d_a.nbytes)                      # every half 0x3838
    device.call("image_loss", d_a.ptr, d_b.ptr, d_a.nbytes, w, h, 6, 0x3F, mask_channel, 0, got)
    value = float(np.array([0x3838], dtype=np.uint16).view(np.float16)[0])
    assert np.allclose(got[:6], value * value, rtol=2e-7, atol=0) and not any(got[6:])
