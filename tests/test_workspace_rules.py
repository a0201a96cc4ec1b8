"""Host-side: which calls ask for scratch memory, and so take the route that needs it (no kernel is launched)."""
import pytest

F32, F16, BF16 = 0, 1, 2


@pytest.fixture(scope="module")
def lib():
    from bittorch_amd import _lib
    return _lib.load()


def _tensor_core_plain(b, k):
    def up(v):
        return -(-v // 256) * 256
    return up(b * (-(-k // 16) * 16)) + up(4 * b)


@pytest.mark.parametrize("n,k", [(4097, 4096), (11007, 4096), (4095, 11008), (16383, 16384), (8193, 3072)])
def test_single_rows_read_odd_packed_rows_as_they_are(lib, n, k):
    """A copy of the weights in tiles costs one row more than the bytes it would read one by one: 11007 x 4096 9.3 us against 17."""
    for dt in (F16, BF16):
        assert lib.bt_packed_forward_workspace_bytes(1, n, k, dt) == 0
    assert lib.bt_tensor_core_workspace_bytes(1, n, k) == _tensor_core_plain(1, k)


@pytest.mark.parametrize("b,n,k,float16,int8", [
    (2, 16383, 4096, False, False), (16, 4095, 16384, False, False), (8, 8193, 4096, False, False), (17, 2049, 8192, False, False),
    (24, 4097, 8192, True, False), (16, 16383, 8192, True, False), (3, 16383, 16384, True, False), (17, 1025, 16384, True, False), (1, 65537, 256, True, False), (2, 16385, 1024, True, False),
    (4, 32769, 1024, True, True), (16, 16383, 16384, True, True), (17, 8191, 2048, True, True), (24, 8191, 8192, True, True),
    (40, 4097, 4096, True, True), (16, 2051, 1040, False, False), (40, 4096, 4096, False, False)])
def test_odd_packed_rows_are_copied_where_that_pays(lib, b, n, k, float16, int8):
    tiles = lib.bt_tiled_weights_bytes(n, k)
    assert lib.bt_packed_forward_workspace_bytes(b, n, k, BF16) == (tiles if float16 else 0)
    assert lib.bt_tensor_core_workspace_bytes(b, n, k) == _tensor_core_plain(b, k) + (tiles if int8 else 0)


def test_fp32_rows_copy_odd_packed_rows_for_two_rows_or_long_ones(lib):
    for b, n, k, copies in ((1, 11007, 4096, False), (1, 8193, 5120, False), (1, 8193, 6144, True), (2, 11007, 4096, True)):
        planes = -(-b * 3 * (-(-k // 64) * 64) * 2 // 256) * 256
        assert lib.bt_packed_forward_workspace_bytes(b, n, k, F32) == planes + (lib.bt_tiled_weights_bytes(n, k) if copies else 0)


@pytest.mark.parametrize("b,k,padded", [(1, 257, False), (3, 257, False), (4, 257, True), (16, 385, True), (16, 258, False), (16, 4092, False),
                                        (17, 258, True), (17, 256, False)])
def test_16_bit_rows_of_odd_length_are_padded_from_four_on(lib, b, k, padded):
    """Their 16-byte loads start on odd halves: 16 rows of 257 bf16 values 11.1 us as they lie, 6.6 through a copy."""
    want = -(-b * (-(-k // 8)) * 16 // 256) * 256 if padded else 0
    for dt in (F16, BF16):
        assert lib.bt_tiled_forward_workspace_bytes(b, 256, k, dt) == want
        assert lib.bt_packed_forward_workspace_bytes(b, 256, k, dt) == want


@pytest.mark.parametrize("m,n,k,scratch", [
    (300, 768, 768, 0), (64, 1024, 1024, 0),                                    # tiles of 128, one of them at most a compute unit
    (16384, 3072, 3072, 144 * 2 * (256 << 10)), (8192, 3072, 3072, 144 * 2 * (256 << 10)),  # 144 tiles of 256: two parts each
    (16384, 3584, 3584, 0), (4096, 4096, 4096, 0)])                             # 196 and 256 tiles: whole
def test_16_bit_weight_gradient_cuts_long_rounds(lib, m, n, k, scratch):
    """One long round over little more than half of the chip, 16384 x 3072 x 3072: 348 us whole, 291 in two parts a tile."""
    assert lib.bt_linear_grad_weight_16_workspace_bytes(m, n, k) == scratch


def test_16_bit_weight_gradient_refuses_what_the_kernel_cannot_take(lib):
    """(every call ends before a launch; the addresses are never read)"""
    from bittorch_amd import _lib
    a = 1 << 20

    def call(dy=a, x=a, dtype=BF16, scale=a, scale_dtype=F32, scale_len=256, dw=a, out=F32, m=64, n=256, k=512, ws=None, nbytes=0):
        return lib.bt_linear_grad_weight_16(dy, x, dtype, scale, scale_dtype, scale_len, dw, out, m, n, k, ws, nbytes, None)

    for bad in (dict(dy=None), dict(m=0), dict(scale_len=255), dict(dtype=F32), dict(out=F16), dict(scale_dtype=9), dict(n=252, scale_len=1),
                dict(k=508), dict(dy=a + 8), dict(x=a + 2), dict(dw=a + 4), dict(scale=a + 2), dict(n=1 << 24, scale_len=1)):
        assert call(**bad) == -1, bad
        assert "bt_linear_grad_weight_16" in _lib.last_error()
    need = lib.bt_linear_grad_weight_16_workspace_bytes(8192, 3072, 3072)
    big = dict(m=8192, n=3072, k=3072, scale_len=1)
    for ws, nbytes in ((None, 0), (a, need - 1), (a + 64, need)):
        assert call(ws=ws, nbytes=nbytes, **big) == -2
        assert "workspace" in _lib.last_error()
