"""Store growth (tp_grow_rows): the stored pages survive, spare slots are zero,
and the bytes between the two are left to the encoder that writes them."""

import ctypes

import pytest
import torch

from turbopolar_amd import TurboPolarConfig, TurboPolarKVCacheRuntime, _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,src_row,dst_row,keep,clear_from", [
    (3, 8192, 16384, 8192, 8192),  # 16-byte chunks, a full doubling
    (2, 64 * 11, 64 * 44, 64 * 7, 64 * 9),  # a gap left alone
    (5, 8, 16, 6, 10),  # fp16 page scales: 2-byte units
    (1, 3, 7, 3, 4),  # odd bytes
    (4, 0, 4096, 0, 0),  # nothing kept: all cleared
    (2, 256, 512, 256, 512),  # nothing cleared
    (2, 1 << 20, 3 << 20, 1 << 20, 2 << 20),  # several workgroups a row
    (70000, 16, 32, 16, 16),  # more rows than the grid's second size
])
def test_grow_rows(device, rows, src_row, dst_row, keep, clear_from):
    print(f"[grow] rows={rows} src={src_row} dst={dst_row} keep={keep} clear={clear_from}", flush=True)
    src = torch.randint(1, 256, (rows, max(src_row, 1)), dtype=torch.uint8, device=device)[:, :src_row].contiguous()
    dst = torch.full((rows, dst_row), 7, dtype=torch.uint8, device=device)
    want = dst.clone()
    want[:, :keep] = src[:, :keep]
    want[:, clear_from:] = 0
    g = (_lib.TPGrow * 1)(_lib.TPGrow(src.data_ptr() if keep else None, dst.data_ptr(), src_row, dst_row, keep, clear_from))
    assert _lib.lib().tp_grow_rows(g, 1, rows, torch.cuda.current_stream().cuda_stream) == 0
    torch.cuda.synchronize()
    assert torch.equal(dst, want)


@pytest.mark.parametrize("int8,l1,deep,split", [(False, 4, 4, 64), (True, 4, 8, 0), (True, 4, 2, 46)])
def test_store_grows_like_one_reservation(device, int8, l1, deep, split):
    """Pages appended a few at a time equal one bulk append; spare slots are zero."""
    cfg = TurboPolarConfig(num_q_heads=4, num_kv_heads=2, use_int8_radii=int8, k_angle_bits_level1=l1,
                           k_angle_bits_deep=deep, split_dim=split)
    g = torch.Generator(device=device).manual_seed(3)
    k, v = (torch.randn((2, 2, 64 * 21, 128), generator=g, device=device).half() for _ in range(2))
    one, many = TurboPolarKVCacheRuntime(cfg), TurboPolarKVCacheRuntime(cfg)
    one.append(k, v)
    for a, b in ((0, 3), (3, 4), (4, 5), (5, 16), (16, 17), (17, 21)):
        many.append(k[:, :, 64 * a:64 * b].contiguous(), v[:, :, 64 * a:64 * b].contiguous())
    torch.cuda.synchronize()
    for name in ("radii", "angle_codes_l1", "angle_codes_deep", "radii_scales"):
        x, y = getattr(one.k_storage, name), getattr(many.k_storage, name)
        assert (x is None) == (y is None)
        if x is not None:
            assert x.shape == y.shape and torch.equal(x, y) and not x[:, :, 21:].any()
    for name in ("codes", "scales"):
        x, y = getattr(one.v_storage, name), getattr(many.v_storage, name)
        assert torch.equal(x, y) and not x[:, :, 21:].any()
    assert one.get_io_telemetry() == many.get_io_telemetry()


def test_reservation_grows_a_store_in_its_own_form(device):
    """The host test's stores on the GPU: two launches of the buffers' own rows."""
    from test_runtime_host import grow_in_own_form

    print("[grow-own-form]", flush=True)
    grow_in_own_form("cuda")


def test_grow_rows_rejects_bad_bounds():
    def call(n=1, rows=1, **kw):
        d = dict(src=4096, dst=8192, src_row=16, dst_row=32, keep=16, clear_from=16)
        d.update(kw)
        return _lib.lib().tp_grow_rows((_lib.TPGrow * 1)(_lib.TPGrow(**d)), n, rows, None)

    for kw in (dict(n=0), dict(n=9), dict(rows=0), dict(dst=None), dict(src=None), dict(keep=17), dict(clear_from=8),
               dict(clear_from=33), dict(keep=-1)):
        assert call(**kw) == _lib.TP_ERR_INVALID, kw
    assert ctypes.sizeof(_lib.TPGrow) == 48
