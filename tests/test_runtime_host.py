"""Runtime host logic without a GPU: the append validation contract
(turbo_polar_cache.py:55-104 of the reference), dense-tail bookkeeping below one
page, telemetry, reset, the storage doubling rule, and that page flushes on a
CPU tensor fail loudly instead of falling back to a CPU path."""

import numpy as np
import pytest
import torch

from turbopolar_amd import PolarKBlockStorage, TurboPolarConfig, TurboPolarFastCache, TurboPolarKVCacheRuntime
from turbopolar_amd.kernels import fp16_scale
from turbopolar_amd.storage import _doublings


def _rt(hkv=4):
    return TurboPolarKVCacheRuntime(TurboPolarConfig(num_q_heads=4, num_kv_heads=hkv))


def _x(B=1, H=4, T=1, D=128, dtype=torch.float16):
    return torch.randn((B, H, T, D)).to(dtype)


def test_rejects_non_tensors():
    with pytest.raises(TypeError):
        _rt().append(np.zeros((1, 4, 1, 128)), np.zeros((1, 4, 1, 128)))


@pytest.mark.parametrize("k,v,msg", [
    (torch.zeros(1, 4, 128), torch.zeros(1, 4, 128), "4-D inputs"),
    (torch.zeros(1, 4, 1, 128), torch.zeros(1, 4, 2, 128), "must match"),
    (torch.zeros(1, 4, 0, 128), torch.zeros(1, 4, 0, 128), "at least one token"),
    (torch.zeros(1, 4, 1, 128), torch.zeros(1, 4, 1, 128, dtype=torch.float16), "dtype"),
    (torch.zeros(1, 4, 1, 128, dtype=torch.bfloat16), torch.zeros(1, 4, 1, 128, dtype=torch.bfloat16),
     "only float16 and float32"),
    (torch.zeros(1, 2, 1, 128), torch.zeros(1, 2, 1, 128), "KV heads"),
    (torch.zeros(1, 4, 1, 64), torch.zeros(1, 4, 1, 64), "head_dim"),
])
def test_append_validation(k, v, msg):
    with pytest.raises(ValueError, match=msg):
        _rt().append(k, v)


def test_nonfinite_rejected():
    k = _x(T=2)
    k[0, 0, 0, 0] = float("inf")
    with pytest.raises(ValueError, match="finite"):
        _rt().append(k, _x(T=2))


def test_invariants_persist_and_reset():
    rt = _rt()
    rt.append(_x(T=3), _x(T=3))
    with pytest.raises(ValueError, match="batch size changed"):
        rt.append(_x(B=2), _x(B=2))
    with pytest.raises(ValueError, match="dtype changed"):
        rt.append(_x(dtype=torch.float32), _x(dtype=torch.float32))
    with pytest.raises(ValueError, match="KV head count changed"):
        rt.append(_x(H=2), _x(H=2))
    rt.reset()
    assert rt.partial_k is None and rt.actual_seq_len == 0
    rt.append(_x(B=2, T=1), _x(B=2, T=1))
    assert rt._batch_size == 2


def test_tail_bookkeeping_below_one_page():
    rt = _rt()
    ks = [_x(T=t) for t in (5, 20, 38)]
    for k in ks:
        rt.append(k, k)
    assert rt.actual_seq_len == 63
    assert torch.equal(rt.partial_k, torch.cat(ks, dim=2))
    tel = rt.get_io_telemetry()
    assert tel["partial_tokens"] == 63 and tel["total_blocks"] == 0
    assert tel["actual_cache_bytes"] == 2 * 4 * 63 * 128 * 2
    assert tel["compression_ratio"] == 1.0
    block, qv, tk, tv, qjl, seq = rt.get_fused_attention_inputs()
    assert block is None and qv is None and qjl is None and seq == 63 and tk.shape == (1, 4, 63, 128)


def test_page_flush_on_cpu_fails_loudly():
    rt = _rt()
    rt.append(_x(T=63), _x(T=63))
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        rt.append(_x(T=1), _x(T=1))


def test_decode_shape_contract():
    cache_cfg = TurboPolarConfig(num_q_heads=4, num_kv_heads=2)
    v = TurboPolarFastCache._validate_decode_shape
    q = torch.zeros(1, 4, 1, 128)
    kv = torch.zeros(1, 2, 1, 128)
    with pytest.raises(NotImplementedError, match="batch size 1"):
        v(torch.zeros(2, 4, 1, 128), torch.zeros(2, 2, 1, 128), torch.zeros(2, 2, 1, 128), cache_cfg)
    with pytest.raises(ValueError, match="single query"):
        v(torch.zeros(1, 4, 2, 128), kv, kv, cache_cfg)
    with pytest.raises(NotImplementedError, match="head_dim == 128"):
        v(torch.zeros(1, 4, 1, 64), torch.zeros(1, 2, 1, 64), torch.zeros(1, 2, 1, 64), cache_cfg)
    with pytest.raises(ValueError, match="GQA ratio"):
        v(torch.zeros(1, 5, 1, 128), kv, kv, cache_cfg)
    with pytest.raises(ValueError, match="4-D"):
        v(torch.zeros(1, 4, 128), kv, kv, cache_cfg)
    v(q, kv, kv, cache_cfg)


def test_storage_doubling_rule():
    """Capacity 4 * 2^k and the reference's _grow call sequence (storage.py:57-87)."""
    assert _doublings(4, 4) == ([], 4)
    assert _doublings(4, 5) == ([4], 8)
    assert _doublings(4, 512) == ([4, 8, 16, 32, 64, 128, 256], 512)
    assert _doublings(8, 2049) == ([8, 16, 32, 64, 128, 256, 512, 1024, 2048], 4096)


def test_storage_append_and_views_on_cpu():
    """PolarKBlockStorage.append: lazy init at capacity 4, doubling, growth bytes."""
    from turbopolar_amd.payload import PolarKeyBlock

    st = PolarKBlockStorage()
    for i in range(5):
        blk = PolarKeyBlock(
            radii=torch.full((1, 2, 64, 64), float(i), dtype=torch.float16),
            angle_codes_l1=torch.full((1, 2, 64, 16), i, dtype=torch.uint8),
            angle_codes_deep=torch.full((1, 2, 64, 16), i, dtype=torch.uint8),
            shape=(1, 2, 64, 128), block_size=64, head_dim=128, metadata={"l1_bits": 4},
        )
        st.append(blk)
    assert st.block_count == 5 and st.capacity == 8 and st.reallocation_count == 1
    assert st.bytes_copied_during_growth == 4 * (1 * 2 * 64 * (64 * 2 + 16 + 16))
    u = st.to_unified_block((1, 2, 5 * 64, 128))
    assert u.radii.shape == (1, 2, 5, 64, 64)
    assert [float(u.radii[0, 0, s, 0, 0]) for s in range(5)] == [0, 1, 2, 3, 4]


def test_reservation_grows_a_store_in_its_own_form():
    """reserve() on a store that holds appended pages keeps their shape, type and
    device, also where they are not the encoder's (32-token blocks, int8 radii), and
    counts the growth by them."""
    grow_in_own_form("cpu")


def grow_in_own_form(device):
    from turbopolar_amd.payload import PolarKeyBlock, QuantizedVBlock
    from turbopolar_amd.codecs import PolarQuantEncoder
    from turbopolar_amd.storage import QuantVBlockStorage

    g = torch.Generator().manual_seed(7)
    rand = lambda shape, dt: torch.randint(-100, 100, shape, generator=g).to(dt).to(device)  # noqa: E731
    st, vs = PolarKBlockStorage(), QuantVBlockStorage()
    blocks = [PolarKeyBlock(radii=rand((2, 3, 32, 64), torch.int8), angle_codes_l1=rand((2, 3, 32, 8), torch.uint8),
                            angle_codes_deep=rand((2, 3, 32, 12), torch.uint8), shape=(2, 3, 32, 128), block_size=32,
                            head_dim=128, radii_scales=rand((2, 3, 1, 1), torch.float16), metadata={"l1_bits": 4})
              for _ in range(3)]
    vblocks = [QuantizedVBlock(codes=rand((2, 3, 1, 64, 128), torch.int8), scales=rand((2, 3, 1, 64, 4), torch.float16),
                               group_size=32) for _ in range(3)]
    for b, v in zip(blocks, vblocks):
        st.append(b)
        vs.append(v)
    other = PolarQuantEncoder(TurboPolarConfig(num_q_heads=4, num_kv_heads=1))
    st.reserve(9, other, 1, 1, "cpu")
    vs.reserve(9, 1, 1, "cpu")
    assert (st.capacity, st.reallocation_count, vs.capacity) == (16, 2, 16)
    assert st.bytes_copied_during_growth == (4 + 8) * 2 * 3 * (32 * (64 + 8 + 12) + 2)
    for name in ("radii", "angle_codes_l1", "angle_codes_deep"):
        t = getattr(st, name)
        assert t.shape == (2, 3, 16) + getattr(blocks[0], name).shape[2:] and t.device.type == torch.device(device).type
        assert t.dtype == getattr(blocks[0], name).dtype
        for i, b in enumerate(blocks):
            assert torch.equal(t[:, :, i], getattr(b, name)), (name, i)
        assert not t[:, :, 3:].any()
    for i, (b, v) in enumerate(zip(blocks, vblocks)):
        assert torch.equal(st.radii_scales[:, :, i], b.radii_scales)
        assert torch.equal(vs.codes[:, :, i], v.codes) and torch.equal(vs.scales[:, :, i], v.scales)
    assert not vs.codes[:, :, 3:].any() and not vs.scales[:, :, 3:].any()


def test_fp16_scale_of_any_number():
    """The scale is taken from what the caller hands over now: NumPy arrays and
    tensors are accepted, one changed in place gives its new value, and a zero
    keeps its sign."""
    for make in (float, np.float32, np.float64, np.array, torch.tensor):
        assert fp16_scale(make(0.088388)) == float(np.float16(0.088388)), make
    for x in (torch.tensor(0.5), np.array(0.5)):
        assert fp16_scale(x) == 0.5
        x *= 4
        assert fp16_scale(x) == 2.0
    assert fp16_scale(1) == fp16_scale(True) == 1.0
    assert [str(fp16_scale(z)) for z in (0.0, -0.0)] == ["0.0", "-0.0"]
    with pytest.raises(TypeError):
        fp16_scale(np.array([0.5, 0.6]))


def test_tail_of_a_refused_first_append_is_not_kept():
    """A cache that has accepted nothing takes any batch and type: the dense tail's
    buffers follow the first accepted append, not a refused one before it."""
    rt = _rt()
    rt._tail_k = rt._tail_v = torch.zeros((1, 4, 64, 128), dtype=torch.float16)  # as the refused append sized it
    k, v = _x(B=3, T=5, dtype=torch.float32), _x(B=3, T=5, dtype=torch.float32)
    rt.append(k, v)
    assert rt._tail_k.shape == (3, 4, 64, 128) and rt._tail_k.dtype == torch.float32
    assert torch.equal(rt.partial_k, k) and torch.equal(rt.partial_v, v)
