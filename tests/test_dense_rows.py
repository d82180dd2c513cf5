"""Packed blocks dequantized into their place of a dense history, at head sizes
and lengths around the tiles of the row kernels, and copies of dense rows."""
import numpy as np
import pytest
import torch

from oracle import oracle
import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,T", [(8, 37), (32, 1), (64, 129), (96, 85), (128, 130), (256, 33), (1024, 9), (66, 20)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_k4_dequantize_sizes(D, T, dtype):
    from inquant.codec import CodecConfig, quantize
    x = torch.from_numpy(synth.normal(D + T, (2, 3, T, D))).cuda().to(dtype)
    packed = quantize(x, CodecConfig(salient_fraction=0.25))
    want = oracle.k4_dequantize({k: v.cpu().numpy() for k, v in packed.tensors.items()}, str(dtype)[6:])
    assert torch.equal(packed.dequantize().float().cpu(), torch.from_numpy(want))


@pytest.mark.parametrize("D,block,vbits,group,dtype", [
    (128, 256, 2, 64, torch.bfloat16), (64, 64, None, 64, torch.float16), (64, 48, 4, 32, torch.float32),
    (96, 100, 2, 32, torch.bfloat16), (66, 32, None, 32, torch.float16), (256, 32, 4, 128, torch.bfloat16)])
def test_materialize_places_every_block(D, block, vbits, group, dtype):
    from inquant.cache import CacheConfig, InQuantCache
    cache = InQuantCache(CacheConfig(block_size=block, residual_length=16, sink_tokens=3, value_bits=vbits,
                                     value_group_size=group))
    x = torch.from_numpy(synth.normal(D + block, (2, 5 * block + 40, 2, D))).cuda().to(dtype)
    k, v = x[0].transpose(0, 1)[None], x[1].transpose(0, 1)[None]
    cache.update(k[:, :, :3 * block + 30], v[:, :, :3 * block + 30], 0)
    cache.update(k[:, :, 3 * block + 30:], v[:, :, 3 * block + 30:], 0)       # a second run of blocks
    layer = cache._layers[0]
    for got, blocks, whole in zip(cache.materialize(0), (layer.key_blocks, layer.value_blocks), (k, v)):
        packed = [b.dequantize(dtype=dtype) for b in blocks]
        at = 3 + block * len(blocks)
        assert torch.equal(got, torch.cat([whole[:, :, :3], *packed, whole[:, :, at:]], 2))


@pytest.mark.parametrize("offset,width", [(0, 64), (1, 64), (2, 62), (0, 3)])
def test_copied_rows(offset, width):
    from inquant.cache import _copy_rows
    src = torch.randn(1, 3, 37, 80, device="cuda").bfloat16()
    dst = torch.zeros(1, 3, 50, 80, device="cuda").bfloat16()
    a, b = src[:, :, :20, offset:offset + width], src[:, :, 20:, offset:offset + width]
    _copy_rows([(a, dst[:, :, 25:45, :width]), (b, dst[:, :, :17, :width]), (a[:, :, :0], dst[:, :, :0, :width])])
    assert torch.equal(dst[:, :, 25:45, :width], a) and torch.equal(dst[:, :, :17, :width], b)
    assert np.count_nonzero(dst.float().cpu().numpy()) <= 3 * 37 * width


def test_rows_and_positions_of_another_device_are_left_to_torch(monkeypatch):
    from inquant.cache import CacheConfig, InQuantCache
    k = torch.randn(1, 2, 9, 64, device="cuda").bfloat16()
    pos = torch.arange(9, device="cuda")
    cache = InQuantCache(CacheConfig(block_size=8, residual_length=4, sink_tokens=2))
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 1)                # as under torch.cuda.device(1)
    monkeypatch.setattr("inquant.cache.nat.lib", lambda: pytest.fail("launched on the current device"))
    cache.update(k[:, :, :7], k[:, :, :7], 0, {"cache_position": pos[:7]})
    with pytest.raises(ValueError, match="contiguous append"):
        cache.update(k[:, :, 7:], k[:, :, 7:], 0, {"cache_position": pos[6:8]})
    for got in cache.update(k[:, :, 7:], k[:, :, 7:], 0, {"cache_position": pos[7:]}):
        assert torch.equal(got, k)


@pytest.mark.parametrize("vbits", [2, None])
def test_every_launch_of_the_cache_runs_on_the_gpu_of_its_tensors(monkeypatch, vbits):
    # GPU 1 is said to be the current one: updates, appends, seals and materialize switch to GPU 0 for their launches
    from inquant import _native
    from inquant.cache import CacheConfig, InQuantCache
    k = torch.randn(1, 2, 60, 128, device="cuda").bfloat16()
    pos = torch.arange(60, device="cuda")

    def session():
        cache = InQuantCache(CacheConfig(block_size=8, residual_length=4, sink_tokens=2, value_bits=vbits))
        out = [*cache.update(k[:, :, :30], k[:, :, :30], 0, {"cache_position": pos[:30]})]
        out += cache.update(k[:, :, 30:45], k[:, :, 30:45], 0, {"cache_position": pos[30:45]})
        for i in range(45, 60):
            view = cache.append_for_attention(k[:, :, i:i + 1], k[:, :, i:i + 1], 0, {"cache_position": pos[i:i + 1]})
            out += [view.residual_key.clone(), view.residual_value.clone()]
        return out + [*cache.materialize(0)]

    want = session()
    current, launches, lib = [1], [], _native.lib()

    class Switch:
        def __init__(self, device):
            self.index = torch.device(device).index

        def __enter__(self):
            self.before, current[0] = current[0], self.index

        def __exit__(self, *error):
            current[0] = self.before

    class Spy:
        def __getattr__(self, name):
            launches.append((name, current[0]))
            return getattr(lib, name)

    row = _native.tail_append_row
    monkeypatch.setattr(torch._C, "_cuda_getDevice", lambda: current[0])        # torch.cuda.current_device() too
    monkeypatch.setattr(torch.cuda, "device", Switch)
    monkeypatch.setattr(_native, "lib", Spy)
    monkeypatch.setattr(_native, "tail_append_row", lambda *args: (launches.append(("append", current[0])), row(*args))[1])
    got = session()
    monkeypatch.undo()
    assert {name for name, _ in launches} >= {"append", "iq_copy_rows", "iq_check_positions", "iq_k4_dequantize_into"}
    assert all(device == 0 for _, device in launches) and current == [1]
    assert all(torch.equal(a, b) for a, b in zip(got, want, strict=True))


@pytest.mark.parametrize("dtype", [torch.int64, torch.int32])
def test_positions_are_checked_before_a_sealing_update_changes_the_layer(dtype):
    from inquant.cache import CacheConfig, InQuantCache
    cache = InQuantCache(CacheConfig(block_size=8, residual_length=4, sink_tokens=2, value_bits=2))
    k = torch.randn(1, 2, 70, 64, device="cuda").bfloat16()
    pos = torch.arange(140, dtype=dtype, device="cuda")[::2] // 2               # a strided view
    wrong = pos.clone()
    wrong[30] += 1
    cache.update(k[:, :, :20], k[:, :, :20], 0, {"cache_position": pos[:20]})
    before, blocks = cache.materialize(0), list(cache._layers[0].key_blocks)
    for bad in (wrong[20:60], pos[21:61]):
        with pytest.raises(ValueError, match="contiguous append"):
            cache.update(k[:, :, 20:60], k[:, :, 20:60], 0, {"cache_position": bad})
        assert cache.get_seq_length() == 20 and len(cache._layers[0].key_blocks) == len(blocks)
        assert all(torch.equal(a, b) for a, b in zip(cache.materialize(0), before))
    cache.update(k[:, :, 20:60], k[:, :, 20:60], 0, {"cache_position": pos[20:60]})
    assert cache.get_seq_length() == 60 and cache._layers[0].key_blocks[0] is blocks[0]
    with pytest.raises(ValueError, match="contiguous append"):
        InQuantCache(cache.config).update(k, k, 0, {"cache_position": wrong})


def test_first_positions_of_a_new_cache_make_no_flag_words():
    from inquant.cache import CacheConfig, InQuantCache
    k = torch.randn(1, 2, 9, 64, device="cuda").bfloat16()
    pos = torch.arange(9, device="cuda")
    cache = InQuantCache(CacheConfig(block_size=8, residual_length=4, sink_tokens=2))
    for wrong in (pos[1:6], pos[:5].flip(0), pos[:5] + 2 ** 40):
        with pytest.raises(ValueError, match="contiguous append"):
            cache.update(k[:, :, :5], k[:, :, :5], 0, {"cache_position": wrong})
    cache.update(k[:, :, :5], k[:, :, :5], 0, {"cache_position": pos[:5]})
    assert cache._flags is None
    with pytest.raises(ValueError, match="contiguous append"):
        cache.update(k[:, :, 5:7], k[:, :, 5:7], 0, {"cache_position": pos[6:8]})
    cache.update(k[:, :, 5:7], k[:, :, 5:7], 0, {"cache_position": pos[5:7]})
    assert cache.get_seq_length() == 7 and not any(cache._flags.tolist())


def test_positions_come_before_the_errors_of_a_sealing_update():
    from inquant.cache import CacheConfig, InQuantCache
    cache = InQuantCache(CacheConfig(block_size=8, residual_length=4, sink_tokens=2, value_bits=2, value_group_size=64))
    k = torch.randn(1, 2, 20, 96, device="cuda").bfloat16()                     # 96 channels: no whole groups of 64
    pos = torch.arange(20, device="cuda")
    with pytest.raises(ValueError, match="contiguous append"):
        cache.update(k, k, 0, {"cache_position": pos + 1})
    with pytest.raises(ValueError) as error:
        cache.update(k, k, 0, {"cache_position": pos})
    assert "contiguous append" not in str(error.value)
    cache.update(k[:, :, :5], k[:, :, :5], 0, {"cache_position": pos[:5]})      # no mismatch is left behind
    assert cache.get_seq_length() == 5


def test_an_argument_error_between_the_encoders_leaves_no_flag_behind():
    # the keys' encoder runs (and raises its flag) before the values' arguments are refused
    from inquant.cache import CacheConfig, InQuantCache
    cache = InQuantCache(CacheConfig(block_size=8, residual_length=4, sink_tokens=2, value_bits=2, value_group_size=64))
    k = torch.randn(1, 2, 24, 96, device="cuda").bfloat16()                     # 96 channels: no whole groups of 64
    k[0, 1, 5, 3] = float("nan")
    with pytest.raises(ValueError, match="divisible by group_size"):
        cache.update(k, k, 0)
    pos = torch.arange(14, device="cuda")
    cache.update(k[:, :, :13], k[:, :, :13], 0, {"cache_position": pos[:13]})   # 13 tokens: nothing to seal yet
    with pytest.raises(ValueError, match="divisible by group_size"):
        cache.append_for_attention(k[:, :, 13:14], k[:, :, 13:14], 0, {"cache_position": pos[13:]})
    good = torch.randn(1, 2, 24, 64, device="cuda").bfloat16()
    cache.update(good, good, 1)                                                 # finite data of another layer
    assert cache.get_seq_length(1) == 24 and not any(cache._flags.tolist())
