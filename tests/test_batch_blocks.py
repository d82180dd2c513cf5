"""Blocks of a batched encode: their fields are views made when they are read,
and the packed decode takes their addresses from the batch."""
import copy
import dataclasses
import pickle

import pytest
import torch


def _batches():
    from inquant.codec import PackedTensor
    from inquant.value_codec import PackedValues
    n, h, t, d, s = 5, 2, 8, 64, 8
    i = torch.arange(n * h * t * d).reshape(n, h, t, d)
    k = PackedTensor((i[..., ::2] % 251).to(torch.uint8), i[:, :, 0].float().contiguous(), (i[:, :, 0, :s] % 60).to(torch.uint8),
                     (i[:, :, 0, s:2 * s] % 59).to(torch.uint8), i[:, :, 1, :s].float().contiguous(), (n, h, t, d), torch.bfloat16)
    v = PackedValues((i[..., ::4] % 249).to(torch.uint8), i[..., ::32].half(), i[..., 1::32].half(), (n, h, t, d),
                     torch.float16, 2, 32)
    return k, v


def test_fields_are_views_of_the_batch():
    from inquant.codec import _blocks_of
    for batch in _batches():
        assert _blocks_of(batch, 1) == [batch] and _blocks_of(batch, 1)[0] is batch
        blocks = _blocks_of(batch, 5)
        for i, block in enumerate(blocks):
            assert type(block) is type(batch) and block.shape == (1, 2, 8, 64)
            assert not any(f in vars(block) for f in batch.tensors)
            for name, field in batch.tensors.items():
                view = getattr(block, name)
                assert torch.equal(view, field[i:i + 1]) and view.data_ptr() == field[i].data_ptr()
                assert getattr(block, name) is view
            for f in dataclasses.fields(batch)[len(batch.tensors) + 1:]:
                assert getattr(block, f.name) == getattr(batch, f.name)
        assert sum(b.nbytes for b in blocks) == batch.nbytes
        assert not hasattr(blocks[0], "nothing") and not hasattr(batch, "nothing")
        with pytest.raises(dataclasses.FrozenInstanceError):
            blocks[0].payload = None


def test_copies_and_pickles_hold_the_fields_alone():
    from inquant.codec import _blocks_of
    for batch in _batches():
        names = {f.name for f in dataclasses.fields(batch)}
        for make in (copy.copy, copy.deepcopy, lambda b: pickle.loads(pickle.dumps(b)), dataclasses.replace):
            for i in (0, 3):
                for source in (_blocks_of(batch, 5)[i], batch):
                    got = make(source)
                    assert type(got) is type(batch) and set(vars(got)) == names
                    for name, field in source.tensors.items():
                        assert torch.equal(getattr(got, name), field)
                    assert (got.shape, got.original_dtype) == (source.shape, source.original_dtype)


def _cache(vbits, tokens, dim=128, block=32):
    from inquant.cache import CacheConfig, InQuantCache
    cache = InQuantCache(CacheConfig(block_size=block, residual_length=16, sink_tokens=4, value_bits=vbits, value_group_size=64))
    g = torch.Generator(device="cuda").manual_seed(tokens)
    k, v = (torch.randn((1, 2, tokens + 60, dim), generator=g, device="cuda").bfloat16() for _ in range(2))
    cache.update(k[:, :, :tokens], v[:, :, :tokens], 0)
    return cache, k, v


@pytest.mark.gpu
@pytest.mark.parametrize("vbits", [2, 4, None])
@pytest.mark.parametrize("tokens", [20, 55, 300])                   # no block, one, nine
def test_packed_steps_after_a_prefill_make_no_views(vbits, tokens):
    from inquant.triton_attention import PackedDecodeState
    cache, k, v = _cache(vbits, tokens)
    q = torch.randn((1, 8, 1, 128), device="cuda").bfloat16()
    state = plain = None
    for i in range(tokens, tokens + 40):                            # a block is sealed on the way, attended from the next step on
        view = cache.append_for_attention(k[:, :, i:i + 1], v[:, :, i:i + 1], 0)
        # blocks whose fields were all made beforehand, as separate tensors of the same memory
        copies = [[copy.copy(b) for b in blocks] for blocks in (view.key_blocks, view.value_blocks)]
        for b in (*view.key_blocks, *view.value_blocks):
            if b._batch is not None:
                for name in b.tensors:
                    del b.__dict__[name]
        if state is None:
            state = PackedDecodeState(view.key_blocks, view.value_blocks)
        else:
            state.extend(view.key_blocks, view.value_blocks)
        plain = PackedDecodeState(*copies)
        outs = [s.decode(q, sink_key=view.sink_key, sink_value=view.sink_value, residual_key=view.residual_key,
                         residual_value=view.residual_value) for s in (state, plain)]
        assert torch.equal(*outs)
        n = len(view.key_blocks)
        assert state.key_blocks == view.key_blocks and state.block_count == n
        if n:
            assert torch.equal(state._tables[:n], plain._tables[:n]) and torch.equal(state._key_map[:n], plain._key_map[:n])
            assert list(state._desc.run.base) == list(plain._desc.run.base)
            assert state._desc.run.blocks == plain._desc.run.blocks
        for b in (*view.key_blocks, *view.value_blocks):
            assert b._batch is None or not any(name in vars(b) for name in b._batch.tensors)
    assert len(view.key_blocks) >= 1


@pytest.mark.gpu
def test_mixed_and_reordered_blocks():
    # runs of a batch, single blocks and plain copies in one state: the same tables as from plain blocks
    from inquant.triton_attention import PackedDecodeState
    cache, _, _ = _cache(2, 300)
    other, _, _ = _cache(2, 400)
    a, b = cache._layers[0], other._layers[0]
    ka, va, kb, vb = a.key_blocks, a.value_blocks, b.key_blocks, b.value_blocks
    for keys, values in (([*ka, *kb], [*va, *vb]), (ka[::-1], va[::-1]), (ka[2:5] + kb[:3] + ka[5:], va[2:5] + vb[:3] + va[5:]),
                         ([ka[0], copy.copy(ka[1]), *ka[2:]], [*va[:4], copy.copy(va[4]), *va[5:]]), (ka[3:], va[1:-2]),
                         (ka[:1], va[1:2])):
        state = PackedDecodeState(keys, values)
        plain = PackedDecodeState([copy.copy(x) for x in keys], [copy.copy(x) for x in values])
        assert torch.equal(state._tables, plain._tables) and torch.equal(state._key_map, plain._key_map)
        assert list(state._desc.run.base) == list(plain._desc.run.base) and state._desc.run.blocks == plain._desc.run.blocks
        first = [x.data_ptr() for x in (keys[-1].payload, keys[-1].scales, keys[-1].padding, values[-1].payload,
                                        values[-1].scales, values[-1].offsets, keys[-1].salient_channels,
                                        keys[-1].donor_channels)]
        assert state._tables[-1].tolist() == first
    four, _, _ = _cache(4, 300)
    longer, _, _ = _cache(2, 300, block=64)
    narrow, _, _ = _cache(2, 300, dim=64)
    for keys, values, message in ((ka, four._layers[0].value_blocks[:1] + va[1:], "same quantizer"),
                                  (ka, va[:1] + four._layers[0].value_blocks[1:], "same quantizer"),
                                  (ka[:2] + longer._layers[0].key_blocks, va[:2] + longer._layers[0].value_blocks, "share shape"),
                                  (narrow._layers[0].key_blocks, narrow._layers[0].value_blocks, "head_dim=128"),
                                  (va, va, None)):
        with pytest.raises((ValueError, AttributeError), match=message):
            PackedDecodeState(keys, values)
