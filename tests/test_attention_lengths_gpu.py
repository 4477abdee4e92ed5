"""The attention drop-in (utils/model.py:24-31) at lengths on and off its 64-key and 256-query tiles, with the strides
and dtypes its operands pass takes, against a dense fp32 softmax of the bf16 operands: bf16 weights and output round
each value by 2^-9 of itself, so errors stay within 2e-2 of the largest value (the bar of the fixed-length tests). Rows
past the last token must neither be read (the tensors end there) nor written."""
import pytest
import torch

from tests.test_attention_gpu import DEV, fp32_reference_gpu, rel_ok

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('T', [1, 2, 31, 32, 33, 63, 64, 65, 100, 255, 257, 320, 511, 1111])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float32])
def test_lengths(T, dtype):
    from noise_amd.model import attention
    for B, H, window in ((1, 1, T), (2, 8, 40), (3, 5, 0)):
        print(B, T, H, window, dtype, flush=True)
        g = torch.Generator(DEV).manual_seed(T)
        q, k, v = (torch.randn(B, T, H, 64, device=DEV, generator=g).to(dtype) for _ in range(3))
        out = attention(q, k, v, window)
        assert out.dtype == dtype and out.is_contiguous()
        rel_ok(out, fp32_reference_gpu(q.bfloat16(), k.bfloat16(), v.bfloat16(), window))
        assert torch.equal(attention(q.bfloat16(), k.bfloat16(), v.bfloat16(), window).to(dtype), out)


def test_views_and_dtypes():
    from noise_amd.model import attention
    g = torch.Generator(DEV).manual_seed(9)
    B, T, H = 2, 203, 3
    qkv = torch.randn(B, T, 3, H, 64, device=DEV, generator=g)
    wide = torch.randn(B, T, H, 3 * 64 + 1, device=DEV, generator=g)
    cases = [qkv.unbind(2), qkv.bfloat16().unbind(2), [qkv[:, :, 0], qkv[:, :, 1].bfloat16(), qkv[:, :, 2].half()],
             [qkv[:, :, 0].half(), qkv[:, :, 1], qkv[:, :, 2].double()], [wide[..., i + 1:i + 65] for i in (0, 64, 128)],
             [t.transpose(1, 2).contiguous().transpose(1, 2) for t in qkv.unbind(2)],
             [t.transpose(2, 3).contiguous().transpose(2, 3) for t in qkv.unbind(2)],
             [qkv[:1, :, i].expand(B, T, H, 64) for i in range(3)]]
    for q, k, v in cases:
        print([(t.dtype, t.stride()) for t in (q, k, v)], flush=True)
        out = attention(q, k, v, 90)
        assert out.dtype == q.dtype
        rel_ok(out, fp32_reference_gpu(q.bfloat16(), k.bfloat16(), v.bfloat16(), 90))


@pytest.mark.parametrize('flags', [0, 2, 4, 6])
def test_rows_past_the_end_are_not_written(flags):
    from noise_amd import _lib
    g = torch.Generator(DEV).manual_seed(4)
    B, T, H, pad = 2, 131, 2, 200
    q, k, v = (torch.nn.functional.rms_norm(torch.randn(B, T, H, 64, device=DEV, generator=g), (64,)).bfloat16()
               for _ in range(3))
    out = torch.full((B, T + pad, H, 64), 9.0, device=DEV, dtype=torch.float32 if flags & 4 else torch.bfloat16)
    dots, vec = torch.full((B * T * H + 64,), 9.0, device=DEV), torch.randn(B, H * 64, device=DEV, generator=g)
    s = [x for t in (q, k, v) for x in (t.stride(0), t.stride(2), t.stride(1))]
    _lib.call('noise_attention_fwd', q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), B, H, T, 64, *s, flags,
              out.stride(0), out.stride(2), out.stride(1), 77, 0.125, vec.data_ptr(), H * 64, 1, dots.data_ptr(),
              _lib.stream_ptr(DEV))
    ref = fp32_reference_gpu(q, k, v, 77)
    rel_ok(out[:, :T], ref)
    assert (out[:, T:] == 9).all() and (dots[B * T * H:] == 9).all()
    expect = (out[:, :T].float() * vec.view(B, 1, H, 64)).sum(-1)
    assert torch.allclose(dots[:B * T * H].view(B, T, H), expect, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize('T', [1, 100, 257])
@pytest.mark.parametrize('flags', [12, 14])
def test_fp32_queries(T, flags):
    """Queries rounded by the kernel: the bits of bf16 queries, in any strides of whole 16 B; odd ones and a bf16 output
    are refused by the kernel's entry and served by the drop-in."""
    from noise_amd import _lib
    from noise_amd.model import attention
    g = torch.Generator(DEV).manual_seed(T)
    B, H = 2, 3
    wide = torch.nn.functional.rms_norm(torch.randn(B, H, T + 1, 68, device=DEV, generator=g), (68,))
    k, v = (torch.nn.functional.rms_norm(torch.randn(B, T, H, 64, device=DEV, generator=g), (64,)).bfloat16()
            for _ in range(2))

    def call(q, flags, dtype):
        out = torch.full((B, T + 3, H, 64), 9.0, device=DEV, dtype=dtype)
        s = [x for t in (q, k, v) for x in (t.stride(0), t.stride(2), t.stride(1))]
        _lib.call('noise_attention_fwd', q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), B, H, T, 64, *s, flags,
                  out.stride(0), out.stride(2), out.stride(1), 77, 0.125, None, 0, 1, None, _lib.stream_ptr(DEV))
        assert (out[:, T:] == 9).all()
        return out[:, :T]

    q = wide[:, :, :T, :64].transpose(1, 2)   # [B, T, H, 64], rows of 68
    assert torch.equal(call(q, flags, torch.float32), call(q.bfloat16().contiguous(), flags & ~8, torch.float32))
    with pytest.raises(RuntimeError):
        call(q, flags & ~4, torch.bfloat16)
    odd = torch.randn(B, T, H, 65, device=DEV, generator=g)[..., :64]
    with pytest.raises(RuntimeError):
        call(odd, flags, torch.float32)
    for t in (q, odd):
        assert torch.equal(attention(t, k, v, 77), attention(t.bfloat16().contiguous(), k, v, 77).float())


@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float32])
def test_more_workgroups_than_one_launch(dtype):
    """2^23 heads and more, of one workgroup of 512 threads each: a launch has fewer than 2^32 threads. A lone token's output
    is its v, a second token's the softmax of two scores."""
    from noise_amd.model import attention
    B, H = 2 ** 20 + 1, 8
    print(B, H, dtype, flush=True)
    g = torch.Generator(DEV).manual_seed(3)
    q, k, v = (torch.randn(B, 1, H, 64, device=DEV, generator=g).to(dtype) for _ in range(3))
    assert torch.equal(attention(q, k, v, 5), v.bfloat16().to(dtype))
    few = (torch.randn(B // 64, 2, H, 64, device=DEV, generator=g).to(dtype) for _ in range(3))
    q, k, v = (t.repeat(64, 1, 1, 1) for t in few)
    n = B // 64
    want = attention(q[:n], k[:n], v[:n], 5)
    rel_ok(want[:64], fp32_reference_gpu(*(t[:64].bfloat16() for t in (q, k, v)), 5))
    out = attention(q, k, v, 5)
    assert out.view(64, n, 2, H, 64).eq(want).all()


def test_more_rows_than_one_cast_launch():
    """2^29 rows and more, eight threads each. Every batch of the source is the same rows."""
    import ctypes
    from noise_amd import _lib
    batch, H = 2 ** 26 + 1, 8
    print(batch, H, flush=True)
    src = torch.randn(1, 1, H, 64, device=DEV)
    dst = torch.empty(batch, H, 64, device=DEV, dtype=torch.bfloat16)
    dst[-4096:] = 9
    cast = _lib.CastHeads()
    cast.count, cast.src[0], cast.dst[0], cast.s_h[0] = 1, src.data_ptr(), dst.data_ptr(), 64
    _lib.call('noise_cast_heads', ctypes.byref(cast), batch, 1, H, _lib.stream_ptr(DEV))
    for part in (dst[:4096], dst[batch // 2:][:4096], dst[-4096:]):
        assert part.eq(src[0].bfloat16()).all()
    del dst, part
    torch.cuda.empty_cache()


@pytest.mark.parametrize('T', [256, 512, 768])
@pytest.mark.parametrize('dtype', [torch.bfloat16, torch.float32])
def test_whole_tiles(T, dtype):
    """Lengths in whole 256-query tiles, without the clamps, give the bits of the same tokens with one more behind them."""
    from noise_amd.model import attention
    test_lengths(T, dtype)
    g = torch.Generator(DEV).manual_seed(T)
    for window in (0, 100, 4096):
        q, k, v = (torch.randn(2, T + 1, 3, 64, device=DEV, generator=g).to(dtype) for _ in range(3))
        assert torch.equal(attention(q[:, :T], k[:, :T], v[:, :T], window), attention(q, k, v, window)[:, :T])
