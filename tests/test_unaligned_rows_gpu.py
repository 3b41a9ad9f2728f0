"""Row operations on rows that are not 16-byte aligned (a length that is no
multiple of four, or an odd base address): the partial last chunk at every
position of the lanes, against float64, with guards around the result."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# 64, 256 and 512 floats are one to eight a lane, 4 and 1024 one chunk and one round
# of 256 lanes; 2048, 8192, 16384 the row lengths at which the kernels change.
SIZES = [1, 2, 3, 5, 7, 63, 64, 65, 255, 257, 511, 513, 779, 1021, 1023, 1025, 1027, 2047, 2049, 4099, 8190, 8193,
         16383, 16386]


def place(torch, a, shift):
    """`a` on the GPU `shift` floats past a 16-byte boundary, guards of 7.0 around it."""
    t = torch.full((a.size + shift + 8,), 7.0, dtype=torch.float32, device="cuda")
    t[4 + shift:4 + shift + a.size] = torch.from_numpy(a.reshape(-1)).cuda()
    return t, t[4 + shift:4 + shift + a.size]


def guarded(t, view):
    before = (view.data_ptr() - t.data_ptr()) // 4
    return bool((t[:before] == 7.0).all()) and bool((t[before + view.numel():] == 7.0).all())


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("shift", [0, 1, 3])
def test_rows(torch_gpu, l2c, size, shift):
    torch = torch_gpu
    print(f"case unaligned rows {size}+{shift}", flush=True)
    rng = np.random.default_rng(size * 10 + shift)
    batch = 3
    x = rng.uniform(-1, 1, (batch, size)).astype(np.float32)
    x[:, -1] = 3.0  # the last element is the maximum
    w = rng.uniform(0.5, 1.5, size).astype(np.float32)
    (_, dx), (_, dw) = place(torch, x, shift), place(torch, w, shift)
    t, out = place(torch, np.full(x.size, np.nan, np.float32), shift)

    def result():
        torch.cuda.synchronize()
        assert guarded(t, out)
        return out.cpu().numpy().reshape(batch, size).astype(np.float64)

    x64 = x.astype(np.float64)
    norm = x64 / np.sqrt((x64 * x64).mean(1, keepdims=True) + 1e-5) * w
    soft = np.exp(x64 - x64.max(1, keepdims=True))
    soft /= soft.sum(1, keepdims=True)
    l2c.rmsnorm(out, dx, dw, size, batch)
    np.testing.assert_allclose(result(), norm, rtol=1e-5)
    l2c.softmax(out, dx, size, batch)
    np.testing.assert_allclose(result(), soft, rtol=1e-5)

    tokens = torch.tensor([2, 0, 1], dtype=torch.int32, device="cuda")
    absmax = torch.zeros(1, dtype=torch.int32, device="cuda")
    for call in (lambda: l2c.decoder_rmsnorm(out, tokens, dx, dw, size, batch, batch),
                 lambda: l2c.decoder_rmsnorm_absmax(out, tokens, dx, dw, size, batch, batch, absmax)):
        out.fill_(float("nan"))
        call()
        np.testing.assert_allclose(result(), norm[[2, 0, 1]], rtol=1e-5)
    assert float(absmax.view(torch.float32)) == float(out.abs().max())
    generated = torch.full((batch,), -2, dtype=torch.int32, device="cuda")
    l2c.decoder_softmax_argmax(out, dx, tokens, generated, size, batch, 1, 0)
    np.testing.assert_allclose(result(), soft, rtol=1e-5)
    assert tokens.tolist() == [size - 1] * batch and generated.tolist() == [size - 1] * batch


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("shift", [0, 1])
def test_matvec(torch_gpu, l2c, size, shift):
    torch = torch_gpu
    print(f"case unaligned matvec {size}+{shift}", flush=True)
    rng = np.random.default_rng(size)
    W = rng.uniform(-1, 1, (7, size)).astype(np.float32)
    x = rng.uniform(-1, 1, size).astype(np.float32)
    (_, dW), (_, dx) = place(torch, W, shift), place(torch, x, shift)
    t, out = place(torch, np.full(7, np.nan, np.float32), shift)
    l2c.matvec(out, dx, dW, size, 7)
    torch.cuda.synchronize()
    assert guarded(t, out)
    # Any order of n fp32 multiply-adds is within n u of the sum of magnitudes.
    bound = (size + 8) * 2.0 ** -24 * (np.abs(W).astype(np.float64) @ np.abs(x).astype(np.float64))
    assert np.all(np.abs(out.cpu().numpy() - W.astype(np.float64) @ x.astype(np.float64)) <= bound)


# Every register-resident instance, aligned and not, and the streamed form.
@pytest.mark.parametrize("vocab,rows", [(701, 2), (1000, 2), (2048, 2), (5003, 2), (8192, 2), (8193, 2), (12288, 2),
                                        (12288, 642), (16383, 2), (16388, 2)])
@pytest.mark.parametrize("ones", [3, 7, 300])
def test_softmax_argmax_rounds_its_smallest_quotients(torch_gpu, l2c, vocab, rows, ones):
    """Exponentials e from 2^-90 to the smallest floats beside `ones` ones: the row
    with a single one has sum 1 and shows e itself, the other has sum `ones`, and
    its probabilities are e / ones correctly rounded."""
    torch = torch_gpu
    print(f"case softmax quotients {rows}x{vocab} ones={ones}", flush=True)
    rng = np.random.default_rng(vocab + ones)
    logits = np.empty((2, vocab), np.float32)
    logits[:] = rng.uniform(-106, -62, vocab)
    at = rng.choice(vocab, ones, replace=False)
    logits[0, at[:1]], logits[1, at] = 0.0, 0.0
    out = torch.empty(rows, vocab, device="cuda")
    tokens, generated = (torch.zeros(rows, dtype=torch.int32, device="cuda") for _ in range(2))
    x = torch.from_numpy(logits).cuda().repeat(rows // 2, 1)
    l2c.decoder_softmax_argmax(out, x, tokens, generated, vocab, rows, 1, 0)
    e, p = out[-2:].cpu().numpy()
    rest = np.setdiff1d(np.arange(vocab), at)
    assert (e[rest] < 2.0 ** -126).any() and (e[rest] > 2.0 ** -100).any()
    np.testing.assert_array_equal(p[rest], e[rest] / np.float32(ones))
    np.testing.assert_array_equal(p[at], np.float32(1) / np.float32(ones))
    assert tokens.tolist() == [at[0], at.min()] * (rows // 2) and generated.tolist() == tokens.tolist()
