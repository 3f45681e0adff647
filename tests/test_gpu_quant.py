"""GPU quant codecs vs the oracle: codes and scales bit-identical."""
import numpy as np
import pytest
import torch

from conftest import golden

pytestmark = pytest.mark.gpu


def _rows(rng):
    yield rng.standard_normal((7, 128)).astype(np.float32)
    yield (rng.standard_normal((33, 4096)) * 0.02).astype(np.float32)
    yield rng.standard_normal((3, 1)).astype(np.float32)
    z = np.zeros((2, 64), np.float32)
    z[1, 5] = -3.0
    yield z
    x = rng.standard_normal((5, 1000)).astype(np.float32) * 50
    x[2, 7] = 1e-30
    yield x
    # exact .5 points after scaling (roundf half away from zero)
    yield np.array([[127.0, 0.5, -0.5, 1.5, -2.5, 63.5, -63.5, 0.0]], np.float32)


def test_quant_int8_rows(be, orc):
    rng = np.random.default_rng(100)
    for x in _rows(rng):
        q, s = be.quant_rows_int8(torch.from_numpy(x).cuda())
        for r in range(x.shape[0]):
            wq, ws = orc.quant_int8(x[r])
            np.testing.assert_array_equal(q[r].cpu().numpy(), wq)
            assert s[r].item() == ws or (np.isnan(ws) and np.isnan(s[r].item()))
            assert np.float32(s[r].item()).view(np.uint32) == np.float32(ws).view(np.uint32)


def test_quant_fp8_rows(be, orc):
    rng = np.random.default_rng(101)
    g = golden("fp8_codec")
    cases = list(_rows(rng)) + [g["direct_in"][None, :]]
    i = 0
    while f"vec{i}_in" in g:
        cases.append(g[f"vec{i}_in"][None, :])
        i += 1
    for x in cases:
        x = np.ascontiguousarray(x, np.float32)
        q, s = be.quant_rows_fp8(torch.from_numpy(x).cuda())
        for r in range(x.shape[0]):
            wq, ws = orc.quant_fp8(x[r])
            np.testing.assert_array_equal(q[r].cpu().numpy(), wq)
            assert np.float32(s[r].item()).view(np.uint32) == np.float32(ws).view(np.uint32)
    # the reference's direct encoder codes (scale == 1 for this vector)
    q, s = be.quant_rows_fp8(torch.from_numpy(np.ascontiguousarray(g["direct_in"][None, :])).cuda())
    np.testing.assert_array_equal(q[0].cpu().numpy(), g["direct_codes"])


def test_fp8_encoder_binade_edges(be, orc):
    """Values a few ulps below every power of two, where log2f rounds up."""
    vals = []
    for e in range(-9, 8):
        p = np.float32(2.0 ** e)
        v = p
        for _ in range(8):
            v = np.nextafter(v, np.float32(0))
            vals.append(v)
        vals.append(p)
    vals = np.array(vals + [224.0], np.float32)     # absmax 224: scale == 1
    q, s = be.quant_rows_fp8(torch.from_numpy(vals[None, :]).cuda())
    assert s.item() == 1.0
    want, _ = orc.quant_fp8(vals)
    np.testing.assert_array_equal(q[0].cpu().numpy(), want)
    # (x * (224 / amax) never exceeds 224, so quant_f32_to_fp8 cannot reach the
    # binades above 2^7.)


def test_fp8_decode_all_codes(be, orc):
    codes = torch.arange(256, dtype=torch.int32).to(torch.uint8).cuda()
    out = be.fp8_decode(codes).cpu().numpy()
    np.testing.assert_array_equal(out.view(np.uint32), orc.fp8_lut().view(np.uint32))


def test_dequant_rows_int8(be, orc):
    rng = np.random.default_rng(102)
    x = rng.standard_normal((9, 130)).astype(np.float32)
    q, s = be.quant_rows_int8(torch.from_numpy(x).cuda())
    out = be.dequant_rows_int8(q, s).cpu().numpy()
    want = q.cpu().numpy().astype(np.float32) * s.cpu().numpy()[:, None]
    np.testing.assert_array_equal(out, want)


@pytest.mark.parametrize("cols", [4, 1020, 1024, 1028, 4096, 4100, 8192, 8196, 16384, 16388, 4098])
def test_quant_rows_vector_edges(be, orc, cols):
    """Row lengths at the edges of the in-register kernel (one to sixteen
    16-byte words per thread) and past them, an absmax in the last element, a
    row of zeros, and a source or destination that is not aligned."""
    rng = np.random.default_rng(cols)
    x = rng.standard_normal((3, cols)).astype(np.float32)
    x[0, -1] = 9.0
    x[1] = 0.0
    dev = torch.from_numpy(x).cuda()
    odd = torch.empty(3 * cols + 1, device="cuda")[1:].view(3, cols)
    odd.copy_(dev)
    for src in (dev, odd):
        for name, quant, want in (("be42_quant_rows_int8", be.quant_rows_int8, orc.quant_int8),
                                  ("be42_quant_rows_fp8", be.quant_rows_fp8, orc.quant_fp8)):
            q, s = quant(src)
            q2 = torch.zeros(3 * cols + 1, dtype=torch.uint8, device="cuda")[1:]
            s2 = torch.zeros(3, device="cuda")
            be._call(name, be.p(q2), be.p(s2), be.p(src), 3, cols, be.stream())
            for r in range(3):
                codes, scale = want(x[r])
                np.testing.assert_array_equal(q[r].cpu().numpy(), codes)
                np.testing.assert_array_equal(q2.view(3, cols)[r].cpu().numpy().view(codes.dtype), codes)
                assert s[r].item() == s2[r].item() == scale
