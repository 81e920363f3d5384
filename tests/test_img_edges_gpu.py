"""The patch-operand producer where its blocks and vector accesses end: rows that are no multiple of four pixels, opaque
and translucent pixels side by side, strips at the largest resample factor, single pixels, crops past the image's edge;
bit for bit against the oracle."""
import ctypes as C

import numpy as np
import pytest
import torch

from tests.test_img_gpu import S, DevImage, _img, _st

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("h,w,pad", [(1, 1, 0), (3, 5, 1), (9, 67, 3), (5, 256, 0), (4, 259, 2), (2, 1023, 1)])
def test_over_white_edges(dev, xt, orc, h, w, pad):
    print(f"over white {w} x {h}, row pad {pad}", flush=True)
    img = _img(h, w, h * w, alpha=True)
    img[:, : w // 2, 3] = 255                                # groups of four: opaque, mixed and translucent
    buf = np.full((h, w + pad, 4), 9, np.uint8)
    buf[:, :w] = img
    d = torch.from_numpy(buf.copy()).to(dev)
    assert xt.lib.eva_img_over_white(xt.ptr(d), (w + pad) * 4, w, h, _st()) == 0
    torch.cuda.synchronize()
    got = d.cpu().numpy()
    assert np.array_equal(got[:, :w], orc.img_over_white(np.ascontiguousarray(img))) and (got[:, w:] == 9).all()


@pytest.mark.parametrize("h,w,crop", [(1, 2400, (0, 0, 2400, 1)), (2400, 1, (0, 0, 1, 2400)), (7, 5, (0, 0, 5, 7)),
                                      (1, 1, (0, 0, 1, 1)), (449, 447, (0, 0, 447, 449)), (900, 895, (0, 0, 895, 900)),
                                      (1791, 1300, (0, 0, 1300, 1791)), (600, 600, (590, 2, 300, 598))])
def test_prep_edges(dev, xt, orc, h, w, crop):
    print(f"prep {w} x {h}, crop {crop}", flush=True)
    img = _img(h, w, 11)
    di = DevImage(xt, dev, img)
    ref, _ = orc.img_prep(orc.img_pyramid(img, S), *crop, S=S)
    nb = xt.lib.eva_img_prep_bytes(S, 6 * S)
    scratch = torch.empty(nb, dtype=torch.uint8, device=dev)
    out = torch.full(((S // 14) ** 2, 592), 0x7E00, dtype=torch.int16, device=dev)
    assert xt.lib.eva_img_prep(C.byref(di.p), *crop, S, xt.ptr(scratch), nb, xt.ptr(out), _st()) == 0
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy().view(np.uint16), ref)
