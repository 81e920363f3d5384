"""What eva_img_prep and eva_img_prep_static refuse, and with which words: every refusal comes from the host before
anything is launched, so the rects here point at no memory. CPU only."""
import ctypes as C

import pytest

STATIC_BYTES = 448 * (4 * 448 - 1) * 16


def _pyr(xt, w, h):
    p = xt.EvaPyr()
    p.nlv, p.lv[0], p.ls[0], p.lw[0], p.lh[0] = 1, 4096, 4 * w, w, h
    return p


@pytest.mark.parametrize("scratch,short,out,S,rect,word", [
    (4096, 0, 0, 448, (0, 0, 900, 700), "out"), (4096, 0, 4104, 448, (0, 0, 900, 700), "out"),
    (4096, 0, 4096, 450, (0, 0, 900, 700), "multiple of 14"), (4096, 0, 4096, 448, (0, 0, 0, 700), "empty"),
    (4096, 0, 4096, 448, (3000, 0, 9, 9), "outside"), (4096, 0, 4096, 448, (0, 0, 3000, 700), "5x"),
    (0, 0, 4096, 448, (0, 0, 900, 700), "scratch"), (4104, 0, 4096, 448, (0, 0, 900, 700), "scratch"),
    (4096, 1, 4096, 448, (0, 0, 900, 700), "scratch")])
def test_prep_refusals(xt, capfd, scratch, short, out, S, rect, word):
    nbytes = xt.lib.eva_img_prep_bytes(S, rect[2]) - short
    assert xt.lib.eva_img_prep(C.byref(_pyr(xt, 3000, 2000)), *rect, S, C.c_void_p(scratch), nbytes, C.c_void_p(out),
                               None) == -1
    err = capfd.readouterr().err
    assert "eva_img_prep:" in err and word in err


@pytest.mark.parametrize("out,S,rect,word", [
    (0, 448, (0, 0, 900, 700), "out"), (4096, 450, (0, 0, 900, 700), "multiple of 14"),
    (4096, 448, (0, 0, 3000, 700), "5x"), (4096, 1008, (0, 0, 3000, 2000), "EVA_IMG_STATIC_BYTES")])
def test_prep_static_refusals(xt, capfd, out, S, rect, word):
    """The rect too wide for the static limit is refused for its width: the caller gave no scratch that could be short
    or misaligned, and `out` must not be taken for one (it holds far less than the limit)."""
    assert word != "EVA_IMG_STATIC_BYTES" or S * rect[2] * 16 > STATIC_BYTES
    assert xt.lib.eva_img_prep_static(C.byref(_pyr(xt, 3000, 2000)), *rect, S, C.c_void_p(out), None) == -1
    err = capfd.readouterr().err
    assert "eva_img_prep_static:" in err and word in err
    assert "scratch must" not in err
