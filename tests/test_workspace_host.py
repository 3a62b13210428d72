"""Workspace sizes of SR-branch solves (at least as many samples as parameters)."""
import pytest

from quantax_amd import _lib

MODES = [_lib.QTX_SOLVE_CHOL_SHIFT, _lib.QTX_SOLVE_EIGH_PINV, _lib.QTX_SOLVE_EIGH_PINV_DIRECT]


def ws(ns, np_, mode):
    return int(_lib.lib().qtx_minsr_ws_bytes(ns, np_, mode, _lib.QTX_GRAM_FP64))


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("np_", [8, 272, 512])
def test_no_obar_where_s_is_formed_from_o(mode, np_):
    """Only the vectors of one entry per sample grow with the samples."""
    assert ws(200000, np_, mode) - ws(1000, np_, mode) <= 2 * 8 * 199000 + 2 * 256
    # the SNR truncation forms Obar, and Obar V, in blocks
    snr = mode | _lib.QTX_SOLVE_SNR
    assert ws(2000, np_, snr) >= ws(2000, np_, mode) + 2 * 8 * 2000 * np_


@pytest.mark.parametrize("mode", MODES)
def test_obar_beyond(mode):
    assert ws(2000, 513, mode) >= 8 * 2000 * 513 + 8 * 513 * 513
