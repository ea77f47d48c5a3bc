"""The shortened square root and division on this device: the correctly rounded
results for every float of the root's range and 2^31 quotients."""
import pytest

from nonnewton_amd import _lib as L

pytestmark = pytest.mark.gpu


def test_shortened_forms_round_correctly():
    assert L.check_roundings(2048) == (0, 0)


def test_bad_arguments():
    assert L.load().nn_check_roundings(-1, None, None) == L.NN_E_ARG
