"""The one-step square root and reciprocals of the fluid terms, exhaustively over significands on the
device (tests/cpp/rsq_identities.hip, built with the library)."""
import pytest

from test_cpp_host import run

pytestmark = pytest.mark.gpu


def test_root_and_reciprocals_are_correctly_rounded():
    assert "checks passed" in run("rsq_identities")
