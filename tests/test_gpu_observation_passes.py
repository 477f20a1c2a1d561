"""The solver's GPU tests once more with FEHIP_NORMAL=0: FP64 and mixed solves
iterate on the observations there, as they do where the level-space form is
not taken (no room for its matrix, too many entries) and where a column starts
over.  Without it those tests' FP64 handles iterate in level space, and the
forms of the passes that they name (pieces, separate launches, the wide map,
schedules) would run in single passes and in FP32 alone."""
import pytest

from test_gpu_configs import *  # noqa: F401,F403
from test_gpu_parity import *  # noqa: F401,F403
from test_gpu_projected import *  # noqa: F401,F403
from test_gpu_warmstart import *  # noqa: F401,F403

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _on_the_observations(monkeypatch):
    monkeypatch.setenv("FEHIP_NORMAL", "0")
