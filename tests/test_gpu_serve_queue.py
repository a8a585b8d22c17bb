"""The serving loop's merging does not depend on how fast requests are submitted or
how long a build takes, as long as they wait in the queue together."""
import time

import pytest

from niq import serve
import test_gpu_serve as base

pytestmark = pytest.mark.gpu


def test_casts_merge_however_slow_the_submits(monkeypatch):
    submit_rays = serve.Server.submit_rays

    def slow(self, *args, **kw):
        time.sleep(0.01)   # a descheduled host
        return submit_rays(self, *args, **kw)

    monkeypatch.setattr(serve.Server, "submit_rays", slow)
    base.test_rays_of_different_models_and_options_share_a_cast()
