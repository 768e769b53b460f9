"""Both sides of the request counts up to which the output cut takes its team form (GPU): passes
of 64, 32 or 16 requests by path length, two up to 11 entries, then one for every four, six at
most."""
from __future__ import annotations

import pytest
import torch

from test_accept_teams_gpu import test_walk_and_cut_equal_the_oracle as walk_and_cut

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("max_depth,requests", [(7, 128), (7, 129), (11, 192), (11, 193), (15, 256), (15, 257), (16, 128),
                                                (16, 129), (31, 192), (31, 193), (32, 96), (32, 97), (63, 96), (63, 97)])
def test_both_sides_of_the_team_form(max_depth, requests):
    walk_and_cut(max_depth, [max_depth + 1 + i % 5 for i in range(requests)], torch.int64)
