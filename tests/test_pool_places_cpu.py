"""Handles lease their worker pools from the process: users that take turns
share one pool, users that overlap never share one, there are never more pools
than users, and none is left once the users are gone."""
import pytest

from tests import oracle_lib


@pytest.mark.parametrize("users,threads", [(1, 3), (3, 2), (4, 4), (3, 1)])
def test_pools_are_shared_and_given_back(users, threads):
    assert oracle_lib.load().oracle_pool_places(users, threads, 50) == 0
