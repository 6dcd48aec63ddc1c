"""Which of the jitconn walks a call takes (bpl_selfcheck_jitconn_by_lane; host code, no device)."""
import ctypes

import numpy as np
import pytest

from brainpylib_amd import _lib
from util import jitconn_by_lane


# (streams, mean synapses, places), either walk measured: by lane at least 5 % faster, or slower
@pytest.mark.parametrize("weights,value_bytes,faster,slower", [
  ("homo", 4, [(4000, 55, 3000), (10_000, 25, 3000), (20_000, 55, 3000), (60_000, 115, 30_000), (500_000, 167, 1_500_000)],
   [(4000, 75, 3000), (4000, 55, 300_000), (9000, 76, 3000), (14_000, 68, 30_000), (20_000, 81, 3000), (80_000, 165, 3000)]),
  ("homo", 8, [(4000, 51, 30_000), (60_000, 115, 30_000)], [(4000, 69, 300_000), (9000, 68, 3000), (20_000, 81, 3000)]),
  ("uniform", 4, [(16_000, 25, 3000), (60_000, 71, 30_000)], [(9000, 52, 3000), (20_000, 63, 3000), (4000, 53, 300_000), (80_000, 102, 3000)]),
  ("uniform", 8, [(4000, 31, 30_000), (60_000, 55, 30_000)], [(9000, 44, 3000), (20_000, 49, 30_000), (4000, 41, 300_000)]),
  ("normal", 4, [(10_000, 8, 3000), (60_000, 31, 3000), (1_000_000, 75, 3000)], [(4000, 18, 3000), (9000, 18, 3000), (20_000, 22, 30_000), (80_000, 53, 3000)]),
  ("normal", 8, [(20_000, 10, 3000), (60_000, 14, 30_000), (8000, 12, 3000)], [(4000, 12, 3000), (9000, 15, 3000), (80_000, 55, 3000)])])
def test_rows_of_either_side_of_the_line(weights, value_bytes, faster, slower):
  for by_lane, rows in ((True, faster), (False, slower)):
    for n_out, mean, n_in in rows:
      assert jitconn_by_lane(weights, value_bytes, n_out, n_in, mean / n_in) == by_lane, (n_out, mean, n_in)


@pytest.mark.parametrize("weights,value_bytes,faster,slower", [
  ("homo", 4, [(10_000, 100, 5000), (32_000, 25, 5000), (130_000, 116, 5000), (1_000_000, 165, 5000)],
   [(2500, 40, 5000), (4000, 40, 5000), (10_000, 130, 5000), (20_000, 55, 5000), (60_000, 100, 5000)]),
  ("homo", 8, [(10_000, 40, 5000), (300_000, 130, 5000)], [(30_000, 45, 5000), (60_000, 77, 5000), (60_000, 77, 500_000)]),
  ("uniform", 8, [(10_000, 26, 5000), (300_000, 55, 100_000)], [(2500, 26, 5000), (60_000, 54, 5000), (60_000, 54, 500_000)]),
  ("normal", 4, [(130_000, 43, 5000), (500_000, 64, 500_000)], [(2500, 13, 5000), (10_000, 15, 5000)]),
  ("normal", 8, [(8000, 3, 5000), (500_000, 32, 5000)], [(2500, 7, 5000), (30_000, 8, 5000), (8000, 15, 5000)])])
def test_columns_of_either_side_of_the_line(weights, value_bytes, faster, slower):
  for by_lane, columns in ((True, faster), (False, slower)):
    for n_in, mean, n_out in columns:
      assert jitconn_by_lane(weights, value_bytes, n_in, n_out, mean / n_out, use=1) == by_lane, (n_in, mean, n_out)


def test_rows_of_events_that_the_l2s_do_not_hold_go_by_wave():
  assert jitconn_by_lane("homo", 8, 500_000, 1_500_000, 167 / 1_500_000, event_bytes=1)
  assert not jitconn_by_lane("homo", 8, 500_000, 1_500_000, 167 / 1_500_000, event_bytes=8)


def test_columns_of_events_with_few_outputs_and_no_bins_go_by_wave():
  for weights, mean in (("homo", 16), ("uniform", 13)):
    assert not jitconn_by_lane(weights, 4, 200_000, 5000, mean / 5000, use=2)
    assert jitconn_by_lane(weights, 4, 200_000, 20_000, mean / 20_000, use=2)
    assert jitconn_by_lane(weights, 4, 1_000_000, 5000, mean / 5000, use=2)  # (bins)
    assert jitconn_by_lane(weights, 4, 20_000, 5000, mean / 5000, use=2)
  assert not jitconn_by_lane("homo", 4, 20_000, 5000, 25 / 5000, use=2)


def test_what_there_is_not_is_an_error():
  check = _lib.lib().bpl_selfcheck_jitconn_by_lane
  for weights, value_bytes, use in ((3, 4, 0), (0, 2, 0), (0, 4, 3)):
    assert check(weights, value_bytes, 100, 100, ctypes.c_double(float(np.log(0.99))), use, 0) == -1
    assert "bpl_selfcheck_jitconn_by_lane" in _lib.last_error()
  _lib.lib().bpl_clear_error()
