"""The polynomials of GeLU and its derivative (thn_act_math.h), read from the source and evaluated in float64 with the numbers as float32
holds them (CPU): the errors of the fits are those that the source states."""
import os
import re

import numpy as np
from scipy.special import log_ndtr

from conftest import ROOT

SOURCE = open(os.path.join(ROOT, "triton-hub_amd", "csrc", "thn_act_math.h")).read()


def fit(function):
    """c and the coefficients that `function` hands to normal_parts."""
    body = SOURCE[SOURCE.index(f"float {function}(float x)"):]
    c, coefficients = re.search(r"normal_parts<7, \w+>\(x, ([0-9.]+)f, \{([^}]*)\}\)", body).groups()
    numbers = [float(np.float32(v.strip().rstrip("f"))) for v in coefficients.split(",")]
    assert len(numbers) == 8
    return float(np.float32(c)), numbers


def test_stated_errors_of_the_fits():
    x = np.linspace(0.0, 13.3, 1_000_001)
    tail = np.exp(log_ndtr(-x) + 0.5 * x * x)               # Phi(-x)*exp(x^2/2), which t*Q(t) stands for
    for function, least, worst in (("normal_cdf", tail, 1.25e-7), ("gelu_slope", x / np.sqrt(2.0 * np.pi) + tail, 4.5e-8)):
        c, coefficients = fit(function)
        t = 1.0 / (1.0 + c * x)
        error = np.abs(t * np.polyval(coefficients[::-1], t) - tail) / least
        assert 0.9 * worst < error.max() <= worst
