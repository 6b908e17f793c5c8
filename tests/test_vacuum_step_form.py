"""The mixed vacuum step's form of Dormand-Prince 5(4) for second-order pairs (csrc/trace_mixed.h dp54_n): its
constants, read from the source, against the tableau of csrc/trace_fp64.h in rational arithmetic. With A the
tableau's matrix (the seventh row the solution's weights b), e the error's weights: c = A 1, n = A^2, f = b A,
g = e A, and e's weights sum to zero, so the estimate does not contain the velocity."""
import os
import re
from fractions import Fraction

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "spacetime-optics_amd", "csrc")


def constants(path, names):
    """name -> exact value of the `name = [-]p.0 / q` constants whose names match."""
    text = open(os.path.join(CSRC, path)).read()
    out = {}
    for body in re.findall(r"constexpr double ([^;{}()]*);", text):
        for name, p, q in re.findall(r"(\w+) = (-?\d+)(?:\.0)? / (\d+)", body):
            if re.fullmatch(names, name):
                assert name not in out, name
                out[name] = Fraction(int(p), int(q))
    return out


def test_form_of_the_method():
    t = constants("trace_fp64.h", r"a\d\d|[be]\d")
    A = [[t.get(f"a{i}{j}", Fraction(0)) for j in range(1, 8)] for i in range(1, 7)]
    b = [t.get(f"b{j}", Fraction(0)) for j in range(1, 8)]
    e = [t.get(f"e{j}", Fraction(0)) for j in range(1, 8)]
    A.append(b)
    assert sum(b) == 1 and sum(e) == 0 and len(t) == 15 + 5 + 6
    n = [[sum(A[i][j] * A[j][k] for j in range(7)) for k in range(7)] for i in range(7)]
    f = [sum(b[j] * A[j][k] for j in range(7)) for k in range(7)]
    g = [sum(e[j] * A[j][k] for j in range(7)) for k in range(7)]
    want = {f"c{i}": sum(A[i - 1]) for i in (3, 4, 5)}
    want.update({f"n{i}{k}": n[i - 1][k - 1] for i in range(3, 7) for k in range(1, i - 1)})
    want.update({f"f{k}": f[k - 1] for k in (1, 3, 4, 5)})
    want.update({f"g{k}": g[k - 1] for k in (1, 3, 4, 5, 6)})
    got = constants("trace_mixed.h", r"c[345]|n\d\d|[fg]\d")
    assert got == want
    # what the step leaves out is zero
    assert sum(A[5]) == sum(A[6]) == 1 and f[1] == f[5] == f[6] == g[1] == g[6] == 0
