"""Writes radix_consts.hpp: cos/sin(2*pi*m/R), m = 0..R-1, for the odd radices
of the Stockham butterflies (OddRadix).  Values are computed in x87 extended
precision and rounded once to double (printed with 17 significant digits)."""
import os
import numpy as np

ODD = [3, 5, 7, 9, 11, 13, 15, 17, 19, 23, 29, 31]


def main(path):
    lines = ["// Generated by gen_radix.py -- do not edit.",
             "#pragma once", "",
             "template <int R> struct OddRadix;", ""]
    two_pi = np.longdouble(2) * np.arccos(np.longdouble(-1))
    for r in ODD:
        m = np.arange(r, dtype=np.longdouble)
        c = np.cos(two_pi * m / r)
        s = np.sin(two_pi * m / r)
        cs = ", ".join(f"{float(x):.17e}" for x in c)
        ss = ", ".join(f"{float(x):.17e}" for x in s)
        lines += [f"template <> struct OddRadix<{r}> {{",
                  f"  static constexpr double c[{r}] = {{{cs}}};",
                  f"  static constexpr double s[{r}] = {{{ss}}};",
                  "};", ""]
    text = "\n".join(lines)
    # rewrite only on change: the kernels' objects depend on this header
    if os.path.exists(path) and open(path).read() == text:
        return
    with open(path, "w") as f:
        f.write(text)


if __name__ == "__main__":
    here = os.path.dirname(os.path.abspath(__file__))
    main(os.path.join(here, "radix_consts.hpp"))
