"""Writes radix_consts.hpp: cos/sin(2*pi*m/R), m = 0..R-1, for the odd radices
of the Stockham butterflies (OddRadix), and for the large ones the rows
cos(2*pi*j*k/R), j = 1..H, then sin, of every output k = 1..H = (R-1)/2
(OddRows, in the precision T of the transform).  Values are computed in x87 extended precision and
rounded once to double (printed with 17 significant digits)."""
import os
import numpy as np

ODD = [3, 5, 7, 9, 11, 13, 15, 17, 19, 23]
ROWS = [29, 31]


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
    lines += ["template <typename T, int R> struct OddRows;", ""]
    for r in ROWS:
        h = (r - 1) // 2
        m = np.outer(np.arange(1, h + 1), np.arange(1, h + 1)) % r
        cs = np.concatenate([np.cos(two_pi * m.astype(np.longdouble) / r),
                             np.sin(two_pi * m.astype(np.longdouble) / r)], axis=1)
        for t, fmt in (("double", lambda x: f"{float(x):.17e}"),
                       ("float", lambda x: f"{np.float32(x):.9e}f")):
            lines += [f"template <> struct OddRows<{t}, {r}> {{",
                      f"  static constexpr {t} cs[{h}][{2 * h}] = {{"]
            lines += ["    {" + ", ".join(fmt(x) for x in row) + "}," for row in cs]
            lines += ["  };", "};", ""]
    text = "\n".join(lines)
    # rewrite only on change: the kernels' objects depend on this header
    if os.path.exists(path) and open(path).read() == text:
        return
    with open(path, "w") as f:
        f.write(text)


if __name__ == "__main__":
    here = os.path.dirname(os.path.abspath(__file__))
    main(os.path.join(here, "radix_consts.hpp"))
