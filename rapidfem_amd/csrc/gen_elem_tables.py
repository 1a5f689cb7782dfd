"""Writes rfhip_elem_tables.hpp: compile-time tables of the equispaced
reference element (dg_basis.rs:270-301) for the component-lane stage kernel,
from the library's own host builder (rfhost_refelem):

  FN[f][m]   the volume node of face node m of local face f;
  DM[k][i]   bit j set where D_k[i][j] is not zero (k = r, s, t). The host
             builder's D_k carries round-off residues of at most 2e-13 where
             the exact entry is zero (the smallest true entry is 1/3), so the
             pattern is |D_k[i][j]| > 1e-9 max |D_k|;
  XM[k][i]   bit j set where D_k[i][j] is not 0.0 (residues included): the
             entries that a kernel keeps to add the terms a dense product adds.

The kernel skips the entries outside DM and indexes its per-lane register
arrays with FN, so both must be known when it is compiled; at operator
creation the library checks that the operator's own tables agree (a
different table makes the variant unavailable).

Usage: python rapidfem_amd/csrc/gen_elem_tables.py [--check]
(--check compares with the committed header and exits 1 on a difference).
"""
from __future__ import annotations

import os
import sys

import numpy as np

HEADER = os.path.join(os.path.dirname(os.path.abspath(__file__)), "rfhip_elem_tables.hpp")
sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.dirname(os.path.abspath(__file__)))))
ORDERS = (1, 2, 3, 4)


def tables(p: int):
    from rapidfem_amd.maxwell import ReferenceElement

    r = ReferenceElement.new(p)
    masks = []
    for d in (r.diff_r, r.diff_s, r.diff_t):
        a = np.abs(d)
        nz = a > 1e-9 * a.max()
        masks.append([sum(1 << j for j in range(d.shape[1]) if nz[i, j]) for i in range(d.shape[0])])
    return r.n_nodes, r.n_face_nodes, r.face_nodes.astype(int).tolist(), masks


def exact_masks(p: int):
    from rapidfem_amd.maxwell import ReferenceElement

    r = ReferenceElement.new(p)
    return [[sum(1 << j for j in range(d.shape[1]) if d[i, j] != 0.0) for i in range(d.shape[0])]
            for d in (r.diff_r, r.diff_s, r.diff_t)]


def render() -> str:
    out = [
        "// Generated by gen_elem_tables.py from the host builder's reference",
        "// element (equispaced nodes, dg_basis.rs:270-301); do not edit.",
        "#pragma once",
        "#include <cstdint>",
        "",
        "namespace rfhip {",
        "",
        "template <int NP>",
        "struct ElemTab;",
    ]
    for p in ORDERS:
        np_, nfp, fn, masks = tables(p)
        out.append("")
        out.append(f"// order {p}: Np = {np_}, Nfp = {nfp}; nonzeros of D_r, D_s, D_t: "
                   + ", ".join(str(sum(bin(m).count('1') for m in mk)) for mk in masks))
        out.append("template <>")
        out.append(f"struct ElemTab<{np_}> {{")
        out.append(f"  static constexpr int NFP = {nfp};")
        rows = ", ".join("{" + ", ".join(str(v) for v in f) + "}" for f in fn)
        out.append(f"  static constexpr int FN[4][{nfp}] = {{{rows}}};")
        out.append(f"  static constexpr uint64_t DM[3][{np_}] = {{")
        for mk in masks:
            out.append("      {" + ", ".join(f"0x{m:x}ull" for m in mk) + "},")
        out.append("  };")
        out.append(f"  static constexpr uint64_t XM[3][{np_}] = {{")
        for mk in exact_masks(p):
            out.append("      {" + ", ".join(f"0x{m:x}ull" for m in mk) + "},")
        out.append("  };")
        out.append("};")
    out.append("")
    out.append("}  // namespace rfhip")
    return "\n".join(out) + "\n"


def main(argv=None) -> int:
    argv = sys.argv[1:] if argv is None else argv
    text = render()
    if "--check" in argv:
        with open(HEADER) as f:
            same = f.read() == text
        print("rfhip_elem_tables.hpp " + ("matches the host builder" if same else "DIFFERS from the host builder"))
        return 0 if same else 1
    with open(HEADER, "w") as f:
        f.write(text)
    print(f"wrote {HEADER}")
    return 0


if __name__ == "__main__":
    sys.exit(main())
