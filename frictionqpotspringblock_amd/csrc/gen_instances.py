"""Generate the resident-kernel instantiation units fq_res_<unit>_<part>.hip and the
header fq_res_units.hpp that declares them.

Each unit instantiates, for its (potential, interaction, forcing) classes and
the variant table of each, k_resident<POT, INT, EXT, PPT, MAXT> (all modes),
for chains k_flow<POT, INT, EXT, PPT, MAXT> (timeSteps / flowSteps), and,
without external forcing, the quasistatic driver (k_quasi_chain, or k_quasi:
see pipelined()); it exposes
launch_resident_<unit>(), launch_flow_<unit>(), launch_quasi_<unit>() and
resident_variants_<unit>(). Small units let hipcc compile them in parallel.
The build (build_ext.py) generates them before compiling; by hand:

    python gen_instances.py
"""

import os

# (particles per thread, max threads per workgroup) variants
HOT = [(1, 1024), (2, 1024), (4, 1024), (4, 512), (8, 1024), (8, 512), (8, 256), (16, 512), (16, 256)]
STD = [(1, 1024), (2, 1024), (4, 1024), (4, 512), (8, 1024), (8, 512), (16, 512), (16, 256)]
MIRROR = [(1, 1024), (2, 1024), (4, 1024), (8, 1024)]
LATTICE = [(1, 1024), (2, 1024), (4, 1024), (4, 512), (8, 1024), (8, 512)]

CHAINS = {"INT_NONE", "INT_LAPLACE1D", "INT_QUARTIC1D", "INT_QUARTICGRADIENT1D"}

# k_flow shapes: those whose registers fit without large spills (other shapes
# of timeSteps / flowSteps run on k_resident)
FLOW_SHAPES = {(1, 1024), (2, 1024), (4, 1024), (4, 512), (8, 512), (8, 256), (16, 256)}
# the one with a form that leaves every refill to the host (fq_flow.hpp)
FLOW_FIXED = (1, 1024)

# unit name -> (potential, [(interaction, forcing values, variants)])
UNITS = {
    "cuspy_laplace": ("POT_CUSPY", [("INT_LAPLACE1D", [0, 1], HOT)]),
    "cuspy_chain": (
        "POT_CUSPY",
        [("INT_QUARTIC1D", [0, 1], STD), ("INT_QUARTICGRADIENT1D", [0], STD), ("INT_NONE", [0, 1], STD)],
    ),
    "cuspy_field": (
        "POT_CUSPY",
        [("INT_LONGRANGE1D", [0, 1], MIRROR), ("INT_LAPLACE2D", [0], LATTICE),
         ("INT_QUARTICGRADIENT2D", [0], LATTICE)],
    ),
    "semismooth": ("POT_SEMISMOOTH", [("INT_LAPLACE1D", [0], STD), ("INT_QUARTIC1D", [0], STD), ("INT_NONE", [0], STD)]),
    "smooth": ("POT_SMOOTH", [("INT_LAPLACE1D", [0], STD), ("INT_QUARTIC1D", [0], STD), ("INT_NONE", [0], STD)]),
}

HEADER = "// Generated by gen_instances.py: resident-kernel instantiations (see fq_launch.hpp).\n"
SIG = (
    "int inter, int ext, int ppt, int maxt, int threads, size_t lds, const SysView* views, int nsys, "
    "const RunArgs& ra, hipStream_t stream"
)
FLOW_SIG = SIG + ", bool unit_mass, bool full, bool moves"
QUASI_SIG = (
    "int inter, int ppt, int maxt, int threads, size_t lds, const SysView* views, int nsys, const RunArgs& ra, "
    "const QsArgs& qa, hipStream_t stream, bool unit_mass, bool full"
)

# units whose quasistatic driver for chains also has the unit-mass and
# full-thread forms (every system's N divisible by the particles per thread)
QUASI_FULL = {"cuspy_laplace"}


def pipelined(pot, it, ppt, mt):
    """Whether a variant's quasistatic driver is k_quasi_chain (fq_quasi.hpp)
    and not k_quasi, and whether minimise alone runs on it as well (else on
    k_resident). k_quasi_chain needs more registers: where it spills hundreds
    of them the general kernels are faster. Three events / a quench of 16
    chains, ms (k_quasi_chain / the general kernels): Cuspy-Laplace of 8192,
    8 x 1024: 72 / 30, 34 / 10; 16 x 512: 59 / 19, 28 / 7.5; of 4096, 4 x 1024:
    7.9 / 8.9, 4.0 / 3.9; 16 x 256: 5.3 / 11.8, 2.8 / 5.7. SemiSmooth-Laplace
    of 8192, 8 x 1024: 188 / 46, 111 / 22; of 4096, 4 x 1024: 43 / 14, 28 / 8.
    Smooth-Laplace, 16 x 256: 73 / 63, 30 / 23."""
    if it == "INT_LONGRANGE1D":
        return False, False
    if ppt <= 2 or (ppt <= 8 and mt <= 512):
        return True, True
    if it not in CHAINS or pot == "POT_SMOOTH":
        return False, False
    if (ppt, mt) == (16, 256):
        return True, True
    return pot == "POT_CUSPY" and (ppt, mt) == (4, 1024), False


def quasi_launcher(name, pot, ints):
    out = [f"bool launch_quasi_{name}({QUASI_SIG})", "{"]
    for it, exts, variants in ints:
        if 0 not in exts:
            continue
        for ppt, mt in variants:
            out.append(f"    if (inter == {it} && ppt == {ppt} && maxt == {mt}) {{")
            driver, alone = pipelined(pot, it, ppt, mt)
            if not alone:
                out.append("        if (qa.plain) { // minimise runs on k_resident")
                out.append("            return false;")
                out.append("        }")
            if driver:
                forms = [("true", "true", "unit_mass && full"), ("true", "false", "unit_mass")] if name in QUASI_FULL else []
                if it not in CHAINS:
                    forms = [("true", "false", "unit_mass")]
                for unit, full, cond in forms:
                    k = f"k_quasi_chain<{pot}, {it}, {ppt}, {mt}, {unit}, {full}>"
                    out.append(f"        if ({cond}) {{")
                    out.append(
                        f"            hipLaunchKernelGGL(({k}), dim3(nsys), dim3(threads), lds, stream, views, ra, qa);"
                    )
                    out.append("            return true;")
                    out.append("        }")
                k = f"k_quasi_chain<{pot}, {it}, {ppt}, {mt}, false, false>"
            else:
                k = f"k_quasi<{pot}, {it}, {ppt}, {mt}, false>"
            out.append(f"        hipLaunchKernelGGL(({k}), dim3(nsys), dim3(threads), lds, stream, views, ra, qa);")
            out.append("        return true;")
            out.append("    }")
    out += ["    return false;", "}"]
    return out


def launcher(name, kernel, pot, ints, chains_only):
    out = [f"bool launch_{kernel}_{name}({FLOW_SIG if chains_only else SIG})", "{"]
    for it, exts, variants in ints:
        if chains_only and it not in CHAINS:
            continue
        for e in exts:
            for ppt, mt in variants:
                if chains_only and (ppt, mt) not in FLOW_SHAPES:
                    continue
                out.append(f"    if (inter == {it} && ext == {e} && ppt == {ppt} && maxt == {mt}) {{")
                if chains_only:  # k_flow: unit mass (and, with it, full threads) compile-time choices
                    for unit, full in (("true", "true"), ("true", "false"), ("false", "false")):
                        k = f"k_{kernel}<{pot}, {it}, {e}, {ppt}, {mt}, {unit}, {full}>"
                        cond = {
                            ("true", "true"): "unit_mass && full",
                            ("true", "false"): "unit_mass && !full",
                            ("false", "false"): "!unit_mass",
                        }[(unit, full)]
                        out.append(f"        if ({cond}) {{")
                        if (ppt, mt) == FLOW_FIXED:
                            out.append("            if (!moves) {")
                            out.append(
                                f"                hipLaunchKernelGGL(({k[:-1]}, false>), dim3(nsys), dim3(threads), lds, "
                                "stream, views, ra);"
                            )
                            out.append("                return true;")
                            out.append("            }")
                        out.append(
                            f"            hipLaunchKernelGGL(({k}), dim3(nsys), dim3(threads), lds, stream, views, ra);"
                        )
                        out.append("            return true;")
                        out.append("        }")
                else:
                    k = f"k_{kernel}<{pot}, {it}, {e}, {ppt}, {mt}>"
                    out.append(f"        hipLaunchKernelGGL(({k}), dim3(nsys), dim3(threads), lds, stream, views, ra);")
                    out.append("        return true;")
                out.append("    }")
    out.append("    return false;")
    out.append("}")
    return out


def variants(name, ints):
    out = [f"int resident_variants_{name}(int inter, int ext, int* ppt, int* maxt, int cap)", "{", "    int n = 0;"]
    for it, exts, shapes in ints:
        for e in exts:
            arr = ", ".join(f"{{{p}, {m}}}" for p, m in shapes)
            out.append(f"    if (inter == {it} && ext == {e}) {{")
            out.append(f"        static const int v[][2] = {{{arr}}};")
            out.append("        for (const auto& x : v) {")
            out.append("            if (n < cap) {")
            out.append("                ppt[n] = x[0];")
            out.append("                maxt[n] = x[1];")
            out.append("            }")
            out.append("            ++n;")
            out.append("        }")
            out.append("        return n;")
            out.append("    }")
    out += ["    return 0;", "}"]
    return out


def unit(name, pot, ints, part):
    """One source of a unit: its k_resident (and the table of variants), its
    k_flow or its quasistatic kernels (separate sources: they compile in
    parallel)."""
    body = {
        "resident": lambda: launcher(name, "resident", pot, ints, False) + [""] + variants(name, ints),
        "flow": lambda: launcher(name, "flow", pot, ints, True),
        "quasi": lambda: quasi_launcher(name, pot, ints),
    }[part]()
    out = [HEADER, '#include "fq_flow.hpp"', '#include "fq_launch.hpp"', '#include "fq_quasi.hpp"',
           '#include "fq_resident.hpp"', "", "namespace fq {", ""]
    return "\n".join(out + body + ["", "} // namespace fq"]) + "\n"


def header():
    out = [HEADER, "#pragma once", "", '#include "fq_common.hpp"', "", "namespace fq {", ""]
    for name in UNITS:
        out.append(f"bool launch_resident_{name}({SIG});")
        out.append(f"bool launch_flow_{name}({FLOW_SIG});")
        out.append(f"bool launch_quasi_{name}({QUASI_SIG});")
        out.append(f"int resident_variants_{name}(int inter, int ext, int* ppt, int* maxt, int cap);")
    out.append("")
    out.append("// the units that instantiate each potential, in the order they are tried")
    for pot in ("POT_CUSPY", "POT_SEMISMOOTH", "POT_SMOOTH"):
        names = [n for n, (p, _) in UNITS.items() if p == pot]
        out.append(f"#define FQ_UNITS_{pot} " + " ".join(f"X({n})" for n in names))
    out.append("")
    out.append("} // namespace fq")
    return "\n".join(out) + "\n"


def _write_if_changed(path, text):
    try:
        with open(path) as fh:
            if fh.read() == text:
                return
    except OSError:
        pass
    with open(path, "w") as fh:
        fh.write(text)


def generate(directory):
    """Write the units and their header into `directory` (files whose text is
    unchanged are left alone); returns the unit file names in build order."""
    names = []
    for name, (pot, ints) in UNITS.items():
        for part in ("resident", "flow", "quasi"):
            fname = f"fq_res_{name}_{part}.hip"
            _write_if_changed(os.path.join(directory, fname), unit(name, pot, ints, part))
            names.append(fname)
    _write_if_changed(os.path.join(directory, "fq_res_units.hpp"), header())
    return names


if __name__ == "__main__":
    generate(os.path.dirname(os.path.abspath(__file__)))
