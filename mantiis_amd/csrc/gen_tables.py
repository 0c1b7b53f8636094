"""Generate mts_tables.inc from the 52-type boundary tables in ../data/system_files.

The tables are data of the reference (include/system_files/*.txt, loaded at
utils.hpp:728-793: direction-major 9x52, icsr 1-based).  They are embedded in
the library so that no file is read at run time.  Run from any directory:
    python mantiis_amd/csrc/gen_tables.py
"""
import os

import numpy as np

HERE = os.path.dirname(os.path.abspath(__file__))
DATA = os.path.join(HERE, "..", "data", "system_files")


def main():
    bt = np.loadtxt(os.path.join(DATA, "bnd_types.txt")).astype(int)
    ifs = np.loadtxt(os.path.join(DATA, "ifstream.txt")).reshape(9, 52).T.astype(int)
    icsr = np.loadtxt(os.path.join(DATA, "icsr.txt")).reshape(9, 52).T.astype(int) - 1
    xy = np.loadtxt(os.path.join(DATA, "xy_norm.txt")).reshape(2, 52).T
    out = ["// Generated by gen_tables.py from data/system_files -- do not edit.",
           "// 52 wall configurations of a cell's 3x3 neighbourhood (utils.hpp:728-793).",
           "#define MTS_NTYPES 52"]
    out.append("static constexpr int MTS_BND_CODE[52] = {" + ", ".join(str(v) for v in bt) + "};")
    out.append("static constexpr unsigned char MTS_IFSTREAM[52][9] = {" +
               ", ".join("{" + ", ".join(str(v) for v in row) + "}" for row in ifs) + "};")
    out.append("static constexpr signed char MTS_ICSR[52][9] = {" +
               ", ".join("{" + ", ".join(str(v) for v in row) + "}" for row in icsr) + "};")
    out.append("static constexpr double MTS_XYNORM[52][2] = {" +
               ", ".join("{%r, %r}" % (float(a), float(b)) for a, b in xy) + "};")
    with open(os.path.join(HERE, "mts_tables.inc"), "w") as f:
        f.write("\n".join(out) + "\n")


if __name__ == "__main__":
    main()
