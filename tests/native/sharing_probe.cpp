// Which wavenumbers of a kxky system share factors (factor_sharing), as plain
// arrays: returns slots per factored system, or -1; the caller's arrays hold
// nkx (NY - 1) representatives, four members each, and three maps of `total`
// rows and columns with their signs.
#include <algorithm>
#include <exception>

#include "../../coral_amd/csrc/assembly.hpp"

extern "C" int sharing_probe(const coral_amd_problem *prob, int isys, int *nrep, int *rep, int *mem, int *row, int *col,
                             unsigned char *rneg, unsigned char *cneg) {
    try {
        const coral::Problem P = coral::assemble(*prob);
        const coral::SystemTables &t = P.kxky.at(isys);
        const coral::FactorSharing f = coral::factor_sharing(t, P.nkx, P.NY, P.kx_box == P.ky_box);
        *nrep = int(f.rep.size());
        std::copy(f.rep.begin(), f.rep.end(), rep);
        std::copy(f.mem.begin(), f.mem.end(), mem);
        for (size_t k = 0; k < f.sym.size(); ++k) {
            std::copy(f.sym[k].row.begin(), f.sym[k].row.end(), row + k * t.total);
            std::copy(f.sym[k].col.begin(), f.sym[k].col.end(), col + k * t.total);
            std::copy(f.sym[k].rneg.begin(), f.sym[k].rneg.end(), rneg + k * t.total);
            std::copy(f.sym[k].cneg.begin(), f.sym[k].cneg.end(), cneg + k * t.total);
        }
        return f.nslot;
    } catch (const std::exception &) {
        return -1;
    }
}
