// The row-program kernels compiled ahead of time for the programs of a decoder block (the norms, the
// causal soft-max): the phases of the interpreter's row kernel unrolled at compile time.
#include "interp.hpp"

namespace cg {

bool launch_compiled_rows(const Pending &p, const FusedArgs &a, uint32_t *rowout, int tpr, dim3 grid, LaunchQueue &s) {
    return aot_rows_dispatch(p, a, rowout, tpr, grid, s, RowsPrograms{});
}

template <class... P> static bool any_matches(const Pending &p, ProgramList<P...>) { return (program_matches<P>(p) || ...); }
bool rows_program_compiled(const Pending &p) { return (p.rowlen + 7) / 8 > 4 && any_matches(p, RowsPrograms{}); } // (shorter rows: four lanes each, interpreted)

template <class P> static bool begins(const Pending &p) {
    if (p.nleaf > P::nleaf || p.ninstr > P::ninstr) return false;
    for (int l = 0; l < p.nleaf; l++)
        if (p.leaf[l].uniform || p.leaf[l].pw) return false;
    for (int i = 0; i < p.ninstr; i++) {
        const Instr &in = p.ins[i];
        if (in.op != P::code[i][0] || in.a != P::code[i][1] || in.b != P::code[i][2] || in.c != P::code[i][3]) return false;
    }
    return true;
}
bool rows_max_program_begun(const Pending &p) { return begins<RowsLogSumExpMax>(p) || begins<RowsLogSumExpMaxKept>(p); }

} // namespace cg
