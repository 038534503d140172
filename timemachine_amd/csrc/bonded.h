#pragma once

#include <vector>

#include "tm_common.h"

namespace tmamd {

enum class BondedKind { Bond = 0, Angle = 1, Torsion = 2 };

inline int bonded_arity(BondedKind k) { return k == BondedKind::Bond ? 2 : (k == BondedKind::Angle ? 3 : 4); }
inline int bonded_nparams(BondedKind k) { return k == BondedKind::Torsion ? 3 : 2; }

// Device view of a list of bonded terms (possibly from many systems).
struct BondedTerms {
    int n;
    const int *idx;      // [n, arity] global atom indices
    const double *params; // [n, nparams]
    const int *mult;     // [n] lambda multiplier (nullptr -> 0)
    const int *offset;   // [n] lambda offset (nullptr -> 1)
    const int *term_sys; // [n] system of each term (nullptr -> 0)
};

// Force slots: a term's force on the atom at position r of term q goes to
// slot slot0[kind] + q * arity + r (3 fixed-point words), written by the term
// kernels instead of a global atomic per atom and component; the incidence
// lists (CSR over global atoms) name the slots of every atom.
struct BondedIncidence {
    int A;            // atoms
    const int *off;   // [A + 1]
    const uint32_t *items; // slot indices
};

// Host side: incidence lists over groups of terms (global atom indices,
// idx[k] = [n_k, arity_k] flattened: position e is slot slot0[k] + e);
// slot0 receives each group's first slot.
void build_bonded_incidence(int A, const std::vector<const std::vector<int> *> &idx, std::vector<int> &off,
                            std::vector<uint32_t> &items, std::vector<int> &slot0);

// The pair tiles' force sums in sorted order: component c of global atom a is
// sorted[c * slots + slot_of[a]], no sums for slot_of[a] < 0 or a >= atoms.
struct SortedForces {
    uint64_t *sorted;
    size_t slots;
    const int *slot_of;
    int atoms; // 0: no sums
};

// du_dx[a] = its slots' sum + its sorted sums (cleared after the read). Nothing
// else may write du_dx or the sums meanwhile. The fixed-point values are those
// the atomics would add, so the sums are bitwise the same. inc.off may be null.
void launch_atom_forces(const BondedIncidence &inc, const uint64_t *slots, const SortedForces &s0,
                        const SortedForces &s1, uint64_t *du_dx, hipStream_t stream);

// All bonded terms of a batch in one launch; the per-atom forces go to force slots
// (see above).
struct BondedSet {
    BondedTerms t[3];   // by BondedKind
    uint64_t *slots[3]; // nullptr: no forces
};
void launch_bonded_all(const BondedSet &b, const double *x, const double *lambdas, const int *red_idx, uint64_t *du_dl,
                       uint64_t *u, hipStream_t stream);

// dl_dp: write d(du/dlambda)/dp into du_dp (every other output must be null).
void launch_bonded(BondedKind kind, const BondedTerms &t, const double *x, const double *lambdas, double lambda0,
                   const int *red_idx, uint64_t *du_dx, uint64_t *du_dp, uint64_t *du_dl, uint64_t *u,
                   hipStream_t stream, bool dl_dp = false);

} // namespace tmamd
