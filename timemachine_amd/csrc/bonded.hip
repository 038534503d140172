// HarmonicBond / HarmonicAngle / PeriodicTorsion kernels, one thread per term,
// over the terms of one or many systems (term_sys maps a term to its system
// for lambda and the reduction index). Atom indices are global. Arithmetic is
// FP64 (bonded_terms.h), accumulation 64-bit fixed point at 2^36. u and
// du/dlambda are summed over the wave per system before one atomic each
// (a per-term atomic on one address per system serialises the whole launch).
#include "bonded.h"
#include "bonded_terms.h"
#include "fixed_point.h"
#include "wave.h"

namespace tmamd {

namespace {

__device__ __forceinline__ void add_fixed(uint64_t *p, double v) {
    const uint64_t f = f64_to_fixed(v, FIXED_SCALE);
    if (f != 0) {
        atomicAdd(reinterpret_cast<unsigned long long *>(p), static_cast<unsigned long long>(f));
    }
}

__device__ __forceinline__ void term_context(const BondedTerms &t, int term, const double *lambdas, double lambda0,
                                             const int *red_idx, double &lam, int &red) {
    const int s = t.term_sys ? t.term_sys[term] : 0;
    lam = lambdas ? lambdas[s] : lambda0;
    red = red_idx ? red_idx[s] : 0;
}

__device__ __forceinline__ void harmonic_bond(const BondedTerms &t, const int b, const double *__restrict__ x,
                                   const double *__restrict__ lambdas, double lambda0,
                                   const int *__restrict__ red_idx, uint64_t *__restrict__ du_dx,
                                   uint64_t *__restrict__ du_dp, uint64_t *__restrict__ du_dl,
                                   uint64_t *__restrict__ u, int dl_dp, uint64_t *__restrict__ slots) {
    const bool active = b < t.n;
    double lam = 0.0;
    int red = -1;
    uint64_t fu = 0, fdl = 0;
    if (active) {
        term_context(t, b, lambdas, lambda0, red_idx, lam, red);
        const int i = t.idx[b * 2 + 0];
        const int j = t.idx[b * 2 + 1];
        const int mult = t.mult ? t.mult[b] : 0;
        const int off = t.offset ? t.offset[b] : 1;
        // dl_dp: d(du/dlambda)/dp = mult * d(shape)/dp, i.e. du/dp at prefactor mult
        const double pf = dl_dp ? static_cast<double>(mult) : lam_prefactor<double>(mult, off, lam);
        const BondOut<double> o =
            bond_term<double>(x + i * 3, x + j * 3, t.params[b * 2 + 0], t.params[b * 2 + 1], mult, pf);
        if (slots) {
            for (int d = 0; d < 3; d++) {
                slots[(b * 2 + 0) * 3 + d] = f64_to_fixed(o.g[0][d], FIXED_SCALE);
                slots[(b * 2 + 1) * 3 + d] = f64_to_fixed(o.g[1][d], FIXED_SCALE);
            }
        } else if (du_dx) {
            for (int d = 0; d < 3; d++) {
                add_fixed(du_dx + i * 3 + d, o.g[0][d]);
                add_fixed(du_dx + j * 3 + d, o.g[1][d]);
            }
        }
        if (du_dp) {
            add_fixed(du_dp + b * 2 + 0, o.dkb);
            add_fixed(du_dp + b * 2 + 1, o.db0);
        }
        fu = f64_to_fixed(o.u, FIXED_SCALE);
        fdl = f64_to_fixed(o.dl, FIXED_SCALE);
    }
    if (u) {
        wave_add_by_key(u, red, fu);
    }
    if (du_dl) {
        wave_add_by_key(du_dl, red, fdl);
    }
}

__device__ __forceinline__ void harmonic_angle(const BondedTerms &t, const int a, const double *__restrict__ x,
                                   const double *__restrict__ lambdas, double lambda0,
                                   const int *__restrict__ red_idx, uint64_t *__restrict__ du_dx,
                                   uint64_t *__restrict__ du_dp, uint64_t *__restrict__ du_dl,
                                   uint64_t *__restrict__ u, int dl_dp, uint64_t *__restrict__ slots) {
    const bool active = a < t.n;
    double lam = 0.0;
    int red = -1;
    uint64_t fu = 0, fdl = 0;
    if (active) {
        term_context(t, a, lambdas, lambda0, red_idx, lam, red);
        const int i = t.idx[a * 3 + 0];
        const int j = t.idx[a * 3 + 1];
        const int k = t.idx[a * 3 + 2];
        const int mult = t.mult ? t.mult[a] : 0;
        const int off = t.offset ? t.offset[a] : 1;
        // dl_dp: d(du/dlambda)/dp = mult * d(shape)/dp, i.e. du/dp at prefactor mult
        const double pf = dl_dp ? static_cast<double>(mult) : lam_prefactor<double>(mult, off, lam);
        const AngleOut<double> o =
            angle_term<double>(x + i * 3, x + j * 3, x + k * 3, t.params[a * 2 + 0], t.params[a * 2 + 1], mult, pf);
        if (slots) {
            for (int d = 0; d < 3; d++) {
                slots[(a * 3 + 0) * 3 + d] = f64_to_fixed(o.g[0][d], FIXED_SCALE);
                slots[(a * 3 + 1) * 3 + d] = f64_to_fixed(o.g[1][d], FIXED_SCALE);
                slots[(a * 3 + 2) * 3 + d] = f64_to_fixed(o.g[2][d], FIXED_SCALE);
            }
        } else if (du_dx) {
            for (int d = 0; d < 3; d++) {
                add_fixed(du_dx + i * 3 + d, o.g[0][d]);
                add_fixed(du_dx + j * 3 + d, o.g[1][d]);
                add_fixed(du_dx + k * 3 + d, o.g[2][d]);
            }
        }
        if (du_dp) {
            add_fixed(du_dp + a * 2 + 0, o.dka);
            add_fixed(du_dp + a * 2 + 1, o.da0);
        }
        fu = f64_to_fixed(o.u, FIXED_SCALE);
        fdl = f64_to_fixed(o.dl, FIXED_SCALE);
    }
    if (u) {
        wave_add_by_key(u, red, fu);
    }
    if (du_dl) {
        wave_add_by_key(du_dl, red, fdl);
    }
}

__device__ __forceinline__ void periodic_torsion(const BondedTerms &t, const int q, const double *__restrict__ x,
                                   const double *__restrict__ lambdas, double lambda0,
                                   const int *__restrict__ red_idx, uint64_t *__restrict__ du_dx,
                                   uint64_t *__restrict__ du_dp, uint64_t *__restrict__ du_dl,
                                   uint64_t *__restrict__ u, int dl_dp, uint64_t *__restrict__ slots) {
    const bool active = q < t.n;
    double lam = 0.0;
    int red = -1;
    uint64_t fu = 0, fdl = 0;
    if (active) {
        term_context(t, q, lambdas, lambda0, red_idx, lam, red);
        const int i = t.idx[q * 4 + 0];
        const int j = t.idx[q * 4 + 1];
        const int k = t.idx[q * 4 + 2];
        const int l = t.idx[q * 4 + 3];
        const int mult = t.mult ? t.mult[q] : 0;
        const int off = t.offset ? t.offset[q] : 1;
        // dl_dp: d(du/dlambda)/dp = mult * d(shape)/dp, i.e. du/dp at prefactor mult
        const double pf = dl_dp ? static_cast<double>(mult) : lam_prefactor<double>(mult, off, lam);
        const TorsionOut<double> o = torsion_term<double>(x + i * 3, x + j * 3, x + k * 3, x + l * 3,
                                                          t.params[q * 3 + 0], t.params[q * 3 + 1],
                                                          t.params[q * 3 + 2], mult, pf);
        if (slots) {
            for (int a = 0; a < 4; a++) {
                for (int d = 0; d < 3; d++) {
                    slots[(q * 4 + a) * 3 + d] = f64_to_fixed(o.g[a][d], FIXED_SCALE);
                }
            }
        } else if (du_dx) {
            const int at[4] = {i, j, k, l};
            for (int a = 0; a < 4; a++) {
                for (int d = 0; d < 3; d++) {
                    add_fixed(du_dx + at[a] * 3 + d, o.g[a][d]);
                }
            }
        }
        if (du_dp) {
            add_fixed(du_dp + q * 3 + 0, o.dk);
            add_fixed(du_dp + q * 3 + 1, o.dphase);
            add_fixed(du_dp + q * 3 + 2, o.dperiod);
        }
        fu = f64_to_fixed(o.u, FIXED_SCALE);
        fdl = f64_to_fixed(o.dl, FIXED_SCALE);
    }
    if (u) {
        wave_add_by_key(u, red, fu);
    }
    if (du_dl) {
        wave_add_by_key(du_dl, red, fdl);
    }
}

template <BondedKind KIND>
__device__ __forceinline__ void bonded_term(const BondedTerms &t, const int term, const double *x,
                                            const double *lambdas, double lambda0, const int *red_idx, uint64_t *du_dx,
                                            uint64_t *du_dp, uint64_t *du_dl, uint64_t *u, int dl_dp, uint64_t *slots) {
    if constexpr (KIND == BondedKind::Bond) {
        harmonic_bond(t, term, x, lambdas, lambda0, red_idx, du_dx, du_dp, du_dl, u, dl_dp, slots);
    } else if constexpr (KIND == BondedKind::Angle) {
        harmonic_angle(t, term, x, lambdas, lambda0, red_idx, du_dx, du_dp, du_dl, u, dl_dp, slots);
    } else {
        periodic_torsion(t, term, x, lambdas, lambda0, red_idx, du_dx, du_dp, du_dl, u, dl_dp, slots);
    }
}

constexpr int TERM_BLOCK = 128;

template <BondedKind KIND>
__global__ __launch_bounds__(TERM_BLOCK) void k_bonded(const BondedTerms t, const double *__restrict__ x,
                                                       const double *__restrict__ lambdas, double lambda0,
                                                       const int *__restrict__ red_idx, uint64_t *__restrict__ du_dx,
                                                       uint64_t *__restrict__ du_dp, uint64_t *__restrict__ du_dl,
                                                       uint64_t *__restrict__ u, int dl_dp,
                                                       uint64_t *__restrict__ slots) {
    bonded_term<KIND>(t, blockIdx.x * TERM_BLOCK + threadIdx.x, x, lambdas, lambda0, red_idx, du_dx, du_dp, du_dl, u,
                      dl_dp, slots);
}

// All three kinds in one launch: workgroups [0, g1) take bonds, [g1, g2) angles
// and the rest torsions. What bounds a single system is the launch itself (4.5 us
// a graph node for ~1 us of work on 6k atoms), so one instead of three.
__global__ __launch_bounds__(TERM_BLOCK) void k_bonded_all(const BondedSet b, const int g1, const int g2,
                                                           const double *__restrict__ x,
                                                           const double *__restrict__ lambdas,
                                                           const int *__restrict__ red_idx,
                                                           uint64_t *__restrict__ du_dl, uint64_t *__restrict__ u) {
    const int g = blockIdx.x;
    if (g < g1) {
        bonded_term<BondedKind::Bond>(b.t[0], g * TERM_BLOCK + threadIdx.x, x, lambdas, 0.0, red_idx, nullptr,
                                      nullptr, du_dl, u, 0, b.slots[0]);
    } else if (g < g2) {
        bonded_term<BondedKind::Angle>(b.t[1], (g - g1) * TERM_BLOCK + threadIdx.x, x, lambdas, 0.0, red_idx, nullptr,
                                       nullptr, du_dl, u, 0, b.slots[1]);
    } else {
        bonded_term<BondedKind::Torsion>(b.t[2], (g - g2) * TERM_BLOCK + threadIdx.x, x, lambdas, 0.0, red_idx, nullptr,
                                         nullptr, du_dl, u, 0, b.slots[2]);
    }
}

// Force of every atom: the fixed-point slots of its terms plus the tiles' sums in
// sorted order, which are cleared for the next launch. GATHER_LANES lanes share an
// atom: one thread an atom walked the longest list alone (a ligand atom of ~60
// slots, two dependent loads each: 17.8 us for one system of 6k atoms) and
// wrote its three words by itself.
constexpr int GATHER_LANES = 4;

__global__ __launch_bounds__(256) void k_atom_forces(const BondedIncidence inc, const uint64_t *__restrict__ slots,
                                                     const SortedForces s0, const SortedForces s1,
                                                     uint64_t *__restrict__ du_dx) {
    const int t = blockIdx.x * 256 + threadIdx.x;
    const int a = t / GATHER_LANES;
    const int q = t % GATHER_LANES;
    if (a >= inc.A) { // whole groups leave
        return;
    }
    uint64_t acc[3] = {0, 0, 0};
    if (inc.off) {
        const int e1 = inc.off[a + 1];
#pragma unroll 2
        for (int e = inc.off[a] + q; e < e1; e += GATHER_LANES) {
            const uint64_t *g = slots + static_cast<size_t>(inc.items[e]) * 3;
            acc[0] += g[0];
            acc[1] += g[1];
            acc[2] += g[2];
        }
    }
    for (int m = 1; m < GATHER_LANES; m <<= 1) {
#pragma unroll
        for (int d = 0; d < 3; d++) {
            acc[d] += __shfl_xor(static_cast<unsigned long long>(acc[d]), m, 64);
        }
    }
    if (q < 3) { // lane q writes component q
        uint64_t f = q == 0 ? acc[0] : q == 1 ? acc[1] : acc[2];
        for (int k = 0; k < 2; k++) {
            const SortedForces &s = k == 0 ? s0 : s1;
            const int slot = a < s.atoms ? s.slot_of[a] : -1;
            if (slot >= 0) {
                uint64_t *p = s.sorted + q * s.slots + slot;
                f += *p;
                *p = 0;
            }
        }
        du_dx[a * 3 + q] = f;
    }
}

} // namespace

void build_bonded_incidence(int A, const std::vector<const std::vector<int> *> &idx, std::vector<int> &off,
                            std::vector<uint32_t> &items, std::vector<int> &slot0) {
    off.assign(static_cast<size_t>(A) + 1, 0);
    slot0.assign(idx.size(), 0);
    size_t n_slots = 0;
    for (size_t k = 0; k < idx.size(); k++) {
        slot0[k] = static_cast<int>(n_slots);
        n_slots += idx[k]->size();
        for (int a : *idx[k]) {
            off[a + 1] += 1;
        }
    }
    if (n_slots >= (1u << 31)) {
        throw Error("bonded incidence: too many terms");
    }
    for (int a = 0; a < A; a++) {
        off[a + 1] += off[a];
    }
    items.assign(off[A], 0);
    std::vector<int> fill(off.begin(), off.end() - 1);
    for (size_t k = 0; k < idx.size(); k++) {
        const std::vector<int> &v = *idx[k];
        for (size_t e = 0; e < v.size(); e++) {
            items[fill[v[e]]++] = static_cast<uint32_t>(slot0[k] + e); // term e / arity, position e % arity
        }
    }
}

void launch_atom_forces(const BondedIncidence &inc, const uint64_t *slots, const SortedForces &s0,
                        const SortedForces &s1, uint64_t *du_dx, hipStream_t stream) {
    if (inc.A == 0) {
        return;
    }
    k_atom_forces<<<ceil_div(inc.A, 256 / GATHER_LANES), 256, 0, stream>>>(inc, slots, s0, s1, du_dx);
    TM_LAUNCH_CHECK();
}

void launch_bonded_all(const BondedSet &b, const double *x, const double *lambdas, const int *red_idx, uint64_t *du_dl,
                       uint64_t *u, hipStream_t stream) {
    const int g1 = ceil_div(b.t[0].n, TERM_BLOCK);
    const int g2 = g1 + ceil_div(b.t[1].n, TERM_BLOCK);
    const int grid = g2 + ceil_div(b.t[2].n, TERM_BLOCK);
    if (grid == 0) {
        return;
    }
    k_bonded_all<<<grid, TERM_BLOCK, 0, stream>>>(b, g1, g2, x, lambdas, red_idx, du_dl, u);
    TM_LAUNCH_CHECK();
}

void launch_bonded(BondedKind kind, const BondedTerms &t, const double *x, const double *lambdas, double lambda0,
                   const int *red_idx, uint64_t *du_dx, uint64_t *du_dp, uint64_t *du_dl, uint64_t *u,
                   hipStream_t stream, bool dl_dp) {
    if (t.n == 0 || (!du_dx && !du_dp && !du_dl && !u)) {
        return;
    }
    if (dl_dp && (du_dx || du_dl || u || !du_dp)) {
        throw Error("launch_bonded: the dl_dp mode writes du_dp only");
    }
    auto kern = kind == BondedKind::Bond    ? k_bonded<BondedKind::Bond>
                : kind == BondedKind::Angle ? k_bonded<BondedKind::Angle>
                                            : k_bonded<BondedKind::Torsion>;
    kern<<<ceil_div(t.n, TERM_BLOCK), TERM_BLOCK, 0, stream>>>(t, x, lambdas, lambda0, red_idx, du_dx, du_dp, du_dl, u,
                                                              dl_dp ? 1 : 0, nullptr);
    TM_LAUNCH_CHECK();
}

} // namespace tmamd
