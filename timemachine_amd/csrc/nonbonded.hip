// Nonbonded pair kernels: the 64x64 tile kernel over the neighborlist and the
// pair-list kernel used for exclusions.
//
// Tile kernel (restates the semantics of kernels/k_nonbonded.cuh:311-671 for
// wave64): one wave per 64 x 64 tile. The reference evaluates every
// (row, column) slot of a tile; here a first pass screens the pairs in FP32
// (on the matrix cores for most tiles) and compacts those inside the cutoff
// into an LDS queue, and a second pass evaluates the queued pairs 64 at a time
// with every lane busy, repeating the exact FP64 cutoff test. Force, du/dp,
// du/dl and energy terms are rounded to
// 64-bit fixed point per pair and summed exactly (LDS u64 atomics per atom,
// registers for u and du/dl). Column atoms leave through 64-bit global
// atomics at the end of each tile, row atoms at the end of a run of tiles of
// the same row block, both to words in sorted order that a second launch moves
// to the atoms (TileOut); u and du/dl leave once per system and wave
// (add_scalars). Integer sums do not depend on the order, so the outputs are
// bitwise those of evaluating the pairs one by one.
//
// Pair-list kernel (kernels/k_nonbonded_pair_list.cuh:17-216): one thread
// per pair; with negated=1 it subtracts exactly what the tile kernel added,
// which is how exclusions cancel.
#include <type_traits>

#include "nb_pair.h"
#include "nb_state.h"
#include "wave.h"

namespace tmamd {

namespace {

// One wave per workgroup: waves share nothing but the output atomics, and a
// one-wave workgroup is scheduled and retired on its own (measured on MI355X at
// an equal wave count: 3% faster per batched step than two-wave workgroups,
// 5% faster than four). Per-wave LDS is 10 KB (forces) to 15 KB (parameter
// derivatives of interpolated parameters).
constexpr int NB_BLOCK = 64;
constexpr int NB_BAD_BOX = NB_STATUS_BOX_TOO_SMALL | NB_STATUS_BOX_NOT_ORTHO;

__device__ __forceinline__ void atomic_add_u64(uint64_t *p, uint64_t v) {
    atomicAdd(reinterpret_cast<unsigned long long *>(p), static_cast<unsigned long long>(v));
}

// A queued item is one row slot and two consecutive column slots, for one lane;
// a batch is 64 items. Fewer than 64 wait in each of the two queues between
// steps of the screen, and a step adds at most 64 to each.
constexpr int ITEM_QUEUE = 2 * TILE;

// LDS index of the atom in row or column place 4 b + j of the screen (block b of
// 16): place j of all blocks together, so that the atoms that a step's items
// take at once (one place of each block) lie in different banks. Columns of the
// second pair are shifted by four blocks against the first's.
__device__ __forceinline__ int row_index(int slot) { return ((slot & 3) << 4) | (slot >> 2); }
__device__ __forceinline__ int col_index(int slot) {
    return ((slot & 3) << 4) | ((slot >> 2) ^ ((slot & 2) << 1));
}
__device__ __forceinline__ int col_place(int index) { // inverse of col_index
    const int j = index >> 4;
    return (((index & 15) ^ ((j & 2) << 1)) << 2) | j;
}
constexpr uint32_t NEXT_COL = 8 * 16; // byte offset of a pair's second column

// dq/dl, dsig/dl, deps/dl of row and column atoms (interpolated parameters only)
template <bool INTERP> struct TileDp {
    float dp[2][3][TILE];
};
template <> struct TileDp<false> {};

// Per-wave LDS of the tile kernel; [0] rows, [1] columns, indexed by slot.
// NACC accumulators per atom: x, y, z forces, then q, sig, eps parameter
// derivatives when requested. Coordinates and charge come in 16-byte pairs: a
// gather of 16 bytes a lane takes the LDS as long as one of 8 (10.8 against
// 10.6 cycles a wave at random slots, 5.7 against 5.0 at consecutive ones).
// The accumulators are 8-byte arrays. 10 KB for the force kernels, so that 16
// waves share a CU (the queue holds 2-byte items, and the 4D coordinates of the
// few lambda-dependent tiles stay in registers for that, see Lane4D).
template <int NACC, bool INTERP> struct TileLds : TileDp<INTERP> {
    double2 xy[2][TILE], zq[2][TILE];
    float2 se[2][TILE]; // sig, eps
    float4 col[TILE];   // screen: column x, y, z and |b|^2 / 2 (FP32, relative to the row block's centre)
    uint32_t idx[2][TILE];      // sorted index: rows always, columns of diagonal tiles
    uint16_t pq[2][ITEM_QUEUE]; // items: row index << 3 | first column index << 9
    uint64_t acc[2][NACC][TILE];
};

// element of an 8-byte array at a byte offset
template <typename T> __device__ __forceinline__ T &at8(T *a, uint32_t off8) {
    return *reinterpret_cast<T *>(reinterpret_cast<char *>(a) + off8);
}
__device__ __forceinline__ double2 at16(const double2 *a, uint32_t off8) {
    return *reinterpret_cast<const double2 *>(reinterpret_cast<const char *>(a) + (off8 << 1));
}
template <typename T> __device__ __forceinline__ T at4(const T *a, uint32_t off8) {
    return *reinterpret_cast<const T *>(reinterpret_cast<const char *>(a) + (off8 >> 1));
}

__device__ __forceinline__ void lds_add_u64(uint64_t *p, uint64_t v) {
    atomicAdd(reinterpret_cast<unsigned long long *>(p), static_cast<unsigned long long>(v));
}
// p -= v modulo 2^64 (one LDS atomic, no separate negation)
__device__ __forceinline__ void lds_sub_u64(uint64_t *p, uint64_t v) {
    __hip_atomic_fetch_sub(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Values of one system that the evaluation reads (wave-uniform).
struct TileSys {
    double bx, by, bz, ibx, iby, ibz; // box edges on the coordinate grid (BoxAxis) and their inverses
    double cut2;                      // squared cutoff: the exact test of pass 2
    double small;                     // fixed_small_factor(cutoff)
    double beta;
};

// 4D coordinate and its lambda derivative of the row with LDS index `lane` and of
// the column in screen place `lane`; lanes read each other's (ds_bpermute).
struct Lane4D {
    double w[2];
    float dwdl[2];
};
__device__ __forceinline__ float push_f32(float v, int to) { // v goes to lane `to`
    return __int_as_float(__builtin_amdgcn_ds_permute(to << 2, __float_as_int(v)));
}
__device__ __forceinline__ double push_f64(double v, int to) {
    const uint64_t b = static_cast<uint64_t>(__double_as_longlong(v));
    const uint32_t lo = __builtin_amdgcn_ds_permute(to << 2, static_cast<int>(static_cast<uint32_t>(b)));
    const uint32_t hi = __builtin_amdgcn_ds_permute(to << 2, static_cast<int>(static_cast<uint32_t>(b >> 32)));
    return __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hi) << 32) | lo));
}
__device__ __forceinline__ float lane_f32(float v, int lane) {
    return __int_as_float(__builtin_amdgcn_ds_bpermute(lane << 2, __float_as_int(v)));
}
__device__ __forceinline__ double lane_f64(double v, int lane) {
    const uint64_t b = static_cast<uint64_t>(__double_as_longlong(v));
    const uint32_t lo = __builtin_amdgcn_ds_bpermute(lane << 2, static_cast<int>(static_cast<uint32_t>(b)));
    const uint32_t hi = __builtin_amdgcn_ds_bpermute(lane << 2, static_cast<int>(static_cast<uint32_t>(b >> 32)));
    return __longlong_as_double(static_cast<long long>((static_cast<uint64_t>(hi) << 32) | lo));
}

// Pass 2: evaluates n <= 64 items, one per lane: its row atom with its two
// column atoms, repeating the exact FP64 cutoff test for each. The row's terms
// of both pairs go to the row's LDS accumulators together, column terms pair by
// pair, u and du/dl to per-lane registers. All sums are 64-bit integers.
// image: the slots' coordinates still need the minimum image (they are in one
// frame otherwise). lj: the items may hold Lennard-Jones pairs. tri: only pairs
// with row index < column index count.
// DLDP: instead of du/dp, accumulate d(du/dlambda)/dp into the du_dp slots
// (same fixed-point exponents); only alchemical tiles contribute.
template <bool ALCH, bool U, bool DX, bool DL, bool DP, bool DLDP, int NACC, bool INTERP>
__device__ __forceinline__ void eval_items(TileLds<NACC, INTERP> &L, const uint16_t *items, const int n,
                                           const bool image, const bool lj, const bool tri, const TileSys &B,
                                           const Lane4D &W, uint64_t &uacc, uint64_t &dlacc) {
    constexpr int PQ = DX ? 3 : 0; // first parameter-derivative component
    // interpolated parameters add du/dp . dp/dl to du/dl, so the LJ parameter gradients are needed
    constexpr bool NEED_DP = DP || (INTERP && ALCH && DL);
    const int lane = threadIdx.x & 63;
    const uint32_t ij = ALCH ? items[min(lane, n - 1)] : (lane < n ? items[lane] : 0u);
    const uint32_t il = ij & 0x1F8u;
    const uint32_t sl0 = (ij >> 6) & 0x1F8u;
    double dw[2] = {0.0, 0.0};
    double dwdl_i = 0.0, dwdl_j[2] = {0.0, 0.0};
    if constexpr (ALCH) { // with every lane active
        const int ri = il >> 3, c0 = col_place(sl0 >> 3), c1 = col_place((sl0 + NEXT_COL) >> 3);
        const double wi = lane_f64(W.w[0], ri);
        dw[0] = wi - lane_f64(W.w[1], c0);
        dw[1] = wi - lane_f64(W.w[1], c1);
        if (DL || DLDP) {
            dwdl_i = lane_f32(W.dwdl[0], ri);
            dwdl_j[0] = lane_f32(W.dwdl[1], c0);
            dwdl_j[1] = lane_f32(W.dwdl[1], c1);
        }
    }
    if (lane >= n) {
        return;
    }
    const double2 xyi = at16(L.xy[0], il), zqi = at16(L.zq[0], il);
    const double qi = zqi.y;
    double dx[2], dy[2], dz[2], d2[2], qj[2];
    bool in[2];
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const uint32_t sl = sl0 + NEXT_COL * t;
        const double2 xyj = at16(L.xy[1], sl), zqj = at16(L.zq[1], sl);
        dx[t] = xyi.x - xyj.x;
        dy[t] = xyi.y - xyj.y;
        dz[t] = zqi.x - zqj.x;
        qj[t] = zqj.y;
    }
    if (image) {
#pragma unroll
        for (int t = 0; t < 2; t++) {
            dx[t] = min_image_d(dx[t], B.bx, B.ibx);
            dy[t] = min_image_d(dy[t], B.by, B.iby);
            dz[t] = min_image_d(dz[t], B.bz, B.ibz);
        }
    }
#pragma unroll
    for (int t = 0; t < 2; t++) {
        d2[t] = pair_d2(dx[t], dy[t], dz[t]);
        if (ALCH) {
            d2[t] = __builtin_fma(dw[t], dw[t], d2[t]);
        }
        in[t] = d2[t] < B.cut2;
    }
    if (tri) {
        const uint32_t ri = at4(L.idx[0], il);
        in[0] = in[0] && ri < at4(L.idx[1], sl0);
        in[1] = in[1] && ri < at4(L.idx[1], sl0 + NEXT_COL);
    }
    EsFactors E[2];
    es_factors_n<U || NEED_DP, 2>(d2, B.beta, E);
    PairTerms T[2];
    float2 si = make_float2(0.f, 0.f), sj[2] = {si, si};
#pragma unroll
    for (int t = 0; t < 2; t++) {
        T[t] = nb_es_terms<U>(E[t], qi, qj[t], 1.0);
    }
    if (lj) {
        si = at8(L.se[0], il);
#pragma unroll
        for (int t = 0; t < 2; t++) {
            sj[t] = at8(L.se[1], sl0 + NEXT_COL * t);
            nb_lj_terms<U, NEED_DP>(T[t], si.x, sj[t].x, si.y, sj[t].y, 1.0);
        }
    }
    uint64_t row[NACC]; // the row's terms of both pairs
#pragma unroll
    for (int c = 0; c < NACC; c++) {
        row[c] = 0;
    }
#pragma unroll
    for (int t = 0; t < 2; t++) {
        if (in[t]) {
            const uint32_t sl = sl0 + NEXT_COL * t;
            if (DX) {
                // fixed(prefactor * d) per component, scaled by 2^36 (exact) before the product
                uint64_t fx, fy, fz;
                product3_to_fixed(T[t].prefactor * FIXED_SCALE, B.small, dx[t], dy[t], dz[t], fx, fy, fz);
                lds_sub_u64(&at8(L.acc[1][0], sl), fx);
                lds_sub_u64(&at8(L.acc[1][1], sl), fy);
                lds_sub_u64(&at8(L.acc[1][2], sl), fz);
                row[0] += fx;
                row[1] += fy;
                row[2] += fz;
            }
            if constexpr (DP) {
                row[PQ] += f64_to_fixed(qj[t] * T[t].erfc_inv_d, FIXED_SCALE);
                lds_add_u64(&at8(L.acc[1][PQ + 0], sl), f64_to_fixed(qi * T[t].erfc_inv_d, FIXED_SCALE));
                if (T[t].lj) {
                    const uint64_t gs = f64_to_fixed(T[t].sig_grad, FIXED_SCALE_DSIG);
                    row[PQ + 1] += gs;
                    row[PQ + 2] += f64_to_fixed(T[t].eps_grad * sj[t].y, FIXED_SCALE_DEPS);
                    lds_add_u64(&at8(L.acc[1][PQ + 1], sl), gs);
                    lds_add_u64(&at8(L.acc[1][PQ + 2], sl), f64_to_fixed(T[t].eps_grad * si.y, FIXED_SCALE_DEPS));
                }
            }
            if constexpr (ALCH && (DL || DLDP)) {
                if constexpr (DL) {
                    if constexpr (INTERP) {
                        dlacc += f64_to_fixed(
                            pair_du_dl(T[t], dw[t], dwdl_i, dwdl_j[t], true, 1.0, qi, qj[t], si.y, sj[t].y,
                                       at4(L.dp[0][0], il), at4(L.dp[1][0], sl), at4(L.dp[0][1], il),
                                       at4(L.dp[1][1], sl), at4(L.dp[0][2], il), at4(L.dp[1][2], sl)),
                            FIXED_SCALE);
                    } else {
                        dlacc += f64_to_fixed(dw[t] * T[t].prefactor * (dwdl_i - dwdl_j[t]), FIXED_SCALE);
                    }
                }
                if constexpr (DLDP) {
                    const PairDlDp D = nb_pair_dl_dp(d2[t], si.x, sj[t].x, si.y, sj[t].y, B.beta, 1.0);
                    const double dd = dw[t] * (dwdl_i - dwdl_j[t]);
                    row[PQ] += f64_to_fixed((qj[t] * D.es_unit) * dd, FIXED_SCALE);
                    lds_add_u64(&at8(L.acc[1][PQ + 0], sl), f64_to_fixed((qi * D.es_unit) * dd, FIXED_SCALE));
                    if (D.lj) {
                        const uint64_t gs = f64_to_fixed(D.lj_dsig * dd, FIXED_SCALE_DSIG);
                        row[PQ + 1] += gs;
                        row[PQ + 2] += f64_to_fixed((D.lj_unit * static_cast<double>(sj[t].y)) * dd, FIXED_SCALE_DEPS);
                        lds_add_u64(&at8(L.acc[1][PQ + 1], sl), gs);
                        lds_add_u64(&at8(L.acc[1][PQ + 2], sl),
                                    f64_to_fixed((D.lj_unit * static_cast<double>(si.y)) * dd, FIXED_SCALE_DEPS));
                    }
                }
            }
            if (U) {
                uacc += f64_to_fixed(T[t].u, FIXED_SCALE);
            }
        }
    }
    if constexpr (DX || DP || DLDP) {
#pragma unroll
        for (int c = 0; c < NACC; c++) {
            lds_add_u64(&at8(L.acc[0][c], il), row[c]);
        }
    }
}

// Row atoms of a run of tiles, per lane: [own] of slot r * 64 + lane, [at slot]
// of the atom in LDS row slot `lane`.
struct RowRegs {
    int index;      // own: its LDS index
    float x, y, z;  // at slot: FP32 position relative to the row block's centre (x NaN for padding)
    float ca[4];    // (screen radius^2 - |a|^2) / 2 of the four row slots 4 (lane / 4) + k
    float cut2;     // squared radius of the imaged screen
    bool image;     // the block is too wide for one frame (small boxes)
    int lj;         // Lennard-Jones rows
    bool moving;    // some row has a 4D coordinate or a parameter that depends on lambda
};

typedef float Vec4f __attribute__((ext_vector_type(4)));

// Where the force and parameter derivative sums go. The rate of device-scope
// 64-bit atomics depends on their addresses: 64 lanes at random atoms of a
// [N, 3] array make 20 G adds/s (MI355X, 6400 atoms), 64 lanes on runs of eight
// or more neighbouring words 120 to 150 G/s. A tile ends with 64 x 3 adds for
// its columns and, once per row run, for its rows; at the random rate they took
// longer than the pairs (38 us for the 800k adds of one system of 6k atoms). So tiles add
// to words in sorted order, sorted[component][slot], and k_add_sorted moves the
// sums to the atoms. Without that scratch (views) they go to the atoms directly.
struct TileOut {
    uint64_t *sorted; // [6][slots]: x, y, z, q, sig, eps; or nullptr
    size_t slots;
    const uint32_t *perm;
};

struct OutAtom {
    uint64_t *dx, *dp;
    size_t step;
    __device__ __forceinline__ OutAtom(const TileOut &O, const NbSys &S, int slot, uint64_t *du_dx, uint64_t *du_dp) {
        const size_t at = static_cast<size_t>(S.slot0) + slot;
        if (O.sorted) {
            dx = O.sorted + at;
            dp = dx + 3 * O.slots;
            step = O.slots;
        } else {
            const size_t atom = static_cast<size_t>(S.atom0) + O.perm[at];
            dx = du_dx + atom * 3;
            dp = du_dp + atom * 3;
            step = 1;
        }
    }
    // component c of the accumulators: forces first if there are any (DX), then parameters
    template <bool DX> __device__ __forceinline__ void add(int c, uint64_t v) const {
        if (v != 0) {
            atomic_add_u64(DX ? (c < 3 ? dx + c * step : dp + (c - 3) * step) : dp + c * step, v);
        }
    }
};

// (row, column pair) items of one step from the hit masks m0 and m1 of two row
// places of every 4 x 4 block (bit 4 b + j: the row of block b with its column
// j). Bit 4 b + 2 p of the result is m0's item of block b and column pair p,
// bit 4 b + 2 p + 1 is m1's item of block b xor 8 and pair p: items that share
// their columns end up apart, so that the lanes that take them in pass 2 do not
// add to one LDS word.
__device__ __forceinline__ uint64_t item_mask(uint64_t m0, uint64_t m1) {
    const uint64_t p0 = (m0 | (m0 >> 1)) & 0x5555555555555555ull;
    const uint64_t p1 = (m1 | (m1 << 1)) & 0xAAAAAAAAAAAAAAAAull;
    const uint32_t lo = static_cast<uint32_t>(p0) | static_cast<uint32_t>(p1 >> 32);
    const uint32_t hi = static_cast<uint32_t>(p0 >> 32) | static_cast<uint32_t>(p1);
    return (static_cast<uint64_t>(hi) << 32) | lo;
}

// One 64 x 64 tile on one wave, rows staged (RowRegs, LDS).
//
// Pass 1 finds the pairs inside the cutoff in FP32 and queues them in LDS as
// items; whenever 64 items wait, pass 2 evaluates them. Fixed-point sums are
// exact, so the order of evaluation does not change any output bit.
//
// The frame. Coordinates are multiples of the box's grid step (BoxAxis), so
// adding a box edge and subtracting two of them is exact whatever the image.
// Every atom is imaged once next to the centre c of the row block. If every
// row atom is within e of c and e + cutoff < L / 2 on every axis, a pair within
// the cutoff has a_i - a_j equal to its minimum-image displacement: any other
// image differs by a multiple of L, so |a_j - a_i| >= L - cutoff > L / 2 + e,
// which a_j - a_i cannot reach; pass 2 then needs no image (9 of ~75
// instructions a pair). c and e come from the block's bounding box of the last
// neighborlist build (block_bounds, FP32): since then the box is unchanged
// and no atom has moved more than padding / 2, so every row atom is within the
// box's half-extent + padding / 2 of its centre, plus 1e-4 nm for the FP32
// rounding of the build. Otherwise ("image", boxes under ~3.4 nm) the screen
// and pass 2 image the difference.
//
// The screen takes 16 steps of 256 pairs (this wave's share of them: k0 to k1);
// step k pairs the row slots of block b
// (4 b .. 4 b + 3) with the column slots of block b xor k. With a, b relative
// to c,
//   |a - b|^2 < R^2  <=>  (R^2 - |a|^2) / 2 + a . b > |b|^2 / 2,
// a 64 x 64 x 3 product: three v_mfma_f32_4x4x1 (16 blocks of 4 x 4) and four
// compares a step, ~17 vector instructions for 256 pairs with the queueing
// where a rotating FP32 screen took 68. FP32 error of the test: 23 roundings of
// 2^-24 R'^2 at most, R' bounding |a| and |b| (block half-diagonal + cutoff);
// R^2 = cutoff^2 (1 + 1e-5) + 2^-19 R'^2. With "image" the nearer of the two
// images per axis is taken pair by pair: both atoms lie in [-L/2, L/2], so
// t = a_j - a_i has |t| <= L and its nearest image at min(|t|, L - |t|); margin
// 1e-4. The 4D coordinate only adds to the distance and is left to pass 2.
//
// What bounds pass 2 is vector issue and LDS (gathers and 64-bit adds; lanes of a
// group of 16 that add to one word take 2 cycles each) together: an item of one
// row and two neighbouring columns shares the row's loads, adds its row terms
// once and gives the lane two independent chains of FP64 arithmetic. Per force
// evaluation with k_add_sorted, against one pair a lane behind a rotating screen,
// accumulators of 12 KB (12 waves a CU) and adds to the atoms: 192 systems of
// 6372 atoms 2.56 -> 2.37 ms (5.7 ns a tile), 24 of 34.5k 1.75 -> 1.58 ms, one
// system of 34.5k 146 -> 107 us, of 6.4k 45 -> 37 us, of 1k 32 -> 13 us.
//
// Lennard-Jones atoms take the first row slots in the order k, 16 blocks each,
// so that with at most 32 of them the second queue (row places 2 and 3) holds
// no Lennard-Jones pair.
template <bool ALCH, bool U, bool DX, bool DL, bool DP, bool DLDP, int NACC, bool INTERP>
__device__ __forceinline__ void tile_body(
    TileLds<NACC, INTERP> &L, const NbSys &S, const TileSys &B, const int r, const uint32_t jl0, double4 pj,
    const float4 aj, const float4 dpj, const float4 bc, const RowRegs &R, const bool row_flush, const int k0, const int k1,
    const TileOut &O, const double4 *__restrict__ pos0, const float4 *__restrict__ par0, uint64_t &uacc,
    uint64_t &dlacc, uint64_t *__restrict__ du_dx, uint64_t *__restrict__ du_dp) {
    constexpr int PQ = DX ? 3 : 0;
    const int lane = threadIdx.x & 63;
    const bool vj = jl0 < static_cast<uint32_t>(S.slot_end); // column slots (NB_INVALID pads) are below this
    const float nan = __builtin_nanf("");
    // padding columns are NaN: they fail every comparison of the screen and of pass 2
    const float qx = vj ? static_cast<float>(min_image_d(pj.x - bc.x, B.bx, B.ibx)) : nan;
    const float qy = static_cast<float>(min_image_d(pj.y - bc.y, B.by, B.iby));
    const float qz = static_cast<float>(min_image_d(pj.z - bc.z, B.bz, B.ibz));
    if (!R.image) {
        pj.x = to_frame(pj.x, bc.x, B.bx, B.ibx);
        pj.y = to_frame(pj.y, bc.y, B.by, B.iby);
        pj.z = to_frame(pj.z, bc.z, B.bz, B.ibz);
    }
    if (!vj) {
        pj.x = __builtin_nan("");
    }
    // columns of the row's own block need i < j (upper triangle); later blocks always pass
    const bool tri = ballot(vj && jl0 < static_cast<uint32_t>((r + 1) * TILE)) != 0;
    const bool lj_cols = ballot(aj.z != 0.f) != 0;
    const bool lj0 = INTERP || (R.lj > 0 && lj_cols), lj1 = INTERP || (R.lj > 32 && lj_cols);
    wave_lds_sync(); // the previous tile's LDS reads are complete
    const int col = col_index(lane); // LDS index of the own column (screen place `lane`)
    L.xy[1][col] = make_double2(pj.x, pj.y);
    L.zq[1][col] = make_double2(pj.z, aj.x);
    L.se[1][col] = make_float2(aj.y, aj.z);
    L.col[lane] = make_float4(qx, qy, qz, 0.5f * __builtin_fmaf(qx, qx, __builtin_fmaf(qy, qy, qz * qz)));
    if (tri) {
        L.idx[1][col] = vj ? jl0 : NB_INVALID;
    }
    if constexpr (INTERP) {
        L.dp[1][0][col] = dpj.x;
        L.dp[1][1][col] = dpj.y;
        L.dp[1][2][col] = dpj.z;
    }
#pragma unroll
    for (int c = 0; c < NACC; c++) {
        L.acc[1][c][lane] = 0;
    }
    wave_lds_sync();

    Lane4D W = {};
    if constexpr (ALCH) { // (the row's block is padded to 64 slots)
        W.w[0] = push_f64(pos0[r * TILE + lane].w, R.index);
        W.w[1] = pj.w;
        W.dwdl[0] = push_f32(par0[r * TILE + lane].w, R.index);
        W.dwdl[1] = aj.w;
    }
    // the item that lane 4 b + t queues (item_mask), before the step's column block
    const int ib = (lane >> 2) ^ ((lane & 1) << 3);
    const uint32_t self = (static_cast<uint32_t>(((lane & 1) << 4) + ib) << 3) |
                          (static_cast<uint32_t>(((lane & 2) << 4) + (ib ^ ((lane & 2) << 1))) << 9);
    const Vec4f ca = {R.ca[0], R.ca[1], R.ca[2], R.ca[3]};
    const float lx = uniform_f(static_cast<float>(B.bx)), ly = uniform_f(static_cast<float>(B.by)),
                lz = uniform_f(static_cast<float>(B.bz));
    int queued0 = 0, queued1 = 0; // items waiting in each queue (wave-uniform)
    float4 cb = L.col[lane ^ (k0 << 2)];
    for (int k = k0; k <= k1; k++) {
        if (k < k1) {
            uint64_t m[4];
            if (!R.image) {
                Vec4f t = __builtin_amdgcn_mfma_f32_4x4x1f32(R.x, cb.x, ca, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_4x4x1f32(R.y, cb.y, t, 0, 0, 0);
                t = __builtin_amdgcn_mfma_f32_4x4x1f32(R.z, cb.z, t, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    m[v] = ballot(t[v] > cb.w);
                }
            } else {
                auto near = [&](float ax, float ay, float az) {
                    float dx = cb.x - ax, dy = cb.y - ay, dz = cb.z - az;
                    dx = __builtin_fminf(__builtin_fabsf(dx), lx - __builtin_fabsf(dx));
                    dy = __builtin_fminf(__builtin_fabsf(dy), ly - __builtin_fabsf(dy));
                    dz = __builtin_fminf(__builtin_fabsf(dz), lz - __builtin_fabsf(dz));
                    // NaN (padding) must survive: fmin drops it from one operand only, and both are NaN
                    return ballot(__builtin_fmaf(dx, dx, __builtin_fmaf(dy, dy, dz * dz)) < R.cut2);
                };
                m[0] = near(quad_bcast<0>(R.x), quad_bcast<0>(R.y), quad_bcast<0>(R.z));
                m[1] = near(quad_bcast<1>(R.x), quad_bcast<1>(R.y), quad_bcast<1>(R.z));
                m[2] = near(quad_bcast<2>(R.x), quad_bcast<2>(R.y), quad_bcast<2>(R.z));
                m[3] = near(quad_bcast<3>(R.x), quad_bcast<3>(R.y), quad_bcast<3>(R.z));
            }
            cb = L.col[lane ^ (((k + 1) & 15) << 2)]; // the next step's columns
            const uint32_t item = self ^ (static_cast<uint32_t>(k) << 9);
            auto push = [&](uint64_t im, uint16_t *queue, int &queued, uint32_t it) {
                if (in_mask(im)) {
                    queue[mbcnt(im, 0) + queued] = static_cast<uint16_t>(it);
                }
                queued += __popcll(im);
            };
            push(item_mask(m[0], m[1]), L.pq[0], queued0, item);
            push(item_mask(m[2], m[3]), L.pq[1], queued1, item + 256u);
        }
        if (k == k1) {
            // the second queue's rest goes on top of the first's
            wave_lds_sync();
            const uint16_t rest = L.pq[1][lane];
            wave_lds_sync();
            if (lane < queued1) {
                L.pq[0][queued0 + lane] = rest;
            }
            queued0 += queued1;
            queued1 = 0;
        }
        // pass 2 from the top of a queue; after the last step whatever is left
        const int least = k < k1 ? TILE : 1;
        while (max(queued0, queued1) >= least) {
            const bool second = queued1 >= least;
            const int waiting = second ? queued1 : queued0;
            const int n = min(waiting, TILE);
            const int from = waiting - n;
            queued0 = second ? queued0 : from;
            queued1 = second ? from : queued1;
            wave_lds_sync();
            eval_items<ALCH, U, DX, DL, DP, DLDP, NACC, INTERP>(L, L.pq[0] + (second ? ITEM_QUEUE : 0) + from, n, R.image,
                                                                second ? lj1 : lj0, tri, B, W, uacc,
                                                                dlacc);
            wave_lds_sync();
        }
    }
    wave_lds_sync();

    if (DX || DP || DLDP) {
        // atomics of neighbouring lanes on neighbouring words travel together
        // (TileOut), so both sides are written in slot order
        const int i = r * TILE + lane;
        if (row_flush && i < S.row_end) {
            const OutAtom o(O, S, i, du_dx, du_dp);
#pragma unroll
            for (int c = 0; c < NACC; c++) {
                o.add<DX>(c, L.acc[0][c][R.index]);
            }
        }
        if (vj) {
            const OutAtom o(O, S, static_cast<int>(jl0), du_dx, du_dp);
#pragma unroll
            for (int c = 0; c < NACC; c++) {
                o.add<DX>(c, L.acc[1][c][col]);
            }
        }
    }
}

// Adds a wave's u and du/dl of system s to the outputs. Device-scope atomics on
// one address take ~10 ns each, one after the other, whoever issues them: the
// 2100 waves of a 6k-atom system kept u and du/dl busy for 21 us. So the waves
// w0 .. w1 that work on the system add to NB_RED_SLOTS partial sums in lines of
// their own, and the last wave of each slot moves its sum to the output and clears
// the slot for the next launch. Up to RED_DIRECT waves the output's queue is
// shorter than the two more round trips of a slot. Measured: 48 evaluations of u
// and du/dl at 4.2k atoms 3.52 -> 3.00 ms, all outputs of 6k atoms with interpolated
// parameters 339 -> 308 us a call.
//
// The order of a wave's sums and its count. The atomics are relaxed, which in the
// language's memory model leaves them unordered; what orders them is this
// hardware. An agent-scope atomic that returns a value returns it from the place
// where all agent-scope atomics on that line meet (a slot is one 128-byte line), so
// a sum whose old value has come back is there, and the count is issued after that
// (it depends on the value). Whoever reads the slot's last count therefore finds
// every sum with an atomic of its own. A release on the count and an acquire by the
// last wave say the same in the language, but the release writes the whole L2 back,
// once a wave: 48 evaluations 2.91 -> 3.71 ms, 30 steps of one 6k system 3.52 -> 4.60
// ms, u and du/dl at 1k atoms 111 -> 155 us a call.
constexpr int RED_DIRECT = 256;

template <bool U, bool DL>
__device__ __forceinline__ void add_scalars(NbRedSlot *slots, const int w, const int w0, const int w1, uint64_t uacc,
                                            uint64_t dlacc, uint64_t *u, uint64_t *dl) {
    const int lane = threadIdx.x & 63;
    const uint64_t ut = U ? wave_sum_u64(uacc) : 0, dt = DL ? wave_sum_u64(dlacc) : 0;
    // lane 0 carries u, lane 1 du/dl
    const bool mine = (U && lane == 0) || (DL && lane == 1);
    uint64_t v = lane == 0 ? ut : dt;
    uint64_t *out = lane == 0 ? u : dl;
    const int n = w1 - w0 + 1;
    if (slots && n > RED_DIRECT) {
        const int j = (w - w0) & (NB_RED_SLOTS - 1);
        const uint32_t expect = static_cast<uint32_t>((n - 1 - j) / NB_RED_SLOTS + 1); // waves of slot j
        NbRedSlot *slot = slots + j;
        uint32_t one = 1;
        if (lane < 2) {
            const uint64_t old = __hip_atomic_fetch_add(slot->v + lane, mine ? v : 0, __ATOMIC_RELAXED,
                                                        __HIP_MEMORY_SCOPE_AGENT);
            // 1, from the value that came back: the sum is in memory before this wave counts
            asm volatile("v_and_b32 %0, 0, %1\n\tv_or_b32 %0, 1, %0" : "=&v"(one) : "v"(static_cast<uint32_t>(old)));
        }
        uint32_t before = 0;
        if (lane == 0) {
            before = __hip_atomic_fetch_add(&slot->waves, one, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (__builtin_amdgcn_readfirstlane(before) + 1 != expect) {
            return;
        }
        if (lane < 2) { // every wave of the slot has added its sums
            v = __hip_atomic_exchange(slot->v + lane, uint64_t(0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (lane == 0) {
            __hip_atomic_store(&slot->waves, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if (mine && v != 0) {
        atomic_add_u64(out, v);
    }
}

// log2 of the waves that share a tile. Few tiles leave most of the GPU's wave
// slots empty while each wave works through a whole tile; but every share stages
// its row and column atoms and writes both again. Kernel with k_add_sorted, us,
// whole / halves / quarters / eighths: 153 tiles (1k atoms) 31 / - / - / 13, 801 tiles
// - / 28 / 22 / 29, 2145 tiles (6k atoms) 48 / 37 / 40 / 56, 4056 tiles 57 / 51 / 62,
// 8556 tiles 91 / 86, 11304 tiles (35k atoms) 107 whole. The lines are tile counts for
// 256 CUs of 16 waves; results do not depend on them.
__device__ __forceinline__ int tile_split(int tiles) {
    return tiles <= 576 ? 3 : tiles <= 1152 ? 2 : tiles <= 9216 ? 1 : 0;
}

// Every wave takes a contiguous range of the tile list of all systems (the
// grid is sized to the machine, the tile count is read on the device).
// WAVES_PER_SIMD = 4 (the default build): at most 128 VGPRs, so four waves
// share a SIMD; 3 and 2 let the compiler use up to 168 and 256 VGPRs with
// fewer waves to hide latency. The engine's instances exist in all three forms
// and the autotuner picks one (NbState::tile_waves).
template <bool U, bool DX, bool DL, bool DP, bool DLDP = false, bool INTERP = false, int WAVES_PER_SIMD = 4>
__global__ __launch_bounds__(NB_BLOCK) __attribute__((amdgpu_waves_per_eu(WAVES_PER_SIMD))) void k_nonbonded_tiles(
    const NbSys *__restrict__ sys,
    const int S,
    const int *__restrict__ tile_prefix,
    const int *__restrict__ tile_order,
    const int *__restrict__ tile_row,
    const uint32_t *__restrict__ tile_atoms,
    const uint32_t *__restrict__ perm,
    const double4 *__restrict__ pos,
    const float4 *__restrict__ par,
    const float4 *__restrict__ dpar,
    const double *__restrict__ boxes,
    const float4 *__restrict__ bb_ctr,
    const float4 *__restrict__ bb_ext,
    const int *__restrict__ status,
    uint64_t *__restrict__ sorted,
    const int slots,
    NbRedSlot *__restrict__ red,
    uint64_t *__restrict__ du_dx,
    uint64_t *__restrict__ du_dp,
    uint64_t *__restrict__ du_dl,
    uint64_t *__restrict__ u) {
    constexpr int NACC = (DX ? 3 : 0) + ((DP || DLDP) ? 3 : 0) > 0 ? (DX ? 3 : 0) + ((DP || DLDP) ? 3 : 0) : 1;
    __shared__ TileLds<NACC, INTERP> L;
    const int lane = threadIdx.x & 63;
    const TileOut O = {sorted, static_cast<size_t>(slots), perm};
    // Each wave takes a contiguous range of the tile list. Tiles of a system
    // are listed grouped by row block (tile_order), so consecutive tiles of a
    // wave mostly share their row atoms: the rows are staged once per such run,
    // and their accumulators stay in LDS over it and go out with one set of
    // global atomics at its end instead of one per tile (device-scope 64-bit
    // atomics are the costly part of a tile's output). The d(du/dlambda)/dp
    // kernel, which skips tiles, writes per tile.
    const int w = uniform(blockIdx.x);
    const int total = tile_prefix[S];
    const int lp = tile_split(total);
    const int units = total << lp;
    const int chunk = (units + static_cast<int>(gridDim.x) - 1) / static_cast<int>(gridDim.x);
    int unit = w * chunk;
    const int unit_end = min(units, unit + chunk);
    if (unit >= unit_end) {
        return;
    }
    int t = unit >> lp;
    int s = 0;
    {
        int lo = 0, hi = S - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (tile_prefix[mid] <= t) {
                lo = mid;
            } else {
                hi = mid - 1;
            }
        }
        s = lo;
    }
    bool open = false; // the row accumulators hold a run that is not written yet
    int have = -1;     // the system B describes
    TileSys B = {};
    RowRegs R = {};
    float4 bc = make_float4(0.f, 0.f, 0.f, 0.f);
    // u and du/dl of the system's tiles so far (per lane); written with one
    // wave-reduced atomic per system and wave, not per tile (every tile of a
    // system adds to the same word)
    uint64_t uacc = 0, dlacc = 0;
    for (; unit < unit_end; unit++) {
        t = unit >> lp;
        const int k0 = (unit & ((1 << lp) - 1)) << (4 - lp);
        const int k1 = k0 + (16 >> lp);
        while (tile_prefix[s + 1] <= t) {
            s++; // tile_prefix[S] = total > t
        }
        if (status[s] & NB_BAD_BOX) {
            continue;
        }
        const NbSys &Sd = sys[s];
        if (have != s) {
            have = s;
            const BoxAxis gx(boxes[s * 9 + 0]), gy(boxes[s * 9 + 4]), gz(boxes[s * 9 + 8]);
            B.bx = uniform_d(gx.edge);
            B.by = uniform_d(gy.edge);
            B.bz = uniform_d(gz.edge);
            B.ibx = uniform_d(gx.inv);
            B.iby = uniform_d(gy.inv);
            B.ibz = uniform_d(gz.inv);
            B.cut2 = uniform_d(Sd.cutoff_d * Sd.cutoff_d);
            B.small = uniform_d(fixed_small_factor(Sd.cutoff_d));
            B.beta = uniform_d(static_cast<double>(Sd.beta));
        }
        const int local = t - tile_prefix[s];
        const int kt = Sd.tile0 + tile_order[Sd.tile0 + local];
        const int r = tile_row[kt];
        bool last = true; // the next tile of this wave has another row (or system)
        if (!DLDP && lp == 0 && unit + 1 < unit_end && t + 1 < tile_prefix[s + 1]) {
            last = tile_row[Sd.tile0 + tile_order[Sd.tile0 + local + 1]] != r;
        }
        const bool fresh = !open;
        open = !last;
        const bool sys_last = unit + 1 >= unit_end || ((unit + 1) >> lp) >= tile_prefix[s + 1];
        const uint32_t jl = tile_atoms[static_cast<size_t>(kt) * TILE + lane];
        const bool vj = jl < static_cast<uint32_t>(Sd.slot_end);
        const double4 pj = vj ? pos[Sd.slot0 + jl] : make_double4(0.0, 0.0, 0.0, 0.0);
        const float4 aj = vj ? par[Sd.slot0 + jl] : make_float4(0.f, 0.f, 0.f, 0.f);
        float4 dpj = make_float4(0.f, 0.f, 0.f, 0.f);
        if (fresh) {
            // stage the row block: LDS slots (Lennard-Jones atoms first) and, per
            // lane, the screen's view of the atom in slot `lane`
            const int i = r * TILE + lane;
            const bool vi = i < Sd.row_end;
            double4 pi = pos[Sd.slot0 + i];
            const float4 ai = par[Sd.slot0 + i];
            bc = bb_ctr[Sd.block0 + r];
            const float4 be = bb_ext[Sd.block0 + r];
            const double slack = 0.5 * Sd.padding_d + 1e-4;
            const double reach = Sd.cutoff_d + 1e-3; // 1e-3 nm covers the FP32 extents
            const bool one_frame = static_cast<double>(be.x) + slack + reach < 0.5 * B.bx &&
                                   static_cast<double>(be.y) + slack + reach < 0.5 * B.by &&
                                   static_cast<double>(be.z) + slack + reach < 0.5 * B.bz;
            R.image = !one_frame;
            const float fx = static_cast<float>(min_image_d(pi.x - bc.x, B.bx, B.ibx));
            const float fy = static_cast<float>(min_image_d(pi.y - bc.y, B.by, B.iby));
            const float fz = static_cast<float>(min_image_d(pi.z - bc.z, B.bz, B.ibz));
            if (one_frame) {
                pi.x = to_frame(pi.x, bc.x, B.bx, B.ibx);
                pi.y = to_frame(pi.y, bc.y, B.by, B.iby);
                pi.z = to_frame(pi.z, bc.z, B.bz, B.ibz);
            }
            const uint64_t m = ballot(vi && ai.z != 0.f);
            R.lj = __popcll(m);
            const int below = lanes_below(m);
            const int place = (vi && ai.z != 0.f) ? below : R.lj + lane - below;
            R.index = place;
            const int slot = ((place & 15) << 2) | (place >> 4); // row_index(slot) = place
            const float fs = static_cast<float>(slack), fr = static_cast<float>(reach);
            const float half_diag =
                __builtin_sqrtf(__builtin_fmaf(be.x + fs, be.x + fs,
                                               __builtin_fmaf(be.y + fs, be.y + fs, (be.z + fs) * (be.z + fs))));
            const float radius = half_diag + fr;
            const float cut2 = static_cast<float>(B.cut2);
            R.cut2 = cut2 * (1.0f + 1e-4f);
            const float mat2 = __builtin_fmaf(0x1p-19f * radius, radius, cut2 * (1.0f + 1e-5f));
            wave_lds_sync(); // the previous run's LDS reads are complete
            L.xy[0][R.index] = make_double2(pi.x, pi.y);
            L.zq[0][R.index] = make_double2(pi.z, ai.x);
            L.se[0][R.index] = make_float2(ai.y, ai.z);
            L.idx[0][R.index] = vi ? static_cast<uint32_t>(i) : NB_INVALID;
            // padding rows are NaN: they fail every comparison of the screen
            L.col[slot] = make_float4(vi ? fx : __builtin_nanf(""), fy, fz,
                                        0.5f * (mat2 - __builtin_fmaf(fx, fx, __builtin_fmaf(fy, fy, fz * fz))));
            bool moves = pi.w != 0.0;
            if (INTERP && Sd.interp) {
                const float4 dpi = dpar[Sd.slot0 + i];
                moves = moves || dpi.x != 0.f || dpi.y != 0.f || dpi.z != 0.f;
                if constexpr (INTERP) {
                    L.dp[0][0][R.index] = dpi.x;
                    L.dp[0][1][R.index] = dpi.y;
                    L.dp[0][2][R.index] = dpi.z;
                }
            } else if constexpr (INTERP) {
                L.dp[0][0][R.index] = 0.f;
                L.dp[0][1][R.index] = 0.f;
                L.dp[0][2][R.index] = 0.f;
            }
            R.moving = ballot(moves) != 0;
#pragma unroll
            for (int c = 0; c < NACC; c++) {
                L.acc[0][c][lane] = 0;
            }
            wave_lds_sync();
            const float4 own = L.col[lane];
            R.x = own.x;
            R.y = own.y;
            R.z = own.z;
#pragma unroll
            for (int c = 0; c < 4; c++) {
                R.ca[c] = L.col[(lane & ~3) + c].w;
            }
        }
        bool moving = pj.w != 0.0;
        if (INTERP && Sd.interp) {
            if (vj) {
                dpj = dpar[Sd.slot0 + jl];
            }
            moving = moving || dpj.x != 0.f || dpj.y != 0.f || dpj.z != 0.f;
        }
        // "vanilla" tiles (no lambda dependence, k_nonbonded.cuh:626-630) skip the 4D terms
        const bool alch = R.moving || ballot(moving) != 0;
        if (alch) {
            tile_body<true, U, DX, DL, DP, DLDP, NACC, INTERP>(L, Sd, B, r, jl, pj, aj, dpj, bc, R, last, k0, k1, O,
                                                               pos + Sd.slot0, par + Sd.slot0, uacc, dlacc, du_dx, du_dp);
        } else if (!DLDP) {
            tile_body<false, U, DX, DL, DP, false, NACC, INTERP>(L, Sd, B, r, jl, pj, aj, dpj, bc, R, last, k0, k1, O,
                                                                 pos + Sd.slot0, par + Sd.slot0, uacc, dlacc, du_dx, du_dp);
        }
        if (sys_last && (U || DL)) {
            const int w0 = (tile_prefix[s] << lp) / chunk, w1 = ((tile_prefix[s + 1] << lp) - 1) / chunk;
            add_scalars<U, DL>(red ? red + s * NB_RED_SLOTS : nullptr, w, w0, w1, uacc, dlacc, u + Sd.red_idx,
                               du_dl + Sd.red_idx);
            uacc = 0;
            dlacc = 0;
        }
    }
}

// Moves the tiles' sums from sorted order to the atoms and clears them for the
// next launch; one thread per slot. Atomic: other streams may add to the outputs.
template <bool DX, bool DP>
__global__ __launch_bounds__(256) void k_add_sorted(const NbSys *__restrict__ sys, const uint32_t *__restrict__ perm,
                                                    const int slots, uint64_t *__restrict__ sorted,
                                                    uint64_t *__restrict__ du_dx, uint64_t *__restrict__ du_dp) {
    const NbSys &S = sys[blockIdx.x];
    const int i = blockIdx.y * 256 + threadIdx.x;
    if (i >= S.nblocks * TILE) {
        return;
    }
    const size_t at = static_cast<size_t>(S.slot0) + i;
    uint64_t v[6];
    bool any = false;
#pragma unroll
    for (int c = DX ? 0 : 3; c < (DP ? 6 : 3); c++) {
        v[c] = sorted[c * static_cast<size_t>(slots) + at];
        any = any || v[c] != 0;
    }
    if (!any) { // padding slots among them
        return;
    }
    const size_t atom = static_cast<size_t>(S.atom0) + perm[at];
#pragma unroll
    for (int c = DX ? 0 : 3; c < (DP ? 6 : 3); c++) {
        if (v[c] != 0) {
            sorted[c * static_cast<size_t>(slots) + at] = 0;
            atomic_add_u64((c < 3 ? du_dx : du_dp) + atom * 3 + c % 3, v[c]);
        }
    }
}

using TileKernel = void (*)(const NbSys *, int, const int *, const int *, const int *, const uint32_t *, const uint32_t *,
                            const double4 *, const float4 *, const float4 *, const double *, const float4 *,
                            const float4 *, const int *, uint64_t *, int, NbRedSlot *, uint64_t *, uint64_t *, uint64_t *, uint64_t *);

// index bits: 8 = u, 4 = du_dx, 2 = du_dl, 1 = du_dp
const TileKernel tile_kernels[16] = {
    k_nonbonded_tiles<0, 0, 0, 0>, k_nonbonded_tiles<0, 0, 0, 1>, k_nonbonded_tiles<0, 0, 1, 0>,
    k_nonbonded_tiles<0, 0, 1, 1>, k_nonbonded_tiles<0, 1, 0, 0>, k_nonbonded_tiles<0, 1, 0, 1>,
    k_nonbonded_tiles<0, 1, 1, 0>, k_nonbonded_tiles<0, 1, 1, 1>, k_nonbonded_tiles<1, 0, 0, 0>,
    k_nonbonded_tiles<1, 0, 0, 1>, k_nonbonded_tiles<1, 0, 1, 0>, k_nonbonded_tiles<1, 0, 1, 1>,
    k_nonbonded_tiles<1, 1, 0, 0>, k_nonbonded_tiles<1, 1, 0, 1>, k_nonbonded_tiles<1, 1, 1, 0>,
    k_nonbonded_tiles<1, 1, 1, 1>,
};

// interpolated parameters: only the outputs that see dp/dl (du_dl) differ, but
// the whole table is instantiated for uniform dispatch
const TileKernel tile_kernels_interp[16] = {
    k_nonbonded_tiles<0, 0, 0, 0, 0, 1>, k_nonbonded_tiles<0, 0, 0, 1, 0, 1>, k_nonbonded_tiles<0, 0, 1, 0, 0, 1>,
    k_nonbonded_tiles<0, 0, 1, 1, 0, 1>, k_nonbonded_tiles<0, 1, 0, 0, 0, 1>, k_nonbonded_tiles<0, 1, 0, 1, 0, 1>,
    k_nonbonded_tiles<0, 1, 1, 0, 0, 1>, k_nonbonded_tiles<0, 1, 1, 1, 0, 1>, k_nonbonded_tiles<1, 0, 0, 0, 0, 1>,
    k_nonbonded_tiles<1, 0, 0, 1, 0, 1>, k_nonbonded_tiles<1, 0, 1, 0, 0, 1>, k_nonbonded_tiles<1, 0, 1, 1, 0, 1>,
    k_nonbonded_tiles<1, 1, 0, 0, 0, 1>, k_nonbonded_tiles<1, 1, 0, 1, 0, 1>, k_nonbonded_tiles<1, 1, 1, 0, 0, 1>,
    k_nonbonded_tiles<1, 1, 1, 1, 0, 1>,
};

// The pair kernel for output set idx (bits as above) at the given waves per
// SIMD: the instances the MD engine launches (du_dx, du_dx + du_dl, u + du_dx,
// u + du_dx + du_dl, plain parameters) exist at 4, 3 and 2; everything else
// only at 4.
TileKernel tile_kernel(const int idx, const bool interp, const int waves) {
    if (!interp && waves == 3) {
        switch (idx) {
        case 4: return k_nonbonded_tiles<0, 1, 0, 0, false, false, 3>;
        case 6: return k_nonbonded_tiles<0, 1, 1, 0, false, false, 3>;
        case 12: return k_nonbonded_tiles<1, 1, 0, 0, false, false, 3>;
        case 14: return k_nonbonded_tiles<1, 1, 1, 0, false, false, 3>;
        default: break;
        }
    }
    if (!interp && waves == 2) {
        switch (idx) {
        case 4: return k_nonbonded_tiles<0, 1, 0, 0, false, false, 2>;
        case 6: return k_nonbonded_tiles<0, 1, 1, 0, false, false, 2>;
        case 12: return k_nonbonded_tiles<1, 1, 0, 0, false, false, 2>;
        case 14: return k_nonbonded_tiles<1, 1, 1, 0, false, false, 2>;
        default: break;
        }
    }
    return interp ? tile_kernels_interp[idx] : tile_kernels[idx];
}

template <bool U, bool DX, bool DL, bool DP, bool DLDP = false>
__global__ __launch_bounds__(256) void k_pair_list(
    const PairListArgs a, uint64_t *__restrict__ du_dx, uint64_t *__restrict__ du_dp, uint64_t *__restrict__ du_dl,
    uint64_t *__restrict__ u) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    const bool neg = a.negated != 0;
    int red = -1;
    uint64_t fu = 0, fdl = 0; // this lane's u and du/dl terms (reduced over the wave below)
    if (p < a.M) {
        const int s = a.pair_sys ? a.pair_sys[p] : 0;
        const int gi = a.pairs[p * 2 + 0];
        const int gj = a.pairs[p * 2 + 1];
        const double *box = a.boxes + s * 9;
        const double lam = a.lambdas ? a.lambdas[s] : a.lambda0;
        const double cutoff_d = a.cutoffs ? a.cutoffs[s] : a.cutoff0;
        const float beta = a.betas ? a.betas[s] : a.beta0;
        red = a.red_idx ? a.red_idx[s] : 0;

        // the tile kernel's displacement: exact on coordinates wrapped to the box's grid
        const BoxAxis ax(box[0]), ay(box[4]), az(box[8]);

        const int pli = a.plane ? a.plane[gi] : 0, plj = a.plane ? a.plane[gj] : 0;
        const int ofi = a.offset ? a.offset[gi] : 0, ofj = a.offset ? a.offset[gj] : 0;
        const double wi = (pli + ofi * lam) * cutoff_d;
        const double wj = (plj + ofj * lam) * cutoff_d;
        const double dwdl_i = static_cast<double>(static_cast<float>(ofi * cutoff_d));
        const double dwdl_j = static_cast<double>(static_cast<float>(ofj * cutoff_d));

        const double dx = ax.delta(a.x[gi * 3 + 0], a.x[gj * 3 + 0]);
        const double dy = ay.delta(a.x[gi * 3 + 1], a.x[gj * 3 + 1]);
        const double dz = az.delta(a.x[gi * 3 + 2], a.x[gj * 3 + 2]);
        const double dw = wi - wj;
        const double d2 = __builtin_fma(dw, dw, pair_d2(dx, dy, dz));
        uint64_t fs[3] = {0, 0, 0}; // force on atom 0 for the slots
        if (d2 < cutoff_d * cutoff_d) {
            // parameters as the tile kernel sees them: FP32 values of p, or of
            // p = (1 - lambda) p0 + lambda p1 when interpolated (k_gather)
            double pv[2][3], dp[2][3] = {{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};
            const int ga[2] = {gi, gj};
            for (int t = 0; t < 2; t++) {
                for (int c = 0; c < 3; c++) {
                    const double p0 = a.params[ga[t] * 3 + c];
                    if (a.params1) {
                        const double p1 = a.params1[ga[t] * 3 + c];
                        pv[t][c] = static_cast<float>((1.0 - lam) * p0 + lam * p1);
                        dp[t][c] = static_cast<float>(p1 - p0);
                    } else {
                        pv[t][c] = static_cast<float>(p0);
                    }
                }
            }
            const double qi = pv[0][0], qj = pv[1][0];
            const double si = pv[0][1], sj = pv[1][1];
            const double ei = pv[0][2], ej = pv[1][2];
            const bool interp = a.params1 != nullptr;
            const double scale_q = a.scales[p * 2 + 0];
            const double scale_lj = a.scales[p * 2 + 1];
            const PairTerms T = (DL && interp) ? nb_pair_terms<U, true>(d2, qi, qj, si, sj, ei, ej,
                                                                      static_cast<double>(beta), scale_q, scale_lj)
                                               : nb_pair_terms<U, DP>(d2, qi, qj, si, sj, ei, ej,
                                                                      static_cast<double>(beta), scale_q, scale_lj);
            auto acc = [neg](uint64_t *dst, uint64_t v) {
                if (v != 0) {
                    atomic_add_u64(dst, neg ? (0ull - v) : v);
                }
            };
            if (DX) {
                const double ps = T.prefactor * FIXED_SCALE; // as the tile kernel rounds
                const uint64_t fx = product_to_fixed(ps, dx);
                const uint64_t fy = product_to_fixed(ps, dy);
                const uint64_t fz = product_to_fixed(ps, dz);
                if (a.slots) {
                    fs[0] = neg ? 0ull - fx : fx;
                    fs[1] = neg ? 0ull - fy : fy;
                    fs[2] = neg ? 0ull - fz : fz;
                } else {
                    acc(du_dx + gi * 3 + 0, fx);
                    acc(du_dx + gi * 3 + 1, fy);
                    acc(du_dx + gi * 3 + 2, fz);
                    acc(du_dx + gj * 3 + 0, 0ull - fx);
                    acc(du_dx + gj * 3 + 1, 0ull - fy);
                    acc(du_dx + gj * 3 + 2, 0ull - fz);
                }
            }
            if (DP) {
                acc(du_dp + gi * 3 + 0, f64_to_fixed((scale_q * qj) * T.erfc_inv_d, FIXED_SCALE));
                acc(du_dp + gj * 3 + 0, f64_to_fixed((scale_q * qi) * T.erfc_inv_d, FIXED_SCALE));
                if (T.lj) {
                    const uint64_t gs = f64_to_fixed(T.sig_grad, FIXED_SCALE_DSIG);
                    acc(du_dp + gi * 3 + 1, gs);
                    acc(du_dp + gj * 3 + 1, gs);
                    acc(du_dp + gi * 3 + 2, f64_to_fixed(T.eps_grad * ej, FIXED_SCALE_DEPS));
                    acc(du_dp + gj * 3 + 2, f64_to_fixed(T.eps_grad * ei, FIXED_SCALE_DEPS));
                }
            }
            const bool vanilla = (wi == 0.0) && (wj == 0.0) && !interp;
            if (DL && !vanilla) {
                if (interp) {
                    fdl = f64_to_fixed(pair_du_dl(T, dw, dwdl_i, dwdl_j, true, scale_q, qi, qj, ei, ej, dp[0][0],
                                                  dp[1][0], dp[0][1], dp[1][1], dp[0][2], dp[1][2]),
                                       FIXED_SCALE);
                } else {
                    fdl = f64_to_fixed(dw * T.prefactor * (dwdl_i - dwdl_j), FIXED_SCALE);
                }
            }
            if (DLDP && !vanilla && !interp) {
                const PairDlDp D = nb_pair_dl_dp(d2, si, sj, ei, ej, static_cast<double>(beta), scale_lj);
                const double dd = dw * (dwdl_i - dwdl_j);
                acc(du_dp + gi * 3 + 0, f64_to_fixed(((scale_q * qj) * D.es_unit) * dd, FIXED_SCALE));
                acc(du_dp + gj * 3 + 0, f64_to_fixed(((scale_q * qi) * D.es_unit) * dd, FIXED_SCALE));
                if (D.lj) {
                    const uint64_t gs = f64_to_fixed(D.lj_dsig * dd, FIXED_SCALE_DSIG);
                    acc(du_dp + gi * 3 + 1, gs);
                    acc(du_dp + gj * 3 + 1, gs);
                    acc(du_dp + gi * 3 + 2, f64_to_fixed((D.lj_unit * ej) * dd, FIXED_SCALE_DEPS));
                    acc(du_dp + gj * 3 + 2, f64_to_fixed((D.lj_unit * ei) * dd, FIXED_SCALE_DEPS));
                }
            }
            if (U) {
                fu = f64_to_fixed(T.u, FIXED_SCALE);
            }
            if (neg) {
                fu = 0ull - fu;
                fdl = 0ull - fdl;
            }
        }
        if (DX && a.slots) {
            for (int c = 0; c < 3; c++) {
                a.slots[static_cast<size_t>(p) * 6 + c] = fs[c];
                a.slots[static_cast<size_t>(p) * 6 + 3 + c] = 0ull - fs[c];
            }
        }
    }
    if (U) {
        wave_add_by_key(u, red, fu);
    }
    if (DL) {
        wave_add_by_key(du_dl, red, fdl);
    }
}

using PairKernel = void (*)(const PairListArgs, uint64_t *, uint64_t *, uint64_t *, uint64_t *);
const PairKernel pair_kernels[16] = {
    k_pair_list<0, 0, 0, 0>, k_pair_list<0, 0, 0, 1>, k_pair_list<0, 0, 1, 0>, k_pair_list<0, 0, 1, 1>,
    k_pair_list<0, 1, 0, 0>, k_pair_list<0, 1, 0, 1>, k_pair_list<0, 1, 1, 0>, k_pair_list<0, 1, 1, 1>,
    k_pair_list<1, 0, 0, 0>, k_pair_list<1, 0, 0, 1>, k_pair_list<1, 0, 1, 0>, k_pair_list<1, 0, 1, 1>,
    k_pair_list<1, 1, 0, 0>, k_pair_list<1, 1, 0, 1>, k_pair_list<1, 1, 1, 0>, k_pair_list<1, 1, 1, 1>,
};

inline int kernel_index(const void *du_dx, const void *du_dp, const void *du_dl, const void *u) {
    return (u ? 8 : 0) | (du_dx ? 4 : 0) | (du_dl ? 2 : 0) | (du_dp ? 1 : 0);
}

int default_tile_grid() {
    // initialised once, thread-safe (engines may be built from several host threads)
    static const int grid = [] {
        int dev = 0;
        TM_HIP_CHECK(hipGetDevice(&dev));
        int cus = 0;
        TM_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        // 128 one-wave workgroups per CU: up to 16 are resident per CU (128 VGPRs,
        // 10 KB LDS per wave for the force kernels) and the rest queue behind
        // them, which balances the uneven per-tile pair counts better than a
        // fully persistent grid (measured on MI355X: -15%)
        return cus * 128;
    }();
    return grid;
}

} // namespace

void NbState::add_sorted(uint64_t *du_dx, uint64_t *du_dp, hipStream_t stream) const {
    if (!sorted_acc.ptr || (!du_dx && !du_dp)) {
        return;
    }
    const dim3 grid(S, ceil_div(max_slots, 256));
    auto kern = du_dx ? (du_dp ? k_add_sorted<true, true> : k_add_sorted<true, false>) : k_add_sorted<false, true>;
    kern<<<grid, 256, 0, stream>>>(sys.ptr, perm.ptr, total_slots, sorted_acc.ptr, du_dx, du_dp);
    TM_LAUNCH_CHECK();
}

void NbState::compute(
    const double *boxes,
    uint64_t *du_dx,
    uint64_t *du_dp,
    uint64_t *du_dl,
    uint64_t *u,
    hipStream_t stream,
    int grid_override,
    bool keep_sorted) const {
    const int idx = kernel_index(du_dx, du_dp, du_dl, u);
    if (idx == 0) {
        return;
    }
    const int grid = grid_override > 0 ? grid_override : default_tile_grid();
    const TileKernel kern = tile_kernel(idx, any_interp, tile_waves);
    kern<<<grid, NB_BLOCK, 0, stream>>>(sys.ptr, S, tile_prefix.ptr, tile_order.ptr, tile_row.ptr, tile_atoms.ptr, perm.ptr, pos.ptr,
                                        par.ptr, any_interp ? dpar.ptr : nullptr, boxes, bb_ctr.ptr, bb_ext.ptr,
                                        status.ptr, sorted_acc.ptr, total_slots, red_slots.ptr, du_dx, du_dp, du_dl, u);
    TM_LAUNCH_CHECK();
    add_sorted(keep_sorted ? nullptr : du_dx, du_dp, stream);
}

void launch_pair_list(
    const PairListArgs &a, uint64_t *du_dx, uint64_t *du_dp, uint64_t *du_dl, uint64_t *u, hipStream_t stream) {
    const int idx = kernel_index(du_dx, du_dp, du_dl, u);
    if (idx == 0 || a.M == 0) {
        return;
    }
    pair_kernels[idx]<<<ceil_div(a.M, 256), 256, 0, stream>>>(a, du_dx, du_dp, du_dl, u);
    TM_LAUNCH_CHECK();
}

void NbState::compute_dl_dp(const double *boxes, uint64_t *dl_dp, hipStream_t stream, int grid_override) const {
    const int grid = grid_override > 0 ? grid_override : default_tile_grid();
    if (any_interp) {
        throw Error("d(du/dlambda)/dp is not available for interpolated parameters");
    }
    k_nonbonded_tiles<false, false, false, false, true><<<grid, NB_BLOCK, 0, stream>>>(
        sys.ptr, S, tile_prefix.ptr, tile_order.ptr, tile_row.ptr, tile_atoms.ptr, perm.ptr, pos.ptr, par.ptr, nullptr, boxes,
        bb_ctr.ptr, bb_ext.ptr, status.ptr, sorted_acc.ptr, total_slots, nullptr, nullptr, dl_dp, nullptr, nullptr);
    TM_LAUNCH_CHECK();
    add_sorted(nullptr, dl_dp, stream);
}

void launch_pair_list_dl_dp(const PairListArgs &a, uint64_t *dl_dp, hipStream_t stream) {
    if (a.M == 0) {
        return;
    }
    if (a.params1) {
        throw Error("d(du/dlambda)/dp is not available for interpolated parameters");
    }
    k_pair_list<false, false, false, false, true><<<ceil_div(a.M, 256), 256, 0, stream>>>(a, nullptr, dl_dp, nullptr,
                                                                                          nullptr);
    TM_LAUNCH_CHECK();
}

} // namespace tmamd
