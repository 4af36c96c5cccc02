// Full-atom protein builder for MI355X (gfx950): FullAtomModel.Angles2Coords
// forward and backward.  The C ABI is include/tpl_a2c.h.
//
// The reference builds a tree of heap-allocated 4x4 transforms per structure
// on the CPU and walks it recursively (Layers/FullAtomModel/cConformation.cpp:
// 29-158); its backward visits, for every angle, every atom below it
// (:160-195), O(atoms x tree depth) with a chain's depth growing with its
// length.  Here one wave takes 64 consecutive residues of a structure, one per
// lane:
//
//   1. each lane multiplies out its residue's step S_i = T_CA(phi_i) T_C(psi_i)
//      T_N(omega_i) (FP64 3x4), the transform from residue i's N frame to
//      residue i+1's;
//   2. a wave scan of those products (DPP), folded with the products of the
//      blocks before, gives each residue its N frame, and a scan of the atom
//      counts its first atom;
//   3. each lane walks its residue: N, CA, the side chain, C, writing atoms.
//
// The backward uses dL/dalpha = u . (sum_{x in subtree} x cross g
// - p cross sum_{x in subtree} g) for a node with x axis u and origin p (the
// reference's g . (F x) with F = M_parent dT M^-1, cConformation.cpp:148,
// 171-184, reduces to this since F x = u cross (x - p)).  u and p follow from
// the forward's coordinates, so the backward reads those and needs no frames.
// The subtree of a backbone node is the rest of its residue plus every later
// residue: again one lane per residue in blocks of 64, whose sums (sum g,
// sum x cross g) a scan over the lanes and the sums of the later blocks join.
// For some batches a run of residues per thread (a2c_fwd_runs, a2c_bwd) or tiles
// of consecutive atoms (a2c_bwd_tiled) are the better form (forward_form,
// backward_form).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>
#include <set>
#include <utility>
#include <vector>

#include "a2c_flagged.h"
#include "a2c_table.h"
#include "report.h"
#include "sincos_tab.h"
#include "tpl_a2c.h"

namespace {

using namespace a2c;

// Workgroup sizes of the run backward: 256 threads, or 512 for long structures
// (see use_large_bwd), where a thread then walks half as many residues.
constexpr int kThreadsSmall = 256, kThreadsLarge = 512;

__constant__ Residue kRes[kTypes] = A2C_RESIDUES;
__constant__ Side kSide[kTypes][kMaxSide] = A2C_SIDES;
__constant__ Atom kAtom[kTypes][kMaxAtoms] = A2C_ATOMS;

// Workgroup-shared tables.  StepTables: what the residue steps and the atom
// counts need.  Tables: also local atom positions, per side-chain node cos/sin
// of beta and of a constant alpha, d, and the packed (row, first atom, count),
// and the names as words.
struct alignas(16) StepTables {
    double tab[128];       // the sincos table of sincos_tab.h
    double bb[3][2];       // cos/sin of beta for the CA, C and N transforms
    int res_i[kTypes];     // natoms | nca << 8 | nside << 16
    uint8_t type[256];     // residue type of a letter, 0xff: none
    uint8_t atoms[256];    // its atoms, 0: none
};
struct alignas(16) Tables : StepTables {
    double loc[kTypes * kMaxAtoms][3];
    double side[kTypes * kMaxSide][5];
    int side_i[kTypes * kMaxSide];
    uint2 name[kTypes * kMaxAtoms];  // the residue's, the atom's
};

// The table sincos (sincos_tab.h) over the workgroup's LDS copy of its table.
struct TabSinCos {
    const double* tab;
    __device__ __forceinline__ void operator()(double x, double* s, double* c) const {
        sincos_tab(x, tab, s, c);
    }
};

// The sines and cosines of the constant angles come from the table sincos
// (within 2.2e-16 of the math library's): the library's FP64 sincos took
// 4-6 us of every workgroup's start.
template <int NT>
__device__ void fill_tables(Tables& tb) {
    for (int k = threadIdx.x; k < 128; k += NT) tb.tab[k] = kTabCS[k];
    __syncthreads();  // tb.tab, for the rest
    const TabSinCos sc{tb.tab};
    for (int k = threadIdx.x; k < kTypes * kMaxAtoms; k += NT) {
        const Atom at = kAtom[k / kMaxAtoms][k % kMaxAtoms];
        local_position_with(at, tb.loc[k], sc);
    }
    for (int k = threadIdx.x; k < kTypes * kMaxSide; k += NT) {
        const Side s = kSide[k / kMaxSide][k % kMaxSide];
        sc(s.beta, &tb.side[k][1], &tb.side[k][0]);
        sc(s.alpha, &tb.side[k][3], &tb.side[k][2]);
        tb.side[k][4] = s.d;
        tb.side_i[k] = (s.row & 0xff) | (s.first << 8) | (s.count << 16);
    }
    for (int k = threadIdx.x; k < kTypes * kMaxAtoms; k += NT)
        tb.name[k] = make_uint2(*reinterpret_cast<const uint32_t*>(kRes[k / kMaxAtoms].name3),
                                *reinterpret_cast<const uint32_t*>(kAtom[k / kMaxAtoms][k % kMaxAtoms].name));
    for (int k = threadIdx.x; k < 256; k += NT) {
        const int t = residue_type((uint8_t)k);
        tb.type[k] = (uint8_t)t;
        tb.atoms[k] = t < 0 ? (uint8_t)0 : (uint8_t)kRes[t].natoms;
    }
    if (threadIdx.x < kTypes) {
        const Residue r = kRes[threadIdx.x];
        tb.res_i[threadIdx.x] = r.natoms | (r.nca << 8) | (r.nside << 16);
    }
    if (threadIdx.x < 3) {
        const double beta = threadIdx.x == 0 ? geo::C_N_CA : (threadIdx.x == 1 ? geo::N_CA_C : geo::CA_C_N);
        sc(beta, &tb.bb[threadIdx.x][1], &tb.bb[threadIdx.x][0]);
    }
}

// The tables are the same for every workgroup and call: a one-workgroup
// kernel computes them once per device into g_tab, and each forward
// workgroup copies that (1.3 us less per workgroup than computing them:
// 32 x 350 residues 17.5 -> 16.2 us, 1024 x 30 15.2 -> 13.4 us).
__device__ Tables g_tab;

__global__ void __launch_bounds__(256) a2c_init_tables() {
    __shared__ Tables tb;
    fill_tables<256>(tb);
    __syncthreads();
    const double* src = reinterpret_cast<const double*>(&tb);
    double* dst = reinterpret_cast<double*>(&g_tab);
    for (int k = threadIdx.x; k < (int)(sizeof(Tables) / 8); k += 256) dst[k] = src[k];
}

template <typename TB>
__device__ __forceinline__ void copy_tables(TB& tb, int nt) {
    const uint4* src = reinterpret_cast<const uint4*>(&static_cast<const TB&>(g_tab));
    uint4* dst = reinterpret_cast<uint4*>(&tb);
    for (int k = threadIdx.x; k < (int)(sizeof(TB) / 16); k += nt) dst[k] = src[k];
}

// m (3x4, row-major) <- m * Ry(beta) Tx(d) Rx(alpha), with cb/sb of beta and
// ca/sa of alpha.  Ry(b) Tx(d) Rx(a) = [[cb, sb sa, sb ca, d cb],
// [0, ca, -sa, 0], [-sb, cb sa, cb ca, -d sb]].
__device__ __forceinline__ void step(double m[12], double cb, double sb, double ca, double sa,
                                     double d) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const double a0 = m[4 * i], a1 = m[4 * i + 1], a2 = m[4 * i + 2];
        const double n0 = a0 * cb - a2 * sb;
        const double t = a0 * sb + a2 * cb;
        m[4 * i] = n0;
        m[4 * i + 1] = t * sa + a1 * ca;
        m[4 * i + 2] = t * ca - a1 * sa;
        m[4 * i + 3] += d * n0;
    }
}

// c = a * b for 3x4 rigid transforms.
__device__ __forceinline__ void compose(const double a[12], const double b[12], double c[12]) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
            c[4 * i + j] = a[4 * i] * b[j] + a[4 * i + 1] * b[4 + j] + a[4 * i + 2] * b[8 + j] +
                           (j == 3 ? a[4 * i + 3] : 0.0);
    }
}

__device__ __forceinline__ void identity(double m[12]) {
#pragma unroll
    for (int k = 0; k < 12; ++k) m[k] = (k == 0 || k == 5 || k == 10) ? 1.0 : 0.0;
}

__device__ __forceinline__ void apply(const double m[12], const double v[3], double x[3]) {
#pragma unroll
    for (int i = 0; i < 3; ++i) x[i] = m[4 * i] * v[0] + m[4 * i + 1] * v[1] + m[4 * i + 2] * v[2] + m[4 * i + 3];
}

// ---- wave-level scans (DPP; all 64 lanes of the wave active) ----
// GFX9 DPP controls: row shifts, row broadcasts, wave shift right by one.
constexpr int kRowShr1 = 0x111, kRowShr2 = 0x112, kRowShr4 = 0x114, kRowShr8 = 0x118;
constexpr int kRowBcast15 = 0x142, kRowBcast31 = 0x143, kWaveShr1 = 0x138;

// DPP move of a double; lanes that receive nothing (or rows masked off)
// keep `old`.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_double(double v, double old) {
    const int lo = __builtin_amdgcn_update_dpp(__double2loint(old), __double2loint(v), CTRL, ROW_MASK, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(__double2hiint(old), __double2hiint(v), CTRL, ROW_MASK, 0xf, false);
    return __hiloint2double(hi, lo);
}
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ int dpp_int(int v) {
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROW_MASK, 0xf, false);
}

__device__ __forceinline__ double ident12(int k) {
    return (k == 0 || k == 5 || k == 10) ? 1.0 : 0.0;
}

// One Hillis-Steele step of the ordered product: m <- (source lane's m) * m,
// with the identity where a lane receives nothing.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ void frame_scan_step(double m[12]) {
    double g[12], r[12];
#pragma unroll
    for (int k = 0; k < 12; ++k) g[k] = dpp_double<CTRL, ROW_MASK>(m[k], ident12(k));
    compose(g, m, r);
#pragma unroll
    for (int k = 0; k < 12; ++k) m[k] = r[k];
}

// Inclusive ordered product over the wave's lanes (lane l ends with
// m_0 * ... * m_l).
__device__ __forceinline__ void wave_scan_frames(double m[12]) {
    frame_scan_step<kRowShr1, 0xf>(m);
    frame_scan_step<kRowShr2, 0xf>(m);
    frame_scan_step<kRowShr4, 0xf>(m);
    frame_scan_step<kRowShr8, 0xf>(m);
    frame_scan_step<kRowBcast15, 0xa>(m);
    frame_scan_step<kRowBcast31, 0xc>(m);
}

// Inclusive prefix sums over the wave's lanes.
__device__ __forceinline__ double wave_scan_double(double v) {
    v += dpp_double<kRowShr1, 0xf>(v, 0.0);
    v += dpp_double<kRowShr2, 0xf>(v, 0.0);
    v += dpp_double<kRowShr4, 0xf>(v, 0.0);
    v += dpp_double<kRowShr8, 0xf>(v, 0.0);
    v += dpp_double<kRowBcast15, 0xa>(v, 0.0);
    v += dpp_double<kRowBcast31, 0xc>(v, 0.0);
    return v;
}
// Inclusive prefix sums within each row of 16 lanes.
__device__ __forceinline__ double row_scan_double(double v) {
    v += dpp_double<kRowShr1, 0xf>(v, 0.0);
    v += dpp_double<kRowShr2, 0xf>(v, 0.0);
    v += dpp_double<kRowShr4, 0xf>(v, 0.0);
    v += dpp_double<kRowShr8, 0xf>(v, 0.0);
    return v;
}
// The value of lane `lane` (wave-uniform) of a double.
__device__ __forceinline__ double readlane_double(double v, int lane) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ int wave_scan_int(int v) {
    v += dpp_int<kRowShr1, 0xf>(v);
    v += dpp_int<kRowShr2, 0xf>(v);
    v += dpp_int<kRowShr4, 0xf>(v);
    v += dpp_int<kRowShr8, 0xf>(v);
    v += dpp_int<kRowBcast15, 0xa>(v);
    v += dpp_int<kRowBcast31, 0xc>(v);
    return v;
}

// The structure's length: the first 0 byte of its sequence row, or
// seq_stride (s_len enters as seq_stride).  Each thread reads 4 consecutive
// bytes per round, the loads issued together.
template <int NT>
__device__ __forceinline__ void find_length(const uint8_t* seq, int seq_stride, int* s_len) {
    constexpr int kPer = 4;
    for (int i0 = (int)threadIdx.x * kPer; i0 < seq_stride; i0 += NT * kPer) {
        uint8_t c[kPer];
#pragma unroll
        for (int e = 0; e < kPer; ++e) c[e] = i0 + e < seq_stride ? seq[i0 + e] : (uint8_t)1;
        int first = -1;
#pragma unroll
        for (int e = kPer - 1; e >= 0; --e)
            if (c[e] == 0) first = i0 + e;
        if (first >= 0) atomicMin(s_len, first);
    }
}

// The side-chain angles xi1..xi5 of a residue in the order its side-chain
// nodes bind them: every template binds rows 3, 4, ... consecutively (the
// table test checks this), so each bound node takes the next one.  Shifting
// keeps the values in registers where an index computed at run time would not.
template <typename T>
struct SideRows {
    T v[5];
    __device__ __forceinline__ explicit SideRows(const T (&a)[8]) {
#pragma unroll
        for (int k = 0; k < 5; ++k) v[k] = a[3 + k];
    }
    __device__ __forceinline__ double pop() {
        const T x = v[0];
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] = v[k + 1];
        return (double)x;
    }
};

// A thread's run of residues [r0, r1) of a structure of L, its first atom and
// the structure's atoms.
struct Run {
    int L, r0, r1, atom0, total;
};

// ---- forward: one wave per block of 64 residues ----
// A structure is cut into blocks of kBlock consecutive residues; a wave builds
// one block's atoms, each lane one residue's, so the lanes' angles and letters
// are consecutive in memory and every wave has the same work, whatever the mix
// of lengths.  A residue needs its N frame (the product of the residue steps
// before it) and its first atom:
//   * a2c_fwd_steps + a2c_fwd_walk: the first kernel multiplies out groups of
//     256 residues, four per lane, and leaves every residue's frame within its
//     group, the groups' products and the atom counts in the caller's
//     workspace; the second puts the groups before in front.  Both wait on
//     latencies (of memory, LDS and dependent FP64) more than half of their
//     waves' time; so the first also writes the zeros past the structures
//     (three quarters of all bytes at mixed lengths), and the frames go through
//     memory (72 bytes per residue) rather than being multiplied out again;
//   * a2c_fwd_single where a structure is one block (angles_stride <= 64): the
//     wave scans its 64 steps;
//   * a2c_fwd_fused: one workgroup per structure, whose waves' scans meet in
//     LDS.  It needs no workspace and one launch, and serves small batches.
// Waves whose residues would lie past the structure write its padding's zeros.
// Against one workgroup of 256 or 512 threads per structure whose threads
// walked runs of up to four residues and wrote their atoms and names one by one
// (names included, us): lengths 30-1000 at B=1024 118 -> 62, in float64
// 159 -> 93; 256 x 1000 60 -> 38; 32 x 350 18.2 -> 13.6; 1024 x 30 16.1 -> 11.2;
// one peptide of 21 in float64 12.8 -> 9.0.
//
// Workgroups go to the 8 XCDs in turn, those of one XCD to its 32 CUs in turn,
// and a workgroup's waves to the CU's SIMDs.  What only some structures have
// (their later groups and blocks) must not always meet the same of these: the
// grids run over the structures first and their groups second, and the waves
// of a workgroup take its shares rotated as the workgroups come round to a CU
// (turned_wave).  With the groups of a structure side by side the XCDs of the
// even workgroups had the first groups: 1024 structures of lengths 30-1000 took
// 55 us in the walk, against 38.
constexpr int kBlock = 64;                   // residues per wave of the walk: one per lane
constexpr int kQuad = 4;                     // residues per lane of the steps
constexpr int kGroup = kBlock * kQuad;       // residues per wave of the steps
constexpr int kGroupWaves = kGroup / kBlock; // blocks per group; waves per workgroup of the steps

// The share of wave `wave` of W in workgroup `wg`.
__device__ __forceinline__ int turned_wave(int wave, int W, int wg) {
    return (int)((uint32_t)(wave + (wg >> 3) + (wg >> 8)) % (uint32_t)W);
}

// A group's products and counts.
struct alignas(16) GroupRec {
    double f[12];             // the product of its residue steps
    int before[kGroupWaves];  // the structure's atoms before each of its blocks
};
// The frames of a group's residues within it: their x and y axes and origins
// (z = x cross y).  Component k of residue 4q + e is at v[k][64e + q], so that
// the steps' stores and the walk's loads are of consecutive doubles.
struct alignas(16) GroupFrames {
    double v[9][kGroup];
};

// The structure of slot b of the batch: order[b], or b without an order; -1
// for an entry outside the batch, which is reported (TPL_A2C_STATUS_ORDER)
// and builds nothing.
__device__ __forceinline__ int structure_at(const int* order, int b, int batch, const Report& rep) {
    if (!order) return b;
    const int o = __builtin_amdgcn_readfirstlane(order[b]);
    if (o >= 0 && o < batch) return o;
    report_bits(rep, TPL_A2C_STATUS_ORDER);
    return -1;
}

// A sequence row read by one wave, 16 loads of 64 consecutive bytes at a time;
// the first 1024 bytes are loaded by load(), so that the caller can do other
// work before it needs them.
struct RowScan {
    static constexpr int kAtOnce = 16;
    uint8_t c[kAtOnce];

    __device__ __forceinline__ void load(const uint8_t* seq, int stride, int lane, int base = 0) {
#pragma unroll
        for (int e = 0; e < kAtOnce; ++e) {
            const int i = base + 64 * e + lane;
            c[e] = i < stride ? seq[i] : (uint8_t)0;
        }
    }
    // The row's length: its first 0 byte, or its stride.  With `atoms`, also
    // the atoms of its letters, those before residue `upto`, and whether one
    // of them is not a residue's.
    template <bool ATOMS>
    __device__ __forceinline__ int finish(const uint8_t* seq, int stride, int lane, const uint8_t* letter_atoms,
                                          int upto, int& atoms, int& before, bool& bad) {
        int n = -1, cnt = 0, bef = 0;
        bool odd = false;
        for (int base = 0; n < 0; base += 64 * kAtOnce) {
            if (base > 0) load(seq, stride, lane, base);
#pragma unroll
            for (int e = 0; e < kAtOnce; ++e) {
                if (n >= 0) continue;
                const uint64_t zero = __builtin_amdgcn_ballot_w64(c[e] == 0);
                const int i = base + 64 * e + lane;
                if (zero) n = base + 64 * e + (int)__builtin_ctzll(zero);
                if (ATOMS && (n < 0 || i < n)) {
                    const int k = letter_atoms[c[e]];
                    odd |= k == 0;
                    cnt += k;
                    if (i < upto) bef += k;
                }
            }
        }
        if (ATOMS) {
            atoms = __builtin_amdgcn_readlane(wave_scan_int(cnt), 63);
            before = __builtin_amdgcn_readlane(wave_scan_int(bef), 63);
            bad = __builtin_amdgcn_ballot_w64(odd) != 0;
        }
        return n;
    }
};

__device__ __forceinline__ int wave_length(const uint8_t* seq, int stride, int lane) {
    RowScan row;
    row.load(seq, stride, lane);
    int atoms, before;
    bool bad;
    return row.finish<false>(seq, stride, lane, nullptr, 0, atoms, before, bad);
}

// Cosines and sines of a residue's phi and psi, for its steps and its walk.
struct Turns {
    double c[2], s[2];
};

// m <- the step of a residue with the angles phi, psi, omega.
__device__ __forceinline__ void first_step(double m[12], const StepTables& tb, double phi, double psi, double omega,
                                           Turns& tu) {
    double s, c;
    sincos_tab(phi, tb.tab, &tu.s[0], &tu.c[0]);
    sincos_tab(psi, tb.tab, &tu.s[1], &tu.c[1]);
    sincos_tab(omega, tb.tab, &s, &c);
    identity(m);
    step(m, tb.bb[0][0], tb.bb[0][1], tu.c[0], tu.s[0], geo::R_N_CA);
    step(m, tb.bb[1][0], tb.bb[1][1], tu.c[1], tu.s[1], geo::R_CA_C);
    step(m, tb.bb[2][0], tb.bb[2][1], c, s, geo::R_C_N);
}

// The lane's residue i: its letter (0 past the structure's length n) and its
// angles.
template <typename T>
__device__ __forceinline__ uint8_t lane_residue(const uint8_t* seq, int n, const T* ang, int stride, int i,
                                                T (&av)[8]) {
    uint8_t code = 0;
#pragma unroll
    for (int r = 0; r < 8; ++r) av[r] = (T)0;
    if (i < n) {
        code = seq[i];
#pragma unroll
        for (int r = 0; r < 8; ++r) av[r] = ang[(size_t)r * stride + i];
    }
    return code;
}

// The type of a letter (-1: none), and its residue's step (the identity for
// -1).
template <typename T>
__device__ __forceinline__ int lane_step(uint8_t code, const StepTables& tb, const T (&av)[8], double m[12],
                                         Turns& tu) {
    const int t = (int)(int8_t)tb.type[code];
    if (t >= 0)
        first_step(m, tb, (double)av[0], (double)av[1], (double)av[2], tu);
    else
        identity(m);
    return t;
}

// P <- P * the products of `count` records, in order (wave-uniform).
template <typename R>
__device__ __forceinline__ void fold(double P[12], const R* rec, int count) {
    for (int k = 0; k < count; ++k) {
        double A[12], Q[12];
#pragma unroll
        for (int e = 0; e < 12; ++e) A[e] = rec[k].f[e];
        compose(P, A, Q);
#pragma unroll
        for (int e = 0; e < 12; ++e) P[e] = Q[e];
    }
}

// An angle that may give coordinates that are NaN, infinite or huge: bounded
// angles give rotations, and positions within 14 A per residue.
template <typename T>
__device__ __forceinline__ bool wild(T a) {
    return !(a < (T)1e8 && a > (T)-1e8);
}

// The atoms of the lane's residue of type t with N frame F, at atom `at` of
// out (wave-uniform).  A group's first atom is its frame's origin.  C and O come
// before the side chain, so that one frame is live in its loop.  The side
// chain's first node is fixed and has no atoms and no length: a turn about x.
template <typename T>
__device__ __forceinline__ void walk_residue(const Tables& tb, int t, const T (&av)[8], const Turns& tu, double F[12],
                                             T* out, uint32_t at) {
    const int ri = tb.res_i[t];
    const int natoms = ri & 0xff, nca = (ri >> 8) & 0xff, nside = ri >> 16;
    const double* loc = tb.loc[t * kMaxAtoms];
    const uint32_t bytes = (uint32_t)(3 * sizeof(T));
    const uint32_t o = bytes * at;  // byte offsets within a block fit 32 bits
    auto origin = [&](int slot, const double m[12]) {
        T* q = reinterpret_cast<T*>(reinterpret_cast<char*>(out) + (o + bytes * (uint32_t)slot));
        q[0] = (T)m[3];
        q[1] = (T)m[7];
        q[2] = (T)m[11];
    };
    auto put = [&](int slot, const double m[12]) {
        double x[3];
        apply(m, loc + 3 * slot, x);
        T* q = reinterpret_cast<T*>(reinterpret_cast<char*>(out) + (o + bytes * (uint32_t)slot));
        q[0] = (T)x[0];
        q[1] = (T)x[1];
        q[2] = (T)x[2];
    };
    origin(0, F);
    step(F, tb.bb[0][0], tb.bb[0][1], tu.c[0], tu.s[0], geo::R_N_CA);  // F: CA
    origin(1, F);
    {
        double C[12];
#pragma unroll
        for (int k = 0; k < 12; ++k) C[k] = F[k];
        step(C, tb.bb[1][0], tb.bb[1][1], tu.c[1], tu.s[1], geo::R_CA_C);
        origin(natoms - 2, C);
        put(natoms - 1, C);
    }
    for (int k = 2; k <= nca; ++k) put(k, F);
    {
        const double c = tb.side[t * kMaxSide][2], s = tb.side[t * kMaxSide][3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const double y = F[4 * i + 1], z = F[4 * i + 2];
            F[4 * i + 1] = y * c + z * s;
            F[4 * i + 2] = z * c - y * s;
        }
    }
    SideRows<T> rows(av);
    for (int n = 1; n < nside; ++n) {
        const int q = t * kMaxSide + n;
        const int si = tb.side_i[q];
        const int row = (int)(int8_t)(si & 0xff), first = (si >> 8) & 0xff, count = si >> 16;
        double c = tb.side[q][2], s = tb.side[q][3];
        if (row >= 0) sincos_tab(rows.pop(), tb.tab, &s, &c);
        step(F, tb.side[q][0], tb.side[q][1], c, s, tb.side[q][4]);
        origin(first, F);
        for (int k = first + 1; k < first + count; ++k) put(k, F);
    }
}

// Wave-scope LDS ordering (the wave's writes before its reads).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The names of a block's `count` atoms at rn, an: each lane notes its
// residue's (type, slot) per atom in the wave's LDS, and the wave writes the
// words of 64 consecutive atoms at a time.  (A lane writing its own residue's
// names, each from a dependent table load, took as long as the coordinates.)
__device__ __forceinline__ void write_names(const Tables& tb, int t, int natoms, int at, int count, uint32_t* rn,
                                            uint32_t* an, uint16_t* s_role, int lane) {
    for (int s = 0; s < natoms; ++s) s_role[at + s] = (uint16_t)(t * kMaxAtoms + s);
    wave_lds_sync();
    for (int k = lane; k < count; k += 64) {
        const uint2 names = tb.name[s_role[k]];
        rn[(uint32_t)k] = names.x;
        an[(uint32_t)k] = names.y;
    }
}

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// The walk's coordinates go through the wave's LDS: a lane writing its own
// residue's atoms to memory makes every store instruction touch 64 lines.  A
// block's atoms are staged at most kStage at a time (64 residues have 525 on
// average, 896 at most; at 576 two workgroups of a2c_fwd_walk fit on a CU).
constexpr int kStage = 576;
template <typename T>
constexpr int stage_values() {
    return 3 * kStage + 16 / (int)sizeof(T);
}
static_assert(stage_values<float>() * sizeof(float) % 16 == 0 && stage_values<double>() * sizeof(double) % 16 == 0,
              "the waves' stages stand one after another at 16-byte alignment");

// Values [0, count) from the wave's LDS to dst, as 16-byte stores where dst is
// aligned; s_w[0] holds the value of dst rounded down to 16 bytes, so that both
// sides are aligned together.
template <typename T>
__device__ __forceinline__ void flush_stage(T* dst, int count, const T* s_w, int lane) {
    constexpr int V = 16 / (int)sizeof(T);
    const int mis = (int)((reinterpret_cast<uintptr_t>(dst) & 15) / sizeof(T));
    T* d0 = dst - mis;
    const int end = mis + count, first = mis ? V : 0, last = end / V * V;
    if (mis && lane >= mis && lane < V && lane < end) d0[lane] = s_w[lane];
    for (int k = first + V * lane; k < last; k += V * 64)
        *reinterpret_cast<uint4*>(d0 + k) = *reinterpret_cast<const uint4*>(s_w + k);
    const int tail = last > first ? last : first;
    if (tail + lane < end) d0[tail + lane] = s_w[tail + lane];
}

// Share f of F of the zeros over words [0, count) of p, by one wave: the waves
// take 1 KB pieces (16-byte streaming stores, whole 128-byte lines) in turn, so
// that they write one stretch of memory together; share 0 also takes the words
// before the first whole line and after the last 16 bytes.
__device__ __forceinline__ void zero_words(uint32_t* p, int64_t count, int f, int F, int lane) {
    if (count <= 0) return;
    const int mis = (int)((128 - (reinterpret_cast<uintptr_t>(p) & 127)) & 127) / 4;
    const int head = (int)(mis < count ? mis : count);
    const int64_t nvec = (count - head) / 4, tail = head + 4 * nvec;
    const u32x4 z = {0u, 0u, 0u, 0u};
    u32x4* q = reinterpret_cast<u32x4*>(p + head);
    for (int64_t v = 64 * f + lane; v < nvec; v += 64 * F) __builtin_nontemporal_store(z, q + v);
    if (f == 0) {
        if (lane < head) p[lane] = 0u;
        if (tail + lane < count) p[tail + lane] = 0u;
    }
}

// Share f of F of the zeros past a structure's `total` atoms, by one wave.
template <typename T>
__device__ __forceinline__ void zero_share(T* out, uint32_t* rn, uint32_t* an, int total, int atoms_stride, int f,
                                           int F, int lane) {
    const int64_t rest = atoms_stride - total;
    constexpr int W = (int)(sizeof(T) / 4);
    zero_words(reinterpret_cast<uint32_t*>(out + 3 * (size_t)total), 3 * W * rest, f, F, lane);
    if (rn) {
        zero_words(rn + total, rest, f, F, lane);
        zero_words(an + total, rest, f, F, lane);
    }
}

// The frames within each group, its product and its atom counts, one wave per
// (structure, group) and four residues per lane; and the zeros past the
// structure.  Every wave reads the whole row of letters (one round of loads)
// and so knows the structure's length, atoms and flags by itself.
template <typename T>
__global__ void __launch_bounds__(64 * kGroupWaves) a2c_fwd_steps(
    const uint8_t* __restrict__ seqs, int seq_stride, const T* __restrict__ angles, int ang_stride,
    int* __restrict__ lens, GroupRec* __restrict__ rec, GroupFrames* __restrict__ frames, T* __restrict__ coords,
    uint32_t* __restrict__ res_names, uint32_t* __restrict__ atom_names, int atoms_stride, Report rep,
    const int* __restrict__ order, int batch, int ng) {
    __shared__ StepTables tb;
    const int wave = turned_wave((int)(threadIdx.x >> 6), kGroupWaves, (int)blockIdx.x);
    const int lane = (int)(threadIdx.x & 63);
    const int w = (int)blockIdx.x * kGroupWaves + wave;
    const int g = w / batch, slot = w - g * batch;
    const int b = g < ng ? structure_at(order, slot, batch, g == 0 ? rep : Report{nullptr, nullptr}) : -1;
    const uint8_t* seq = seqs + (size_t)(b < 0 ? 0 : b) * seq_stride;
    const T* ang = angles + (size_t)(b < 0 ? 0 : b) * 8 * ang_stride;
    // All loads go out before the first wait: the row, and this lane's letters
    // and angles (zeros where the strides end; unused past the structure).
    RowScan row;
    row.load(seq, seq_stride, lane);
    const int i0 = kGroup * g + kQuad * lane;
    uint8_t code[kQuad];
    T a[3][kQuad];
#pragma unroll
    for (int e = 0; e < kQuad; ++e) {
        const bool in = i0 + e < ang_stride;
        code[e] = in && i0 + e < seq_stride ? seq[i0 + e] : (uint8_t)0;
#pragma unroll
        for (int r = 0; r < 3; ++r) a[r][e] = in ? ang[(size_t)r * ang_stride + i0 + e] : (T)0;
    }
    copy_tables(tb, 64 * kGroupWaves);
    __syncthreads();
    if (b < 0) {
        if (g == 0 && lane == 0) lens[slot] = 0;
        return;
    }
    int total = 0, before = 0, flags = 0;
    bool bad = false;
    int n = row.finish<true>(seq, seq_stride, lane, tb.atoms, kGroup * g, total, before, bad);
    if (n > ang_stride) {
        flags = TPL_A2C_STATUS_LENGTH;
    } else {
        if (bad) flags |= TPL_A2C_STATUS_SEQ;
        if (total > atoms_stride) flags |= TPL_A2C_STATUS_ATOMS;
    }
    if (flags) {  // a flagged structure is all zeros
        if (g == 0 && lane == 0) report_bits(rep, (uint32_t)flags);
        n = total = 0;
    }
    T* out = coords + (size_t)b * 3 * atoms_stride;
    uint32_t* rn = res_names ? res_names + (size_t)b * atoms_stride : nullptr;
    uint32_t* an = atom_names ? atom_names + (size_t)b * atoms_stride : nullptr;
    const int here = (n + kGroup - 1) / kGroup;  // groups that hold residues
    GroupRec* r = rec + (size_t)b * ng + g;
    if (g == 0 && lane == 0) lens[slot] = n;
    if (g < here) {
        double m[12], turn[kQuad - 1][3][2];  // the first residues' (cos, sin), for their frames
        identity(m);
        int cnt = 0;
#pragma unroll
        for (int e = 0; e < kQuad; ++e) {
            const bool in = i0 + e < n;
            cnt += in ? tb.atoms[code[e]] : 0;
            double v[3][2];
#pragma unroll
            for (int r = 0; r < 3; ++r) sincos_tab((double)a[r][e], tb.tab, &v[r][1], &v[r][0]);
            if (in) {
                step(m, tb.bb[0][0], tb.bb[0][1], v[0][0], v[0][1], geo::R_N_CA);
                step(m, tb.bb[1][0], tb.bb[1][1], v[1][0], v[1][1], geo::R_CA_C);
                step(m, tb.bb[2][0], tb.bb[2][1], v[2][0], v[2][1], geo::R_C_N);
            }
            if (e < kQuad - 1) {
#pragma unroll
                for (int r = 0; r < 3; ++r) turn[e][r][0] = v[r][0], turn[e][r][1] = v[r][1];
            }
        }
        const int cinc = wave_scan_int(cnt);
        wave_scan_frames(m);
        if ((lane & 15) == 0) r->before[lane >> 4] = before + cinc - cnt;
        if (lane == 63) {
#pragma unroll
            for (int k = 0; k < 12; ++k) r->f[k] = m[k];
        }
#pragma unroll
        for (int k = 0; k < 12; ++k) m[k] = dpp_double<kWaveShr1, 0xf>(m[k], ident12(k));
        GroupFrames* gf = frames + ((size_t)b * ng + g);
#pragma unroll
        for (int e = 0; e < kQuad; ++e) {
            if (i0 + e < n) {
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    gf->v[i][64 * e + lane] = m[4 * i];
                    gf->v[3 + i][64 * e + lane] = m[4 * i + 1];
                    gf->v[6 + i][64 * e + lane] = m[4 * i + 3];
                }
            }
            if (e < kQuad - 1) {
                step(m, tb.bb[0][0], tb.bb[0][1], turn[e][0][0], turn[e][0][1], geo::R_N_CA);
                step(m, tb.bb[1][0], tb.bb[1][1], turn[e][1][0], turn[e][1][1], geo::R_CA_C);
                step(m, tb.bb[2][0], tb.bb[2][1], turn[e][2][0], turn[e][2][1], geo::R_C_N);
            }
        }
    }
    // the padding: by the groups past the structure, or by all where none is
    if (here == ng)
        zero_share(out, rn, an, total, atoms_stride, g, ng, lane);
    else if (g >= here)
        zero_share(out, rn, an, total, atoms_stride, g - here, ng - here, lane);
}

// The atoms (and names) of a block of `total` atoms, by one wave: the lane's
// residue has the type t, the N frame F and `cnt` atoms from `at` on; out, rn
// and an are the block's.
template <typename T>
__device__ __forceinline__ void build_block(const Tables& tb, int t, const T (&av)[8], const Turns& tu, double F[12],
                                            int at, int cnt, int total, T* out, uint32_t* rn, uint32_t* an, T* s_w,
                                            int lane) {
    for (int base = 0; base < total;) {  // once, unless the block has more than kStage atoms
        const uint64_t later = __builtin_amdgcn_ballot_w64(at + cnt > base + kStage);
        const int end = later ? __builtin_amdgcn_readlane(at, (int)__builtin_ctzll(later)) : total;
        T* dst = out + 3 * (size_t)base;
        const int mis = (int)((reinterpret_cast<uintptr_t>(dst) & 15) / sizeof(T));
        if (t >= 0 && at >= base && at < end) walk_residue(tb, t, av, tu, F, s_w + mis, (uint32_t)(at - base));
        wave_lds_sync();
        flush_stage(dst, 3 * (end - base), s_w, lane);
        wave_lds_sync();
        base = end;
    }
    if (rn) {
        write_names(tb, t, cnt, at, total, rn, an, reinterpret_cast<uint16_t*>(s_w), lane);
        wave_lds_sync();
    }
}

// Whether an angle may give coordinates out of range.
template <typename T>
__device__ __forceinline__ bool any_wild(const T (&av)[8]) {
    bool suspect = false;
#pragma unroll
    for (int r = 0; r < 8; ++r) suspect |= wild(av[r]);
    return suspect;
}

// The atoms of structures of one block (ang_stride <= kBlock), one wave each.
template <typename T>
__global__ void __launch_bounds__(64 * kGroupWaves) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 3 : 2, 8)))
a2c_fwd_single(const uint8_t* __restrict__ seqs, int seq_stride, const T* __restrict__ angles, int ang_stride,
               T* __restrict__ coords, uint32_t* __restrict__ res_names, uint32_t* __restrict__ atom_names,
               int atoms_stride, Report rep, const int* __restrict__ order, int batch) {
    __shared__ Tables tb;
    __shared__ __align__(16) T s_stage[kGroupWaves][stage_values<T>()];
    const int wave = (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63);
    const int slot = (int)blockIdx.x * kGroupWaves + wave;
    const int b = slot < batch ? structure_at(order, slot, batch, rep) : -1;
    const uint8_t* seq = seqs + (size_t)(b < 0 ? 0 : b) * seq_stride;
    int n = b < 0 ? 0 : wave_length(seq, seq_stride, lane), flags = 0;
    if (n > ang_stride) {
        flags = TPL_A2C_STATUS_LENGTH;
        n = 0;
    }
    T av[8];
    const uint8_t code =
        lane_residue(seq, n, angles + (size_t)(b < 0 ? 0 : b) * 8 * ang_stride, ang_stride, lane, av);
    copy_tables(tb, 64 * kGroupWaves);
    __syncthreads();
    if (b < 0) return;
    T* out = coords + (size_t)b * 3 * atoms_stride;
    uint32_t* rn = res_names ? res_names + (size_t)b * atoms_stride : nullptr;
    uint32_t* an = atom_names ? atom_names + (size_t)b * atoms_stride : nullptr;
    double m[12];
    Turns tu;
    const int t = lane_step(code, tb, av, m, tu);
    const int cnt = t >= 0 ? tb.res_i[t] & 0xff : 0;
    const int cinc = wave_scan_int(cnt);
    const int total = __builtin_amdgcn_readlane(cinc, 63);
    if (__builtin_amdgcn_ballot_w64(lane < n && t < 0)) flags |= TPL_A2C_STATUS_SEQ;
    if (total > atoms_stride) flags |= TPL_A2C_STATUS_ATOMS;
    if (flags) {  // a flagged structure is all zeros
        if (lane == 0) report_bits(rep, (uint32_t)flags);
        zero_share(out, rn, an, 0, atoms_stride, 0, 1, lane);
        return;
    }
    if (any_wild(av)) report_flag(rep, TPLX_A2C_RANGE);
    wave_scan_frames(m);
#pragma unroll
    for (int k = 0; k < 12; ++k) m[k] = dpp_double<kWaveShr1, 0xf>(m[k], ident12(k));
    build_block(tb, t, av, tu, m, cinc - cnt, cnt, total, out, rn, an, s_stage[wave], lane);
    zero_share(out, rn, an, total, atoms_stride, 0, 1, lane);
}

// The blocks that hold residues, as a list that a resident grid's waves share:
// structure by structure, a segment of the batch at a time.  Every workgroup
// sums up the structures' block counts from their lengths, and wave w of W
// takes blocks w, w + W, ... of the list.  One block per wave in a grid over all
// blocks left a CU's slots to waves that found their block past the structure
// and to workgroups with one wave at work, each copying the tables anew: the
// walk of lengths 30-1000 at B=1024 took 38 us, against 31.
constexpr int kWalkWaves = 8;
constexpr int kSegment = 2048;  // structures per segment: their block counts' sums live in LDS
struct BlockList {
    int first[kSegment + 1];  // blocks before a structure of the segment
    uint8_t last[kSegment];   // residues of its last block, less one
    int sum[kWalkWaves];
};

// Fills the list for m structures from their lengths; returns its blocks.
// meanwhile() runs while the lengths are loaded.  Ends with a barrier.
template <typename Meanwhile>
__device__ __forceinline__ int list_blocks(BlockList& l, const int* lens, int m, int wave, int lane,
                                           Meanwhile meanwhile) {
    constexpr int NT = 64 * kWalkWaves, kPer = kSegment / NT;
    int nb[kPer], last[kPer], sum = 0;
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
        const int k = kPer * (int)threadIdx.x + e;
        last[e] = k < m ? lens[k] : 0;
    }
    meanwhile();
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
        nb[e] = (last[e] + kBlock - 1) / kBlock;
        last[e] = (last[e] - 1) & (kBlock - 1);
        sum += nb[e];
    }
    const int inc = wave_scan_int(sum);
    __syncthreads();  // a list before this one is done with
    if (lane == 63) l.sum[wave] = inc;
    __syncthreads();
    int at = inc - sum, blocks = 0;
#pragma unroll
    for (int k = 0; k < kWalkWaves; ++k) {
        at += k < wave ? l.sum[k] : 0;
        blocks += l.sum[k];
    }
#pragma unroll
    for (int e = 0; e < kPer; ++e) {
        l.first[kPer * (int)threadIdx.x + e] = at;
        l.last[kPer * (int)threadIdx.x + e] = (uint8_t)last[e];
        at += nb[e];
    }
    if (threadIdx.x == NT - 1) l.first[kSegment] = at;
    __syncthreads();
    return blocks;
}

// Block `it` of the list: its structure k of the segment (the last one that
// starts at or before it: empty ones share the start of the next), which block
// j of it, and that structure's length n.  All wave-uniform.
__device__ __forceinline__ void find_block(const BlockList& l, int it, int lane, int& k, int& j, int& n) {
    static_assert(kSegment == 64 * 32, "two rounds of comparisons: every 32nd, then 32");
    const int hi = 32 * (__builtin_popcountll(__builtin_amdgcn_ballot_w64(l.first[32 * lane] <= it)) - 1);
    k = hi + __builtin_popcountll(__builtin_amdgcn_ballot_w64(lane < 32 && l.first[hi + (lane & 31)] <= it)) - 1;
    const int first = __builtin_amdgcn_readfirstlane(l.first[k]);
    j = it - first;
    n = kBlock * (__builtin_amdgcn_readfirstlane(l.first[k + 1]) - first - 1) +
        __builtin_amdgcn_readfirstlane((int)l.last[k]) + 1;
}

// The atoms after a2c_fwd_steps, which also took care of the flags and the
// padding: the blocks of the list above.
template <typename T>
__global__ void __launch_bounds__(64 * kWalkWaves) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 4 : 2, 8)))
a2c_fwd_walk(const uint8_t* __restrict__ seqs, int seq_stride, const T* __restrict__ angles, int ang_stride,
             const int* __restrict__ lens, const GroupRec* __restrict__ rec, const GroupFrames* __restrict__ frames,
             T* __restrict__ coords, uint32_t* __restrict__ res_names, uint32_t* __restrict__ atom_names,
             int atoms_stride, Report rep, const int* __restrict__ order, int batch, int ng) {
    __shared__ Tables tb;
    __shared__ __align__(16) T s_stage[kWalkWaves][stage_values<T>()];
    __shared__ BlockList s_list;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (int)(threadIdx.x & 63);
    const int step = (int)gridDim.x * kWalkWaves;
    bool suspect = false;
    for (int base = 0; base < batch; base += kSegment) {
        const int blocks =
            list_blocks(s_list, lens + base, batch - base < kSegment ? batch - base : kSegment, wave, lane, [&] {
                if (base == 0) copy_tables(tb, 64 * kWalkWaves);
            });
        for (int it = (int)blockIdx.x * kWalkWaves + wave; it < blocks; it += step) {
            int k, j, bn;
            find_block(s_list, it, lane, k, j, bn);
            const int b = structure_at(order, base + k, batch, Report{nullptr, nullptr});
            const int g = j / kGroupWaves, part = j % kGroupWaves;
            const int i = kBlock * j + lane;
            const GroupRec* rb = rec + (size_t)b * ng;
            const GroupFrames* gf = frames + ((size_t)b * ng + g);
            T av[8];
            const uint8_t code = lane_residue(seqs + (size_t)b * seq_stride, bn,
                                              angles + (size_t)b * 8 * ang_stride, ang_stride, i, av);
            const int before = __builtin_amdgcn_readfirstlane(rb[g].before[part]);
            double G[12];
            {
                const uint32_t r = kBlock * part + lane, at4 = 64 * (r & 3) + (r >> 2);
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    G[4 * c] = i < bn ? gf->v[c][at4] : 0.0;
                    G[4 * c + 1] = i < bn ? gf->v[3 + c][at4] : 0.0;
                    G[4 * c + 3] = i < bn ? gf->v[6 + c][at4] : 0.0;
                }
            }
            const int t = (int)(int8_t)tb.type[code];
            const int cnt = t >= 0 ? tb.res_i[t] & 0xff : 0;
            const int cinc = wave_scan_int(cnt);
            suspect |= any_wild(av);
#pragma unroll
            for (int c = 0; c < 3; ++c) {  // z = x cross y
                const int p = (c + 1) % 3, q = (c + 2) % 3;
                G[4 * c + 2] = G[4 * p] * G[4 * q + 1] - G[4 * q] * G[4 * p + 1];
            }
            for (int h = g - 1; h >= 0; --h) {  // the groups before
                double M[12];
#pragma unroll
                for (int c = 0; c < 12; ++c) M[c] = G[c];
                compose(rb[h].f, M, G);
            }
            Turns tu;
            sincos_tab((double)av[0], tb.tab, &tu.s[0], &tu.c[0]);
            sincos_tab((double)av[1], tb.tab, &tu.s[1], &tu.c[1]);
            const size_t row = (size_t)b * atoms_stride + before;
            build_block(tb, t, av, tu, G, cinc - cnt, cnt, __builtin_amdgcn_readlane(cinc, 63), coords + 3 * row,
                        res_names ? res_names + row : nullptr, atom_names ? atom_names + row : nullptr,
                        s_stage[wave], lane);
        }
    }
    if (suspect) report_flag(rep, TPLX_A2C_RANGE);
}

// One workgroup per structure, of at most MAXW waves (blockDim / 64, one per
// block of the stride where that fits): the waves take their blocks together,
// whose products meet in LDS.  EU: the waves per SIMD it is held to.
struct BlockRec {
    double f[12];  // the product of its residue steps
    int atoms, flags;
};
template <int MAXW, int EU, typename T>
__global__ void __launch_bounds__(64 * MAXW) __attribute__((amdgpu_waves_per_eu(EU, 8))) a2c_fwd_fused(
    const uint8_t* __restrict__ seqs, int seq_stride, const T* __restrict__ angles, int ang_stride,
    T* __restrict__ coords, uint32_t* __restrict__ res_names, uint32_t* __restrict__ atom_names, int atoms_stride,
    Report rep, const int* __restrict__ order, int batch) {
    __shared__ Tables tb;
    __shared__ uint16_t s_role[MAXW][kBlock * kMaxAtoms];
    __shared__ BlockRec s_rec[MAXW];
    __shared__ int s_sum[2];  // atoms and flags of a structure of more than NW blocks
    const int NW = (int)(blockDim.x >> 6);
    const int wave = turned_wave((int)(threadIdx.x >> 6), NW, (int)blockIdx.x), lane = (int)(threadIdx.x & 63);
    const int b = structure_at(order, (int)blockIdx.x, batch, rep);
    if (b < 0) return;
    const uint8_t* seq = seqs + (size_t)b * seq_stride;
    const T* ang = angles + (size_t)b * 8 * ang_stride;
    copy_tables(tb, 64 * NW);
    if (threadIdx.x < 2) s_sum[threadIdx.x] = 0;
    int n = wave_length(seq, seq_stride, lane), flags = 0;  // every wave alike
    if (n > ang_stride) {
        flags = TPL_A2C_STATUS_LENGTH;
        n = 0;
    }
    const int nb = (n + kBlock - 1) / kBlock;
    __syncthreads();
    int total = 0;
    if (nb > NW) {  // the whole structure's atoms and flags before its first block is written
        int cnt = 0;
        bool bad = false;
        for (int i = (int)threadIdx.x; i < n; i += 64 * NW) {
            const int t = (int)(int8_t)tb.type[seq[i]];
            bad |= t < 0;
            if (t >= 0) cnt += tb.res_i[t] & 0xff;
        }
        atomicAdd(&s_sum[0], cnt);
        if (bad) atomicOr(&s_sum[1], (int)TPL_A2C_STATUS_SEQ);
        __syncthreads();
        total = s_sum[0];
        flags |= s_sum[1];
    }
    T* out = coords + (size_t)b * 3 * atoms_stride;
    uint32_t* rn = res_names ? res_names + (size_t)b * atoms_stride : nullptr;
    uint32_t* an = atom_names ? atom_names + (size_t)b * atoms_stride : nullptr;
    double P[12];
    identity(P);
    int before = 0;
    bool suspect = false;
    if (total > atoms_stride) flags |= TPL_A2C_STATUS_ATOMS;
    for (int k0 = 0; k0 < nb && !flags; k0 += NW) {
        const int j = k0 + wave, i = kBlock * j + lane;
        T av[8];
        double m[12];
        Turns tu;
        int t = -1, cnt = 0, cinc = 0;
        if (j < nb) {
            t = lane_step(lane_residue(seq, n, ang, ang_stride, i, av), tb, av, m, tu);
            cnt = t >= 0 ? tb.res_i[t] & 0xff : 0;
            const bool bad = __builtin_amdgcn_ballot_w64(i < n && t < 0) != 0;
            cinc = wave_scan_int(cnt);
            wave_scan_frames(m);
            if (lane == 63) {
#pragma unroll
                for (int k = 0; k < 12; ++k) s_rec[wave].f[k] = m[k];
                s_rec[wave].atoms = cinc;
                s_rec[wave].flags = bad ? (int)TPL_A2C_STATUS_SEQ : 0;
            }
        }
        __syncthreads();
        const int here = nb - k0 < NW ? nb - k0 : NW;
        int mine = before;
        for (int k = 0; k < here; ++k) {
            if (k < wave) mine += s_rec[k].atoms;
            before += s_rec[k].atoms;
            if (nb <= NW) flags |= s_rec[k].flags;
        }
        if (nb <= NW) {
            total = before;
            if (total > atoms_stride) flags |= TPL_A2C_STATUS_ATOMS;
        }
        if (!flags) {
            fold(P, s_rec, wave < here ? wave : here);
            if (j < nb) {
                double E[12], G[12];
#pragma unroll
                for (int k = 0; k < 12; ++k) E[k] = dpp_double<kWaveShr1, 0xf>(m[k], ident12(k));
                compose(P, E, G);
#pragma unroll
                for (int r = 0; r < 8; ++r) suspect |= wild(av[r]);
                const int at = cinc - cnt;
                if (t >= 0) walk_residue(tb, t, av, tu, G, out + 3 * (size_t)mine, (uint32_t)at);
                if (rn)
                    write_names(tb, t, cnt, at, __builtin_amdgcn_readlane(cinc, 63), rn + mine, an + mine,
                                s_role[wave], lane);
            }
            if (k0 + NW < nb) fold(P, s_rec + wave, here - wave);  // here is NW: P for the next NW blocks
        }
        __syncthreads();
    }
    if (suspect) report_flag(rep, TPLX_A2C_RANGE);
    if (flags) {
        if (threadIdx.x == 0) report_bits(rep, (uint32_t)flags);
        zero_share(out, rn, an, 0, atoms_stride, wave, NW, lane);
    } else if (nb < NW) {  // the waves without a block
        if (wave >= nb) zero_share(out, rn, an, total, atoms_stride, wave - nb, NW - nb, lane);
    } else {
        zero_share(out, rn, an, total, atoms_stride, wave, NW, lane);
    }
}

// ---- forward: a run of residues per thread ----
// One workgroup of 256 or 512 threads per structure, a thread multiplying out
// the steps of up to four consecutive residues and walking them; a workgroup
// scan joins the threads.  Each thread writes its own atoms, so this is the
// better form only where little is written or there is little else to wait for
// (forward_form).

// The 8 angles of residue i, loaded together at the top of the residue so
// that their latencies overlap (one global-load latency per residue walk
// instead of one per transform).
template <typename T>
struct ResAngles {
    T v[8];
    __device__ __forceinline__ void load(const T* ang, int stride, int i) {
#pragma unroll
        for (int r = 0; r < 8; ++r) v[r] = ang[(size_t)r * stride + i];
    }
};

// The residue step S_i applied to m: m <- m T_CA(phi) T_C(psi) T_N(omega).
template <typename T>
__device__ __forceinline__ void residue_step(double m[12], const Tables& tb, const T* ang, int stride, int i) {
    const double phi = (double)ang[i], psi = (double)ang[(size_t)stride + i], omega = (double)ang[(size_t)2 * stride + i];
    double s, c;
    sincos_tab(phi, tb.tab, &s, &c);
    step(m, tb.bb[0][0], tb.bb[0][1], c, s, geo::R_N_CA);
    sincos_tab(psi, tb.tab, &s, &c);
    step(m, tb.bb[1][0], tb.bb[1][1], c, s, geo::R_CA_C);
    sincos_tab(omega, tb.tab, &s, &c);
    step(m, tb.bb[2][0], tb.bb[2][1], c, s, geo::R_C_N);
}

// Per structure: the sequence length (first 0 byte), the residues' validity,
// this thread's run [r0, r1), and the workgroup scans giving the N frame of
// residue r0 (frame) and its first atom (atom0); nothing is left to build if the
// structure is flagged.
template <int NT, typename T>
__device__ void prepare(const uint8_t* seq, int seq_stride, const T* ang, int ang_stride,
                        int atoms_stride, const Report& rep, const Tables& tb, double (*s_m)[NT / 64],
                        int* s_c, int* s_flag, Run& run, double frame[12], ResAngles<T>& av0,
                        uint8_t& code0) {
    const int tid = threadIdx.x;
    if (tid == 0) {
        s_flag[0] = seq_stride;  // length
        s_flag[1] = 0;           // status bits
    }
    __syncthreads();
    find_length<NT>(seq, seq_stride, &s_flag[0]);
    __syncthreads();
    int L = s_flag[0];
    if (L > ang_stride) {
        if (tid == 0) atomicOr(&s_flag[1], (int)TPL_A2C_STATUS_LENGTH);
        L = 0;
    }
    const int chunk = (L + NT - 1) / NT;
    const int r0 = min(L, tid * chunk), r1 = min(L, r0 + chunk);
    // The walk's first residue: its angles and letter are loaded now, so
    // that they arrive while the workgroup scans.
    if (r0 < r1) {
        av0.load(ang, ang_stride, r0);
        code0 = seq[r0];
    }
    double P[12];
    identity(P);
    int cnt = 0;
    bool bad = false;
    for (int i = r0; i < r1; ++i) {
        const int t = residue_type(seq[i]);
        if (t < 0) {
            bad = true;
            continue;
        }
        cnt += tb.res_i[t] & 0xff;
        residue_step(P, tb, ang, ang_stride, i);
    }
    if (bad) atomicOr(&s_flag[1], (int)TPL_A2C_STATUS_SEQ);
    // Ordered product of the runs' steps and sum of their atom counts over
    // the workgroup: inclusive within each wave by DPP, then across waves
    // through LDS (the waves' totals; each wave composes those before it).
    // frame = product of the earlier runs' steps, atom0 = their atoms.
    constexpr int NW = NT / 64;
    const int wv = tid >> 6;
    int cinc = cnt;
    if ((tid & ~63) * chunk < L) {  // a wave whose runs are all past the structure holds identities and zeros
        cinc = wave_scan_int(cnt);
        wave_scan_frames(P);
    }
    if ((tid & 63) == 63) {
#pragma unroll
        for (int k = 0; k < 12; ++k) s_m[k][wv] = P[k];
        s_c[wv] = cinc;
    }
    double E[12];
#pragma unroll
    for (int k = 0; k < 12; ++k) E[k] = dpp_double<kWaveShr1, 0xf>(P[k], ident12(k));
    __syncthreads();
    double W[12];
    identity(W);
    int before = 0, total = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        if (w < wv) {
            double Tw[12], R2[12];
#pragma unroll
            for (int k = 0; k < 12; ++k) Tw[k] = s_m[k][w];
            compose(W, Tw, R2);
#pragma unroll
            for (int k = 0; k < 12; ++k) W[k] = R2[k];
            before += s_c[w];
        }
        total += s_c[w];
    }
    compose(W, E, frame);
    run.atom0 = before + cinc - cnt;
    run.total = total;
    if (run.total > atoms_stride && tid == 0) atomicOr(&s_flag[1], (int)TPL_A2C_STATUS_ATOMS);
    __syncthreads();
    const int flags = s_flag[1];
    if (flags && tid == 0) report_bits(rep, (uint32_t)flags);
    run.L = L;
    run.r0 = r0;
    run.r1 = r1;
    if (flags) run.L = run.r0 = run.r1 = run.total = 0;
}

// At 256 threads the forward is held to four waves per SIMD (<= 128 VGPRs,
// a few dwords spilled) so that four workgroups fit on a CU, as LDS allows:
// 85 -> 71 us at mixed lengths 30-1000, B=1024, against three workgroups.
template <int NT, typename T>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(NT == 256 ? 4 : 1, 8))) a2c_fwd_runs(
    const uint8_t* __restrict__ seqs, int seq_stride, const T* __restrict__ angles, int ang_stride,
    T* __restrict__ coords, uint32_t* __restrict__ res_names, uint32_t* __restrict__ atom_names, int atoms_stride,
    Report rep, const int* __restrict__ order) {
    __shared__ Tables tb;
    __shared__ double s_m[12][NT / 64];  // the waves' products
    __shared__ int s_c[NT / 64];          // the waves' atom counts
    __shared__ int s_flag[2];
    const int b = structure_at(order, (int)blockIdx.x, (int)gridDim.x, rep);
    if (b < 0) return;
    const uint8_t* seq = seqs + (size_t)b * seq_stride;
    const T* ang = angles + (size_t)b * 8 * ang_stride;
    T* out = coords + (size_t)b * 3 * atoms_stride;
    copy_tables(tb, NT);
    __syncthreads();
    Run run;
    double G[12];
    ResAngles<T> av;
    uint8_t code = 0;
    prepare<NT>(seq, seq_stride, ang, ang_stride, atoms_stride, rep, tb, s_m, s_c, s_flag, run, G, av, code);
    int a = run.atom0;
    uint32_t* rn = res_names ? res_names + (size_t)b * atoms_stride : nullptr;
    uint32_t* an = atom_names ? atom_names + (size_t)b * atoms_stride : nullptr;
    for (int i = run.r0; i < run.r1; ++i) {
        if (__builtin_expect(any_wild(av.v), 0)) report_flag(rep, TPLX_A2C_RANGE);
        // the next residue's angles and letter go out before this one's work
        ResAngles<T> nav;
        uint8_t ncode = 0;
        if (i + 1 < run.r1) {
            nav.load(ang, ang_stride, i + 1);
            ncode = seq[i + 1];
        }
        const int t = residue_type(code);
        const int ri = tb.res_i[t];
        const int natoms = ri & 0xff, nca = (ri >> 8) & 0xff, nside = ri >> 16;
        const double* loc = tb.loc[t * kMaxAtoms];
        double x[3];
        auto put = [&](int slot, const double m[12]) {
            apply(m, loc + 3 * slot, x);
            T* o = out + 3 * (size_t)(a + slot);
            o[0] = (T)x[0];
            o[1] = (T)x[1];
            o[2] = (T)x[2];
        };
        put(0, G);
        double s, c, F[12], CA[12];
#pragma unroll
        for (int k = 0; k < 12; ++k) CA[k] = G[k];
        sincos_tab((double)av.v[0], tb.tab, &s, &c);
        step(CA, tb.bb[0][0], tb.bb[0][1], c, s, geo::R_N_CA);
        for (int k = 1; k <= nca; ++k) put(k, CA);
#pragma unroll
        for (int k = 0; k < 12; ++k) F[k] = CA[k];
        SideRows<T> rows(av.v);
        for (int n = 0; n < nside; ++n) {
            const int q = t * kMaxSide + n;
            const int si = tb.side_i[q];
            const int row = (int)(int8_t)(si & 0xff), first = (si >> 8) & 0xff, count = si >> 16;
            double ca = tb.side[q][2], sa = tb.side[q][3];
            if (row >= 0) sincos_tab(rows.pop(), tb.tab, &sa, &ca);
            step(F, tb.side[q][0], tb.side[q][1], ca, sa, tb.side[q][4]);
            for (int k = first; k < first + count; ++k) put(k, F);
        }
        sincos_tab((double)av.v[1], tb.tab, &s, &c);
        step(CA, tb.bb[1][0], tb.bb[1][1], c, s, geo::R_CA_C);  // CA now holds the C frame
        put(natoms - 2, CA);
        put(natoms - 1, CA);
        if (rn) {
            for (int k = 0; k < natoms; ++k) {
                const uint2 names = tb.name[t * kMaxAtoms + k];
                rn[a + k] = names.x;
                an[a + k] = names.y;
            }
        }
        sincos_tab((double)av.v[2], tb.tab, &s, &c);
        step(CA, tb.bb[2][0], tb.bb[2][1], c, s, geo::R_C_N);
#pragma unroll
        for (int k = 0; k < 12; ++k) G[k] = CA[k];
        a += natoms;
        av = nav;
        code = ncode;
    }
    for (int k = 3 * run.total + threadIdx.x; k < 3 * atoms_stride; k += NT) out[k] = (T)0;
    if (rn)
        for (int k = run.total + threadIdx.x; k < atoms_stride; k += NT) rn[k] = an[k] = 0u;
}

struct Sums {
    double g[3], xg[3];
};

__device__ __forceinline__ void sums_zero(Sums& s) {
#pragma unroll
    for (int c = 0; c < 3; ++c) s.g[c] = s.xg[c] = 0.0;
}

__device__ __forceinline__ void sums_add(Sums& s, const double x[3], const double g[3]) {
#pragma unroll
    for (int c = 0; c < 3; ++c) s.g[c] += g[c];
    s.xg[0] += x[1] * g[2] - x[2] * g[1];
    s.xg[1] += x[2] * g[0] - x[0] * g[2];
    s.xg[2] += x[0] * g[1] - x[1] * g[0];
}

// Backward from the forward's coordinates.  A node bound to an angle turns
// its subtree about its x axis through its origin; the origin is the node's
// first atom (every group's first atom sits at the group origin), and the x
// axis is the unit bond vector from the parent node's origin (the transform
// Ry Tx(d) Rx moves the origin by d along Ry's x axis, which Rx keeps), so
// the gradient needs no frames: dL/dalpha = u . (sum x cross g - p cross
// sum g) over the subtree, with u = (p - q) / |p - q| for parent origin q.

// Per structure, without frames: length, validity, this thread's run and its
// first atom (workgroup scan of the atom counts).  Flags as in prepare().
// With s_ra, also each residue's first atom | type << 24 (visible to the
// workgroup after its next barrier).
template <int NT>
__device__ void count_run(const uint8_t* seq, int seq_stride, int ang_stride, int atoms_stride,
                          const Report& rep, const int* res_i, int* s_c, int* s_flag, Run& run,
                          int* s_ra = nullptr) {
    const int tid = threadIdx.x;
    if (tid == 0) {
        s_flag[0] = seq_stride;
        s_flag[1] = 0;
    }
    __syncthreads();
    find_length<NT>(seq, seq_stride, &s_flag[0]);
    __syncthreads();
    int L = s_flag[0];
    if (L > ang_stride) {
        if (tid == 0) atomicOr(&s_flag[1], (int)TPL_A2C_STATUS_LENGTH);
        L = 0;
    }
    // Runs go to threads in reverse order (run q = NT - 1 - tid), so that
    // sums over a run and every later run are prefix sums over threads.
    const int chunk = (L + NT - 1) / NT;
    const int q = NT - 1 - tid;
    const int r0 = min(L, q * chunk), r1 = min(L, r0 + chunk);
    int cnt = 0;
    bool bad = false;
    for (int i = r0; i < r1; ++i) {
        const int t = residue_type(seq[i]);
        if (t < 0) {
            bad = true;
        } else {
            if (s_ra) s_ra[i] = cnt | (t << 24);
            cnt += res_i[t] & 0xff;
        }
    }
    if (bad) atomicOr(&s_flag[1], (int)TPL_A2C_STATUS_SEQ);
    // atoms of this run and the later ones: prefix over threads, by DPP
    // within the wave and the earlier waves' totals through LDS
    constexpr int NW = NT / 64;
    const int wv = tid >> 6;
    const int cinc = wave_scan_int(cnt);
    if ((tid & 63) == 63) s_c[wv] = cinc;
    __syncthreads();
    int before = 0, total = 0;
#pragma unroll
    for (int w = 0; w < NW; ++w) {
        if (w < wv) before += s_c[w];
        total += s_c[w];
    }
    run.total = total;
    run.atom0 = total - (before + cinc);  // atoms of the runs before this one
    if (s_ra)
        for (int i = r0; i < r1; ++i) s_ra[i] += run.atom0;
    if (run.total > atoms_stride && tid == 0) atomicOr(&s_flag[1], (int)TPL_A2C_STATUS_ATOMS);
    __syncthreads();
    const int flags = s_flag[1];
    if (flags && tid == 0) report_bits(rep, (uint32_t)flags);
    run.L = L;
    run.r0 = r0;
    run.r1 = r1;
    if (flags) run.L = run.r0 = run.r1 = run.total = 0;
}

template <typename T>
__device__ __forceinline__ void load3(const T* p, double v[3]) {
    v[0] = (double)p[0];
    v[1] = (double)p[1];
    v[2] = (double)p[2];
}

// Sums over atoms [k0, k1) of a structure.  With UNROLL, four atoms at a time
// with their loads issued first.  This kernel now serves small batches,
// where it is latency-bound: at 512 threads, 32 x 350 residues 18.0 -> 16.9
// us, one structure of 1000 36.0 -> 33.9, 64 x 1000 43.9 -> 41.0.  At 256
// threads the extra registers cost a wave per SIMD (1024 x 30: 13.9 -> 18.7
// us), so it stays off there.  (When this kernel also served B=1024 of
// mixed lengths 30-1000, unrolling measured slower there: 153 -> 204 us.)
template <bool UNROLL, typename T>
__device__ __forceinline__ void atom_sums(const T* xs, const T* gs, int k0, int k1, Sums& acc) {
    int k = k0;
    if (UNROLL) {
        for (; k + 4 <= k1; k += 4) {
            double x[4][3], g[4][3];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                load3(xs + 3 * (size_t)(k + j), x[j]);
                load3(gs + 3 * (size_t)(k + j), g[j]);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) sums_add(acc, x[j], g[j]);
        }
    }
    for (; k < k1; ++k) {
        double x[3], g[3];
        load3(xs + 3 * (size_t)k, x);
        load3(gs + 3 * (size_t)k, g);
        sums_add(acc, x, g);
    }
}

// u . (xg - p cross g) with u the unit vector from q to p.
__device__ __forceinline__ double bond_torque(const double p[3], const double q[3], const Sums& s) {
    const double d0 = p[0] - q[0], d1 = p[1] - q[1], d2 = p[2] - q[2];
    const double inv = 1.0 / sqrt(d0 * d0 + d1 * d1 + d2 * d2);
    const double v0 = s.xg[0] - (p[1] * s.g[2] - p[2] * s.g[1]);
    const double v1 = s.xg[1] - (p[2] * s.g[0] - p[0] * s.g[2]);
    const double v2 = s.xg[2] - (p[0] * s.g[1] - p[1] * s.g[0]);
    return (d0 * v0 + d1 * v1 + d2 * v2) * inv;
}

template <int NT, typename T>
__global__ void __launch_bounds__(NT) a2c_bwd(const uint8_t* __restrict__ seqs, int seq_stride,
                                              const T* __restrict__ coords, const T* __restrict__ grad_coords,
                                              int atoms_stride, T* __restrict__ grad_angles, int ang_stride,
                                              Report rep, const int* __restrict__ order) {
    __shared__ int s_res[kTypes];
    __shared__ int s_side[kTypes * kMaxSide];
    __shared__ double s_v[6][NT / 64];  // the waves' sums
    __shared__ int s_c[NT / 64];        // the waves' atom counts
    __shared__ int s_flag[2];
    const int b = structure_at(order, (int)blockIdx.x, (int)gridDim.x, rep), tid = threadIdx.x;
    if (b < 0) return;
    const uint8_t* seq = seqs + (size_t)b * seq_stride;
    const T* xs = coords + (size_t)b * 3 * atoms_stride;
    const T* gs = grad_coords + (size_t)b * 3 * atoms_stride;
    T* ga = grad_angles + (size_t)b * 8 * ang_stride;
    for (int k = tid; k < kTypes * kMaxSide; k += NT) {
        const Side sd = kSide[k / kMaxSide][k % kMaxSide];
        s_side[k] = (sd.row & 0xff) | (sd.first << 8) | (sd.count << 16);
    }
    if (tid < kTypes) {
        const Residue r = kRes[tid];
        s_res[tid] = r.natoms | (r.nca << 8) | (r.nside << 16);
    }
    __syncthreads();
    Run run;
    count_run<NT>(seq, seq_stride, ang_stride, atoms_stride, rep, s_res, s_c, s_flag, run);
    // pass A: this run's (sum g, sum x cross g)
    Sums run_sum;
    sums_zero(run_sum);
    {
        int a = run.atom0;
        for (int i = run.r0; i < run.r1; ++i) a += s_res[residue_type(seq[i])] & 0xff;
        atom_sums<NT == kThreadsLarge>(xs, gs, run.atom0, a, run_sum);
    }
    // incl = sums over every atom from this run on: runs are in reverse
    // thread order, so an inclusive prefix sum over threads (DPP within the
    // wave, then the earlier waves' totals through LDS)
    double v[6];
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        v[c] = run_sum.g[c];
        v[3 + c] = run_sum.xg[c];
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) v[k] = wave_scan_double(v[k]);
    if ((tid & 63) == 63) {
#pragma unroll
        for (int k = 0; k < 6; ++k) s_v[k][tid >> 6] = v[k];
    }
    __syncthreads();
    for (int w = 0; w < (tid >> 6); ++w) {
#pragma unroll
        for (int k = 0; k < 6; ++k) v[k] += s_v[k][w];
    }
    Sums incl;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        incl.g[c] = v[c];
        incl.xg[c] = v[3 + c];
    }
    // pass B: gradients, residue by residue
    int a = run.atom0;
    bool range = false;
    const auto put = [&](size_t at, double v) {
        ga[at] = (T)v;
        range |= out_of_range((T)v);
    };
    for (int i = run.r0; i < run.r1; ++i) {
        const int t = residue_type(seq[i]);
        const int ri = s_res[t];
        const int natoms = ri & 0xff, nca = (ri >> 8) & 0xff, nside = ri >> 16;
        Sums sN, sCA, sSide, sC, excl, s;
        sums_zero(sN);
        sums_zero(sCA);
        sums_zero(sSide);
        sums_zero(sC);
        atom_sums<NT == kThreadsLarge>(xs, gs, a, a + 1, sN);
        atom_sums<NT == kThreadsLarge>(xs, gs, a + 1, a + 1 + nca, sCA);
        atom_sums<NT == kThreadsLarge>(xs, gs, a + natoms - 2, a + natoms, sC);
        double pN[3], pCA[3], pC[3];
        load3(xs + 3 * (size_t)a, pN);
        load3(xs + 3 * (size_t)(a + 1), pCA);
        load3(xs + 3 * (size_t)(a + natoms - 2), pC);
        for (int r = 3; r < 8; ++r) ga[(size_t)r * ang_stride + i] = (T)0;
        // side chain, last node first, so that sSide holds node n's group and
        // the later nodes' groups when node n is reached (each atom read
        // once).  Node n hangs on node n-1, or on CA when n-1 is the fixed
        // first node (no atoms, at CA's origin; every other node has atoms).
        for (int n = nside - 1; n >= 0; --n) {
            const int si = s_side[t * kMaxSide + n];
            const int row = (int)(int8_t)(si & 0xff), first = (si >> 8) & 0xff, count = si >> 16;
            if (count == 0) continue;
            atom_sums<NT == kThreadsLarge>(xs, gs, a + first, a + first + count, sSide);
            if (row >= 0) {
                const int sp = n > 0 ? s_side[t * kMaxSide + n - 1] : 0;
                const int pfirst = (sp >> 8) & 0xff, pcount = sp >> 16;
                double p[3], q[3];
                load3(xs + 3 * (size_t)(a + first), p);
                if (pcount > 0)
                    load3(xs + 3 * (size_t)(a + pfirst), q);
                else
                    q[0] = pCA[0], q[1] = pCA[1], q[2] = pCA[2];
                put((size_t)row * ang_stride + i, bond_torque(p, q, sSide));
            }
        }
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            excl.g[c] = incl.g[c] - (sN.g[c] + sCA.g[c] + sSide.g[c] + sC.g[c]);
            excl.xg[c] = incl.xg[c] - (sN.xg[c] + sCA.xg[c] + sSide.xg[c] + sC.xg[c]);
        }
        // omega of residue i-1 binds N_i (on the previous C): the whole residue and everything after
        if (i > 0) {
            double pCp[3];
            load3(xs + 3 * (size_t)(a - 2), pCp);
            put((size_t)2 * ang_stride + i - 1, bond_torque(pN, pCp, incl));
        }
        if (i == run.L - 1) ga[(size_t)2 * ang_stride + i] = (T)0;
        // phi binds CA (on N): all but N
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            s.g[c] = incl.g[c] - sN.g[c];
            s.xg[c] = incl.xg[c] - sN.xg[c];
        }
        put(i, bond_torque(pCA, pN, s));
        // psi binds C (on CA): the C group and everything after
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            s.g[c] = sC.g[c] + excl.g[c];
            s.xg[c] = sC.xg[c] + excl.xg[c];
        }
        put((size_t)ang_stride + i, bond_torque(pC, pCA, s));
        incl = excl;
        a += natoms;
    }
    if (range) report_flag(rep, TPLX_A2C_RANGE);
    // angles past the sequence (and every angle of a flagged structure)
    for (int k = tid; k < 8 * ang_stride; k += NT)
        if (k % ang_stride >= run.L) ga[k] = (T)0;
}

// ---- backward over atom tiles ----
// The run-per-thread backward above makes every load of a wave touch 64
// cache lines (the lanes' runs lie far apart), and it reads each atom twice.
// This one walks a structure from its end in tiles of up to kTileAtoms
// consecutive atoms, cut at residue starts: thread t takes the tile's atoms
// hi-1-Kt ... hi-K-Kt, so a wave's loads cover consecutive atoms, and each
// atom is read once.  Per tile: a workgroup prefix scan over threads (in
// descending atom order, so a suffix over atoms) of (sum g, sum x cross g)
// plus the carry from the later tiles gives the suffix sum SUF[k] at every
// atom; every node's subtree is a suffix (backbone nodes: from the node's
// origin on) or a suffix minus the suffix at the residue's C (side-chain
// nodes: side groups are contiguous and end right before C), so the thread
// holding a node's origin atom writes that node's gradient.  The next tile's
// atoms are loaded while the current one is processed.
constexpr int kTileThreads = 512;
constexpr int kTileK = 2;                                   // atoms per thread and tile
constexpr int kTileAtoms = kTileThreads * kTileK;           // 1024
constexpr int kTileRes = kTileAtoms / 4;                    // residues per tile at most (4 atoms or more each)
constexpr int kTileStride = kTileAtoms - (kMaxAtoms - 1);   // tile p starts at the first residue starting at or after p * this
constexpr int kTileMaxRes = 2048;                           // residues per structure (the residue starts live in LDS)
constexpr int kTileMaxTiles = kTileMaxRes * kMaxAtoms / kTileStride + 1;

// 1 / sqrt(x) for x > 0: the hardware estimate and two Newton steps
// (each squares the relative error).
__device__ __forceinline__ double rsqrt_nr(double x) {
    double y = __builtin_amdgcn_rsq(x);
    const double h = 0.5 * x;
    y = y * (1.5 - h * y * y);
    y = y * (1.5 - h * y * y);
    return y;
}

// u . (xg - p cross g) with u the unit vector from q to p (bond_torque with
// the reciprocal square root above).
__device__ __forceinline__ double bond_torque_rsq(const double p[3], const double q[3], const double s[6]) {
    const double d0 = p[0] - q[0], d1 = p[1] - q[1], d2 = p[2] - q[2];
    const double v0 = s[3] - (p[1] * s[2] - p[2] * s[1]);
    const double v1 = s[4] - (p[2] * s[0] - p[0] * s[2]);
    const double v2 = s[5] - (p[0] * s[1] - p[1] * s[0]);
    return (d0 * v0 + d1 * v1 + d2 * v2) * rsqrt_nr(d0 * d0 + d1 * d1 + d2 * d2);
}

// The tile's atoms of this thread; atoms below lo read atom lo (in bounds)
// and are zeroed.
template <typename T>
__device__ __forceinline__ void load_tile_atoms(const T* xs, const T* gs, int lo, int hi, T (&x)[kTileK][3],
                                                T (&g)[kTileK][3]) {
#pragma unroll
    for (int m = 0; m < kTileK; ++m) {
        const int k = hi - 1 - (kTileK * (int)threadIdx.x + m);
        const size_t kc = 3 * (size_t)(k >= lo ? k : lo);
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            x[m][c] = xs[kc + c];
            g[m][c] = gs[kc + c];
        }
        if (k < lo) {
#pragma unroll
            for (int c = 0; c < 3; ++c) x[m][c] = g[m][c] = (T)0;
        }
    }
}

template <typename T>
__global__ void __launch_bounds__(kTileThreads) __attribute__((amdgpu_waves_per_eu(4, 8))) a2c_bwd_tiled(const uint8_t* __restrict__ seqs, int seq_stride,
                                                              const T* __restrict__ coords,
                                                              const T* __restrict__ grad_coords, int atoms_stride,
                                                              T* __restrict__ grad_angles, int ang_stride,
                                                              Report rep, const int* __restrict__ order) {
    constexpr int NT = kTileThreads, NW = NT / 64, K = kTileK;
    __shared__ int s_res[kTypes];                   // natoms | nca << 8 | nside << 16 | bound rows << 24
    __shared__ int s_side[kTypes * kMaxSide];       // row & 0xff | first << 8 | count << 16
    __shared__ uint32_t s_slot[kTypes * kMaxAtoms]; // per (type, slot): the role bits (tile_roles)
    __shared__ int s_ra[kTileMaxRes];               // residue's first atom | type << 24
    __shared__ int s_tile[kTileMaxTiles];           // each tile's first residue
    __shared__ uint32_t s_role[2][kTileAtoms];      // tile atoms' roles (tile_roles)
    __shared__ T s_x[2][3 * kTileAtoms];            // tile atoms' positions
    __shared__ double s_cs[kTileRes][6];            // suffix sums at each tile residue's C
    __shared__ double s_v[6][NW];                   // the waves' sums
    __shared__ int s_c[NW];
    __shared__ int s_flag[2];
    const int b = structure_at(order, (int)blockIdx.x, (int)gridDim.x, rep), tid = threadIdx.x;
    if (b < 0) return;
    const uint8_t* seq = seqs + (size_t)b * seq_stride;
    const T* xs = coords + (size_t)b * 3 * atoms_stride;
    const T* gs = grad_coords + (size_t)b * 3 * atoms_stride;
    T* ga = grad_angles + (size_t)b * 8 * ang_stride;
    for (int k = tid; k < kTypes * kMaxSide; k += NT) {
        const Side sd = kSide[k / kMaxSide][k % kMaxSide];
        s_side[k] = (sd.row & 0xff) | (sd.first << 8) | (sd.count << 16);
    }
    if (tid < kTypes) {
        const Residue r = kRes[tid];
        s_res[tid] = r.natoms | (r.nca << 8) | (r.nside << 16);
    }
    __syncthreads();
    // Per (type t, atom slot s), the role bits of tile_roles but the
    // residue's index: whether the atom is the origin of a node with an
    // angle, the angle's row, whether that angle belongs to the previous
    // residue (omega, on N, from the previous C two atoms back), how many
    // atoms back the parent node's origin lies, whether the node is a side
    // one, whether the atom is C.  A side node hangs on the node before it,
    // or on CA when that one is the fixed first node without atoms.  And per
    // type, the side rows (3..7) it writes: nodes with atoms and a bound
    // angle.
    for (int k = tid; k < kTypes * kMaxAtoms; k += NT) {
        const int t = k / kMaxAtoms, s = k % kMaxAtoms;
        const int natoms = s_res[t] & 0xff, nside = (s_res[t] >> 16) & 0xff;
        uint32_t role = s == natoms - 2 ? 1u << 18 : 0u;
        if (s == 0)
            role |= (1u << 8) | (2u << 9) | (1u << 12) | (2u << 13);  // omega: N on the previous C
        else if (s == 1)
            role |= (1u << 8) | (0u << 9) | (1u << 13);  // phi: CA on N
        else if (s == natoms - 2)
            role |= (1u << 8) | (1u << 9) | ((uint32_t)(s - 1) << 13);  // psi: C on CA
        else if (s < natoms)
            for (int n = 0; n < nside; ++n) {
                const int si = s_side[t * kMaxSide + n];
                const int row = (int)(int8_t)(si & 0xff), first = (si >> 8) & 0xff, count = si >> 16;
                if (count > 0 && row >= 0 && first == s) {
                    const int sp = n > 0 ? s_side[t * kMaxSide + n - 1] : 0;
                    const int parent = (sp >> 16) > 0 ? (sp >> 8) & 0xff : 1;
                    role |= (1u << 8) | ((uint32_t)row << 9) | ((uint32_t)(s - parent) << 13) | (1u << 17);
                }
            }
        s_slot[k] = role;
    }
    int bound = 0;
    if (tid < kTypes) {
        for (int n = 0; n < ((s_res[tid] >> 16) & 0xff); ++n) {
            const int si = s_side[tid * kMaxSide + n];
            if ((si >> 16) > 0 && (int)(int8_t)(si & 0xff) >= 0) bound |= 1 << (si & 0xff);
        }
    }
    __syncthreads();
    if (tid < kTypes) s_res[tid] |= bound << 24;
    Run run;
    count_run<NT>(seq, seq_stride, ang_stride, atoms_stride, rep, s_res, s_c, s_flag, run, s_ra);
    __syncthreads();
    const int L = run.L;
    for (int i = tid; i < L; i += NT) {
        const int p = (s_ra[i] & 0xffffff) / kTileStride;
        if (i == 0 || p != (s_ra[i - 1] & 0xffffff) / kTileStride) s_tile[p] = i;
    }
    __syncthreads();
    const int ntiles = L > 0 ? (s_ra[L - 1] & 0xffffff) / kTileStride + 1 : 0;
    const size_t stride = (size_t)ang_stride;
    // Roles of tile p's atoms into s_role[p & 1], one residue per thread:
    // bits 0-7 the residue's index in the tile, bit 8 set if the atom is the
    // origin of a node with an angle, bits 9-11 that angle's row, bit 12 if
    // it belongs to the previous residue (omega, on N), bits 13-16 how many
    // atoms back the parent node's origin lies, bit 17 for side-chain nodes
    // (the suffix at C is subtracted), bit 18 if the atom is the residue's
    // C.  The thread also writes the residue's angles that no node carries:
    // the side rows its type does not bind, and omega of the last residue.
    auto tile_roles = [&](int p) {
        const int ilo = s_tile[p], ihi = p + 1 < ntiles ? s_tile[p + 1] : L;
        const int lo = s_ra[ilo] & 0xffffff;
        if (tid < ihi - ilo) {
            const int i = ilo + tid, ra = s_ra[i];
            const int a = ra & 0xffffff, t = ra >> 24, rt = s_res[t], n = rt & 0xff;
#pragma unroll
            for (int s = 0; s < kMaxAtoms; ++s)
                if (s < n) {
                    uint32_t role = s_slot[t * kMaxAtoms + s] | (uint32_t)tid;
                    if (s == 0 && i == 0) role &= ~(1u << 8);  // the first residue has no omega before it
                    s_role[p & 1][a - lo + s] = role;
                }
            const int bnd = (int)((uint32_t)rt >> 24);
            for (int r = 3; r < 8; ++r)
                if (!((bnd >> r) & 1)) ga[r * stride + i] = (T)0;
            if (i == L - 1) ga[2 * stride + i] = (T)0;
        }
    };
    double carry[6];
#pragma unroll
    for (int c = 0; c < 6; ++c) carry[c] = 0.0;
    bool range = false;
    T cx[K][3], cg[K][3];
    int lo = 0, hi = 0;
    if (ntiles > 0) {
        lo = s_ra[s_tile[ntiles - 1]] & 0xffffff;
        hi = run.total;
        load_tile_atoms(xs, gs, lo, hi, cx, cg);
        tile_roles(ntiles - 1);
        __syncthreads();
    }
    for (int p = ntiles - 1; p >= 0; --p) {
        const int buf = p & 1;
        const int ilo = s_tile[p];
        // the previous residue's C (omega of residue ilo - 1 turns about the
        // bond from it), then the next (lower) tile's atoms
        T qprev[3] = {(T)0, (T)0, (T)0};
        if (ilo > 0) {
#pragma unroll
            for (int c = 0; c < 3; ++c) qprev[c] = xs[3 * (size_t)(lo - 2) + c];
        }
        T nx[K][3], ng[K][3];
        const int nlo = p > 0 ? s_ra[s_tile[p - 1]] & 0xffffff : 0;
        load_tile_atoms(xs, gs, nlo, p > 0 ? lo : nlo, nx, ng);
        // this tile's positions, for the parent origins; the next tile's roles
#pragma unroll
        for (int m = 0; m < K; ++m) {
            const int k = hi - 1 - (K * tid + m);
            if (k >= lo) {
#pragma unroll
                for (int c = 0; c < 3; ++c) s_x[buf][3 * (k - lo) + c] = cx[m][c];
            }
        }
        if (p > 0) tile_roles(p - 1);
        // per atom: the node whose origin it is, its angle's slot in ga, its
        // parent's origin in s_x (-1: qprev), whether the suffix at C is
        // subtracted, and whether the atom is a C
        int dst[K], qi[K], il[K];
        bool sub[K], isc[K];
#pragma unroll
        for (int m = 0; m < K; ++m) {
            const int k = hi - 1 - (K * tid + m);
            const uint32_t role = k >= lo ? s_role[buf][k - lo] : 0u;
            il[m] = role & 0xff;
            dst[m] = (role >> 8) & 1 ? (int)((role >> 9) & 7) * ang_stride + ilo + il[m] - (int)((role >> 12) & 1) : -1;
            qi[m] = k - (int)((role >> 13) & 15) - lo;
            sub[m] = (role >> 17) & 1;
            isc[m] = k >= lo && ((role >> 18) & 1);
        }
        // (g, x cross g) per atom; the thread's sum; prefix over threads
        double w[K][6], tot[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) tot[c] = 0.0;
#pragma unroll
        for (int m = 0; m < K; ++m) {
            const double x0 = (double)cx[m][0], x1 = (double)cx[m][1], x2 = (double)cx[m][2];
            const double g0 = (double)cg[m][0], g1 = (double)cg[m][1], g2 = (double)cg[m][2];
            w[m][0] = g0;
            w[m][1] = g1;
            w[m][2] = g2;
            w[m][3] = x1 * g2 - x2 * g1;
            w[m][4] = x2 * g0 - x0 * g2;
            w[m][5] = x0 * g1 - x1 * g0;
#pragma unroll
            for (int c = 0; c < 6; ++c) tot[c] += w[m][c];
        }
        double incl[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) incl[c] = wave_scan_double(tot[c]);
        if ((tid & 63) == 63) {
#pragma unroll
            for (int c = 0; c < 6; ++c) s_v[c][tid >> 6] = incl[c];
        }
        __syncthreads();
        // SUF at the thread's atoms: carry (later tiles) + later waves +
        // later lanes + the thread's atoms from the highest down.  Lane v of
        // every wave takes wave v's total and a row scan makes them
        // inclusive over waves (NW <= 16), read back with readlane.
        const int lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
        double wt[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) wt[c] = row_scan_double(lane < NW ? s_v[c][lane] : 0.0);
        double suf[K][6];
#pragma unroll
        for (int c = 0; c < 6; ++c) {
            const double all = readlane_double(wt[c], NW - 1);
            const double before = wv > 0 ? readlane_double(wt[c], wv - 1) : 0.0;
            double acc = carry[c] + before + (incl[c] - tot[c]);
#pragma unroll
            for (int m = 0; m < K; ++m) {
                acc += w[m][c];
                suf[m][c] = acc;
            }
            carry[c] += all;
        }
#pragma unroll
        for (int m = 0; m < K; ++m)
            if (isc[m]) {
#pragma unroll
                for (int c = 0; c < 6; ++c) s_cs[il[m]][c] = suf[m][c];
            }
        __syncthreads();
        // gradients of the nodes whose origins this thread holds
#pragma unroll
        for (int m = 0; m < K; ++m) {
            if (dst[m] < 0) continue;
            const double p3[3] = {(double)cx[m][0], (double)cx[m][1], (double)cx[m][2]};
            double q[3], sm[6];
            const int qk = qi[m] >= 0 ? qi[m] : 0;
#pragma unroll
            for (int c = 0; c < 3; ++c) q[c] = (double)(qi[m] >= 0 ? s_x[buf][3 * qk + c] : qprev[c]);
#pragma unroll
            for (int c = 0; c < 6; ++c) sm[c] = sub[m] ? suf[m][c] - s_cs[il[m]][c] : suf[m][c];
            const T v = (T)bond_torque_rsq(p3, q, sm);
            range |= out_of_range(v);
            ga[dst[m]] = v;
        }
        hi = lo;
        lo = nlo;
#pragma unroll
        for (int m = 0; m < K; ++m)
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                cx[m][c] = nx[m][c];
                cg[m][c] = ng[m][c];
            }
    }
    if (range) report_flag(rep, TPLX_A2C_RANGE);
    // angles past the sequence (and every angle of a flagged structure)
    for (int k = tid; k < 8 * ang_stride; k += NT)
        if (k % ang_stride >= L) ga[k] = (T)0;
}

// ---- backward: one lane per residue ----
// As in the forward, a wave takes a block of 64 consecutive residues, one per
// lane, the last residue first: sums over a residue's subtree run over the
// later residues, so they are prefixes over the lanes.  The block's atoms and
// their gradients come through the wave's LDS (coalesced loads, each read
// once), and a lane sums its residue's groups from the end: C and O, then the
// side chain, whose angles' gradients follow at once (their subtrees end
// with the residue), CA, N.  A scan of the residues' sums over the lanes and
// the sums of the later blocks give the backbone angles' subtrees.
//   * a2c_bwd_sums + a2c_bwd_walk: the first kernel leaves each block's sums in
//     the caller's workspace (and writes the zeros past the structures), the
//     second takes the blocks of the list (list_blocks);
//   * a2c_bwd_fused: one workgroup per structure, whose waves' sums meet in
//     LDS.  One launch, no workspace.
// Against runs of residues per thread, or atom tiles walked by one workgroup per
// structure (which some batches still take: backward_form), us: lengths 30-1000 at
// B=1024 94 -> 60 (60 -> 60 with the structures ordered by size), in float64 168 ->
// 95; 256 x 1000 50 -> 33, 1 x 1000 34 -> 17, 32 x 350 16.8 -> 15.1, 1024 x 128
// 39 -> 15, 1024 x 30 13.6 -> 9.0, one peptide of 21 in float64 11.3 -> 7.8.  What
// bounds it: the LDS that a block's atoms take holds eight
// waves on a CU, and those wait on latencies two thirds of their time.
struct alignas(16) BackTables {
    int res_i[kTypes];              // natoms | nca << 8 | nside << 16
    int side_i[kTypes * kMaxSide];  // row & 0xff | first << 8 | count << 16
    uint8_t type[256];              // residue type of a letter, 0xff: none
    uint8_t atoms[256];             // its atoms, 0: none
};

constexpr BackTables make_back_tables() {
    constexpr Residue res[kTypes] = A2C_RESIDUES;
    constexpr Side side[kTypes][kMaxSide] = A2C_SIDES;
    BackTables t{};
    for (int c = 0; c < 256; ++c) t.type[c] = 0xff;
    for (int k = 0; k < kTypes; ++k) {
        t.res_i[k] = res[k].natoms | (res[k].nca << 8) | (res[k].nside << 16);
        for (int n = 0; n < kMaxSide; ++n)
            t.side_i[k * kMaxSide + n] = (side[k][n].row & 0xff) | (side[k][n].first << 8) | (side[k][n].count << 16);
        t.type[(uint8_t)kCodes[k]] = (uint8_t)k;
        t.atoms[(uint8_t)kCodes[k]] = (uint8_t)res[k].natoms;
    }
    return t;
}
__constant__ BackTables kBack = make_back_tables();

__device__ __forceinline__ void copy_back_tables(BackTables& tb, int nt) {
    const uint4* src = reinterpret_cast<const uint4*>(&kBack);
    uint4* dst = reinterpret_cast<uint4*>(&tb);
    for (int k = threadIdx.x; k < (int)(sizeof(BackTables) / 16); k += nt) dst[k] = src[k];
}

// Atoms staged at a time (in float64 a block takes two rounds, so that eight
// waves fit on a CU), and the values per array: those atoms', two more atoms
// before them (the C and O of the residue before), the offset that aligns both
// sides, and what makes it whole 16-byte blocks: the gradients' array follows
// the coordinates', and both are written in such blocks.
template <typename T>
constexpr int back_stage() {
    return sizeof(T) == 4 ? 576 : 288;
}
template <typename T>
constexpr int back_values() {
    constexpr int V = 16 / (int)sizeof(T);
    return (3 * (back_stage<T>() + 2) + V + V - 1) / V * V;
}
static_assert(back_values<float>() * sizeof(float) % 16 == 0 && back_values<double>() * sizeof(double) % 16 == 0,
              "the staged arrays stand one after another at 16-byte alignment");

// A run of values on its way from memory to the wave's LDS: fetch() issues the
// loads (16 bytes per lane where src is aligned), commit() writes them to LDS,
// whose s_w[0] holds the value of src rounded down to 16 bytes (flush_stage's
// layout).  The two stand apart, so that other work hides the loads.
template <typename T>
struct Fetch {
    static constexpr int V = 16 / (int)sizeof(T);
    static constexpr int kBody = (back_values<T>() + 64 * V - 1) / (64 * V);
    uint4 body[kBody];
    T head, tail;

    __device__ __forceinline__ static int offset(const T* src) {
        return (int)((reinterpret_cast<uintptr_t>(src) & 15) / sizeof(T));
    }
    __device__ __forceinline__ void fetch(const T* src, int count, int lane) {
        const int mis = offset(src), end = mis + count, first = mis ? V : 0, last = end / V * V;
        const T* d0 = src - mis;
        head = tail = (T)0;
        if (mis && lane >= mis && lane < V && lane < end) head = d0[lane];
#pragma unroll
        for (int e = 0; e < kBody; ++e) {
            const int k = first + V * (64 * e + lane);
            body[e] = make_uint4(0, 0, 0, 0);
            if (k < last) body[e] = *reinterpret_cast<const uint4*>(d0 + k);
        }
        const int t = (last > first ? last : first) + lane;
        if (t < end) tail = d0[t];
    }
    __device__ __forceinline__ void commit(const T* src, int count, T* s_w, int lane) const {
        const int mis = offset(src), end = mis + count, first = mis ? V : 0, last = end / V * V;
        if (mis && lane >= mis && lane < V && lane < end) s_w[lane] = head;
#pragma unroll
        for (int e = 0; e < kBody; ++e) {
            const int k = first + V * (64 * e + lane);
            if (k < last) *reinterpret_cast<uint4*>(s_w + k) = body[e];
        }
        const int t = (last > first ? last : first) + lane;
        if (t < end) s_w[t] = tail;
    }
};

// s += the sums (g, x cross g) of atoms [k0, k1) of the staged x and g.
template <typename T>
__device__ __forceinline__ void staged_sums(const T* x, const T* g, int k0, int k1, double s[6]) {
    for (int k = k0; k < k1; ++k) {
        double p[3], h[3];
        load3(x + 3 * k, p);
        load3(g + 3 * k, h);
        s[0] += h[0];
        s[1] += h[1];
        s[2] += h[2];
        s[3] += p[1] * h[2] - p[2] * h[1];
        s[4] += p[2] * h[0] - p[0] * h[2];
        s[5] += p[0] * h[1] - p[1] * h[0];
    }
}

// What a lane keeps of its residue for the backbone angles.
template <typename T>
struct BackResidue {
    double sc[6];  // sums over C and O
    double sa[6];  // over the side chain and CA's group
    double sn[6];  // over N
    T n[3], ca[3], c[3], prev[3];  // origins, prev: the C before
};

// The lane's residue of type t from its staged atoms x and g: its sums and
// origins, and its side chain's gradients (0 for the rows it does not bind).
// Returns whether a gradient is out of range.
template <typename T>
__device__ __forceinline__ bool back_residue(const BackTables& tb, int t, bool first, const T* x, const T* g,
                                             BackResidue<T>& r, T* ga, uint32_t stride, uint32_t i) {
    const int ri = tb.res_i[t];
    const int natoms = ri & 0xff, nca = (ri >> 8) & 0xff, nside = ri >> 16;
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        r.n[c] = x[c];
        r.ca[c] = x[3 + c];
        r.c[c] = x[3 * (natoms - 2) + c];
        r.prev[c] = first ? (T)0 : x[c - 6];
    }
#pragma unroll
    for (int k = 0; k < 6; ++k) r.sc[k] = r.sa[k] = r.sn[k] = 0.0;
    staged_sums(x, g, natoms - 2, natoms, r.sc);
    bool range = false;
    int bound = 0;
    int si = nside > 0 ? tb.side_i[t * kMaxSide + nside - 1] : 0;
    for (int n = nside - 1; n > 0; --n) {  // node 0 is fixed and has no atoms
        const int sp = tb.side_i[t * kMaxSide + n - 1];
        const int row = (int)(int8_t)(si & 0xff), first_atom = (si >> 8) & 0xff, count = si >> 16;
        staged_sums(x, g, first_atom, first_atom + count, r.sa);
        if (row >= 0) {
            // the parent's origin: the node before, or CA for the first
            const int parent = (sp >> 16) > 0 ? (sp >> 8) & 0xff : 1;
            double p[3], q[3];
            load3(x + 3 * first_atom, p);
            load3(x + 3 * parent, q);
            const T v = (T)bond_torque_rsq(p, q, r.sa);
            range |= out_of_range(v);
            ga[(uint32_t)row * stride + i] = v;
            bound |= 1 << row;
        }
        si = sp;
    }
#pragma unroll
    for (int row = 3; row < 8; ++row)
        if (!((bound >> row) & 1)) ga[(uint32_t)row * stride + i] = (T)0;
    staged_sums(x, g, 1, 1 + nca, r.sa);
    staged_sums(x, g, 0, 1, r.sn);
    return range;
}

// The backbone angles of the lane's residue i of n, whose later residues'
// atoms sum to `after`: psi turns C and what follows, phi CA's group and the
// side chain too, omega of the residue before everything from N on.
template <typename T>
__device__ __forceinline__ bool back_backbone(const BackResidue<T>& r, const double after[6], T* ga, uint32_t stride,
                                              uint32_t i, uint32_t n) {
    double s[6], p[3], q[3], a[3], c[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) p[k] = (double)r.n[k], a[k] = (double)r.ca[k], c[k] = (double)r.c[k], q[k] = (double)r.prev[k];
#pragma unroll
    for (int k = 0; k < 6; ++k) s[k] = after[k] + r.sc[k];
    const T psi = (T)bond_torque_rsq(c, a, s);
#pragma unroll
    for (int k = 0; k < 6; ++k) s[k] += r.sa[k];
    const T phi = (T)bond_torque_rsq(a, p, s);
    ga[i] = phi;
    ga[stride + i] = psi;
    bool range = out_of_range(phi) || out_of_range(psi);
    if (i > 0) {
#pragma unroll
        for (int k = 0; k < 6; ++k) s[k] += r.sn[k];
        const T omega = (T)bond_torque_rsq(p, q, s);
        range |= out_of_range(omega);
        ga[2 * stride + i - 1] = omega;
    }
    if (i == n - 1) ga[2 * stride + i] = (T)0;
    return range;
}

// v <- the sum over the lanes before (exclusive prefix); all: the wave's sum.
__device__ __forceinline__ void lanes_before(double v[6], double all[6]) {
#pragma unroll
    for (int k = 0; k < 6; ++k) {
        const double inc = wave_scan_double(v[k]);
        all[k] = readlane_double(inc, 63);
        v[k] = dpp_double<kWaveShr1, 0xf>(inc, 0.0);
    }
}

// The atoms of a block that starts at atom a0 and has `total`, on their way to
// LDS: at first as many as are staged at a time, with the C and O before them.
template <typename T>
struct BackFetch {
    Fetch<T> x, g;

    __device__ __forceinline__ static int lead(int a0) { return a0 >= 2 ? 2 : 0; }
    __device__ __forceinline__ static int values(int a0, int total) {
        return 3 * ((total < back_stage<T>() ? total : back_stage<T>()) + lead(a0));
    }
    __device__ __forceinline__ void fetch(const T* xs, const T* gs, int a0, int total, int lane) {
        const size_t from = 3 * (size_t)(a0 - lead(a0));
        x.fetch(xs + from, values(a0, total), lane);
        g.fetch(gs + from, values(a0, total), lane);
    }
    __device__ __forceinline__ void commit(const T* xs, const T* gs, int a0, int total, T* s_x, T* s_g, int lane) const {
        const size_t from = 3 * (size_t)(a0 - lead(a0));
        x.commit(xs + from, values(a0, total), s_x, lane);
        g.commit(gs + from, values(a0, total), s_g, lane);
    }
};

// A block's residues, by one wave: lane l holds residue i0 + 63 - l, of type t
// (-1: none) with cnt atoms from `at` on; f holds the block's first atoms.
// Fills r; returns whether a gradient is out of range.
template <typename T>
__device__ __forceinline__ bool back_block(const BackTables& tb, int t, int at, int cnt, int total, int a0, const T* xs,
                                           const T* gs, BackFetch<T>& f, BackResidue<T>& r, T* ga, uint32_t stride,
                                           uint32_t i, T* s_x, T* s_g, int lane) {
    bool range = false;
    for (int base = 0; base < total;) {
        // residues go down the lanes: the first one that does not fit is in the highest of those lanes
        const uint64_t later = __builtin_amdgcn_ballot_w64(t >= 0 && at + cnt > base + back_stage<T>());
        const int end = later ? __builtin_amdgcn_readlane(at, 63 - (int)__builtin_clzll(later)) : total;
        const int from = a0 + base, lead = BackFetch<T>::lead(from);
        if (base > 0) f.fetch(xs, gs, from, total - base, lane);
        f.commit(xs, gs, from, total - base, s_x, s_g, lane);
        wave_lds_sync();
        if (t >= 0 && at >= base && at < end) {
            const size_t first = 3 * (size_t)(from - lead);
            const int o = 3 * (at - base + lead);
            range |= back_residue(tb, t, a0 + at == 0, s_x + Fetch<T>::offset(xs + first) + o,
                                  s_g + Fetch<T>::offset(gs + first) + o, r, ga, stride, i);
        }
        wave_lds_sync();
        base = end;
    }
    return range;
}

// A block's sums, for the blocks before it.
struct alignas(16) BackRec {
    double s[6];
    int a0, total;  // its first atom and its atoms
    int pad[2];
};

// Zeros for residues [r0, r1) of a structure's 8 rows, by one wave.
template <typename T>
__device__ __forceinline__ void zero_rows(T* ga, uint32_t stride, int r0, int r1, int lane) {
    for (int row = 0; row < 8; ++row)
        for (int i = r0 + lane; i < r1; i += 64) ga[(size_t)row * stride + i] = (T)0;
}

// Each block's sums, one wave per (structure, block), structures first; and the
// zeros of the blocks past the structure.  Every wave reads the whole row of
// letters and so knows the structure's length, atoms and flags by itself.
constexpr int kSumWaves = 4;
template <typename T>
__global__ void __launch_bounds__(64 * kSumWaves) a2c_bwd_sums(
    const uint8_t* __restrict__ seqs, int seq_stride, const T* __restrict__ coords, const T* __restrict__ grads,
    int atoms_stride, int* __restrict__ lens, BackRec* __restrict__ rec, T* __restrict__ grad_angles, int ang_stride,
    Report rep, const int* __restrict__ order, int batch, int nslot) {
    __shared__ BackTables tb;
    const int wave = (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63);
    const int w = __builtin_amdgcn_readfirstlane((int)blockIdx.x * kSumWaves + wave);
    const int j = w / batch, slot = w - j * batch;
    const int b = j < nslot ? structure_at(order, slot, batch, j == 0 ? rep : Report{nullptr, nullptr}) : -1;
    const uint8_t* seq = seqs + (size_t)(b < 0 ? 0 : b) * seq_stride;
    RowScan row;
    row.load(seq, seq_stride, lane);
    const int i = kBlock * j + lane;
    const uint8_t code = b >= 0 && i < ang_stride && i < seq_stride ? seq[i] : (uint8_t)0;
    copy_back_tables(tb, 64 * kSumWaves);
    __syncthreads();
    if (b < 0) {
        if (j == 0 && slot < batch && lane == 0) lens[slot] = 0;
        return;
    }
    int total = 0, before = 0, flags = 0;
    bool bad = false;
    int n = row.finish<true>(seq, seq_stride, lane, tb.atoms, kBlock * j, total, before, bad);
    if (n > ang_stride) {
        flags = TPL_A2C_STATUS_LENGTH;
    } else {
        if (bad) flags |= TPL_A2C_STATUS_SEQ;
        if (total > atoms_stride) flags |= TPL_A2C_STATUS_ATOMS;
    }
    if (flags) {  // a flagged structure's gradients are zeros
        if (j == 0 && lane == 0) report_bits(rep, (uint32_t)flags);
        n = 0;
    }
    if (j == 0 && lane == 0) lens[slot] = n;
    T* ga = grad_angles + (size_t)b * 8 * ang_stride;
    if (kBlock * j >= n) {
        const int r1 = kBlock * (j + 1) < ang_stride ? kBlock * (j + 1) : ang_stride;
        zero_rows(ga, (uint32_t)ang_stride, kBlock * j, r1, lane);
        return;
    }
    const int here = __builtin_amdgcn_readlane(wave_scan_int(i < n ? (int)tb.atoms[code] : 0), 63);
    const T* xs = coords + 3 * ((size_t)b * atoms_stride + before);
    const T* gs = grads + 3 * ((size_t)b * atoms_stride + before);
    double s[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    constexpr int kAtOnce = 3;  // atoms per lane in flight
    for (int k0 = lane; k0 < here; k0 += 64 * kAtOnce) {
        T p[kAtOnce][3], h[kAtOnce][3];
#pragma unroll
        for (int e = 0; e < kAtOnce; ++e) {
            const int k = k0 + 64 * e < here ? k0 + 64 * e : k0;
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                p[e][c] = xs[3 * k + c];
                h[e][c] = gs[3 * k + c];
            }
        }
#pragma unroll
        for (int e = 0; e < kAtOnce; ++e)
            if (k0 + 64 * e < here) staged_sums(p[e], h[e], 0, 1, s);
    }
    double all[6];
    lanes_before(s, all);
    if (lane == 0) {
        BackRec* r = rec + (size_t)b * nslot + j;
#pragma unroll
        for (int k = 0; k < 6; ++k) r->s[k] = all[k];
        r->a0 = before;
        r->total = here;
    }
}

// The gradients after a2c_bwd_sums: the blocks of the list.
template <typename T>
__global__ void __launch_bounds__(64 * kWalkWaves) a2c_bwd_walk(
    const uint8_t* __restrict__ seqs, int seq_stride, const T* __restrict__ coords, const T* __restrict__ grads,
    int atoms_stride, const int* __restrict__ lens, const BackRec* __restrict__ rec, T* __restrict__ grad_angles,
    int ang_stride, Report rep, const int* __restrict__ order, int batch, int nslot) {
    __shared__ BackTables tb;
    __shared__ BlockList s_list;
    extern __shared__ __align__(16) unsigned char s_dyn[];
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = (int)(threadIdx.x & 63);
    T* s_x = reinterpret_cast<T*>(s_dyn) + (size_t)wave * 2 * back_values<T>();
    T* s_g = s_x + back_values<T>();
    const int step = (int)gridDim.x * kWalkWaves;
    const uint32_t stride = (uint32_t)ang_stride;
    bool range = false;
    for (int base = 0; base < batch; base += kSegment) {
        const int blocks =
            list_blocks(s_list, lens + base, batch - base < kSegment ? batch - base : kSegment, wave, lane, [&] {
                if (base == 0) copy_back_tables(tb, 64 * kWalkWaves);
            });
        // A block's letters and record are loaded while the one before it is
        // walked, and its atoms while that one's backbone is.
        int it = (int)blockIdx.x * kWalkWaves + wave, b = 0, j = 0, n = 0, a0 = 0, total = 0;
        uint8_t code = 0;
        BackFetch<T> f;
        const auto find = [&](int at) {
            int k;
            find_block(s_list, at, lane, k, j, n);
            b = structure_at(order, base + k, batch, Report{nullptr, nullptr});
            const int i = kBlock * j + 63 - lane;
            code = i < n ? seqs[(size_t)b * seq_stride + i] : (uint8_t)0;
            const BackRec* rb = rec + (size_t)b * nslot + j;
            a0 = rb->a0;
            total = rb->total;
        };
        const auto fetch = [&]() {
            a0 = __builtin_amdgcn_readfirstlane(a0);
            total = __builtin_amdgcn_readfirstlane(total);
            f.fetch(coords + 3 * (size_t)b * atoms_stride, grads + 3 * (size_t)b * atoms_stride, a0, total, lane);
        };
        if (it < blocks) {
            find(it);
            fetch();
        }
        for (; it < blocks; it += step) {
            const int cb = b, cj = j, cn = n, ca0 = a0, ctotal = total;
            const int i = kBlock * cj + 63 - lane;
            const int t = (int)(int8_t)tb.type[code];
            const int cnt = t >= 0 ? tb.res_i[t] & 0xff : 0;
            // the lanes up to this one hold its residue's atoms and the later ones'
            const int at = ctotal - wave_scan_int(cnt);
            // the later blocks' sums, one block per lane
            const BackRec* rb = rec + (size_t)cb * nslot + cj;
            double carry[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
            const int nb = (cn + kBlock - 1) / kBlock;
            for (int h = cj + 1 + lane; h < nb + lane; h += 64) {
#pragma unroll
                for (int c = 0; c < 6; ++c) carry[c] += h < nb ? rb[h - cj].s[c] : 0.0;
            }
            const T* xs = coords + 3 * (size_t)cb * atoms_stride;
            const T* gs = grads + 3 * (size_t)cb * atoms_stride;
            T* ga = grad_angles + (size_t)cb * 8 * ang_stride;
            const bool more = it + step < blocks;
            if (more) find(it + step);
            BackResidue<T> r;
            range |= back_block(tb, t, at, cnt, ctotal, ca0, xs, gs, f, r, ga, stride, (uint32_t)i, s_x, s_g, lane);
            if (more) fetch();
            double after[6], all[6];
            if (nb > cj + 1) {
                double later[6];
                lanes_before(carry, later);
#pragma unroll
                for (int c = 0; c < 6; ++c) carry[c] = later[c];
            }
#pragma unroll
            for (int c = 0; c < 6; ++c) after[c] = t >= 0 ? r.sc[c] + r.sa[c] + r.sn[c] : 0.0;
            lanes_before(after, all);
#pragma unroll
            for (int c = 0; c < 6; ++c) after[c] += carry[c];
            if (t >= 0)
                range |= back_backbone(r, after, ga, stride, (uint32_t)i, (uint32_t)cn);
            else if (i < ang_stride)
                for (int row = 0; row < 8; ++row) ga[(uint32_t)row * stride + (uint32_t)i] = (T)0;
        }
    }
    if (range) report_flag(rep, TPLX_A2C_RANGE);
}

// One workgroup per structure, of blockDim / 64 waves: the waves take their
// blocks together, from the structure's end, as many at a time as there are
// waves.
constexpr int kBackWaves = 8;
template <typename T>
__global__ void __launch_bounds__(64 * kBackWaves) a2c_bwd_fused(
    const uint8_t* __restrict__ seqs, int seq_stride, const T* __restrict__ coords, const T* __restrict__ grads,
    int atoms_stride, T* __restrict__ grad_angles, int ang_stride, Report rep, const int* __restrict__ order,
    int batch) {
    __shared__ BackTables tb;
    __shared__ double s_sum[kBackWaves][6];
    __shared__ int s_cnt[kBackWaves];
    extern __shared__ __align__(16) unsigned char s_dyn[];
    const int NW = (int)(blockDim.x >> 6);
    const int wave = turned_wave(__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), NW, (int)blockIdx.x);
    const int lane = (int)(threadIdx.x & 63);
    T* s_x = reinterpret_cast<T*>(s_dyn) + (size_t)wave * 2 * back_values<T>();
    T* s_g = s_x + back_values<T>();
    const int b = structure_at(order, (int)blockIdx.x, batch, rep);
    if (b < 0) return;
    const uint8_t* seq = seqs + (size_t)b * seq_stride;
    RowScan row;
    row.load(seq, seq_stride, lane);
    copy_back_tables(tb, 64 * NW);
    __syncthreads();
    // every wave alike
    int atoms = 0, unused = 0, flags = 0;
    bool bad = false;
    int n = row.finish<true>(seq, seq_stride, lane, tb.atoms, 0, atoms, unused, bad);
    if (n > ang_stride) {
        flags = TPL_A2C_STATUS_LENGTH;
    } else {
        if (bad) flags |= TPL_A2C_STATUS_SEQ;
        if (atoms > atoms_stride) flags |= TPL_A2C_STATUS_ATOMS;
    }
    if (flags) {
        if (threadIdx.x == 0) report_bits(rep, (uint32_t)flags);
        n = 0;
    }
    const T* xs = coords + 3 * (size_t)b * atoms_stride;
    const T* gs = grads + 3 * (size_t)b * atoms_stride;
    T* ga = grad_angles + (size_t)b * 8 * ang_stride;
    const uint32_t stride = (uint32_t)ang_stride;
    const int nb = (n + kBlock - 1) / kBlock;
    double carry[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};  // sums past the blocks at hand
    bool range = false;
    for (int hi = nb; hi > 0; hi -= NW) {
        const int lo = hi > NW ? hi - NW : 0, j = hi - 1 - wave;  // wave 0 takes the last block
        const int i = kBlock * j + 63 - lane;
        const bool real = j >= lo;
        const uint8_t code = real && i < n ? seq[i] : (uint8_t)0;
        const int t = (int)(int8_t)tb.type[code];
        const int cnt = t >= 0 ? tb.res_i[t] & 0xff : 0;
        const int inc = wave_scan_int(cnt);
        const int total = __builtin_amdgcn_readlane(inc, 63);
        // this block's first atom, from the later blocks' counts
        if (lane == 0) s_cnt[wave] = total;
        __syncthreads();
        const int here = hi - lo;
        int a0 = atoms - total;
        for (int k = 0; k < here; ++k) {
            if (k < wave) a0 -= s_cnt[k];
            atoms -= s_cnt[k];
        }
        BackResidue<T> r;
        double after[6], all[6];
        if (real) {
            BackFetch<T> f;
            f.fetch(xs, gs, a0, total, lane);
            range |= back_block(tb, t, total - inc, cnt, total, a0, xs, gs, f, r, ga, stride, (uint32_t)i, s_x, s_g,
                                lane);
#pragma unroll
            for (int c = 0; c < 6; ++c) after[c] = t >= 0 ? r.sc[c] + r.sa[c] + r.sn[c] : 0.0;
            lanes_before(after, all);
            if (lane == 0) {
#pragma unroll
                for (int c = 0; c < 6; ++c) s_sum[wave][c] = all[c];
            }
        }
        __syncthreads();
        double past[6];
#pragma unroll
        for (int c = 0; c < 6; ++c) past[c] = carry[c];
        for (int k = 0; k < here; ++k) {
#pragma unroll
            for (int c = 0; c < 6; ++c) {
                if (k < wave) past[c] += s_sum[k][c];
                carry[c] += s_sum[k][c];
            }
        }
        if (t >= 0) {
#pragma unroll
            for (int c = 0; c < 6; ++c) after[c] += past[c];
            range |= back_backbone(r, after, ga, stride, (uint32_t)i, (uint32_t)n);
        }
        __syncthreads();  // the sums, before the next blocks'
    }
    if (range) report_flag(rep, TPLX_A2C_RANGE);
    // angles past the sequence (and every angle of a flagged structure)
    for (int row8 = wave; row8 < 8; row8 += NW)
        for (int i = n + lane; i < ang_stride; i += 64) ga[(uint32_t)row8 * stride + (uint32_t)i] = (T)0;
}

// Run backward: 512-thread workgroups when some structure may be longer than
// 256 residues (mixed lengths 30-1000 at B=1024: 155 -> 129 us).
bool use_large_bwd(int ang_stride) {
    return ang_stride > kThreadsSmall;
}

// g_tab of the current device, filled on the first forward there: the
// kernel runs on the caller's stream, which is then synchronised once, so
// that forwards on any stream of the device find the tables.
bool tables_ready(hipStream_t s) {
    static std::mutex mu;
    static std::vector<char> ready;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0) return false;
    std::lock_guard<std::mutex> lock(mu);
    if ((int)ready.size() <= dev) ready.resize(dev + 1, 0);
    if (ready[dev]) return true;
    hipLaunchKernelGGL(a2c_init_tables, dim3(1), dim3(256), 0, s);
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(s) != hipSuccess) return false;
    ready[dev] = 1;
    return true;
}

int check(int dtype, int B, int seq_stride, int ang_stride, int atoms_stride) {
    if (dtype != TPL_A2C_F32 && dtype != TPL_A2C_F64) return TPL_A2C_ERR_ARG;
    if (B < 0 || seq_stride < 0 || ang_stride < 0 || atoms_stride < 0) return TPL_A2C_ERR_ARG;
    if ((int64_t)8 * ang_stride > INT32_MAX || (int64_t)3 * atoms_stride > INT32_MAX)
        return TPL_A2C_ERR_SIZE;
    return TPL_A2C_OK;
}

int blocks_of(int residues) { return residues <= kBlock ? 1 : (residues + kBlock - 1) / kBlock; }
int groups_of(int residues) { return (residues + kGroup - 1) / kGroup; }

// The workspace: the structures' lengths by slot of the batch (0 for flagged
// ones), the groups' records, the residues' frames.
size_t lens_bytes(int batch) { return ((size_t)batch * sizeof(int) + 15) / 16 * 16; }
size_t recs_bytes(int batch, int angles_stride) {
    return (size_t)batch * groups_of(angles_stride) * sizeof(GroupRec);
}
size_t frames_bytes(int batch, int angles_stride) {
    return (size_t)batch * groups_of(angles_stride) * sizeof(GroupFrames);
}

// CUs of the current device (256 where it cannot be asked).
int compute_units() {
    static std::mutex mu;
    static std::vector<int> cus;
    int dev = 0, n = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0) return 256;
    std::lock_guard<std::mutex> lock(mu);
    if ((int)cus.size() <= dev) cus.resize(dev + 1, 0);
    if (cus[dev] == 0)
        cus[dev] = hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && n > 0 ? n : 256;
    return cus[dev];
}

// The residues that the longest structure is likely to have: callers give the
// atoms of the largest one as atoms_stride, 8.2 to a residue on average, while
// the angles' stride may be a longer one that they keep.  For choosing only.
int likely_residues(int angles_stride, int atoms_stride) {
    const int n = atoms_stride / 8 > 1 ? atoms_stride / 8 : 1;
    return n < angles_stride ? n : angles_stride;
}

// Run forward: 512 threads for structures that may be longer than 256 residues,
// up to twice as many structures as CUs (B=256 of 1000 residues: 33.7 -> 28.6
// us; B=512 of 300: 23.8 -> 21.8 us; at B=1024 512 threads measured slower, with
// fewer workgroups per CU: mixed lengths 30-1000 48.4 -> 55.7 us, 1024 x 270
// 32.0 -> 39.6 us).
bool use_large_fwd(int batch, int ang_stride) {
    return batch <= 512 && ang_stride > kThreadsSmall;
}

// Whether the group kernels' grids can be counted.
bool forward_groups_fit(int batch, int angles_stride) {
    return (int64_t)batch * groups_of(angles_stride) <= INT32_MAX / kGroup;
}
// What AUTO takes.  us of the forms (U: lengths uniform; structures x stride):
//   GROUPS share the blocks evenly over the GPU, and win where the structures need
//   more than one round of workgroups, or where there are fewer long ones than
//   CUs.  Without it -> GROUPS, with names, float32: 1024 x 1000 U 90 -> 63, 2048 x 300
//   U 58 -> 47, 300 x 600 40 -> 36, 4096 x 200 U 74 -> 70, 100 x 1400 41 -> 37, 8 x 3000 65
//   -> 28, 64 x 1000 28.2 -> 26.5, 4096 x 128 U 62 -> 55; not 1024 x 200 27 -> 37, 512 x 450 30 -> 38, 64 x 600 21.5
//   -> 24.7, 256 x 1000 35 -> 40; float64: 200 x 800 U 34 -> 30, not 256 x 600 33 -> 40.
//   FUSED against RUNS: a wave per block wins while every structure has a CU to
//   itself, and where RUNS would have 512 threads for little more than 256
//   residues; otherwise a run per thread does, most where no names are written.
//   RUNS -> FUSED without names / with names, float32: 256 x 300 16.1 -> 13.6 / 18.9 ->
//   16.2, 256 x 1000 26.6 -> 31.3 / 37.6 -> 34.7, 512 x 300 21.7 -> 20.8 / 25.9 -> 23.8, 1024 x
//   300 32 -> 46 / 41 -> 53, 1024 x 128 16.9 -> 18.5 / 20.6 -> 22.0, 8 x 3000 56 -> 75 / 65 ->
//   82; float64: 256 x 300 18.1 -> 17.1 / 21.2 -> 19.5, 256 x 600 28.6 -> 30.4 / 35.9 -> 32.9,
//   512 x 200 20 -> 23 / 23 -> 26, 512 x 450 40 -> 38 / 46 -> 42, 64 x 1000 26 -> 33 / 32 -> 37.
//   With names and 14 to 16 blocks many structures win too in float32 (1024 x 1000 131 -> 112,
//   U longest first 89 -> 76; not 300 x 1000 50 -> 55, float64 188 -> 194).
// A structure of one block needs no groups, whatever the form.
bool forward_groups_pay(bool f64, int batch, int nb) {
    const int cus = compute_units();
    if (nb > 16) return true;
    if (batch <= cus) return f64 ? nb > 10 : nb > 13 && batch <= cus / 2;
    return nb > 8 || (int64_t)batch * nb >= (nb > 4 ? 5000 : 8000);
}
int forward_form(bool f64, int batch, int angles_stride, int atoms_stride, bool names, bool workspace) {
    const int nb = blocks_of(likely_residues(angles_stride, atoms_stride)), cus = compute_units();
    if (blocks_of(angles_stride) == 1) return TPLX_A2C_FWD_FUSED;
    if (workspace && forward_groups_fit(batch, angles_stride) && forward_groups_pay(f64, batch, nb))
        return TPLX_A2C_FWD_GROUPS;
    const int most = (f64 ? 8 : 13) + (names ? f64 ? 2 : 3 : 0);
    const bool fused = batch <= cus                ? nb <= most
                       : names && !f64 && nb > 13  ? nb <= 16 && batch >= 2 * cus
                                                   : batch <= 2 * cus && nb >= 5 && nb <= (f64 ? 10 : 7);
    return fused ? TPLX_A2C_FWD_FUSED : TPLX_A2C_FWD_RUNS;
}

template <typename T>
void launch_forward(int form, hipStream_t s, const uint8_t* sequences, int seq_stride, const T* a, int angles_stride,
                    T* c, uint32_t* rn, uint32_t* an, int atoms_stride, void* workspace, const Report& rep,
                    const int32_t* order, int batch) {
    const int nslot = blocks_of(angles_stride), ng = groups_of(angles_stride);
    const dim3 block(64 * kGroupWaves);
    if (nslot == 1 && form != TPLX_A2C_FWD_RUNS) {
        hipLaunchKernelGGL((a2c_fwd_single<T>), dim3((batch + kGroupWaves - 1) / kGroupWaves), block, 0, s, sequences,
                           seq_stride, a, angles_stride, c, rn, an, atoms_stride, rep, order, batch);
        return;
    }
    if (form == TPLX_A2C_FWD_GROUPS) {
        char* ws = static_cast<char*>(workspace);
        int* lens = reinterpret_cast<int*>(ws);
        GroupRec* rec = reinterpret_cast<GroupRec*>(ws + lens_bytes(batch));
        GroupFrames* frames =
            reinterpret_cast<GroupFrames*>(ws + lens_bytes(batch) + recs_bytes(batch, angles_stride));
        hipLaunchKernelGGL((a2c_fwd_steps<T>), dim3((batch * ng + kGroupWaves - 1) / kGroupWaves), block, 0, s,
                           sequences, seq_stride, a, angles_stride, lens, rec, frames, c, rn, an, atoms_stride, rep,
                           order, batch, ng);
        // what stays resident: two workgroups per CU (one in float64), as their LDS allows
        const int fill = (sizeof(T) == 4 ? 2 : 1) * compute_units();
        const int wgs = (batch * nslot + kWalkWaves - 1) / kWalkWaves;
        hipLaunchKernelGGL((a2c_fwd_walk<T>), dim3(wgs < fill ? wgs : fill), dim3(64 * kWalkWaves), 0, s, sequences,
                           seq_stride, a, angles_stride, lens, rec, frames, c, rn, an, atoms_stride, rep, order,
                           batch, ng);
        return;
    }
    if (form == TPLX_A2C_FWD_RUNS) {
        const int nt = use_large_fwd(batch, angles_stride) ? kThreadsLarge : kThreadsSmall;
        const auto kernel = nt == kThreadsLarge ? a2c_fwd_runs<kThreadsLarge, T> : a2c_fwd_runs<kThreadsSmall, T>;
        hipLaunchKernelGGL(kernel, dim3(batch), dim3(nt), 0, s, sequences, seq_stride, a, angles_stride, c, rn, an,
                           atoms_stride, rep, order);
        return;
    }
    // One wave per block up to 8, or up to 16 where every structure can have a
    // CU; above that the waves go round.  Beyond one structure per CU the
    // kernel is held to 128 VGPRs, so that two workgroups of 8 waves fit, and
    // spills: 100 bytes in float32 (512 x 300: 30 -> 25 us), 152 in float64 (512
    // x 300 31.7 -> 29.0, 512 x 600 60.8 -> 53.5).
    const bool few = batch <= compute_units();
    const int most = few ? 16 : 8, rounds = (nslot + most - 1) / most, nw = (nslot + rounds - 1) / rounds;
    const auto kernel = nw > 8 ? a2c_fwd_fused<16, 4, T> : few ? a2c_fwd_fused<8, 2, T> : a2c_fwd_fused<8, 4, T>;
    hipLaunchKernelGGL(kernel, dim3(batch), dim3(64 * nw), 0, s, sequences, seq_stride, a, angles_stride, c, rn, an,
                       atoms_stride, rep, order, batch);
}

// form: TPLX_A2C_FWD_*; GROUPS needs the workspace (where a structure is more
// than one block), AUTO uses it if there is one.
int forward_on(int form, const int32_t* order, int dtype, const uint8_t* sequences, int seq_stride,
               const void* angles, int angles_stride, void* coords, uint8_t* res_names, uint8_t* atom_names,
               int atoms_stride, void* workspace, const Report& rep, int batch, tpl_a2c_stream_t stream) {
    const int rc = check(dtype, batch, seq_stride, angles_stride, atoms_stride);
    if (rc != TPL_A2C_OK) return rc;
    if (batch == 0) return TPL_A2C_OK;
    if (!sequences || (angles_stride > 0 && !angles) || (atoms_stride > 0 && !coords) ||
        (!res_names) != (!atom_names))
        return TPL_A2C_ERR_ARG;
    if (form == TPLX_A2C_FWD_AUTO)
        form = forward_form(dtype == TPL_A2C_F64, batch, angles_stride, atoms_stride, res_names != nullptr,
                            workspace != nullptr);
    if (form == TPLX_A2C_FWD_GROUPS && blocks_of(angles_stride) > 1 &&
        !(workspace && forward_groups_fit(batch, angles_stride)))
        return TPL_A2C_ERR_ARG;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (!tables_ready(s)) return TPL_A2C_ERR_LAUNCH;
    uint32_t* rn = reinterpret_cast<uint32_t*>(res_names);
    uint32_t* an = reinterpret_cast<uint32_t*>(atom_names);
    if (dtype == TPL_A2C_F32)
        launch_forward<float>(form, s, sequences, seq_stride, static_cast<const float*>(angles), angles_stride,
                              static_cast<float*>(coords), rn, an, atoms_stride, workspace, rep, order, batch);
    else
        launch_forward<double>(form, s, sequences, seq_stride, static_cast<const double*>(angles), angles_stride,
                               static_cast<double*>(coords), rn, an, atoms_stride, workspace, rep, order, batch);
    return hipGetLastError() == hipSuccess ? TPL_A2C_OK : TPL_A2C_ERR_LAUNCH;
}

// The backward's workspace: the structures' lengths by slot of the batch, the
// blocks' sums.
size_t back_recs_bytes(int batch, int angles_stride) {
    return (size_t)batch * blocks_of(angles_stride) * sizeof(BackRec);
}

// Dynamic LDS beyond 64 KB has to be allowed per kernel and device, once.
bool allow_lds(const void* kernel, size_t bytes) {
    static std::mutex mu;
    static std::set<std::pair<int, const void*>> allowed;
    if (bytes <= 60u << 10) return true;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    std::lock_guard<std::mutex> lock(mu);
    if (allowed.count({dev, kernel})) return true;
    if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess) return false;
    allowed.insert({dev, kernel});
    return true;
}

bool backward_groups_fit(int batch, int angles_stride) {
    return (int64_t)batch * blocks_of(angles_stride) <= INT32_MAX / kBlock;
}
// What AUTO takes.  us of the forms (U: lengths uniform):
//   GROUPS as in the forward, from 5 blocks on; FUSED -> GROUPS, float32: 1024 x 1000 U 91 ->
//   77, 2048 x 300 U 85 -> 52, 700 x 300 40 -> 37, 64 x 600 23 -> 21, 8 x 3000 70 -> 25; not
//   1024 x 200 27 -> 40, 256 x 1000 33 -> 41, 512 x 450 34 -> 39.
//   FUSED otherwise, but for
//   - TILES in float32, whose workgroup of one structure has two on a CU: with 5 to 7
//     blocks beyond a structure per CU, with 5 to 10 up to two (FUSED -> TILES: 400 x 300 26.5 ->
//     24.5, 1024 x 300 52 -> 48, 512 x 600 48 -> 45, 1500 x 400 U longest first 67 -> 59; not
//     260 x 450 27 -> 30, 2048 x 500 U 98 -> 109);
//   - RUNS in float64, where a block's atoms are staged in two rounds, for up to a
//     structure of 256 residues per CU (FUSED -> RUNS: 128 x 64 15.4 -> 13.1, 128 x 128 15.9
//     -> 14.7, 64 x 200 18.0 -> 16.0; not 320 x 200 19.7 -> 29, 256 x 300 20.5 -> 27, 1 x 128
//     12.9 -> 13.9) and two of 64 (512 x 64 17.1 -> 15.0);
//   - TILES for short structures in a long stride, whose workgroups of a wave per
//     block of the stride would be nearly idle (FUSED -> TILES: 500 x 20..100 at 800 22.5
//     -> 15.0, float64 31.5 -> 22.1; 1024 x 25..125 at 1000 39 -> 32, GROUPS 28).
int backward_form(bool f64, int batch, int angles_stride, int atoms_stride, bool workspace) {
    const int nb = blocks_of(angles_stride), cus = compute_units();
    const bool tiles_fit = angles_stride <= kTileMaxRes, two_each = 2 * batch >= 3 * cus && batch <= 2 * cus;
    if (4 * likely_residues(angles_stride, atoms_stride) <= angles_stride && batch > cus && tiles_fit &&
        (!workspace || batch <= 2 * cus))
        return TPLX_A2C_BWD_TILES;
    if (workspace && backward_groups_fit(batch, angles_stride) && nb > 4 && !(two_each && nb <= 10)) {
        if (nb > 16 || (batch <= cus ? nb > 8 && batch <= cus / 2 : (int64_t)batch * nb >= 3000))
            return TPLX_A2C_BWD_GROUPS;
    }
    if (f64) {
        const bool runs = angles_stride > 36 && nb <= 4 && batch >= 16 && batch <= (nb == 1 ? 2 * cus : cus);
        return runs ? TPLX_A2C_BWD_RUNS : TPLX_A2C_BWD_FUSED;
    }
    const bool tiles = nb >= 5 && (nb <= 7 ? 4 * batch >= 5 * cus : nb <= 10 && two_each);
    return tiles && tiles_fit ? TPLX_A2C_BWD_TILES : TPLX_A2C_BWD_FUSED;
}

template <typename T>
int launch_backward(int form, hipStream_t s, const uint8_t* sequences, int seq_stride, const T* x, const T* g,
                    int atoms_stride, T* ga, int angles_stride, void* workspace, const Report& rep,
                    const int32_t* order, int batch) {
    const int nslot = blocks_of(angles_stride);
    constexpr size_t per_wave = 2 * back_values<T>() * sizeof(T);
    if (form == TPLX_A2C_BWD_TILES) {
        hipLaunchKernelGGL((a2c_bwd_tiled<T>), dim3(batch), dim3(kTileThreads), 0, s, sequences, seq_stride, x, g,
                           atoms_stride, ga, angles_stride, rep, order);
    } else if (form == TPLX_A2C_BWD_RUNS) {
        const int nt = use_large_bwd(angles_stride) ? kThreadsLarge : kThreadsSmall;
        const auto kernel = nt == kThreadsLarge ? a2c_bwd<kThreadsLarge, T> : a2c_bwd<kThreadsSmall, T>;
        hipLaunchKernelGGL(kernel, dim3(batch), dim3(nt), 0, s, sequences, seq_stride, x, g, atoms_stride, ga,
                           angles_stride, rep, order);
    } else if (form == TPLX_A2C_BWD_GROUPS) {
        int* lens = static_cast<int*>(workspace);
        BackRec* rec = reinterpret_cast<BackRec*>(static_cast<char*>(workspace) + lens_bytes(batch));
        const int wgs = (batch * nslot + kWalkWaves - 1) / kWalkWaves, fill = compute_units();
        const size_t lds = kWalkWaves * per_wave;
        if (!allow_lds(reinterpret_cast<const void*>(a2c_bwd_walk<T>), lds)) return TPL_A2C_ERR_LAUNCH;
        hipLaunchKernelGGL((a2c_bwd_sums<T>), dim3((batch * nslot + kSumWaves - 1) / kSumWaves), dim3(64 * kSumWaves),
                           0, s, sequences, seq_stride, x, g, atoms_stride, lens, rec, ga, angles_stride, rep, order,
                           batch, nslot);
        hipLaunchKernelGGL((a2c_bwd_walk<T>), dim3(wgs < fill ? wgs : fill), dim3(64 * kWalkWaves), lds, s, sequences,
                           seq_stride, x, g, atoms_stride, lens, rec, ga, angles_stride, rep, order, batch, nslot);
    } else {
        const int rounds = (nslot + kBackWaves - 1) / kBackWaves, nw = (nslot + rounds - 1) / rounds;
        if (!allow_lds(reinterpret_cast<const void*>(a2c_bwd_fused<T>), kBackWaves * per_wave))
            return TPL_A2C_ERR_LAUNCH;
        hipLaunchKernelGGL((a2c_bwd_fused<T>), dim3(batch), dim3(64 * nw), nw * per_wave, s, sequences, seq_stride, x,
                           g, atoms_stride, ga, angles_stride, rep, order, batch);
    }
    return hipGetLastError() == hipSuccess ? TPL_A2C_OK : TPL_A2C_ERR_LAUNCH;
}

int backward_on(int form, const int32_t* order, int dtype, const uint8_t* sequences, int seq_stride,
                const void* coords, const void* grad_coords, int atoms_stride, void* grad_angles, int angles_stride,
                void* workspace, const Report& rep, int batch, tpl_a2c_stream_t stream) {
    const int rc = check(dtype, batch, seq_stride, angles_stride, atoms_stride);
    if (rc != TPL_A2C_OK) return rc;
    if (form == TPLX_A2C_BWD_TILES && angles_stride > kTileMaxRes) return TPL_A2C_ERR_SIZE;
    if (batch == 0 || angles_stride == 0) return TPL_A2C_OK;
    if (!sequences || !grad_angles || (atoms_stride > 0 && (!coords || !grad_coords))) return TPL_A2C_ERR_ARG;
    if (form == TPLX_A2C_BWD_AUTO)
        form = backward_form(dtype == TPL_A2C_F64, batch, angles_stride, atoms_stride, workspace != nullptr);
    if (form == TPLX_A2C_BWD_GROUPS && !(workspace && backward_groups_fit(batch, angles_stride)))
        return TPL_A2C_ERR_ARG;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == TPL_A2C_F32)
        return launch_backward<float>(form, s, sequences, seq_stride, static_cast<const float*>(coords),
                                      static_cast<const float*>(grad_coords), atoms_stride,
                                      static_cast<float*>(grad_angles), angles_stride, workspace, rep, order, batch);
    return launch_backward<double>(form, s, sequences, seq_stride, static_cast<const double*>(coords),
                                   static_cast<const double*>(grad_coords), atoms_stride,
                                   static_cast<double*>(grad_angles), angles_stride, workspace, rep, order, batch);
}

}  // namespace

extern "C" {

const char* tpl_a2c_strerror(int code) {
    switch (code) {
        case TPL_A2C_OK: return "ok";
        case TPL_A2C_ERR_ARG: return "invalid argument (null pointer, negative size or unknown dtype)";
        case TPL_A2C_ERR_LAUNCH: return "kernel launch failed";
        case TPL_A2C_ERR_SIZE: return "sizes too large";
        default: return "unknown error code";
    }
}

int tpl_a2c_num_atoms(const char* sequence) {
    // Atoms by letter, -1 outside the 20 (32 sequences of 350 letters: 78 -> 7
    // us against looking up each letter's residue).
    struct Counts {
        int8_t of[256];
    };
    static const Counts counts = [] {
        static const Residue res[kTypes] = A2C_RESIDUES;
        Counts c;
        for (int k = 0; k < 256; ++k) {
            const int t = residue_type((uint8_t)k);
            c.of[k] = (int8_t)(t < 0 ? -1 : res[t].natoms);
        }
        return c;
    }();
    if (!sequence) return -1;
    int n = 0, bad = 0;
    for (const char* p = sequence; *p; ++p) {
        const int k = counts.of[(uint8_t)*p];
        bad |= k;  // negative once a letter is
        n += k;
    }
    return bad < 0 ? -1 : n;
}

int tpl_a2c_forward_ordered(const int32_t* order, int dtype, const uint8_t* sequences, int seq_stride,
                            const void* angles, int angles_stride, void* coords, uint8_t* res_names,
                            uint8_t* atom_names, int atoms_stride, uint32_t* status, int batch,
                            tpl_a2c_stream_t stream) {
    return forward_on(TPLX_A2C_FWD_AUTO, order, dtype, sequences, seq_stride, angles, angles_stride, coords,
                      res_names, atom_names, atoms_stride, nullptr, Report{status, nullptr}, batch, stream);
}

int tplx_a2c_forward(int form, const int32_t* order, int dtype, const uint8_t* sequences, int seq_stride,
                     const void* angles, int angles_stride, void* coords, uint8_t* res_names, uint8_t* atom_names,
                     int atoms_stride, void* workspace, uint32_t* status, uint32_t* flags, int batch,
                     tpl_a2c_stream_t stream) {
    return forward_on(form, order, dtype, sequences, seq_stride, angles, angles_stride, coords, res_names,
                      atom_names, atoms_stride, workspace, Report{status, flags}, batch, stream);
}

int tplx_a2c_forward_form(int dtype, int batch, int angles_stride, int atoms_stride, int names, int workspace) {
    return forward_form(dtype == TPL_A2C_F64, batch, angles_stride, atoms_stride, names != 0, workspace != 0);
}

int tplx_a2c_backward_form(int dtype, int batch, int angles_stride, int atoms_stride, int workspace) {
    return backward_form(dtype == TPL_A2C_F64, batch, angles_stride, atoms_stride, workspace != 0);
}

size_t tplx_a2c_workspace_bytes(int batch, int angles_stride) {
    if (batch <= 0 || blocks_of(angles_stride) == 1) return 0;
    return lens_bytes(batch) + recs_bytes(batch, angles_stride) + frames_bytes(batch, angles_stride);
}

size_t tplx_a2c_backward_workspace_bytes(int batch, int angles_stride) {
    return batch <= 0 ? 0 : lens_bytes(batch) + back_recs_bytes(batch, angles_stride);
}

int tplx_a2c_backward(int form, const int32_t* order, int dtype, const uint8_t* sequences, int seq_stride,
                      const void* coords, const void* grad_coords, int atoms_stride, void* grad_angles,
                      int angles_stride, void* workspace, uint32_t* status, uint32_t* flags, int batch,
                      tpl_a2c_stream_t stream) {
    return backward_on(form, order, dtype, sequences, seq_stride, coords, grad_coords, atoms_stride, grad_angles,
                       angles_stride, workspace, Report{status, flags}, batch, stream);
}

int tpl_a2c_forward(int dtype, const uint8_t* sequences, int seq_stride, const void* angles,
                    int angles_stride, void* coords, uint8_t* res_names, uint8_t* atom_names,
                    int atoms_stride, uint32_t* status, int batch, tpl_a2c_stream_t stream) {
    return tpl_a2c_forward_ordered(nullptr, dtype, sequences, seq_stride, angles, angles_stride, coords,
                                   res_names, atom_names, atoms_stride, status, batch, stream);
}

int tpl_a2c_backward_form(int form, const int32_t* order, int dtype, const uint8_t* sequences, int seq_stride,
                          const void* coords, const void* grad_coords, int atoms_stride, void* grad_angles,
                          int angles_stride, uint32_t* status, int batch, tpl_a2c_stream_t stream) {
    static_assert(TPLX_A2C_BWD_AUTO == TPL_A2C_BWD_AUTO, "one name for both");
    if (form != TPL_A2C_BWD_AUTO && form != TPL_A2C_BWD_RUNS && form != TPL_A2C_BWD_TILES) return TPL_A2C_ERR_ARG;
    form = form == TPL_A2C_BWD_RUNS ? TPLX_A2C_BWD_RUNS : form == TPL_A2C_BWD_TILES ? TPLX_A2C_BWD_TILES : form;
    return backward_on(form, order, dtype, sequences, seq_stride, coords, grad_coords, atoms_stride, grad_angles,
                       angles_stride, nullptr, Report{status, nullptr}, batch, stream);
}

int tpl_a2c_backward(int dtype, const uint8_t* sequences, int seq_stride, const void* coords,
                     const void* grad_coords, int atoms_stride, void* grad_angles, int angles_stride,
                     uint32_t* status, int batch, tpl_a2c_stream_t stream) {
    return tpl_a2c_backward_form(TPL_A2C_BWD_AUTO, nullptr, dtype, sequences, seq_stride, coords, grad_coords,
                                 atoms_stride, grad_angles, angles_stride, status, batch, stream);
}

}  // extern "C"
