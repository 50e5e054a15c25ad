// Host-side mechanism: parse the compiled .mech tables and build the device
// tables used by every kernel.  Replaces the reference's mechanism assembly
// (newSolution -> BulkKinetics::addReaction; src/kinetics/BulkKinetics.cpp:16-84,
// src/kinetics/Kinetics.cpp:709-800) for the ideal-gas bulk path.
#pragma once
#include <string>
#include <utility>
#include <vector>

#include <hip/hip_runtime.h>

namespace cg {

constexpr int kMaxSide = 4;   // species entries per reaction side on the device
constexpr int kMaxTB = 32;    // explicit efficiencies per reaction
constexpr int kTbPad = 8;     // efficiency lists are padded to a multiple of this many entries
constexpr int kDummy = 64;    // sentinel species slots K .. K+63 in the kernels' scratch

enum RxnType { kElementary = 0, kThreeBody = 1, kLindemann = 2, kTroe = 3, kPlog = 4, kChebyshev = 5, kSri = 6, kTsang = 7 };

struct HostReaction {
    int type = 0;
    bool rev = false;
    double dn = 0, A = 0, b = 0, EaR = 0, A0 = 0, b0 = 0, EaR0 = 0;
    double troe[4] = {0, 0, 0, 0};   // a, 1/T3, 1/T1, T2
    double sri[5] = {0, 0, 0, 1, 0}; // kSri: a, b, c, d, e
    double tsang[2] = {0, 0};        // kTsang: A, B
    bool chem_act = false;           // chemically activated falloff: k = k0 F / (1 + Pr)
    std::vector<int> rk;             // reactant species (name order)
    std::vector<double> rs, ro;      // stoich, order
    std::vector<int> pk;
    std::vector<double> ps;
    double tbdef = 0;
    std::vector<int> tbk;
    std::vector<double> tbe;         // efficiency - default
    std::vector<double> plog;        // kPlog: (P [Pa], A, b, Ea/R) per entry, sorted by P
    std::vector<double> cheb;        // kChebyshev: Tmin, Tmax, Pmin, Pmax, nT, nP, nT x nP coefficients
    std::string equation;
};

struct HostMech {
    std::string phase;
    int K = 0, I = 0, E = 0;
    std::vector<std::string> elements, names;
    std::vector<double> aw, mw, comp;              // comp: K x E
    std::vector<double> tmin, tmid, tmax, pref;
    std::vector<double> clow, chigh;               // K x 7
    std::vector<HostReaction> rxn;
};

// Parse a .mech file written by cantera_amd/mechc.py.  Throws std::runtime_error.
HostMech load_mech(const std::string& path);

// Per-reaction device record (integer part).  Species lists follow the
// reference StoichManagerN convention: unit-stoichiometry sides with at most
// three molecules are expanded into repeated species ("kRep", C1/C2/C3); other
// sides are "general" (C_AnyN: species, order, stoich).  Unused entries of
// rk/pk hold K, a sentinel species whose concentration is 1 and chemical
// potential 0 in the kernels' scratch.
struct RxnI {
    int flags;      // bit0 reversible, bits1-2 type (0..3), bit3 reactant side general, bit4 product side general,
                    // bit5 third body, bit6 PLOG, bit7 Chebyshev (those two with type 0),
                    // bit8 SRI (with type 3), bit9 chemically activated (types 2, 3)
    int nr, np;     // entries in rk/pk
    int tbo, tbn;   // third-body efficiency list offset/count
    int fo;         // falloff record index, or PLOG / Chebyshev record offset in pdd (-1 if none)
    int gen;        // general-order record index (-1 if none)
    int orig;       // reaction index in mechanism order
    short rk[kMaxSide];
    short pk[kMaxSide];
};
static_assert(sizeof(RxnI) == 48, "RxnI layout");

constexpr int kDummyWide = 8;  // sentinel slots where several states share a wavefront's scratch

// Compact record of a standard reaction: both sides unit-stoichiometry lists of
// at most three molecules (four products if irreversible), a rate constant of
// Arrhenius, three-body, Lindemann or Troe form.  Each entry is the byte offset
// of the species' (C, mu) pair in the kernels' scratch (16 x slot).  Unused entries
// point at the sentinel slot K + (reaction % kDummy), where C = 1 and mu = 0:
// every sum and product runs without tests, and the lanes of a pass, which
// hold consecutive reactions, add their unused entries to slots of their own
// instead of serialising on one address.
struct alignas(16) RxnS {
    unsigned short r[3], p[4];
    unsigned short flags;        // bit0 reversible, bit1 a fourth product
};
static_assert(sizeof(RxnS) == 16, "RxnS layout");

// Device view of a mechanism (all pointers are device pointers).
struct DevMech {
    int K, I, N, E;          // species, reactions, state size (K+2), elements
    int n_el, n_tb, n_fo;    // reactions of each class, in permuted order:
                             // [Chebyshev | PLOG | other non-standard | Troe | Lindemann | three-body | elementary]
    int gen_end, tb_end;     // wavefront passes of 64 reactions: [0, gen_end) hold the non-standard reactions
                             // (evaluated by the general code), [gen_end, tb_end) the other falloff and
                             // three-body ones, the rest is elementary
    int n_pd;                // PLOG + Chebyshev reactions (the first n_pd, at most 64)
    double pref, rpref;      // reference pressure and its reciprocal
    const double* mw;        // K
    const double* rmw;       // K
    const double* nasa;      // K x 16: low[7], tmid, high[7], pad
    // per-reaction tables: I entries and null reactions (A = 0, no species) up to a multiple of 64
    const double* rd;        // 4 each: A, b, EaR, dn
    const double* tbdef;
    const RxnI* ri;
    const RxnS* rs;          // valid for standard and null reactions
    const RxnS* rsw;         // the same with sentinel slots K + (reaction % kDummyWide), for scratch with
                             // several states per wavefront
    int n_gen, n_nonplain;   // non-standard reactions; reactions up to the last that is not elementary
    const double* fod;       // (n_fo + 1) x 8, the last all zero: A0, b0, EaR0, then Troe a, 1/T3, 1/T1, T2, B (Tsang: a = A, 1/T3 = inf,
                             // 1/T1 = 0, T2 = 0, B) or SRI a, b, c, d, e
    const double* gend;      // n_gen x 12: reactant order[4], reactant stoich[4], product stoich[4]
    const int* tbk;          // efficiency species
    const double* tbe;       // efficiency - default
    const double* comp;      // K x E element composition
    const double* pdd;       // PLOG and Chebyshev records (see DeviceMech)
    int const_volume;        // reactor model of an integrator launch: 0 IdealGasConstPressureReactor
                             // (the P argument is the pressure), 1 IdealGasReactor (it is the volume)
};

// Tables of the batched Jacobian without atomics (jac_tile.hip; nd = 0 if the
// mechanism does not qualify).  Each reaction stores its derivatives in
// consecutive slots: one per reactant, one per product if reversible, one for
// [M] if it has explicit efficiencies.  Each entry of the K x K matrix
// d wdot / d C is a list of (slot, coefficient), long ones cut into pieces;
// pieces are ranked by length, 256 to a group, and the 64 lists of a wavefront
// in a group lie interleaved in rows of 64, padded with (nd, 0), whose slot
// holds 0.
struct JacTables {
    int nd, ncoef, groups, nsplit, nover;
    const unsigned* rxn;          // per reaction (permuted, padded): slot | reactants << 16 | products << 19 | [M] << 22
    const unsigned* ell;          // slot | coefficient index << 16
    const int2* seg;              // per group and wavefront: first row, rows
    const unsigned short* pos;    // per lane of a group: k K + j, K K + overflow piece, or 0xffff
    const int2* split;            // entries in several pieces: k K + j, overflow pieces
    const double* coef;
};

// Owns device memory for a DevMech.
class DeviceMech {
public:
    explicit DeviceMech(const HostMech& h);
    ~DeviceMech();
    DeviceMech(const DeviceMech&) = delete;
    DeviceMech& operator=(const DeviceMech&) = delete;
    const DevMech& view() const { return d_; }
    const JacTables& jac() const { return jac_; }
    const HostMech& host() const { return h_; }
    const std::vector<int>& perm() const { return perm_; }   // permuted index -> mechanism index
    size_t table_bytes() const { return bytes_; }

private:
    HostMech h_;
    DevMech d_{};
    JacTables jac_{};
    void build_jac();
    void* tables_ = nullptr;
    std::vector<int> perm_;
    size_t bytes_ = 0;
    // tables are collected in one host image and copied with one allocation
    // (finish_upload), which then sets the pointers
    template <class T> void upload(const std::vector<T>& v, const T*& dst);
    void finish_upload();
    std::vector<char> image_;
    std::vector<std::pair<const void**, size_t>> fix_;
};

}  // namespace cg
