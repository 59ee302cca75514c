// Internal handle types of libflygpu (host side).
#pragma once

#include <istream>
#include <memory>
#include <string>
#include <vector>

#include "common.hpp"

namespace flyg {

  // Raw setfl contents (host, FP64).
  struct SetflData {
    int ntypes = 0;
    std::vector<std::string> names;
    std::vector<double> mass;
    double drho = 0, dr = 0, rcut = 0;
    std::vector<std::vector<double>> F, phi, V;   // phi[a + n*b], V[max + n*min]
  };

  SetflData read_setfl(std::string const& path);
  SetflData read_setfl_stream(std::istream& in);
  std::vector<double4> spline_coefficients(std::vector<double> y, double dx);

}  // namespace flyg

// ------------------------------------------------------------------------------------------------
// Handles (the opaque types of flygpu.h).
// ------------------------------------------------------------------------------------------------

struct flyg_ctx_s {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  int cus = 0;
  flyg::DBuf<unsigned> dflags;   // [0] error bits, [1..] scratch counters
  // Pinned: [0] error bits read by take_flags, [1] those a kernel left, [2] a count, [3] set by an L-BFGS step that
  // gave up waiting (lb_newton), [4] by one of a rotor, which may be under way beside it.
  unsigned* hflags = nullptr;
  double* hpart = nullptr;       // pinned: block partial sums that kernels write for the host, then scalars

  unsigned step_polls = 1u << 14;   // polls before a workgroup of lb_newton gives up (about 10 ms)

  int refs = 1;                  // the context lives until its creator and every handle released it

  void set_device() const;
  unsigned take_flags();         // sync, read and clear the error bits
  void retain() { ++refs; }
  void release();
};

struct flyg_eam_s {
  flyg_ctx_s* ctx = nullptr;
  flyg::SetflData data;
  flyg::EAMTables tab{};   // device view
  // The same in device memory, for kernels that are launched often: 1.5 KB of arguments by value cost 0.6 us a
  // launch on the host.
  flyg::DBuf<flyg::EAMTables> dtab;
  flyg::DBuf<double4> c64;
  flyg::DBuf<float4> c32;
  int precision = FLYG_FP64;
  // scratch
  flyg::DBuf<double4> posf;     // positions + F' (pass 1 -> pass 2)
  flyg::DBuf<double2> dfp;      // HVP: (F', dF') per atom
  flyg::DBuf<double> eatom;     // per-atom energies
  flyg::DBuf<uint32_t> types;   // staged host inputs
  flyg::DBuf<uint32_t> gtype;   // types in the list's slot order (gradients with several species)
  long types_stamp = 0;         // renewed (process-wide unique) whenever the staged host types change
  long gtype_build = -1, gtype_stamp = -1;   // gtype holds the staged types in the layout of this build
  flyg::DBuf<uint8_t> frozen;
  flyg::DBuf<double> vec_in, vec_out;
  flyg::DBuf<double> hess;      // workspace of hessian_eigenvalues, kept between calls while it is small
  flyg::DBuf<int> hess_ids;     // its atom indices
  std::vector<uint32_t> last_types;
  std::vector<uint8_t> last_frozen;
  int lanes = 0;                // lanes per atom row, 0 = the library's choice
  int staged_single = -1;       // one species in the staged host types, else -1
  long staged_n = -1;           // atoms in the staged copy (types/frozen), -1 = none
  // Optional kernel timing of gradient calls: one event pair around each call's kernels.
  bool timing = false;
  std::vector<std::pair<hipEvent_t, hipEvent_t>> events;
  std::size_t events_used = 0;
  ~flyg_eam_s() {
    for (auto& e : events) {
      (void)hipEventDestroy(e.first);
      (void)hipEventDestroy(e.second);
    }
  }
};

struct flyg_list_s {
  flyg_ctx_s* ctx = nullptr;
  flyg::BoxDesc box{};
  flyg::GridDesc grid{};
  double rc = 0;
  long n = 0;
  long nghost = 0;
  int K = 0;       // row capacity of the neighbour table
  bool built = false;
  long build_id = 0;   // unique per successful rebuild (process-wide), names the slot layout in use
  flyg::DBuf<double4> pos;       // live positions (x, y, z, 0)
  flyg::DBuf<double4> ent;       // reals + ghost images at build time (chained positions)
  flyg::DBuf<unsigned> eid;      // packed (shift, real) of ent
  flyg::DBuf<int> ecell;         // cell of ent
  flyg::DBuf<int> earr;          // its place in the cell in arrival order
  flyg::DBuf<int> ccount, cstart;
  flyg::DBuf<double4> spos;      // ent sorted by cell (packed-id order inside a cell)
  flyg::DBuf<unsigned> usid;     // packed ids scattered by cell, unordered inside a cell
  flyg::DBuf<int> rslot;         // sorted slot of each real atom
  flyg::DBuf<unsigned> sid;
  flyg::DBuf<unsigned> nbr;      // n x K packed entries
  flyg::DBuf<int> ncnt;          // entries per atom
  // The gradient passes' layout, made at each rebuild: the real atoms in cell order (slot k holds atom
  // order[k], rank[i] is atom i's slot) and their positions by slot (kept current by update).
  flyg::DBuf<int> order, rank;
  // gpos's w slot holds the species of each slot for a multi-species gradient (written with the slot-order
  // types; update keeps it): those of the staged host types with stamp wtype_stamp, if wtype_build is the
  // current build_id, else of the last gradient call's types.
  flyg::DBuf<double4> gpos;
  long wtype_stamp = -1, wtype_build = -1;
  // Tiles (boxes of cells): a pair kernel's workgroup stages the positions of a tile's cells and of the cells
  // around it in LDS and walks its atoms' rows through 16-bit indices into that stage.  sslot: the
  // sorted entries (reals and images, cell by cell) as (shift, slot); rows: by slot, rowK entries of
  // room, in blocks of 32 whose entry k lies at 2 (k mod 16) + (k / 16 mod 2), so a lane of 16 loads two at a time.
  // Lists that are not tiled keep packed (shift, slot) entries there instead, nbr's in the slot order.
  flyg::TileGrid tile{};
  bool tiled = false;            // rows and sslot belong to this build
  int tile_most = 0;             // entries staged by the fullest tile
  // Of the last build, for every tile shape: entries of the fullest tile, and tiles that hold atoms.  Valid for the
  // next one while the atom count and the grid stay the same (tile_seen).
  unsigned tile_full[flyg::TILE_KINDS] = {}, tile_used[flyg::TILE_KINDS] = {};
  bool tile_seen = false;
  int tile_shape[3] = {};        // the grid they belong to
  int rowK = 0;
  double mean_row = 0;           // entries of a row, roughly
  flyg::DBuf<unsigned> sslot;
  flyg::DBuf<unsigned> rows;
  flyg::DBuf<int> gcnt;          // entries per slot
  // The plain rows in slot order of a tiled list, K entries of room each, made when a build's first call needs them.
  flyg::DBuf<unsigned> srows;
  long srows_build = -1;
  bool grad_rows = false;        // a tiled list whose gradients are faster by rows, from a build's second on
  long grad_build = -1;          // the build of the last gradient
  flyg::DBuf<int> scan_tmp;
  flyg::DBuf<double> stage;      // host staging of xyz vectors
  flyg::DBuf<unsigned> lstate;   // device build counters: two sets of LIST_STATE words, used in turn
  int parity = 0;                // the set of the next build
  // ccount and that set are zero for a grid of so many cells + 1 (the search server gives one list object
  // system after system, each with its own box and grid).
  long clear_cells = -1;
  unsigned* hstate = nullptr;    // pinned mirror
  long gcap = 0;                 // ghost slots
  ~flyg_list_s() {
    if (hstate) (void)hipHostFree(hstate);
  }
};

namespace flyg {
  // Shift vectors of the 27 image codes (sum of +-basis columns), for pair arithmetic.
  void shift_table(BoxDesc const& b, double3* out27);

  // What take_flags returned, as an error: whoever clears the bits reports every one of them.
  inline void throw_flags(unsigned fl) {
    if (fl & ERR_SPLINE_OOB) throw Error(FLYG_SPLINE_OOB, "x is outside tabulated region of a spline");
    if (fl & ERR_TYPE) throw Error(FLYG_INVALID_ARG, "TypeID out of range");
    if (fl) throw Error(FLYG_DEVICE_ERROR, "device error flag set");
  }

  // neigh.hip
  void list_rebuild(flyg_list_s& nl, double const* d_xyz, long n);
  void list_update(flyg_list_s& nl, double const* d_delta, long n);
  // Exclusive scan of src into dst (they may be the same; both hold scan_room(n) values, whatever lies past the
  // n-th); clear_state: src and the LIST_STATE words there are zeroed.
  constexpr int LIST_STATE = 16;
  constexpr long scan_room(long n) { return (n + 3) & ~3l; }
  void exclusive_scan(flyg_ctx_s& ctx, int* src, int* dst, int n, flyg::DBuf<int>& tmp, unsigned* clear_state = nullptr);

  // eam.hip
  struct PairArgs {
    double4 const* pos;
    unsigned const* nbr;
    int const* cnt;
    int K;
    long n;
    uint32_t const* types;
    uint8_t const* frozen;
    int t0;   // the one species present (-1: several or unknown); read by the single-species kernels
    // Null: rows, positions and types are by atom.  Otherwise they are by slot of the list's cell-order
    // layout (types gathered into slot order) and order[slot] is the atom, for frozen flags and gradients.
    int const* order = nullptr;
    // The w slot of pos holds each atom's species (as a double), so a neighbour's species arrives with
    // its position; set for the slot layout with several species.
    bool type_in_w = false;
  };
  // Image shift of a packed entry: sum_a s_a * basis column a, s_a in {-1, 0, 1}.  Exact for
  // orthorhombic boxes (each component is 0 or +-L), computed in registers (no table lookup).
  struct Shifts {
    double b[3][3];   // b[row][col]
    __device__ double3 of(unsigned code) const {
      int s0 = static_cast<int>(code % 3u) - 1;
      int s1 = static_cast<int>((code / 3u) % 3u) - 1;
      int s2 = static_cast<int>(code / 9u) - 1;
      return make_double3(s0 * b[0][0] + s1 * b[0][1] + s2 * b[0][2], s0 * b[1][0] + s1 * b[1][1] + s2 * b[1][2],
                          s0 * b[2][0] + s1 * b[2][1] + s2 * b[2][2]);
    }
  };
  inline Shifts shifts_of(BoxDesc const& b) {
    Shifts s;
    for (int r = 0; r < 3; ++r)
      for (int c = 0; c < 3; ++c) s.b[r][c] = b.B[r][c];
    return s;
  }
  __device__ inline int vidx(EAMTables const& T, int a, int b) { return a > b ? a + T.ntypes * b : b + T.ntypes * a; }
  PairArgs pair_args(flyg_eam_s const& E, flyg_list_s& nl, uint32_t const* types, uint8_t const* frozen);

  void eam_setup_tables(flyg_eam_s& e);
  double eam_energy(flyg_eam_s& e, flyg_list_s& nl, uint32_t const* d_types, uint8_t const* d_frozen);
  void eam_gradient(flyg_eam_s& e, flyg_list_s& nl, uint32_t const* d_types, uint8_t const* d_frozen, double* d_grad,
                    int precision);
  // Allocation-free gradient: the pass-1 output lives in a file-scope device array of NOALLOC_MAX_ATOMS
  // entries; noalloc_scratch_init(device) looks its address up once per device (that device current).
  constexpr long NOALLOC_MAX_ATOMS = 131072;
  void noalloc_scratch_init(int device);
  void eam_gradient_noalloc(flyg_eam_s& e, flyg_list_s& nl, uint32_t const* d_types, uint8_t const* d_frozen,
                            double* d_grad, int precision);
  // Sorted eigenvalues of the mass-weighted Hessian block of the non-frozen atoms (hessian.hip).
  std::vector<double> hessian_eigenvalues(flyg_eam_s& e, flyg_list_s& nl, uint32_t const* d_types,
                                          uint8_t const* d_frozen, std::vector<uint8_t> const& h_frozen,
                                          std::vector<uint32_t> const& h_types);
  void eam_hvp(flyg_eam_s& e, flyg_list_s& nl, uint32_t const* d_types, uint8_t const* d_frozen, double const* d_v,
               double* d_hv);
  void eam_table_eval(flyg_eam_s& e, int kind, int a, int b, double const* x, long m, int deriv, double* out);

  // Stage host per-atom inputs into the potential handle (re-uploads only when they changed); device
  // inputs pass through; types = frozen = null selects the staged copy.
  void stage_atoms(flyg_eam_s& e, uint32_t const* types, uint8_t const* frozen, long n, int where,
                   uint32_t const** d_types, uint8_t const** d_frozen);
  // Copy device per-atom inputs into the handle's staged buffers.
  void stage_atoms_device(flyg_eam_s& e, uint32_t const* types, uint8_t const* frozen, long n);

  // Block partial sums of x and the error flags, for the host (vecops.hip).
  void dev_sum(flyg_ctx_s& ctx, double const* x, long n, double* part, unsigned* hflag);
}  // namespace flyg
