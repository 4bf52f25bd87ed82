// Host setup of one instance: geometry, stencils, least-squares
// pseudo-inverses and the structure-of-arrays image the kernels read.
#pragma once

#include <cstdint>
#include <functional>
#include <vector>

#include "common.hpp"

namespace zfv {

// Compile-time shape family of the kernels (see kernels.hip for the
// instantiations that exist).
struct Shape {
  int dim = 2;      // 2 or 3
  int nvars = 4;    // conserved variables stored: rho, m (dim), E
  int nfaces = 3;   // faces per cell
  int q = 2;        // quadrature points per face
  int qv = 6;       // quadrature points per cell (volume rule)
  int dofc = 6;     // dof of the highest-order (central) stencil's polynomial
  int rc = 10;      // rows of the central LSQ system (members - 1)
  int nb = 3;       // number of one-sided stencils
  int dofb = 3;     // dof of the one-sided polynomials
  int rb = 3;       // rows of each one-sided LSQ system
  int m = 68;       // pseudo-inverse entries per cell
  int nrows = 19;   // stencil rows per cell = rc + nb*rb
  int nmom = 3;     // stored moments (indices 3 .. dofc-1)
};

// Per-cell meta bits
enum : int32_t {
  META_KHIGH_MASK = 0x7,      // index of the stencil that receives the CWENO correction
  META_FIRST_ORDER = 1 << 3,  // single one-cell stencil: constant reconstruction
  META_GHOST = 1 << 4,        // frozen ghost cell
};

// cface bits: (face_id << 2) | (side << 0) | (exterior << 1)
constexpr int CFACE_SIDE_R = 1;
constexpr int CFACE_EXTERIOR = 2;
// a face between two ghost cells: no flux and no flux BC, geometry only
// (include/zisa/fvm_loops/flux_loop.hpp:71-83 leaves such faces out)
constexpr int CFACE_GHOST_PAIR = CFACE_EXTERIOR | CFACE_SIDE_R;

struct HostImage {
  Shape s;
  int64_t n = 0;   // cells
  int64_t n_near = 0;  // cells that are not ghosts away from the interior: the first ones
  int64_t ne = 0;  // interior faces
  std::vector<double> P;         // m * n in tiles of one wavefront's cells (p_central)
  std::vector<int32_t> rows;     // nrows * n   (product numbering)
  // one-sided row r (rc <= r < nrows) whose member (cell and translation) is
  // also central row twin[(r - rc) * n + i]: its equilibrium average is the
  // central row's; -1 if none
  std::vector<int8_t> twin;      // (nrows - rc) * n
  std::vector<double> crn;       // (nfaces*dim) * n, corner k coordinate d at (k*dim+d)
  std::vector<double> xc;        // dim * n
  std::vector<double> len, vol, inr;
  std::vector<double> mom;       // nmom * n
  std::vector<int32_t> meta;     // n
  std::vector<int32_t> cface;    // 4 * n: per cell its face words (2D: the fourth unused)
  // the cell-face slots (i * nfaces + k, product numbering) of each interior
  // face's left (side 0, first ne entries) and right (side 1) cell: where the
  // reconstruction leaves the face's point values
  std::vector<int32_t> fslot;    // ne pairs (left slot, right slot)
  std::vector<uint32_t> fperm;   // n: own-corner index of the face's left-cell vertex order
  std::vector<int32_t> perm;     // product index -> caller index
  std::vector<int32_t> iperm;    // caller index -> product index
  std::vector<uint8_t> ghost;    // product numbering
  // reference-layout bookkeeping for zfv_get_stencils (caller numbering)
  std::vector<int32_t> l2g_off, l2g;               // CSR of the combined stencil
  std::vector<int32_t> mem_off, members;           // CSR of [order, size, ids...]
  // normalized quadrature rules used by the kernels (device constants)
  std::vector<double> face_w, face_x;  // q weights; face_x: q * (dim) barycentric / GL coordinates
  std::vector<double> vol_w, vol_x;    // qv weights; vol_x: qv * (dim+1) barycentric
  // periodic translations of stencil members: row code c (bits 27..30 of a
  // row entry) adds shift[3c..3c+2] to the member's coordinates; code 0 = none
  std::vector<double> shift = std::vector<double>(48, 0.0);
  double max_cond = 0.0;               // largest estimated condition number of A^T A
  double linear_weights[ZFV_MAX_STENCILS] = {0};
};

// Hilbert index of integer coordinates with `bits` bits per axis (bits <= 32
// in 2D, <= 21 in 3D): the cell order of the instances and of the mesh
// renumbering tool.
uint64_t hilbert2(uint32_t x, uint32_t y, int bits);
uint64_t hilbert3(uint32_t x, uint32_t y, uint32_t z, int bits);

// Builds everything on the host.  Throws ZfvError on unsupported input.
void build_image(const zfv_mesh &mesh, const zfv_params &p, HostImage &img);

// Shape implied by the parameters (throws if the GPU kernels have no
// instantiation for it).
Shape shape_for(const zfv_params &p);
// true when the volume rule and the cell moments both integrate the central
// polynomial's basis exactly: then the quadrature mean of a reconstruction
// over its cell is its constant coefficient (every other basis function has
// mean zero), which the light set's gravity volume term uses
bool volume_mean_is_constant_term(const zfv_params &p, const Shape &s);

// The faces of the update kernel's tiles of `cells` consecutive cells: per tile
// its interior faces once each (both sides where both cells are in the tile)
// and, with the constant flux BC, its boundary faces: 64 UpdateFace entries a
// tile, tile t's further ones in more from off[t]; per cell a word naming its
// faces' entries.
void build_update_tiles(const HostImage &img, int cells, bool flux_bc, std::vector<int32_t> &entries,
                        std::vector<int32_t> &off, std::vector<int32_t> &more, std::vector<uint32_t> &cell_words);

// The caller's n x 5 row-major state (AllVariables::cvars) to and from the
// product's nvars x n planes in product order (perm: product index -> caller
// index), on the host's threads.  from_soa adds into aos when accumulate.
void to_soa(const HostImage &img, const double *aos, double *soa);
void from_soa(const HostImage &img, const double *soa, double *aos, bool accumulate);
// The same with the kernels' layout: nvars values per cell in product order
// (state_at with AOS).
void to_cells(const HostImage &img, const double *aos, double *cells);
enum class Into { Set, Add, FromZero };  // aos = c, aos += c, aos = 0 + c (which turns -0 into 0)
void from_cells(const HostImage &img, const double *cells, double *aos, Into into);
// Has pages of a caller's output array of n doubles mapped while the device
// computes or copies (busy), its contents unchanged: a fresh array's page faults
// are otherwise waited for afterwards.  Up to kMapWhole bytes all at once (one
// call takes 90 us a MB of small pages, 50 of huge ones; 16 writing threads that
// meet their faults take longer: a state of 2.0 MB is read into small pages in
// 0.24 instead of 0.41 ms, 3.1 MB 0.34 / 0.41).  Larger ones piece by piece as
// long as the device is busy; the rest is left to the threads that write, which
// map it faster than one call does (read into small pages: 8.2 MB 0.47 instead
// of 0.86 ms, 16.3 MB 0.89 / 1.72, 32.8 MB 1.68 / 3.5; huge pages 0.35 / 0.53,
// 0.58 / 0.84, 1.08 / 1.8; at 4.1 MB both take 0.44).  Where the threads read
// before they write (all), the rest is mapped by all of them first, beyond twice
// kMapWhole: a first read costs a page a second fault (a rate added into untouched
// small pages, one call / piece by piece: 4.1 MB 0.51 / 0.67 ms, 8.2 MB 0.97 /
// 0.86, 16.3 MB 1.90 / 1.62; nothing mapped ahead 7.2, 7.5 and 14 ms).
constexpr size_t kMapWhole = 3500000;
void map_pages(double *out, size_t n, bool all, const std::function<bool()> &busy);

}  // namespace zfv
