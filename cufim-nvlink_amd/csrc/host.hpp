// host.hpp -- host-side data structures of the FIM solver (mesh, partition,
// device pack).  Internal to libcufim.so; the public surface is include/cufim.h.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <mutex>
#include <stdexcept>
#include <string>
#include <thread>
#include <vector>

#include "cufim.h"

namespace fim {

// f(begin, end) over [0, n) on up to eight host threads, at least `least` each
// (starting and joining four took 20 to 50 us).  f may not throw.
template <class F>
void parallel_ranges(size_t n, size_t least, F &&f) {
  const size_t nt = std::max<size_t>(1, std::min<size_t>({8, (size_t)std::thread::hardware_concurrency(), n / least}));
  std::vector<std::thread> ts;
  ts.reserve(nt);
  size_t t = 1;
  try {
    for (; t < nt; ++t) ts.emplace_back([&f, n, nt, t] { f(n * t / nt, n * (t + 1) / nt); });
  } catch (const std::exception &) {  // no more threads: the rest on this one
  }
  f(0, n / nt);
  if (t < nt) f(n * t / nt, n);
  for (auto &w : ts) w.join();
}

// error carried to the C ABI as (code, message)
struct Error : std::runtime_error {
  int code;
  Error(int c, const std::string &m) : std::runtime_error(m), code(c) {}
};

void set_last_error(const std::string &msg);

// ---------------------------------------------------------------------------
// Mesh: tetrahedra only.  Element node lists are kept sorted ascending, the
// order the reference establishes in compute_base_connectivity
// (src/core/types.cpp:63-67) and writes to its VTK output.
// ---------------------------------------------------------------------------
struct Mesh {
  int64_t nn = 0, ne = 0;
  std::vector<double> xyz;      // 3*nn
  std::vector<int64_t> e2n;     // 4*ne, sorted per element
  std::vector<double> fib;      // 3*ne unit fibre
  std::vector<double> vel;      // 2*ne (v_fibre, v_cross)
  std::vector<int32_t> etags;   // ne, written as elemTag
  std::vector<int32_t> atags;   // ne partition tags (may be empty)
  std::vector<uint8_t> region;  // ne region ids 0..3 (may be empty)

  // vertex -> incident elements, ascending element id
  std::vector<int64_t> n2e_dsp;  // nn+1
  std::vector<int64_t> n2e_con;  // 4*ne

  void finalize();  // sorts element nodes, validates, builds n2e
};

// metric tensor M = f f^T / vf^2 + (I - f f^T) / vs^2 packed (xx xy xz yy yz zz)
void metric_tensor(const double f[3], double vf, double vs, double M[6]);
// 6 squared metric edge lengths e12 e13 e23 e14 e24 e34 of element e in the
// element's (sorted) node order
void element_geo(const Mesh &m, int64_t e, double geo[6]);
double front_width(const Mesh &m);

Mesh load_vtk(const std::string &path);
void save_vtk(const Mesh &m, const std::string &path, const double *phi,
              const int32_t *state);
std::vector<int32_t> read_tags(const std::string &path);
Mesh gen_box(double lx, double ly, double lz, int nx, int ny, int nz, double jitter,
             uint64_t seed, double a0, double a1, double vf, double vc);
Mesh gen_shell(double ao, double bo, double ai, double bi, double h, int n_scars, double r0,
               double r1, uint64_t seed, double vf, double vc, double vs);

// ---------------------------------------------------------------------------
// Partition: elements grouped into submeshes, vertices duplicated per
// submesh ("copies"), copies of one submesh contiguous.
// ---------------------------------------------------------------------------
struct Partition {
  int64_t nsub = 0;
  std::vector<int64_t> e2s;        // ne
  std::vector<int64_t> s_edsp;     // nsub+1 offsets into s_elems
  std::vector<int64_t> s_elems;    // element ids in submesh order
  std::vector<int64_t> s_vdsp;     // nsub+1 offsets into l2g
  std::vector<int64_t> l2g;        // copy -> global vertex
};

Partition partition_from_tags(const Mesh &m, const std::vector<int32_t> &tags);
Partition partition_rcb(const Mesh &m, int max_nn, int max_ne, uint64_t seed);

// ---------------------------------------------------------------------------
// Pack: device layout.  All offsets are absolute indices into the flat
// arrays below.
// ---------------------------------------------------------------------------
struct SubInfo {
  uint32_t eoff, ne;   // elements [eoff, eoff+ne)
  uint32_t coff, nn;   // copies   [coff, coff+nn)
  uint32_t ioff, ni;   // interface entries [ioff, ioff+ni)
};

struct Pack {
  int64_t nn_global = 0, ne_global = 0, nsub = 0, ncopy = 0;
  int32_t nn_max = 0, ne_max = 0;
  int32_t source = FIM_PART_RCB;
  Partition part;
  std::vector<SubInfo> sub;        // nsub
  std::vector<uint16_t> e2n_l;     // 4 per element: local copy ids, sorted
  std::vector<float> geo32;        // 6 per element
  std::vector<float> hgt32;        // 4 per element: metric height of each node
                                   // above its opposite face, rounded down
  std::vector<double> geo64;       // 6 per element
  std::vector<uint8_t> ereg;       // 1 per element
  std::vector<uint32_t> c2g;       // per copy
  std::vector<uint32_t> c2s;       // per copy
  std::vector<uint32_t> g2c_dsp;   // nn_global+1
  std::vector<uint32_t> g2c;       // ncopy, ascending submesh
  std::vector<uint32_t> grp_v;     // global vertices with >= 2 copies
  // interface (converge mode): per submesh entries [ioff, ioff+ni)
  std::vector<uint16_t> if_l;      // local copy id of the entry
  std::vector<uint32_t> if_dsp;    // n_if+1 offsets into if_other
  std::vector<uint32_t> if_other;  // other copies (global copy ids)
  // compat extras: per copy CSR into local element / vertex lists
  std::vector<uint32_t> n2e_dsp;   // ncopy+1
  std::vector<uint16_t> n2e_le;    // local element id
  std::vector<uint8_t> n2e_pos;    // position of the owner in that element
  std::vector<uint32_t> n2n_dsp;   // ncopy+1
  std::vector<uint16_t> n2n_lv;    // local copy ids, sorted, self included
  double front_width = 0.0;
};

Pack build_pack(const Mesh &m, const Partition &p, int32_t source);

// Candidate bounds of the elements (cand_bounds), for the band kernel's records
struct ElementBounds {
  std::vector<uint8_t> b;      // 12 per element: for each node as target, lower bounds
                               // n . (x_target - x_i) of the other three nodes for a unit
                               // direction n, (byte - 128) * scale
  std::vector<float> scale;    // 1 per element
};
ElementBounds element_bounds(const Pack &k);

// element-list entries the converge-mode band kernel keeps per pass at least
// (more marked elements take further passes)
constexpr uint32_t kElistCap = 2032;
// (element, target) pair ring of one wave in the band kernel: pairs left from
// earlier rounds of 64 ilp plus 4 targets of 64 elements
constexpr uint32_t pair_ring(int ilp) { return 64u * (uint32_t)ilp + 256u; }
// the band kernel evaluates pairs with workgroups of 256 and 512, where local
// element ids fit 14 bits
inline bool band_with_pairs(int block, int32_t ne_max) {
  return (block == 256 || block == 512) && ne_max < (1 << 14);
}
// A list of at most one unit per submesh leaves the CUs with a few waves each
// when the mesh has few submeshes: the band kernel gets registers for two pair
// rounds side by side then
inline bool few_submeshes(int64_t nsub, int cus) { return nsub <= 4 * (int64_t)cus; }

// Elements per wave of a workgroup up to which a submesh's sweeps are listed by
// few waves (GATHER of k_conv_band): always, and while the launch's units fill
// at least half of its workgroups
constexpr uint32_t kGatherAlways = 256, kGatherFull = 640;

// Dynamic LDS of the converge-mode kernels for the largest submesh: byte
// offsets, the entries of the element list, all bytes.
struct ConvergeCarve {
  uint32_t o_phin, o_flg, o_tch, o_dfr, o_e2n, o_geo, o_list, o_vlist, o_misc, o_wrt, o_ifc, elcap, bytes;
};
// ilp: pair rounds side by side, 0 without pairs
ConvergeCarve converge_carve(int32_t nn_max, int32_t ne_max, int block, bool staged, int ilp);

// solver-context hooks for the surrogate (csrc/surrogate.hip); device
// pointers, work queued on the context's stream
void *ctx_stream(fim_ctx *c);
int32_t ctx_device(const fim_ctx *c);
uint32_t ctx_vertices(const fim_ctx *c);
int32_t ctx_instances(const fim_ctx *c);
bool ctx_converge(const fim_ctx *c);
// per-vertex map of an instance (min over copies) in the context's field buffer
const float *ctx_gather(fim_ctx *c, int32_t inst);
// the context's field buffer (nn floats): fill it, then ctx_init_field
float *ctx_field_buffer(fim_ctx *c);
// instance field := field buffer; all_active marks every copy dirty and
// queues every submesh (warm start), otherwise only the times are set
void ctx_init_field(fim_ctx *c, int32_t inst, bool all_active);

}  // namespace fim

// for tests of long runs, not part of cufim.h: the context's next iteration
// gets the number n, or n + 1; in compat mode its next window, higher than
// the last one's
extern "C" int fim_ctx_renumber(fim_ctx *c, uint32_t n);

struct fim_mesh {
  fim::Mesh m;
};
struct fim_pack {
  fim::Pack p;
  // worked out for the first context that runs the band kernel (0.1 s for 2M
  // elements), kept for those after it
  mutable fim::ElementBounds bounds;
  mutable std::once_flag bounds_once;
};
