// Host driver of the nuclear-derivative integral kernels (integrals_grad.hpp):
// launches every shell class with its response weights and reduces the
// per-task / per-function partial derivatives to atoms in a fixed order, so
// the gradient is bitwise reproducible run to run.
#include <algorithm>

#include "integrals_grad.hpp"
#include "integrals_gradient.hpp"

namespace vqc {
using namespace detail;
namespace {

void dispatch_pair_grad(int la, int lb, int lc, bool cart, const ThreeCenterGradArgs& args, int nchunk, hipStream_t s) {
  switch (la * 10 + lb) {
    case 0: dispatch_3c_grad_00(lc, cart, args, nchunk, s); break;
    case 10: dispatch_3c_grad_10(lc, cart, args, nchunk, s); break;
    case 11: dispatch_3c_grad_11(lc, cart, args, nchunk, s); break;
    case 20: dispatch_3c_grad_20(lc, cart, args, nchunk, s); break;
    case 21: dispatch_3c_grad_21(lc, cart, args, nchunk, s); break;
    case 22: dispatch_3c_grad_22(lc, cart, args, nchunk, s); break;
    case 30: dispatch_3c_grad_30(lc, cart, args, nchunk, s); break;
    case 31: dispatch_3c_grad_31(lc, cart, args, nchunk, s); break;
    case 32: dispatch_3c_grad_32(lc, cart, args, nchunk, s); break;
    case 33: dispatch_3c_grad_33(lc, cart, args, nchunk, s); break;
    default: throw NotImplemented("orbital angular momentum above f");
  }
}

void dispatch_metric_grad(int la, int lc, bool cart, const ThreeCenterGradArgs& args, int nchunk, hipStream_t s) {
  switch (la) {
    case 0: dispatch_metric_grad_0(lc, cart, args, nchunk, s); break;
    case 1: dispatch_metric_grad_1(lc, cart, args, nchunk, s); break;
    case 2: dispatch_metric_grad_2(lc, cart, args, nchunk, s); break;
    case 3: dispatch_metric_grad_3(lc, cart, args, nchunk, s); break;
    default: throw NotImplemented("auxiliary angular momentum above f");
  }
}

void dispatch_1e_grad(int la, int lb, const OneElectronGradArgs& args, hipStream_t s) {
  switch (la * 10 + lb) {
    case 0: dispatch_1e_grad_00(args, s); break;
    case 10: dispatch_1e_grad_10(args, s); break;
    case 11: dispatch_1e_grad_11(args, s); break;
    case 20: dispatch_1e_grad_20(args, s); break;
    case 21: dispatch_1e_grad_21(args, s); break;
    case 22: dispatch_1e_grad_22(args, s); break;
    case 30: dispatch_1e_grad_30(args, s); break;
    case 31: dispatch_1e_grad_31(args, s); break;
    case 32: dispatch_1e_grad_32(args, s); break;
    case 33: dispatch_1e_grad_33(args, s); break;
    default: throw NotImplemented("orbital angular momentum above f");
  }
}

constexpr int kReduceThreads = 256;

// The partial derivatives of every class of a gradient share one layout, so
// a few launches sum them, whatever the number of classes (one launch per
// class, whose blocks each read all of its partials, took 80 to 120 us; with
// the uploads and allocations of each class the (H2O)6 gradient took 12.0 ms
// and takes 6.4):
//   ab[task][slot][6]  d/dA, d/dB of the shell pairs of all classes (a slot
//                      is a block of 64 functions),
//   c[row][3 column]   d/dC of each function or nucleus; a class' launch
//                      writes the columns of its functions in its own rows.
// Every sum has a fixed order.

// task_sum[task][6] = sum over slots.
__global__ __launch_bounds__(kReduceThreads) void sum_slots_kernel(const double* __restrict__ ab, std::size_t ntask,
                                                                   int nslot, double* __restrict__ task_sum) {
  const std::size_t e = static_cast<std::size_t>(blockIdx.x) * kReduceThreads + threadIdx.x;
  if (e >= ntask * 6) return;
  const double* p = ab + (e / 6) * nslot * 6 + e % 6;
  double s = 0.0;
#pragma unroll 8
  for (int k = 0; k < nslot; ++k) s += p[k * 6];
  task_sum[e] = s;
}

// out[col] = sum over rows of c[row][col]: 64 columns a block, 16 row groups.
constexpr int kColumns = 64, kRowGroups = 16;
__global__ __launch_bounds__(kColumns* kRowGroups) void sum_columns_kernel(const double* __restrict__ c, int rows,
                                                                           int cols, double* __restrict__ out) {
  __shared__ double red[kRowGroups][kColumns];
  const int lane = threadIdx.x % kColumns, g = threadIdx.x / kColumns;
  const int col = blockIdx.x * kColumns + lane;
  double s = 0.0;
  if (col < cols) {
#pragma unroll 8
    for (int r = g; r < rows; r += kRowGroups) s += c[static_cast<std::size_t>(r) * cols + col];
  }
  red[g][lane] = s;
  __syncthreads();
  if (g == 0 && col < cols) {
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < kRowGroups; ++k) t += red[k][lane];
    out[col] = t;
  }
}

// grad[atom] += the A part of the tasks whose bra shell sits on the atom, the
// B part of those whose ket shell does, and the functions (nuclei) on it.
// One block per atom; the thread-to-entry map and the tree are fixed.
__global__ __launch_bounds__(kReduceThreads) void gather_atoms_kernel(const double* __restrict__ task_sum, int ntask,
                                                                      const int2* __restrict__ task_atoms,
                                                                      const double* __restrict__ fn_sum, int nfn,
                                                                      const int* __restrict__ fn_atoms,
                                                                      double* __restrict__ grad) {
  const int atom = blockIdx.x, tid = threadIdx.x;
  double s[3] = {0.0, 0.0, 0.0};
  for (int t = tid; t < ntask; t += kReduceThreads) {
    const int2 ta = task_atoms[t];
    const double* o = task_sum + static_cast<std::size_t>(t) * 6;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      if (ta.x == atom) s[d] += o[d];
      if (ta.y == atom) s[d] += o[3 + d];
    }
  }
  for (int f = tid; f < nfn; f += kReduceThreads) {
    if (fn_atoms[f] != atom) continue;
#pragma unroll
    for (int d = 0; d < 3; ++d) s[d] += fn_sum[static_cast<std::size_t>(f) * 3 + d];
  }
  __shared__ double red[3][kReduceThreads];
#pragma unroll
  for (int d = 0; d < 3; ++d) red[d][tid] = s[d];
  __syncthreads();
  for (int w = kReduceThreads / 2; w > 0; w >>= 1) {
    if (tid < w)
#pragma unroll
      for (int d = 0; d < 3; ++d) red[d][tid] += red[d][tid + w];
    __syncthreads();
  }
  if (tid < 3) grad[atom * 3 + tid] += red[tid][0];
}

// The shell pairs of all classes of one gradient, class by class, and the
// atoms of their shells and of the columns (functions or nuclei).
struct GradTasks {
  struct Class {
    int la, lb, begin, count;
  };
  std::vector<Class> classes;
  std::vector<int2> tasks, atoms;
  std::vector<int> columns;

  void add(int la, int lb, const std::vector<int2>& pairs, const System& sys) {
    if (pairs.empty()) return;
    classes.push_back({la, lb, static_cast<int>(tasks.size()), static_cast<int>(pairs.size())});
    for (const int2& t : pairs) {
      tasks.push_back(t);
      atoms.push_back(make_int2(static_cast<int>(sys.shells[t.x].atom), static_cast<int>(sys.shells[t.y].atom)));
    }
  }
};

// Device copies of the lists (one upload) and the partial buffers.
struct GradPartials {
  int ntask, ncol;
  DeviceArray<int2> lists;
  DeviceArray<double> ab, sums;
  const int2* tasks;
  const int2* atoms;
  const int* columns;

  GradPartials(const GradTasks& g, int nslot, hipStream_t s)
      : ntask(static_cast<int>(g.tasks.size())), ncol(static_cast<int>(g.columns.size())) {
    std::vector<int2> host(g.tasks);
    host.insert(host.end(), g.atoms.begin(), g.atoms.end());
    host.resize(2 * static_cast<std::size_t>(ntask) + (ncol + 1) / 2);
    std::copy(g.columns.begin(), g.columns.end(), reinterpret_cast<int*>(host.data() + 2 * static_cast<std::size_t>(ntask)));
    lists.upload(host, s);
    tasks = lists.data();
    atoms = tasks + ntask;
    columns = reinterpret_cast<const int*>(tasks + 2 * static_cast<std::size_t>(ntask));
    ab.resize(static_cast<std::size_t>(ntask) * nslot * 6);
    sums.resize(static_cast<std::size_t>(ntask) * 6 + static_cast<std::size_t>(ncol) * 3);
  }
  double* column_sums() { return sums.data() + static_cast<std::size_t>(ntask) * 6; }
  void sum_columns(const double* c, int rows, int first, int count, hipStream_t s) {
    const int cols = 3 * count;
    hipLaunchKernelGGL(sum_columns_kernel, dim3((cols + kColumns - 1) / kColumns), dim3(kColumns * kRowGroups), 0, s, c,
                       rows, cols, column_sums() + 3 * static_cast<std::size_t>(first));
    VQC_LAUNCH("sum_columns_kernel");
  }
  void gather(int nslot, int natom, double* grad, hipStream_t s) {
    const std::size_t entries = static_cast<std::size_t>(ntask) * 6;
    hipLaunchKernelGGL(sum_slots_kernel, dim3(static_cast<unsigned>((entries + kReduceThreads - 1) / kReduceThreads)),
                       dim3(kReduceThreads), 0, s, ab.data(), static_cast<std::size_t>(ntask), nslot, sums.data());
    VQC_LAUNCH("sum_slots_kernel");
    hipLaunchKernelGGL(gather_atoms_kernel, dim3(natom), dim3(kReduceThreads), 0, s, sums.data(), ntask, atoms,
                       column_sums(), ncol, columns, grad);
    VQC_LAUNCH("gather_atoms_kernel");
  }
};

// Task lists of unordered orbital shell pairs grouped by (larger l, smaller l).
std::vector<std::vector<int2>> grad_pair_tasks(const System& sys) {
  std::vector<std::vector<int2>> classes(100);
  const int n = static_cast<int>(sys.shells.size());
  for (int i = 0; i < n; ++i)
    for (int j = 0; j <= i; ++j) {
      const int li = sys.shells[i].l, lj = sys.shells[j].l;
      const int2 t = li >= lj ? make_int2(i, j) : make_int2(j, i);
      classes[std::max(li, lj) * 10 + std::min(li, lj)].push_back(t);
    }
  return classes;
}

// Enough blocks to fill the GPU while each block reuses its 64 functions'
// coefficients over several tasks.
int tasks_per_block(int ntask, int nfnblk) {
  const long long blocks = static_cast<long long>(ntask) * nfnblk;
  return static_cast<int>(std::max<long long>(1, std::min<long long>(ntask, blocks / 4096)));
}

// Every (class, auxiliary l) launch of a three-centre or metric gradient into
// the shared partials, then their sums.  `dispatch` launches one of them.
template <class Dispatch>
void contract_classes(const GradTasks& g, const AuxiliaryLayout& aux, int natom, ThreeCenterGradArgs args, double* grad,
                      hipStream_t s, Dispatch dispatch) {
  int nslot = 0;
  for (int lc = 0; lc <= kMaxAuxiliaryL; ++lc) nslot += (aux.class_begin[lc + 1] - aux.class_begin[lc] + 63) / 64;
  if (g.tasks.empty() || nslot == 0) return;
  GradPartials p(g, nslot, s);
  struct Launch {
    int tpb, nchunk;
  };
  std::vector<DeviceArray<double>> c(kMaxAuxiliaryL + 1);
  int slot = 0;
  for (int lc = 0; lc <= kMaxAuxiliaryL; ++lc) {
    const int begin = aux.class_begin[lc], nfn = aux.class_begin[lc + 1] - begin;
    if (nfn <= 0) continue;
    const int nfnblk = (nfn + 63) / 64;
    std::vector<Launch> launches;
    int rows = 0;
    for (const auto& k : g.classes) {
      const int tpb = tasks_per_block(k.count, nfnblk);
      launches.push_back({tpb, (k.count + tpb - 1) / tpb});
      rows += launches.back().nchunk;
    }
    c[lc].resize(static_cast<std::size_t>(rows) * nfn * 3);
    args.fns = aux.functions.data() + begin;
    args.nfn = nfn;
    args.ab_stride = static_cast<std::size_t>(nslot) * 6;
    int row = 0;
    for (std::size_t q = 0; q < g.classes.size(); ++q) {
      const auto& k = g.classes[q];
      args.tasks = p.tasks + k.begin;
      args.ntask = k.count;
      args.tasks_per_block = launches[q].tpb;
      args.out_ab = p.ab.data() + static_cast<std::size_t>(k.begin) * args.ab_stride + static_cast<std::size_t>(slot) * 6;
      args.out_c = c[lc].data() + static_cast<std::size_t>(row) * nfn * 3;
      dispatch(k, lc, args, launches[q].nchunk);
      row += launches[q].nchunk;
    }
    p.sum_columns(c[lc].data(), rows, begin, nfn, s);
    slot += nfnblk;
  }
  p.gather(nslot, natom, grad, s);
  VQC_HIP(hipStreamSynchronize(s));
}

std::vector<int> auxiliary_atoms(const System& aux_sys, const DeviceBasis& b) {
  std::vector<int> atoms(b.nfunctions);
  for (int sh = 0; sh < b.nshell; ++sh)
    for (int m = 0; m < aux_sys.functions(b.host_shells[sh].l); ++m)
      atoms[b.host_shells[sh].fn_off + m] = static_cast<int>(aux_sys.shells[sh].atom);
  return atoms;
}

ThreeCenterGradArgs auxiliary_args(const AuxiliaryLayout& aux, const double* boys, const double* W, std::size_t ld) {
  const auto& b = aux.basis;
  ThreeCenterGradArgs args{};
  args.aux_shells = b.shells.data();
  args.aux_exps = b.exps.data();
  args.aux_coefs = b.coefs.data();
  args.hermite = aux.hermite.data();
  args.boys = boys;
  args.w = W;
  args.ld = ld;
  return args;
}

}  // namespace

void compute_three_center_gradient(const System& orb, const DeviceBasis& basis, const System& aux_sys,
                                   const AuxiliaryLayout& aux, const double* boys, const double* W, std::size_t ld,
                                   double screening, double* grad, hipStream_t s) {
  const auto& b = aux.basis;
  const bool cart = b.representation == GENERATIVEQC_BASIS_CARTESIAN;
  GradTasks g;
  const auto classes = grad_pair_tasks(orb);
  for (int key = 0; key < 100; ++key) g.add(key / 10, key % 10, classes[key], orb);
  g.columns = auxiliary_atoms(aux_sys, b);
  ThreeCenterGradArgs args = auxiliary_args(aux, boys, W, ld);
  args.bra_shells = basis.shells.data();
  args.bra_exps = basis.exps.data();
  args.bra_coefs = basis.coefs.data();
  args.prim_cutoff = screening;
  contract_classes(g, aux, static_cast<int>(orb.atoms.size()), args, grad, s,
                   [&](const GradTasks::Class& k, int lc, ThreeCenterGradArgs& a, int nchunk) {
                     a.ta = basis.transform.data() + basis.transform_off[k.la];
                     a.tb = basis.transform.data() + basis.transform_off[k.lb];
                     a.nfa = orb.functions(k.la);
                     a.nfb = orb.functions(k.lb);
                     dispatch_pair_grad(k.la, k.lb, lc, cart && lc >= 2, a, nchunk, s);
                   });
}

void compute_metric_gradient(const System& aux_sys, const AuxiliaryLayout& aux, const double* boys, const double* W,
                             std::size_t ld, int natom, double* grad, hipStream_t s) {
  const auto& b = aux.basis;
  const bool cart = b.representation == GENERATIVEQC_BASIS_CARTESIAN;
  GradTasks g;
  for (int la = 0; la <= kMaxAuxiliaryL; ++la) {
    std::vector<int2> tasks;
    for (int i = 0; i < b.nshell; ++i)
      if (b.host_shells[i].l == la) tasks.push_back(make_int2(i, i));
    g.add(la, 0, tasks, aux_sys);
  }
  g.columns = auxiliary_atoms(aux_sys, b);
  ThreeCenterGradArgs args = auxiliary_args(aux, boys, W, ld);
  args.bra_shells = b.shells.data();
  args.bra_exps = b.exps.data();
  args.bra_coefs = b.coefs.data();
  args.tb = b.transform.data() + b.transform_off[0];
  args.nfb = 1;
  args.prim_cutoff = 0.0;
  contract_classes(g, aux, natom, args, grad, s, [&](const GradTasks::Class& k, int lc, ThreeCenterGradArgs& a, int nchunk) {
    a.ta = b.transform.data() + b.transform_off[k.la];
    a.nfa = b.representation == GENERATIVEQC_BASIS_SPHERICAL ? 2 * k.la + 1 : ncart(k.la);
    dispatch_metric_grad(k.la, lc, cart && lc >= 2, a, nchunk, s);
  });
}

void compute_one_electron_gradient(const System& sys, const DeviceBasis& basis, const double* boys,
                                   const double* dens, const double* edens, double* grad, hipStream_t s) {
  std::vector<double4> atoms;
  for (const auto& a : sys.atoms) atoms.push_back(make_double4(a.xyz[0], a.xyz[1], a.xyz[2], a.z));
  const int natom = static_cast<int>(atoms.size());
  DeviceArray<double4> datoms;
  datoms.upload(atoms, s);
  GradTasks g;
  const auto classes = grad_pair_tasks(sys);
  for (int key = 0; key < 100; ++key) g.add(key / 10, key % 10, classes[key], sys);
  for (int k = 0; k < natom; ++k) g.columns.push_back(k);
  if (g.tasks.empty()) return;
  GradPartials p(g, 1, s);
  // Lanes of a pair: up to eight split the nuclei (as many as LDS needs), then
  // its Cartesian entries, then more nuclei, while the class' pairs leave the
  // chip without eight waves a CU.
  struct Shape {
    int sub, esub, nblock;
  };
  std::vector<Shape> shapes;
  int rows = 0;
  for (const auto& k : g.classes) {
    const int entries = ((k.la + 1) * (k.la + 2) / 2) * ((k.lb + 1) * (k.lb + 2) / 2);
    int sub = one_electron_lanes(natom, one_electron_grad_bytes(k.la, k.lb)), esub = 1;
    auto more = [&] { return sub * esub < 64 && static_cast<long long>(k.count) * sub * esub < 64 * 2048; };
    while (more() && 2 * esub <= entries) esub *= 2;
    while (more() && sub < natom) sub *= 2;
    const int nblock = one_electron_grad_blocks(k.count, sub * esub);
    shapes.push_back({sub, esub, nblock});
    rows += nblock;
  }
  DeviceArray<double> c(static_cast<std::size_t>(rows) * natom * 3);
  int row = 0;
  for (std::size_t q = 0; q < g.classes.size(); ++q) {
    const auto& k = g.classes[q];
    OneElectronGradArgs args{};
    args.shells = basis.shells.data();
    args.exps = basis.exps.data();
    args.coefs = basis.coefs.data();
    args.tasks = p.tasks + k.begin;
    args.ntask = k.count;
    args.atoms = datoms.data();
    args.natom = natom;
    args.ta = basis.transform.data() + basis.transform_off[k.la];
    args.tb = basis.transform.data() + basis.transform_off[k.lb];
    args.nfa = sys.functions(k.la);
    args.nfb = sys.functions(k.lb);
    args.boys = boys;
    args.dens = dens;
    args.edens = edens;
    args.n = static_cast<int>(basis.nfunctions);
    args.out_ab = p.ab.data() + static_cast<std::size_t>(k.begin) * 6;
    args.out_c = c.data() + static_cast<std::size_t>(row) * natom * 3;
    args.sub = shapes[q].sub;
    args.esub = shapes[q].esub;
    dispatch_1e_grad(k.la, k.lb, args, s);
    row += shapes[q].nblock;
  }
  p.sum_columns(c.data(), rows, 0, natom, s);
  p.gather(1, natom, grad, s);
  VQC_HIP(hipStreamSynchronize(s));
}

}  // namespace vqc
