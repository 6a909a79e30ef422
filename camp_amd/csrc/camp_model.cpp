// Host model: packed-parameter store, CAMP sparsity pattern and ids, and
// compilation into the flat tables the HIP kernels read.
#include "camp_model.hpp"

#include "camp_aero.hpp"

#include <algorithm>
#include <cstdio>
#include <cstring>
#include <functional>
#include <limits>

namespace camp {

int Csc::find(int dep, int ind) const {
  for (int e = colptr[ind]; e < colptr[ind + 1]; ++e)
    if (rowval[e] == dep) return e;
  return -1;
}

namespace {

// Registration-then-build semantics of Jacobian.c:105-214: unique (dep,
// ind) pairs per column, each column sorted ascending at build time.
struct PatternBuilder {
  std::vector<std::vector<int>> cols;
  explicit PatternBuilder(int n) : cols(n) {}
  void add(int dep, int ind) {
    auto& c = cols[ind];
    if (std::find(c.begin(), c.end(), dep) == c.end()) c.push_back(dep);
  }
  Csc build() {
    Csc m;
    m.n = (int)cols.size();
    m.colptr.assign(m.n + 1, 0);
    for (int j = 0; j < m.n; ++j) {
      std::sort(cols[j].begin(), cols[j].end());
      m.colptr[j + 1] = m.colptr[j] + (int)cols[j].size();
      m.rowval.insert(m.rowval.end(), cols[j].begin(), cols[j].end());
    }
    return m;
  }
};

bool mass_action(int t) {
  return t == kRxnArrhenius || t == kRxnTroe || t == kRxnPhotolysis || t == kRxnCmaqH2O2 ||
         t == kRxnCmaqOhHno3;
}

// Packed layout of the mass-action types (rxn_arrhenius.c:20-36,
// rxn_troe.c:20-39, rxn_CMAQ_H2O2.c:19-35, rxn_CMAQ_OH_HNO3.c:19-41,
// rxn_photolysis.c:20-33); d points after the type slot.
struct MassActionView {
  int* d;
  double* f;
  int t;
  int npi() const { return t == kRxnPhotolysis ? 3 : 2; }
  int npf() const {
    return t == kRxnArrhenius ? 6 : t == kRxnTroe ? 10 : t == kRxnCmaqH2O2 ? 7
                                  : t == kRxnCmaqOhHno3 ? 11 : 1;
  }
  int nr() const { return d[0]; }
  int np() const { return d[1]; }
  int react(int x) const { return d[npi() + x] - 1; }
  int prod(int x) const { return d[npi() + nr() + x] - 1; }
  int& deriv_id(int x) { return d[npi() + nr() + np() + x]; }
  int& jac_id(int x) { return d[npi() + 2 * (nr() + np()) + x]; }
  double yield(int x) const { return f[npf() + x]; }
};

// aero_phase_get_used_jac_elem (aero_phase_solver.c:40-63)
int phase_used_jac_elem(const Model& m, int p, int state_id, std::vector<char>& flags) {
  PhaseView v{&m.ph_int[m.ph_int_idx[p]], &m.ph_flt[m.ph_flt_idx[p]]};
  int n = 0;
  for (int i = 0; i < v.n(); ++i)
    if (v.counted(i)) {
      flags[state_id + i] = 1;
      ++n;
    }
  return n;
}

BinnedRepView rep_view(Model& m, int r) {
  return BinnedRepView{&m.rep_int[m.rep_int_idx[r]] + 1, &m.rep_flt[m.rep_flt_idx[r]]};
}

// aero_rep_modal_binned_mass_get_used_jac_elem (:84-113): flags the species
// of every phase in the bin that holds phase instance aero_phase_idx and
// records each phase's count in the representation's int data
int rep_used_jac_elem(Model& m, int r, int aero_phase_idx, std::vector<char>& flags) {
  BinnedRepView v = rep_view(m, r);
  int n = 0;
  for (int s = 0; s < v.nsec() && aero_phase_idx >= 0; s++)
    for (int b = 0; b < v.nbin(s) && aero_phase_idx >= 0; b++)
      for (int p = 0; p < v.nph(s) && aero_phase_idx >= 0; p++) {
        if (aero_phase_idx == 0)
          for (int j = 0; j < v.nph(s); j++) {
            v.phase_njac(s, j, b) =
                phase_used_jac_elem(m, v.phase_model(s, j, b), v.phase_state(s, j, b), flags);
            n += v.phase_njac(s, j, b);
          }
        aero_phase_idx -= 1;
      }
  return n;
}

}  // namespace

void Model::size_aero(int n_ph, int n_ph_int, int n_ph_flt, int n_rp, int n_rp_int,
                      int n_rp_flt, int n_sb, int n_sb_int, int n_sb_flt) {
  n_phase = n_ph;
  ph_int.assign(std::max(n_ph_int, 0), 0);
  ph_flt.assign(std::max(n_ph_flt, 0), 0.0);
  ph_int_idx.assign(n_ph + 1, 0);
  ph_flt_idx.assign(n_ph + 1, 0);
  n_rep = n_rp;
  rep_int.assign(std::max(n_rp_int, 0) + n_rp, 0);
  rep_flt.assign(std::max(n_rp_flt, 0), 0.0);
  rep_int_idx.assign(n_rp + 1, 0);
  rep_flt_idx.assign(n_rp + 1, 0);
  rep_env_idx.assign(n_rp + 1, 0);
  n_sub = n_sb;
  sub_int.assign(std::max(n_sb_int, 0) + n_sb, 0);
  sub_flt.assign(std::max(n_sb_flt, 0), 0.0);
  sub_int_idx.assign(n_sb + 1, 0);
  sub_flt_idx.assign(n_sb + 1, 0);
  sub_env_idx.assign(n_sb + 1, 0);
}

// aero_phase_solver.c:165-194
void Model::add_phase(int n_int, int n_float, const int* ip, const double* fp) {
  int k = n_added_phase;
  if (k >= n_phase) return;
  ph_int_idx[k + 1] = ph_int_idx[k] + n_int;
  ph_flt_idx[k + 1] = ph_flt_idx[k] + n_float;
  std::memcpy(&ph_int[ph_int_idx[k]], ip, sizeof(int) * n_int);
  if (n_float) std::memcpy(&ph_flt[ph_flt_idx[k]], fp, sizeof(double) * n_float);
  ++n_added_phase;
}

// aero_rep_solver.c:443-482
void Model::add_rep(int type, int n_int, int n_float, int n_env_param, const int* ip,
                    const double* fp) {
  int k = n_added_rep;
  if (k >= n_rep) return;
  rep_int_idx[k + 1] = rep_int_idx[k] + n_int + 1;
  rep_flt_idx[k + 1] = rep_flt_idx[k] + n_float;
  rep_env_idx[k + 1] = rep_env_idx[k] + n_env_param;
  int* id = &rep_int[rep_int_idx[k]];
  id[0] = type;
  std::memcpy(id + 1, ip, sizeof(int) * n_int);
  if (n_float) std::memcpy(&rep_flt[rep_flt_idx[k]], fp, sizeof(double) * n_float);
  n_rep_env += n_env_param;
  ++n_added_rep;
}

// sub_model_solver.c:413-453
void Model::add_sub(int type, int n_int, int n_float, int n_env_param, const int* ip,
                    const double* fp) {
  int k = n_added_sub;
  if (k >= n_sub) return;
  sub_int_idx[k + 1] = sub_int_idx[k] + n_int + 1;
  sub_flt_idx[k + 1] = sub_flt_idx[k] + n_float;
  sub_env_idx[k + 1] = sub_env_idx[k] + n_env_param;
  int* id = &sub_int[sub_int_idx[k]];
  id[0] = type;
  std::memcpy(id + 1, ip, sizeof(int) * n_int);
  if (n_float) std::memcpy(&sub_flt[sub_flt_idx[k]], fp, sizeof(double) * n_float);
  n_sub_env += n_env_param;
  ++n_added_sub;
}

void Model::add_rxn(int type, int n_int, int n_float, int n_env_param,
                    const int* int_param, const double* float_param) {
  int k = n_added;
  if (k >= n_rxn) return;
  rxn_int_idx[k + 1] = rxn_int_idx[k] + n_int + 1;
  rxn_float_idx[k + 1] = rxn_float_idx[k] + n_float;
  rxn_env_idx[k + 1] = rxn_env_idx[k] + n_env_param;
  int* id = &rxn_int[rxn_int_idx[k]];
  id[0] = type;
  std::memcpy(id + 1, int_param, sizeof(int) * n_int);
  if (n_float) std::memcpy(&rxn_float[rxn_float_idx[k]], float_param, sizeof(double) * n_float);
  n_env += n_env_param;
  ++n_added;
}

bool Model::update_data(int cell, int* rxn_id, int type, int uid, double rate) {
  for (; *rxn_id < n_rxn; (*rxn_id)++) {
    int* id = rint(*rxn_id);
    int t = id[0];
    if (t != type) continue;
    int my_id;
    if (t == kRxnPhotolysis) my_id = id[3];
    else if (t == kRxnEmission || t == kRxnFirstOrderLoss) my_id = id[1];
    else continue;
    if (uid == my_id && my_id > 0) {
      double* e = &rxn_env[(size_t)cell * n_env + rxn_env_idx[*rxn_id]];
      e[1] = rate;
      e[0] = rflt(*rxn_id)[0] * e[1];
      return true;
    }
  }
  return false;
}

std::vector<int> markowitz_order(int n, const std::vector<int>& colptr,
                                 const std::vector<int>& rowval) {
  std::vector<char> A((size_t)n * n, 0);
  for (int j = 0; j < n; ++j)
    for (int k = colptr[j]; k < colptr[j + 1]; ++k) A[(size_t)rowval[k] * n + j] = 1;
  // entries of each row and column among the pivots left, the diagonal aside
  std::vector<long> row(n, -1), col(n, -1);
  for (int i = 0; i < n; ++i)
    for (int j = 0; j < n; ++j)
      if (A[(size_t)i * n + j]) {
        ++row[i];
        ++col[j];
      }
  std::vector<int> order, left(n), across;
  for (int j = 0; j < n; ++j) left[j] = j;
  while (!left.empty()) {
    int b = left[0];
    for (int j : left)
      if (row[j] * col[j] < row[b] * col[b]) b = j;
    left.erase(std::find(left.begin(), left.end(), b));
    across.clear();
    for (int c : left)
      if (A[(size_t)b * n + c]) {
        across.push_back(c);
        --col[c];
      }
    for (int i : left) {
      char* r = &A[(size_t)i * n];
      if (!r[b]) continue;
      --row[i];
      for (int c : across)
        if (!r[c]) {
          r[c] = 1;
          ++row[i];
          ++col[c];
        }
    }
    order.push_back(b);
  }
  return order;
}

// J records of contiguous element runs with near-equal record counts, one
// run per lane of G (the layout of Program::gj_rec); an element without
// records gets one record of coefficient 0, so that every element is
// written.  kc maps the rxn_env slot of a record's rate constant to its
// compact index; nullptr keeps the slot itself.
static void build_j_runs(const Program& P, int G, const std::vector<int>* kc,
                         std::vector<int>& gj, int& rows_out) {
  auto put_coef = [](int* r, double c) {
    uint64_t bits;
    std::memcpy(&bits, &c, sizeof(bits));
    r[0] = (int)(uint32_t)(bits & 0xFFFFFFFFu);
    r[1] = (int)(uint32_t)(bits >> 32);
  };
  const int nnz = P.nnz;
  auto nrec = [&](int e) { return std::max(1, P.j_ptr[e + 1] - P.j_ptr[e]); };
  std::vector<long> acc(nnz + 1, 0);
  for (int e = 0; e < nnz; ++e) acc[e + 1] = acc[e] + nrec(e);
  const long total = acc[nnz];
  std::vector<int> first(G + 1, nnz);
  first[0] = 0;
  for (int j = 1; j < G; ++j) {
    long target = total * j / G;
    int e = first[j - 1];
    while (e < nnz && acc[e] < target) ++e;
    first[j] = e;
  }
  int rows = 1;
  for (int j = 0; j < G; ++j) rows = std::max(rows, (int)(acc[first[j + 1]] - acc[first[j]]));
  rows_out = (rows + 3) / 4 * 4;
  // plus 4 rows that the kernels' look-ahead loads but never processes
  const int j_alloc = rows_out + 4;
  gj.assign((size_t)8 * G * j_alloc, 0);
  for (int j = 0; j < G; ++j) {
    int r = 0;
    for (int e = first[j]; e < first[j + 1]; ++e) {
      if (P.j_ptr[e] == P.j_ptr[e + 1]) {
        int* d = &gj[(size_t)8 * ((size_t)r * G + j)];
        d[0] = e | (1 << 30);
        d[1] = -1;
        put_coef(&d[2], 0.0);
        d[4] = 0;
        d[5] = d[6] = -1;
        d[7] = 0;
        ++r;
        continue;
      }
      for (int q = P.j_ptr[e]; q < P.j_ptr[e + 1]; ++q, ++r) {
        int* d = &gj[(size_t)8 * ((size_t)r * G + j)];
        d[0] = e | ((q + 1 == P.j_ptr[e + 1]) ? (1 << 30) : 0);
        d[1] = P.je_b[q];
        put_coef(&d[2], P.je_c[q]);
        d[4] = kc ? (*kc)[P.je_a[4 * q]] : P.je_a[4 * q];
        d[5] = P.je_a[4 * q + 1];
        d[6] = P.je_a[4 * q + 2];
        d[7] = P.je_a[4 * q + 3];
      }
    }
    for (; r < j_alloc; ++r) {
      int* d = &gj[(size_t)8 * ((size_t)r * G + j)];
      d[0] = nnz | (1 << 30);
      d[1] = -1;
      put_coef(&d[2], 0.0);
      d[4] = 0;
      d[5] = d[6] = -1;
      d[7] = 0;
    }
  }
}

// The lane-group f and J program (see Program::gf_rec): whole species
// packed longest first into G bins for f, contiguous element runs
// of near-equal record counts for J, and the compact k index map.
static void build_group_program(Program& P, int w) {
  const int G = kGroupWidths[w], nv = P.nv;
  // compact k: the rxn_env slot of each term, in term order
  std::vector<int> kc_of_slot(std::max(P.n_env, 1), -1);
  P.k_slot.clear();
  for (int t = 0; t < P.n_terms; ++t) {
    int sl = P.t_kidx[t];
    if (kc_of_slot[sl] < 0) {
      kc_of_slot[sl] = (int)P.k_slot.size();
      P.k_slot.push_back(sl);
    }
  }
  P.n_k = (int)P.k_slot.size();
  if (P.k_slot.empty()) P.k_slot.push_back(0);
  auto put_coef = [](int* r, double c) {
    uint64_t bits;
    std::memcpy(&bits, &c, sizeof(bits));
    r[0] = (int)(uint32_t)(bits & 0xFFFFFFFFu);
    r[1] = (int)(uint32_t)(bits >> 32);
  };
  // f: species into bins, longest first, each to the least-loaded bin
  P.f_count.assign(nv, 0);
  P.f_zero.clear();
  std::vector<int> sp(nv);
  for (int i = 0; i < nv; ++i) {
    sp[i] = i;
    P.f_count[i] = P.f_ptr[i + 1] - P.f_ptr[i];
    if (P.f_count[i] == 0) P.f_zero.push_back(i);
  }
  std::stable_sort(sp.begin(), sp.end(),
                   [&](int a, int b) { return P.f_count[a] > P.f_count[b]; });
  std::vector<std::vector<int>> fbin(G);
  std::vector<int> load(G, 0);
  for (int i : sp) {
    if (P.f_count[i] == 0) continue;
    int b = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    fbin[b].push_back(i);
    load[b] += P.f_count[i];
  }
  // each bin walks its species in index order
  for (auto& b : fbin) std::sort(b.begin(), b.end());
  // rows: the longest bin, rounded up to a multiple of 4, plus 4 rows that
  // the kernels' look-ahead loads but never processes
  P.g_f_rows[w] = (std::max(1, *std::max_element(load.begin(), load.end())) + 3) / 4 * 4;
  const int f_alloc = P.g_f_rows[w] + 4;
  std::vector<int>& gf = P.gf_rec[w];
  gf.assign((size_t)8 * G * f_alloc, 0);
  for (int j = 0; j < G; ++j) {
    int r = 0;
    for (int i : fbin[j])
      for (int q = P.f_ptr[i]; q < P.f_ptr[i + 1]; ++q, ++r) {
        int* d = &gf[(size_t)8 * ((size_t)r * G + j)];
        int t = P.f_term[q];
        d[0] = i | ((q + 1 == P.f_ptr[i + 1]) ? (1 << 30) : 0);
        d[1] = P.f_guard[q];
        put_coef(&d[2], P.f_coef[q]);
        d[4] = kc_of_slot[P.t_kidx[t]] | (P.t_flags[t] << 28);
        for (int m = 0; m < 3; ++m) d[5 + m] = m < P.t_nreact[t] ? P.t_react[3 * t + m] : -1;
      }
    for (; r < f_alloc; ++r) {
      int* d = &gf[(size_t)8 * ((size_t)r * G + j)];
      d[0] = nv | (1 << 30);
      d[1] = -1;
      put_coef(&d[2], 0.0);
      d[4] = 0;
      d[5] = d[6] = d[7] = -1;
    }
  }
  build_j_runs(P, G, &kc_of_slot, P.gj_rec[w], P.g_j_rows[w]);
}

// The per-cell kernels' J_rxn assembly order for multi-phase programs:
// reaction elements grouped by their record signature (the number of
// mass-action records, then the kinds of the special records in order), so
// that a row of 64 lanes runs one code path.
static void build_mp_j_order(Program& P) {
  const int rn = P.rnnz;
  std::vector<std::vector<int>> sig(rn);
  for (int e = 0; e < rn; ++e) {
    sig[e].push_back(P.j_ptr[e + 1] - P.j_ptr[e]);
    for (int q = P.js_ptr[e]; q < P.js_ptr[e + 1]; ++q) sig[e].push_back(P.js_a[4 * q]);
  }
  std::vector<int> order(rn);
  for (int e = 0; e < rn; ++e) order[e] = e;
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return sig[x] < sig[y]; });
  P.mj_rows = (rn + 63) / 64;
  P.mj_elist.assign((size_t)64 * std::max(P.mj_rows, 1), -1);
  for (int i = 0; i < rn; ++i) P.mj_elist[i] = order[i];
  // the rows' record streams
  auto put = [&](int* d, int k0, int k1, int k2, int k3, int k4, int k5, double c) {
    uint64_t bits;
    std::memcpy(&bits, &c, sizeof(bits));
    d[0] = k0; d[1] = k1; d[2] = k2; d[3] = k3; d[4] = k4; d[5] = k5;
    d[6] = (int)(uint32_t)(bits & 0xFFFFFFFFu);
    d[7] = (int)(uint32_t)(bits >> 32);
  };
  P.mj_rec.clear();
  P.mj_rhdr.clear();
  int rec_rows = 0;
  for (int r = 0; r < P.mj_rows; ++r) {
    int len = 1;
    for (int l = 0; l < 64; ++l) {
      int e = P.mj_elist[(size_t)64 * r + l];
      if (e >= 0)
        len = std::max(len, (P.j_ptr[e + 1] - P.j_ptr[e]) + (P.js_ptr[e + 1] - P.js_ptr[e]));
    }
    P.mj_rhdr.push_back(rec_rows);
    P.mj_rhdr.push_back(len);
    P.mj_rec.resize((size_t)8 * 64 * (rec_rows + len), 0);  // zeros: padding records
    for (int l = 0; l < 64; ++l) {
      int e = P.mj_elist[(size_t)64 * r + l];
      if (e < 0) continue;
      int k = 0;
      for (int q = P.j_ptr[e]; q < P.j_ptr[e + 1]; ++q, ++k)
        put(&P.mj_rec[(size_t)8 * (64 * (size_t)(rec_rows + k) + l)], -1, P.je_a[4 * q],
            P.je_a[4 * q + 1], P.je_a[4 * q + 2], P.je_a[4 * q + 3], P.je_b[q], P.je_c[q]);
      for (int q = P.js_ptr[e]; q < P.js_ptr[e + 1]; ++q, ++k)
        put(&P.mj_rec[(size_t)8 * (64 * (size_t)(rec_rows + k) + l)], P.js_a[4 * q],
            P.js_a[4 * q + 1], P.js_a[4 * q + 2], P.js_a[4 * q + 3], 0, 0, P.js_c[q]);
    }
    rec_rows += len;
  }
  P.mj_rec.resize((size_t)8 * 64 * (rec_rows + 1), 0);  // the look-ahead's padding row
}

// One chain of the triangular solves' batches: a row's entries {LU position,
// pivot} in elimination order.
struct TriRow {
  int row;
  std::vector<std::pair<int, int>> ent;
};

// Packs the rows' chains into batches of 64 lanes (the layout of
// Program::tri_e / tri_r) and returns their number.  done[k]: pivot k's
// unknown is final before the first batch; a row that ends makes its own
// final for the next batch.  Where more than 64 rows can go on, those with
// the longest way to the end of the sweep go first.
static int pack_tri_batches(const std::vector<TriRow>& rows, std::vector<char> done,
                            const std::vector<int>& xi, const std::vector<int>& diag, int zero,
                            bool empty_rows, std::vector<int>& te, std::vector<int>& tr) {
  const int n = (int)rows.size();
  std::vector<int> at(n, 0), left(n, 0);
  // entries on the longest chain of rows that waits on each row
  std::vector<long> weight(n, 0);
  std::vector<int> row_of(done.size(), -1);
  for (int i = 0; i < n; ++i) row_of[rows[i].row] = i;
  for (int i = n - 1; i >= 0; --i)  // rows come in an order that respects the chains
    for (int q = 0; q < (int)rows[i].ent.size(); ++q) {
      int j = row_of[rows[i].ent[q].second];
      if (j >= 0)
        weight[j] = std::max(weight[j], weight[i] + 8 + (long)rows[i].ent.size() - q);
    }
  std::vector<char> open(n, 1);
  int n_open = 0, batches = 0;
  for (int i = 0; i < n; ++i) {
    if (rows[i].ent.empty() && !empty_rows) {
      done[rows[i].row] = 1;
      open[i] = 0;
    } else {
      ++n_open;
    }
  }
  while (n_open) {
    std::vector<int> cand;
    for (int i = 0; i < n; ++i) {
      if (!open[i]) continue;
      const auto& e = rows[i].ent;
      int r = 0;
      while (r < 8 && at[i] + r < (int)e.size() && done[e[at[i] + r].second]) ++r;
      left[i] = r;
      if (r > 0 || e.empty()) cand.push_back(i);
    }
    if (cand.size() > 64) {
      std::stable_sort(cand.begin(), cand.end(), [&](int a, int b) {
        return weight[a] + (long)rows[a].ent.size() - at[a] >
               weight[b] + (long)rows[b].ent.size() - at[b];
      });
      cand.resize(64);
    }
    const size_t e0 = te.size(), r0 = tr.size();
    te.resize(e0 + 2 * 64 * 4, zero);
    tr.resize(r0 + 2 * 64, 0);
    for (int l = 0; l < 64; ++l) tr[r0 + 2 * l] = 0xFFFF;
    std::vector<int> ended;
    for (int l = 0; l < (int)cand.size(); ++l) {
      const int i = cand[l];
      const auto& e = rows[i].ent;
      const int x = xi[rows[i].row];
      const bool first = at[i] == 0, last = at[i] + left[i] == (int)e.size();
      for (int u = 0; u < 8; ++u) {
        int w = zero | (x << 16);
        if (u < left[i]) w = e[at[i] + u].first | (xi[e[at[i] + u].second] << 16);
        te[e0 + ((size_t)(u / 4) * 64 + l) * 4 + u % 4] = w;
      }
      at[i] += left[i];
      tr[r0 + 2 * l] = x | (first << 16) | (last << 17);
      tr[r0 + 2 * l + 1] = diag[rows[i].row];
      if (last) ended.push_back(i);
    }
    for (int i : ended) {
      open[i] = 0;
      --n_open;
      done[rows[i].row] = 1;
    }
    ++batches;
  }
  return batches;
}

// The triangular solves' program (Program::tri_e and following) of the
// filled pattern F with value positions pos (row-major, nv x nv, pivot
// order).
static void build_tri_program(Program& P, const std::vector<char>& F,
                              const std::vector<int>& pos) {
  const int nv = P.nv, zero = P.lu_nnz + 64;
  const int d = P.tri_d = std::min(64, nv), s = P.tri_s = nv - d;
  std::vector<int> xi(nv);
  for (int k = 0; k < nv; ++k) xi[k] = nv <= kTriInPlace ? P.perm[k] : k;
  auto pad = [&](std::vector<int>& e, std::vector<int>& r) {
    e.resize(e.size() + (size_t)kTriPad * 2 * 64 * 4, zero);
    for (int q = 0; q < kTriPad * 64; ++q) {
      r.push_back(0xFFFF);
      r.push_back(0);
    }
  };
  P.tri_e.clear();
  P.tri_r.clear();
  std::vector<TriRow> rows;
  for (int i = 0; i < nv; ++i) {
    TriRow t{i, {}};
    for (int k = 0; k < std::min(i, s); ++k)
      if (F[(size_t)i * nv + k]) t.ent.push_back({pos[(size_t)i * nv + k], k});
    rows.push_back(t);
  }
  P.tri_nf = pack_tri_batches(rows, std::vector<char>(nv, 0), xi, P.diag_pos, zero, false,
                              P.tri_e, P.tri_r);
  pad(P.tri_e, P.tri_r);
  rows.clear();
  std::vector<char> done(nv, 0);
  for (int k = s; k < nv; ++k) done[k] = 1;
  for (int i = s - 1; i >= 0; --i) {
    TriRow t{i, {}};
    for (int k = nv - 1; k > i; --k)
      if (F[(size_t)i * nv + k]) t.ent.push_back({pos[(size_t)i * nv + k], k});
    rows.push_back(t);
  }
  P.tri_nb = pack_tri_batches(rows, done, xi, P.diag_pos, zero, true, P.tri_e, P.tri_r);
  pad(P.tri_e, P.tri_r);
  // the tail: blocks of 8 pivots in the order the sweeps visit them
  P.tt.clear();
  auto block = [&](int kb, int dir) {
    for (int l = 0; l < 64; ++l)
      for (int u = 0; u < 8; u += 2) {
        int w = 0;
        for (int h = 0; h < 2; ++h) {
          const int k = kb + dir * (u + h), r = l;
          int p = zero;
          if (k >= 0 && k < d && r < d && (dir > 0 ? r > k : r < k) &&
              F[(size_t)(s + r) * nv + s + k])
            p = pos[(size_t)(s + r) * nv + s + k];
          w |= p << (16 * h);
        }
        P.tt.push_back(w);
      }
  };
  P.lu_at.resize(P.lu_nnz);
  for (int p = 0; p < P.lu_nnz; ++p) P.lu_at[p] = p;
  P.tt_nf = P.tt_nb = 0;
  for (int kb = 0; kb < d - 1; kb += 8, ++P.tt_nf) block(kb, 1);
  for (int q = 0; q < kTriPad; ++q) block(d, 1);
  for (int kb = d - 1; kb >= 0; kb -= 8, ++P.tt_nb) block(kb, -1);
  for (int q = 0; q < kTriPad; ++q) block(-1, -1);
  // renumber the LU values in the order the batches and blocks read them,
  // lane after lane for each entry, the diagonals first: a load of one entry
  // per lane is then a run of addresses (whole cache lines, no bank conflicts)
  std::vector<int> to(zero + 1, -1);
  int n_to = 0;
  to[zero] = zero;
  auto take = [&](int p) { return to[p] >= 0 ? to[p] : to[p] = n_to++; };
  for (int k = 0; k < nv; ++k) take(P.diag_pos[k]);
  auto head = [&](int b0, int nb) {
    for (int b = b0; b < b0 + nb; ++b)
      for (int u = 0; u < 8; ++u)
        for (int l = 0; l < 64; ++l) {
          int& w = P.tri_e[(((size_t)2 * b + u / 4) * 64 + l) * 4 + u % 4];
          w = take(w & 0xFFFF) | (int)((unsigned)w & 0xFFFF0000u);
        }
  };
  auto tail = [&](int b0, int nb) {
    for (int b = b0; b < b0 + nb; ++b)
      for (int u = 0; u < 8; ++u)
        for (int l = 0; l < 64; ++l) {
          int& w = P.tt[((size_t)b * 64 + l) * 4 + u / 2];
          const int sh = 16 * (u % 2);
          const int p = take((int)(((unsigned)w >> sh) & 0xFFFF));
          w = (int)(((unsigned)w & ~(0xFFFFu << sh)) | ((unsigned)p << sh));
        }
  };
  head(0, P.tri_nf);
  tail(0, P.tt_nf);
  tail(P.tt_nf + kTriPad, P.tt_nb);
  head(P.tri_nf + kTriPad, P.tri_nb);
  for (size_t q = 0; q < P.tri_r.size(); q += 2)
    if ((P.tri_r[q] & 0xFFFF) != 0xFFFF) P.tri_r[q + 1] = to[P.tri_r[q + 1]];
  for (int p = 0; p < P.lu_nnz; ++p) P.lu_at[p] = take(p);
  for (int k = 0; k < nv; ++k) P.diag_pos[k] = to[P.diag_pos[k]];
}

// The factorisation's tasks (Program::lg_rec) for a filled pattern: what does not
// depend on the register block's size, so that sizes can be compared.
struct LuProduct {
  uint16_t dst, l, u;
};
struct LuTasks {
  int nv = 0;
  std::vector<int> pos;               // (row, column) -> task (LU position) or -1
  std::vector<int> row, col;          // of each task
  std::vector<int> k_ptr, k;          // per task: the pivots whose products it takes, in order
  std::vector<int> out_ptr, out;      // per task: the tasks that read it
  std::vector<int> order;             // the tasks from the last pivot back
  std::vector<int> j_of;              // Jacobian element or -1

  LuTasks(const Program& P, const std::vector<LuProduct>& products,
          const std::vector<int>& positions)
      : nv(P.nv), pos(positions) {
    const int n = P.lu_nnz;
    row.resize(n);
    col.resize(n);
    for (int i = 0; i < nv; ++i)
      for (int j = 0; j < nv; ++j) {
        const int p = pos[(size_t)i * nv + j];
        if (p < 0) continue;
        row[p] = i;
        col[p] = j;
      }
    k_ptr.assign(n + 1, 0);
    out_ptr.assign(n + 1, 0);
    for (const LuProduct& x : products) {
      ++k_ptr[x.dst + 1];
      ++out_ptr[x.l + 1];
      ++out_ptr[x.u + 1];
    }
    for (int p = 0; p < n; ++p)
      if (row[p] > col[p]) ++out_ptr[diag(col[p]) + 1];
    for (int p = 0; p < n; ++p) {
      k_ptr[p + 1] += k_ptr[p];
      out_ptr[p + 1] += out_ptr[p];
    }
    k.resize(k_ptr[n]);
    out.resize(out_ptr[n]);
    std::vector<int> k_at(k_ptr.begin(), k_ptr.end() - 1), at(out_ptr.begin(), out_ptr.end() - 1);
    for (const LuProduct& x : products) {
      k[k_at[x.dst]++] = col[x.l];
      out[at[x.l]++] = x.dst;
      out[at[x.u]++] = x.dst;
    }
    for (int p = 0; p < n; ++p)
      if (row[p] > col[p]) out[at[diag(col[p])]++] = p;
    // min(row, column) orders the tasks; within one pivot the diagonal and its
    // row precede the column
    order.resize(n);
    for (int p = 0; p < n; ++p) order[p] = p;
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) {
      const int mx = pivot(x), my = pivot(y);
      return mx != my ? mx > my : (row[x] > col[x]) > (row[y] > col[y]);
    });
    j_of.assign(n, -1);
    for (int e = 0; e < P.nnz; ++e) j_of[P.lu_at[P.m_to_lu[e]]] = e;
  }
  int diag(int k) const { return pos[(size_t)k * nv + k]; }
  // the pivot at which a task's value is final (and read by others)
  int pivot(int p) const { return std::min(row[p], col[p]); }
};

// What a lane does in a group: step `step` of a task, 4 products.
struct LuSlot {
  int group, lane, task, step;
};
// Schedules the tasks for a register block of the last `tail` pivots into slots
// and returns the number of groups, or `most` where it takes as many or more.
static int schedule_lu(const LuTasks& T, int tail, int most, std::vector<LuSlot>& slots) {
  slots.clear();
  const int n = (int)T.row.size();
  if (n == 0) return 0;
  const int s = T.nv - std::min(tail, T.nv);
  std::vector<int> groups(n), waits(n);
  for (int p = 0; p < n; ++p) {
    const int* k0 = T.k.data() + T.k_ptr[p];
    const int c = (int)(std::lower_bound(k0, T.k.data() + T.k_ptr[p + 1], s) - k0);
    groups[p] = std::max(1, (c + 3) / 4);
    waits[p] = 2 * c + (T.row[p] > T.col[p] && T.col[p] < s ? 1 : 0);
  }
  // longest chains (groups from a task's start), from the last tasks back
  std::vector<int> path(n, 0);
  for (int p : T.order) {
    if (T.pivot(p) < s)
      for (int q = T.out_ptr[p]; q < T.out_ptr[p + 1]; ++q)
        path[p] = std::max(path[p], path[T.out[q]] + kLuDist - 1);
    path[p] += groups[p];
  }
  // (no schedule is shorter than the longest chain, or than the lanes allow)
  const int longest = *std::max_element(path.begin(), path.end());
  long total = 0;
  for (int c : groups) total += c;
  if (std::max<long>(longest, (total + 63) / 64) >= most) return most;
  // list scheduling: the ready task with the longest chain (of equals the first)
  // to a free lane; ready[c]: the ready tasks with a chain of c, a heap of their
  // numbers, top: the longest
  std::vector<std::vector<int>> ready(1 + longest);
  int top = 0;
  // tasks that become ready at a group: linked lists (a group's tasks enter the
  // heap together, so their order does not matter)
  std::vector<int> due, next(n, -1), ready_at(n, 0);
  auto put = [&](int g, int p) {
    if ((int)due.size() <= g) due.resize(g + 1, -1);
    next[p] = due[g];
    due[g] = p;
  };
  for (int p = 0; p < n; ++p)
    if (waits[p] == 0) put(0, p);
  int lane_task[64], lane_step[64], left = n, g = 0;
  std::fill(lane_task, lane_task + 64, -1);
  for (; left > 0; ++g) {
    if (g == most) return most;
    if (g < (int)due.size())
      for (int p = due[g]; p >= 0; p = next[p]) {
        auto& h = ready[path[p]];
        h.push_back(p);
        std::push_heap(h.begin(), h.end(), std::greater<int>());
        top = std::max(top, path[p]);
      }
    for (int l = 0; l < 64; ++l) {
      if (lane_task[l] < 0) {
        while (top > 0 && ready[top].empty()) --top;
        if (top == 0) continue;
        auto& h = ready[top];
        std::pop_heap(h.begin(), h.end(), std::greater<int>());
        lane_task[l] = h.back();
        lane_step[l] = 0;
        h.pop_back();
      }
      const int p = lane_task[l];
      slots.push_back({g, l, p, lane_step[l]});
      if (++lane_step[l] < groups[p]) continue;
      lane_task[l] = -1;
      --left;
      if (T.pivot(p) >= s) continue;
      for (int q = T.out_ptr[p]; q < T.out_ptr[p + 1]; ++q) {
        const int t = T.out[q];
        ready_at[t] = std::max(ready_at[t], g + kLuDist);
        if (--waits[t] == 0) put(ready_at[t], t);
      }
    }
  }
  return g;
}

// The factorisation's program (Program::lg_rec) of a schedule for a register
// block of the last `tail` pivots.
static void build_lu_program(Program& P, const LuTasks& T, int tail, int n_groups,
                             const std::vector<LuSlot>& slots) {
  const int nv = P.nv, zero = P.lu_nnz + 64;
  const int d = P.lu_d = std::min(tail, nv), s = nv - d;
  P.lg_n = n_groups;
  P.lg_rec.resize((size_t)(n_groups + kLuPad) * 64 * 8);
  for (size_t q = 0; q < P.lg_rec.size(); q += 4) {
    const bool rec = q / 256 % 2 == 0;
    int* w = &P.lg_rec[q];
    w[0] = rec ? zero | (zero << 16) : -1;
    w[1] = zero | (zero << 16);
    w[2] = w[3] = rec ? zero | (zero << 16) : 0;
  }
  for (const LuSlot& x : slots) {
    int* rec = &P.lg_rec[(size_t)x.group * 64 * 8 + (size_t)x.lane * 4];
    int* hdr = rec + 64 * 4;
    const int p = x.task, i = T.row[p], j = T.col[p];
    const int* k0 = T.k.data() + T.k_ptr[p];
    const int c = (int)(std::lower_bound(k0, T.k.data() + T.k_ptr[p + 1], s) - k0);
    for (int u = 0; u < 4 && x.step * 4 + u < c; ++u) {
      const int k = k0[x.step * 4 + u];
      rec[u] = T.pos[(size_t)i * nv + k] | (T.pos[(size_t)k * nv + j] << 16);
    }
    const bool scaled = i > j && j < s, first = x.step == 0,
               last = x.step + 1 == std::max(1, (c + 3) / 4);
    if (first) hdr[0] = T.j_of[p];
    hdr[1] = p | ((scaled ? T.diag(j) : zero) << 16);
    hdr[2] = (first ? 1 : 0) | (last ? 2 : 0) | (scaled && last ? 4 : 0) | (i == j ? 8 : 0) |
             (i == j && j < s ? 16 : 0);
  }
  P.lt_pos.clear();
  const int nb = (d + 7) / 8;
  for (int a = 0; a < nb; ++a)
    for (int b = 0; b < nb; ++b)
      for (int l = 0; l < 64; ++l) {
        const int i = 8 * a + l / 8, j = 8 * b + l % 8;
        P.lt_pos.push_back(i < d && j < d ? T.pos[(size_t)(s + i) * nv + s + j] : -1);
      }
}

std::string Model::initialize() {
  if (n_added != n_rxn) return "not all reactions were added before solver_initialize";
  // --- reaction Jacobian pattern: diagonal + per-type used elements -------
  PatternBuilder rb(ns);
  for (int i = 0; i < ns; ++i) rb.add(i, i);
  for (int r = 0; r < n_rxn; ++r) {
    int* id = rint(r);
    int t = id[0];
    if (mass_action(t)) {
      MassActionView v{id + 1, rflt(r), t};
      for (int i = 0; i < v.nr(); ++i) {
        for (int d = 0; d < v.nr(); ++d) rb.add(v.react(d), v.react(i));
        for (int d = 0; d < v.np(); ++d) rb.add(v.prod(d), v.react(i));
      }
    } else if (t == kRxnFirstOrderLoss) {
      rb.add(id[2] - 1, id[2] - 1);
    } else if (t == kRxnAqueousEquilibrium) {
      // rxn_aqueous_equilibrium_get_used_jac_elem (:80-126)
      AqEqView v{id + 1, rflt(r)};
      int nr = v.nr(), np = v.np();
      for (int p = 0; p < v.nph(); p++) {
        for (int ri = p * nr; ri < (p + 1) * nr; ri++) {
          for (int rd = p * nr; rd < (p + 1) * nr; rd++) rb.add(v.react(rd), v.react(ri));
          for (int pd = p * np; pd < (p + 1) * np; pd++) rb.add(v.prod(pd), v.react(ri));
        }
        for (int pi = p * np; pi < (p + 1) * np; pi++) {
          for (int rd = p * nr; rd < (p + 1) * nr; rd++) rb.add(v.react(rd), v.prod(pi));
          for (int pd = p * np; pd < (p + 1) * np; pd++) rb.add(v.prod(pd), v.prod(pi));
        }
        for (int rd = p * nr; rd < (p + 1) * nr; rd++) rb.add(v.react(rd), v.water(p));
        for (int pd = p * np; pd < (p + 1) * np; pd++) rb.add(v.prod(pd), v.water(p));
        if (v.act(p) < 0) continue;
        for (int rd = p * nr; rd < (p + 1) * nr; ++rd) rb.add(v.react(rd), v.act(p));
        for (int pd = p * np; pd < (p + 1) * np; ++pd) rb.add(v.prod(pd), v.act(p));
      }
    } else if (t == kRxnSimpolPhaseTransfer) {
      // rxn_SIMPOL_phase_transfer_get_used_jac_elem (:86-149)
      SimpolView v{id + 1, rflt(r)};
      std::vector<char> flags(ns);
      rb.add(v.gas(), v.gas());
      for (int i = 0; i < v.n(); i++) {
        rb.add(v.aero(i), v.gas());
        rb.add(v.gas(), v.aero(i));
        rb.add(v.aero(i), v.aero(i));
        if (v.act(i) > 0) {
          rb.add(v.gas(), v.act(i));
          rb.add(v.aero(i), v.act(i));
        }
        std::fill(flags.begin(), flags.end(), 0);
        if (v.rep(i) < 0 || v.rep(i) >= n_rep || rep_int[rep_int_idx[v.rep(i)]] !=
                                                      kAeroRepModalBinnedMass)
          return "SIMPOL phase transfer needs a modal/binned-mass aerosol representation";
        int n_elem = rep_used_jac_elem(*this, v.rep(i), v.phase(i), flags);
        if (n_elem > v.njac(i))
          return "SIMPOL phase transfer: more Jacobian elements than expected";
        int used = 0;
        for (int k = 0; k < ns; ++k)
          if (flags[k]) {
            rb.add(v.gas(), k);
            rb.add(v.aero(i), k);
            v.phase_jac(i, 0, used) = k;
            v.phase_jac(i, 1, used) = k;
            ++used;
          }
        for (; used < v.njac(i); ++used) v.phase_jac(i, 0, used) = v.phase_jac(i, 1, used) = -1;
      }
    } else if (t != kRxnEmission) {
      char buf[96];
      std::snprintf(buf, sizeof buf, "unsupported reaction type %d", t);
      return buf;
    }
  }
  rjac = rb.build();

  // --- derivative ids and in-place id update (rxn_*_update_ids) ----------
  deriv_ids.assign(ns, -1);
  dep_state.clear();
  for (int i = 0; i < ns; ++i)
    if (var_type[i] == kVariable) {
      deriv_ids[i] = (int)dep_state.size();
      dep_state.push_back(i);
    }
  nv = (int)dep_state.size();
  for (int r = 0; r < n_rxn; ++r) {
    int* id = rint(r);
    int t = id[0];
    if (mass_action(t)) {
      MassActionView v{id + 1, rflt(r), t};
      for (int i = 0; i < v.nr(); ++i) v.deriv_id(i) = deriv_ids[v.react(i)];
      for (int i = 0; i < v.np(); ++i) v.deriv_id(v.nr() + i) = deriv_ids[v.prod(i)];
      int e = 0;
      for (int i = 0; i < v.nr(); ++i) {
        for (int d = 0; d < v.nr(); ++d) v.jac_id(e++) = rjac.find(v.react(d), v.react(i));
        for (int d = 0; d < v.np(); ++d) v.jac_id(e++) = rjac.find(v.prod(d), v.react(i));
      }
    } else if (t == kRxnEmission) {
      id[3] = deriv_ids[id[2] - 1];
    } else if (t == kRxnFirstOrderLoss) {
      id[3] = deriv_ids[id[2] - 1];
      id[4] = rjac.find(id[2] - 1, id[2] - 1);
    } else if (t == kRxnAqueousEquilibrium) {
      // rxn_aqueous_equilibrium_update_ids (:138-230)
      AqEqView v{id + 1, rflt(r)};
      int nr = v.nr(), np = v.np();
      for (int p = 0, k = 0; p < v.nph(); p++) {
        for (int q = 0; q < nr; q++) v.deriv_id(k++) = deriv_ids[v.react(p * nr + q)];
        for (int q = 0; q < np; q++) v.deriv_id(k++) = deriv_ids[v.prod(p * np + q)];
      }
      for (int p = 0, j = 0; p < v.nph(); p++) {
        for (int ri = p * nr; ri < (p + 1) * nr; ri++) {
          for (int rd = p * nr; rd < (p + 1) * nr; rd++) v.jac_id(j++) = rjac.find(v.react(rd), v.react(ri));
          for (int pd = p * np; pd < (p + 1) * np; pd++) v.jac_id(j++) = rjac.find(v.prod(pd), v.react(ri));
        }
        for (int pi = p * np; pi < (p + 1) * np; pi++) {
          for (int rd = p * nr; rd < (p + 1) * nr; rd++) v.jac_id(j++) = rjac.find(v.react(rd), v.prod(pi));
          for (int pd = p * np; pd < (p + 1) * np; pd++) v.jac_id(j++) = rjac.find(v.prod(pd), v.prod(pi));
        }
        for (int rd = p * nr; rd < (p + 1) * nr; rd++) v.jac_id(j++) = rjac.find(v.react(rd), v.water(p));
        for (int pd = p * np; pd < (p + 1) * np; pd++) v.jac_id(j++) = rjac.find(v.prod(pd), v.water(p));
        for (int rd = p * nr; rd < (p + 1) * nr; ++rd)
          v.jac_id(j++) = v.act(p) < 0 ? -1 : rjac.find(v.react(rd), v.act(p));
        for (int pd = p * np; pd < (p + 1) * np; ++pd)
          v.jac_id(j++) = v.act(p) < 0 ? -1 : rjac.find(v.prod(pd), v.act(p));
      }
      for (int p = 0; p < v.nph(); p++) {
        v.small_conc(p) = 99999.0;
        for (int q = 0; q < nr; q++)
          if (v.small_conc(p) > abs_tol[v.react(p * nr + q)] / 100.0)
            v.small_conc(p) = abs_tol[v.react(p * nr + q)] / 100.0;
        for (int q = 0; q < np; q++)
          if (v.small_conc(p) > abs_tol[v.prod(p * np + q)] / 100.0)
            v.small_conc(p) = abs_tol[v.prod(p * np + q)] / 100.0;
      }
      for (int p = 0; p < v.nph(); p++) v.small_water(p) = abs_tol[v.water(p)] / 10.0;
    } else if (t == kRxnSimpolPhaseTransfer) {
      // rxn_SIMPOL_phase_transfer_update_ids (:160-207)
      SimpolView v{id + 1, rflt(r)};
      v.deriv_id(0) = deriv_ids[v.gas()];
      for (int i = 0; i < v.n(); i++) v.deriv_id(i + 1) = deriv_ids[v.aero(i)];
      int j = 0;
      v.jac_id(j++) = rjac.find(v.gas(), v.gas());
      for (int i = 0; i < v.n(); i++) {
        v.jac_id(j++) = rjac.find(v.aero(i), v.gas());
        v.jac_id(j++) = rjac.find(v.gas(), v.aero(i));
        v.jac_id(j++) = rjac.find(v.aero(i), v.aero(i));
        v.gas_act_jac(i) = v.act(i) > 0 ? rjac.find(v.gas(), v.act(i)) : -1;
        v.aero_act_jac(i) = v.act(i) > 0 ? rjac.find(v.aero(i), v.act(i)) : -1;
        for (int k = 0; k < v.njac(i); ++k) {
          if (v.phase_jac(i, 0, k) > 0) v.phase_jac(i, 0, k) = rjac.find(v.gas(), v.phase_jac(i, 0, k));
          if (v.phase_jac(i, 1, k) > 0)
            v.phase_jac(i, 1, k) = rjac.find(v.aero(i), v.phase_jac(i, 1, k));
        }
      }
    }
  }

  // --- parameter (sub-model) pattern: the dummy (0,0) element, then the
  // sub models' elements (camp_solver.c:1509-1552) --------------------------
  PatternBuilder pb(ns);
  pb.add(0, 0);
  for (int k = 0; k < n_sub; ++k) {
    int* id = &sub_int[sub_int_idx[k]];
    if (id[0] != kSubModelZsrAerosolWater) return "unsupported sub model type";
    ZsrView z{id + 1, &sub_flt[sub_flt_idx[k]]};
    for (int p = 0; p < z.nph(); ++p) {
      pb.add(z.phase(p), z.gas_water());
      for (int x = 0; x < z.npair(); ++x) {
        if (z.type(x) != kZsrJacobson) return "ZSR ion pairs other than JACOBSON are not supported";
        pb.add(z.phase(p), z.phase(p) + z.cation(x));
        pb.add(z.phase(p), z.phase(p) + z.anion(x));
      }
    }
  }
  pjac = pb.build();
  for (int k = 0; k < n_sub; ++k) {
    ZsrView z{&sub_int[sub_int_idx[k]] + 1, &sub_flt[sub_flt_idx[k]]};
    for (int p = 0; p < z.nph(); ++p)
      for (int x = 0; x < z.npair(); ++x) {
        z.gw_jac(p, x) = pjac.find(z.phase(p), z.gas_water());
        z.cation_jac(p, x) = pjac.find(z.phase(p), z.phase(p) + z.cation(x));
        z.anion_jac(p, x) = pjac.find(z.phase(p), z.phase(p) + z.anion(x));
      }
  }

  // --- solver Jacobian pattern and jac_map --------------------------------
  PatternBuilder sb(ns);
  for (int i_ind = 0; i_ind < ns; ++i_ind)
    for (int i_dep = 0; i_dep < ns; ++i_dep) {
      if (var_type[i_dep] != kVariable || rjac.find(i_dep, i_ind) == -1) continue;
      if (var_type[i_ind] == kVariable) {
        sb.add(i_dep, i_ind);
        continue;
      }
      for (int j_ind = 0; j_ind < ns; ++j_ind)
        if (pjac.find(i_ind, j_ind) != -1 && var_type[j_ind] == kVariable) sb.add(i_dep, j_ind);
    }
  sjac = sb.build();
  map_solver.clear();
  map_rxn.clear();
  map_param.clear();
  for (int i_ind = 0; i_ind < ns; ++i_ind)
    for (int e = rjac.colptr[i_ind]; e < rjac.colptr[i_ind + 1]; ++e) {
      int i_dep = rjac.rowval[e];
      if (var_type[i_dep] != kVariable) continue;
      if (var_type[i_ind] == kVariable) {
        map_solver.push_back(sjac.find(i_dep, i_ind));
        map_rxn.push_back(e);
        map_param.push_back(0);
        continue;
      }
      for (int j_ind = 0; j_ind < ns; ++j_ind)
        if (pjac.find(i_ind, j_ind) != -1 && var_type[j_ind] == kVariable) {
          map_solver.push_back(sjac.find(i_dep, j_ind));
          map_rxn.push_back(e);
          map_param.push_back(pjac.find(i_ind, j_ind));
        }
    }
  bool chained = false;
  for (int p : map_param) chained |= p != 0;
  if (chained && !multiphase()) return "sub-model Jacobian parameters without sub models";

  // --- compile the kernel program ----------------------------------------
  Program& P = prog;
  P = Program();
  P.ns = ns;
  P.nv = nv;
  P.n_env = n_env;
  P.nnz = sjac.nnz();
  P.dep_state = dep_state;
  P.colptr.assign(nv + 1, 0);
  for (int c = 0; c < ns; ++c)
    if (deriv_ids[c] >= 0) P.colptr[deriv_ids[c]] = sjac.colptr[c];
  P.colptr[nv] = P.nnz;
  P.rowval.resize(P.nnz);
  for (int e = 0; e < P.nnz; ++e) P.rowval[e] = deriv_ids[sjac.rowval[e]];
  // Jacobian gather space: solver elements directly when the map is the
  // identity (gas phase), reaction-pattern elements otherwise (the solver
  // Jacobian is then J_rxn * J_params over the map, camp_solver.c:1100-1106)
  const bool mp = multiphase();
  const int jn = mp ? rjac.nnz() : P.nnz;
  std::vector<int> rxn_to_solver(rjac.nnz(), -1);
  if (mp) {
    for (int e = 0; e < rjac.nnz(); ++e) rxn_to_solver[e] = e;
  } else {
    for (size_t m = 0; m < map_rxn.size(); ++m) rxn_to_solver[map_rxn[m]] = map_solver[m];
  }
  // multi-phase instances: slots of f contributions per solver variable
  std::vector<std::vector<int>> f_slots(nv);
  if (mp) {
    std::string err = compile_multiphase(f_slots);
    if (!err.empty()) return err;
  }

  // rate terms: one per reaction
  P.n_terms = n_rxn;
  P.t_kidx.resize(n_rxn);
  P.t_react.assign(3 * n_rxn, -1);
  P.t_nreact.resize(n_rxn);
  P.t_flags.resize(n_rxn);
  std::vector<std::vector<int>> f_term(nv), f_guard(nv), j_term(jn), j_skip(jn), j_guard(jn),
      j_rind(jn);
  std::vector<std::vector<double>> f_coef(nv), j_coef(jn);
  for (int r = 0; r < n_rxn; ++r) {
    int* id = rint(r);
    int t = id[0];
    P.t_kidx[r] = rxn_env_idx[r];
    if (mass_action(t)) {
      MassActionView v{id + 1, rflt(r), t};
      if (v.nr() > 3) return "reactions with more than 3 reactants are not supported";
      P.t_nreact[r] = v.nr();
      P.t_flags[r] = kTermMassAction;
      for (int i = 0; i < v.nr(); ++i) P.t_react[3 * r + i] = v.react(i);
      int dv = 0;
      for (int i = 0; i < v.nr(); ++i, ++dv)
        if (v.deriv_id(dv) >= 0) {
          f_term[v.deriv_id(dv)].push_back(r);
          f_coef[v.deriv_id(dv)].push_back(-1.0);
          f_guard[v.deriv_id(dv)].push_back(-1);
        }
      for (int i = 0; i < v.np(); ++i, ++dv)
        if (v.deriv_id(dv) >= 0) {
          f_term[v.deriv_id(dv)].push_back(r);
          f_coef[v.deriv_id(dv)].push_back(v.yield(i));
          f_guard[v.deriv_id(dv)].push_back(v.prod(i));
        }
      int el = 0;
      for (int i_ind = 0; i_ind < v.nr(); ++i_ind) {
        for (int d = 0; d < v.nr(); ++d, ++el) {
          int je = v.jac_id(el);
          if (je < 0 || rxn_to_solver[je] < 0) continue;
          int se = rxn_to_solver[je];
          j_term[se].push_back(r);
          j_skip[se].push_back(i_ind);
          j_coef[se].push_back(-1.0);
          j_guard[se].push_back(-1);
          j_rind[se].push_back(v.react(i_ind));
        }
        for (int d = 0; d < v.np(); ++d, ++el) {
          int je = v.jac_id(el);
          if (je < 0 || rxn_to_solver[je] < 0) continue;
          int se = rxn_to_solver[je];
          j_term[se].push_back(r);
          j_skip[se].push_back(i_ind);
          j_coef[se].push_back(v.yield(d));
          j_guard[se].push_back(v.prod(d));
          j_rind[se].push_back(v.react(i_ind));
        }
      }
    } else if (t == kRxnEmission) {
      P.t_nreact[r] = 0;
      P.t_flags[r] = 0;
      if (id[3] >= 0) {
        f_term[id[3]].push_back(r);
        f_coef[id[3]].push_back(1.0);
        f_guard[id[3]].push_back(-1);
      }
    } else if (t == kRxnFirstOrderLoss) {
      P.t_nreact[r] = 1;
      P.t_flags[r] = kTermRoundRate;
      P.t_react[3 * r] = id[2] - 1;
      if (id[3] >= 0) {
        f_term[id[3]].push_back(r);
        f_coef[id[3]].push_back(-1.0);
        f_guard[id[3]].push_back(-1);
      }
      if (id[4] >= 0 && rxn_to_solver[id[4]] >= 0) {
        int se = rxn_to_solver[id[4]];
        j_term[se].push_back(r);
        j_skip[se].push_back(0);
        j_coef[se].push_back(-1.0);
        j_guard[se].push_back(-1);
        j_rind[se].push_back(id[2] - 1);
      }
    }
  }
  // slot records (term -1 - slot): contributions of the multi-phase types
  for (int i = 0; i < nv; ++i)
    for (int sl : f_slots[i]) {
      f_term[i].push_back(-1 - sl);
      f_coef[i].push_back(1.0);
      f_guard[i].push_back(-1);
    }
  P.f_ptr.assign(1, 0);
  for (int i = 0; i < nv; ++i) {
    P.f_term.insert(P.f_term.end(), f_term[i].begin(), f_term[i].end());
    P.f_coef.insert(P.f_coef.end(), f_coef[i].begin(), f_coef[i].end());
    P.f_guard.insert(P.f_guard.end(), f_guard[i].begin(), f_guard[i].end());
    P.f_ptr.push_back((int)P.f_term.size());
    P.max_f_len = std::max(P.max_f_len, (int)f_term[i].size());
  }
  P.j_ptr.assign(1, 0);
  for (int e = 0; e < jn; ++e) {
    P.j_term.insert(P.j_term.end(), j_term[e].begin(), j_term[e].end());
    P.j_skip.insert(P.j_skip.end(), j_skip[e].begin(), j_skip[e].end());
    P.j_coef.insert(P.j_coef.end(), j_coef[e].begin(), j_coef[e].end());
    P.j_guard.insert(P.j_guard.end(), j_guard[e].begin(), j_guard[e].end());
    P.j_rind.insert(P.j_rind.end(), j_rind[e].begin(), j_rind[e].end());
    P.j_ptr.push_back((int)P.j_term.size());
    P.max_j_len = std::max(P.max_j_len, (int)j_term[e].size());
  }
  for (size_t q = 0; q < P.f_term.size(); ++q) {
    int t = P.f_term[q];
    if (t < 0) {  // slot record
      P.fe_c.push_back(1.0);
      P.fe_tb.push_back(-1 - t);
      P.fe_tb.push_back(0xFFFFFF | (kTermSlot << 24));
      continue;
    }
    P.fe_tb.push_back(t);
    P.fe_tb.push_back((P.f_guard[q] & 0xFFFFFF) | (P.t_flags[t] << 24));
    P.fe_c.push_back(P.f_coef[q]);
  }
  for (size_t q = 0; q < P.j_term.size(); ++q) {
    int t = P.j_term[q], skip = P.j_skip[q];
    int others[2] = {-1, -1}, n_o = 0;
    for (int j = 0; j < P.t_nreact[t]; ++j)
      if (j != skip) others[n_o++] = P.t_react[3 * t + j];
    P.je_a.push_back(P.t_kidx[t]);
    P.je_a.push_back(others[0]);
    P.je_a.push_back(others[1]);
    P.je_a.push_back(P.j_rind[q]);
    P.je_b.push_back(P.j_guard[q]);
    P.je_c.push_back(P.j_coef[q]);
  }
  if (P.fe_c.empty()) {
    P.fe_c.push_back(0.0);
    P.fe_tb.assign(2, -1);
  }
  if (P.je_c.empty()) {
    P.je_a.assign(4, -1); P.je_b.push_back(-1); P.je_c.push_back(0.0);
  }
  if (P.f_term.empty()) { P.f_term.push_back(0); P.f_coef.push_back(0); P.f_guard.push_back(-1); }
  if (P.j_term.empty()) {
    P.j_term.push_back(0); P.j_skip.push_back(0); P.j_coef.push_back(0);
    P.j_guard.push_back(-1); P.j_rind.push_back(0);
  }

  P.t_rec.assign(4 * (size_t)std::max(P.n_terms, 1), -1);
  for (int t = 0; t < P.n_terms; ++t) {
    P.t_rec[4 * t] = P.t_kidx[t] | (P.t_flags[t] << 28);
    for (int j = 0; j < 3; ++j) P.t_rec[4 * t + 1 + j] = j < P.t_nreact[t] ? P.t_react[3 * t + j] : -1;
  }
  P.fe_rec.resize(2 * P.fe_tb.size());
  for (size_t q = 0; q < P.fe_c.size(); ++q) {
    uint64_t bits;
    std::memcpy(&bits, &P.fe_c[q], sizeof(bits));
    P.fe_rec[4 * q] = P.fe_tb[2 * q];
    P.fe_rec[4 * q + 1] = P.fe_tb[2 * q + 1];
    P.fe_rec[4 * q + 2] = (int)(uint32_t)(bits & 0xFFFFFFFFu);
    P.fe_rec[4 * q + 3] = (int)(uint32_t)(bits >> 32);
  }

  if (!P.mp) {
    for (int w = 0; w < 3; ++w) build_group_program(P, w);
    build_j_runs(P, 64, nullptr, P.cj_rec, P.cj_rows);
  } else {
    build_mp_j_order(P);
  }

  // row view of the solver pattern (entries of each row in column order)
  P.r_ptr.assign(nv + 1, 0);
  for (int e = 0; e < P.nnz; ++e) P.r_ptr[P.rowval[e] + 1]++;
  for (int i = 0; i < nv; ++i) P.r_ptr[i + 1] += P.r_ptr[i];
  P.r_elem.resize(P.nnz);
  P.r_col.resize(P.nnz);
  {
    std::vector<int> fill(P.r_ptr.begin(), P.r_ptr.end() - 1);
    for (int j = 0; j < nv; ++j)
      for (int e = P.colptr[j]; e < P.colptr[j + 1]; ++e) {
        int i = P.rowval[e];
        P.r_elem[fill[i]] = e;
        P.r_col[fill[i]++] = j;
      }
  }
  {
    const int W = 64;
    std::vector<int> order(nv);
    for (int i = 0; i < nv; ++i) order[i] = i;
    std::stable_sort(order.begin(), order.end(), [&](int a, int b) {
      return P.r_ptr[a + 1] - P.r_ptr[a] > P.r_ptr[b + 1] - P.r_ptr[b];
    });
    P.fs_species = order;
    P.es_hdr.clear();
    P.es_col.clear();
    P.es_src.clear();
    const int npass = (nv + W - 1) / W;
    for (int pass = 0; pass < npass; ++pass) {
      auto len = [&](int l) {
        int slot = pass * W + l;
        return slot < nv ? P.r_ptr[order[slot] + 1] - P.r_ptr[order[slot]] : 0;
      };
      for (int j = 0; j == 0 || j < len(0); j += kEstBatch) {
        int cnt = 0;
        while (cnt < W && len(cnt) > j) ++cnt;
        const bool last = j + kEstBatch >= len(0);
        for (int l = 0; l < W; ++l) {
          P.es_hdr.push_back((int)P.es_src.size() + std::max(0, std::min(l, cnt - 1)));
          P.es_hdr.push_back(cnt | (last ? (pass + 1) << 16 : 0));
        }
        for (int l = 0; l < W; ++l)
          for (int u = 0; u < kEstBatch; u += 2) {
            int w = 0;
            for (int h = 0; h < 2; ++h) {
              int c = j + u + h < len(l) ? P.r_col[P.r_ptr[order[pass * W + l]] + j + u + h]
                                         : 0xFFFF;
              w |= c << (16 * h);
            }
            P.es_col.push_back(w);
          }
        for (int u = 0; u < kEstBatch; ++u)
          for (int l = 0; l < cnt; ++l)
            P.es_src.push_back(j + u < len(l) ? P.r_elem[P.r_ptr[order[pass * W + l]] + j + u]
                                              : -1);
      }
    }
    P.es_n = (int)P.es_src.size();
    for (int q = 0; q < kEstPad; ++q) {
      P.es_hdr.insert(P.es_hdr.end(), (size_t)2 * W, 0);
      P.es_col.insert(P.es_col.end(), (size_t)W * kEstBatch / 2, -1);
    }
  }
  {
    // balanced bins of the f gather
    const int W = 64;
    int total = P.f_ptr[nv];
    if (P.n_terms >= 65536 || P.n_slots >= 65536) return "more than 65535 f terms or slots";
    struct Piece { int species, first, count, part; };
    // Pieces: species longer than L split into near-equal pieces, placed
    // longest first into the fullest bin that holds them; a piece that no
    // bin holds fills the emptiest bin and its rest goes on.  L grows until
    // the pieces fit with at most kMaxParts partials (LDS of the gather).
    const int kMaxParts = 64;
    std::vector<std::vector<Piece>> bins;
    int L = std::max(1, (total + W - 1) / W);
    for (;; ++L) {
      std::vector<Piece> pieces;
      for (int i = 0; i < nv; ++i) {
        int cnt = P.f_ptr[i + 1] - P.f_ptr[i];
        if (cnt == 0) continue;
        int np = (cnt + L - 1) / L, at = P.f_ptr[i];
        for (int k = 0; k < np; ++k) {
          int c = cnt / np + (k < cnt % np ? 1 : 0);
          pieces.push_back({i, at, c, -1});
          at += c;
        }
      }
      std::stable_sort(pieces.begin(), pieces.end(),
                       [](const Piece& a, const Piece& b) { return a.count > b.count; });
      bins.assign(W, {});
      std::vector<int> fill(W, 0);
      bool ok = true;
      for (Piece pc : pieces) {
        while (pc.count > 0) {
          int best = -1, most = -1;
          for (int b = 0; b < W; ++b) {
            int room = L - fill[b];
            if (room >= pc.count && (best < 0 || room < L - fill[best])) best = b;
            if (room > 0 && (most < 0 || room > L - fill[most])) most = b;
          }
          if (best >= 0) {
            bins[best].push_back(pc);
            fill[best] += pc.count;
            break;
          }
          if (most < 0) {
            ok = false;
            break;
          }
          int r = L - fill[most];
          bins[most].push_back({pc.species, pc.first, r, -1});
          fill[most] += r;
          pc.first += r;
          pc.count -= r;
        }
        if (!ok) break;
      }
      if (!ok) continue;
      // partials: the pieces of a species in record order get consecutive ids
      std::vector<std::vector<Piece*>> of(nv);
      for (auto& b : bins)
        for (Piece& pc : b) of[pc.species].push_back(&pc);
      int np_total = 0;
      for (int i = 0; i < nv; ++i) {
        if (of[i].size() < 2) continue;
        std::sort(of[i].begin(), of[i].end(),
                  [](const Piece* a, const Piece* b) { return a->first < b->first; });
        for (Piece* pc : of[i]) pc->part = np_total++;
      }
      if (np_total <= kMaxParts || L >= P.max_f_len) {
        P.fb_nparts = np_total;
        break;
      }
    }
    if (2 * nv + 3 * P.fb_nparts + 3 >= 65536) return "more than 65535 f gather targets";
    P.fb_rows = L;
    // rows padded to a multiple of 4 plus 4 more, so that the gather's
    // batches of 4 and its loads 4 rows ahead need no bounds checks
    const int L_alloc = (L + 3) / 4 * 4 + 4;
    P.fb_rec.assign((size_t)4 * W * L_alloc, 0);
    for (int l = 0; l < W; ++l) {
      int j = 0;
      for (const Piece& pc : bins[l])
        for (int r = 0; r < pc.count; ++r, ++j) {
          const int* src = &P.fe_rec[4 * (size_t)(pc.first + r)];
          int* dst = &P.fb_rec[4 * ((size_t)j * W + l)];
          // the piece's sum goes to s_fb[target]: a whole species' value at
          // [species] (its magnitude sum at [nv + species]), a partial's
          // (hi, lo, magnitudes) at [2 nv + 3 part ..] (flag 32)
          int target = pc.part >= 0 ? 2 * nv + 3 * pc.part : pc.species;
          dst[0] = (src[0] & 0xFFFF) | (target << 16);
          dst[1] = src[1] | (r + 1 == pc.count ? (16 << 24) : 0) | (pc.part >= 0 ? (32 << 24) : 0);
          dst[2] = src[2];
          dst[3] = src[3];
        }
      // padding: no contribution, running sums stored to a spare partial
      for (; j < L_alloc; ++j) {
        int* dst = &P.fb_rec[4 * ((size_t)j * W + l)];
        dst[0] = (2 * nv + 3 * P.fb_nparts) << 16;
        dst[1] = ((8 | 32) << 24) | 0xFFFFFF;
        dst[2] = dst[3] = 0;
      }
    }
    P.fb_fin.assign(2 * (size_t)std::max(nv, 1), 0);
    for (int i = 0; i < nv; ++i) {
      int cnt = P.f_ptr[i + 1] - P.f_ptr[i];
      P.fb_fin[2 * i] = 0;
      P.fb_fin[2 * i + 1] = cnt == 0 ? -1 : 0;
    }
    for (const auto& b : bins)
      for (const Piece& pc : b)
        if (pc.part >= 0) {
          int* f = &P.fb_fin[2 * pc.species];
          if (f[1] == 0) f[0] = pc.part;
          f[0] = std::min(f[0], pc.part);
          f[1] += 1;
        }
    // the packing must cover every species' records exactly once, in pieces
    // of consecutive records, with consecutive partial ids in record order
    std::vector<std::vector<const Piece*>> by(nv);
    for (const auto& b : bins) {
      int fill = 0;
      for (const Piece& pc : b) {
        by[pc.species].push_back(&pc);
        fill += pc.count;
      }
      if (fill > L) return "f gather packing: a bin exceeds its rows";
    }
    for (int i = 0; i < nv; ++i) {
      std::sort(by[i].begin(), by[i].end(),
                [](const Piece* a, const Piece* b) { return a->first < b->first; });
      int at = P.f_ptr[i];
      for (size_t k = 0; k < by[i].size(); ++k) {
        const Piece* pc = by[i][k];
        bool ok = pc->first == at && pc->count > 0 &&
                  (by[i].size() == 1 ? pc->part < 0 : pc->part == P.fb_fin[2 * i] + (int)k);
        if (!ok) return "f gather packing: species records not covered exactly once";
        at += pc->count;
      }
      if (at != P.f_ptr[i + 1]) return "f gather packing: species records not covered";
    }
  }

  // --- LU: Markowitz ordering, symbolic fill, per-pivot programs ----------
  P.perm = markowitz_order(nv, P.colptr, P.rowval);
  P.iperm.assign(nv, 0);
  for (int k = 0; k < nv; ++k) P.iperm[P.perm[k]] = k;
  std::vector<char> F((size_t)nv * nv, 0);
  for (int j = 0; j < nv; ++j)
    for (int e = P.colptr[j]; e < P.colptr[j + 1]; ++e)
      F[(size_t)P.iperm[P.rowval[e]] * nv + P.iperm[j]] = 1;
  for (int k = 0; k < nv; ++k)
    for (int i = k + 1; i < nv; ++i)
      if (F[(size_t)i * nv + k])
        for (int j = k + 1; j < nv; ++j)
          if (F[(size_t)k * nv + j]) F[(size_t)i * nv + j] = 1;
  std::vector<int> pos((size_t)nv * nv, -1);
  int p = 0;
  for (int i = 0; i < nv; ++i)
    for (int j = 0; j < nv; ++j)
      if (F[(size_t)i * nv + j]) pos[(size_t)i * nv + j] = p++;
  P.lu_nnz = p;
  if (P.lu_nnz > 65535) return "LU fill exceeds 65535 entries per cell";
  P.m_to_lu.resize(P.nnz);
  for (int j = 0; j < nv; ++j)
    for (int e = P.colptr[j]; e < P.colptr[j + 1]; ++e) {
      P.m_to_lu[e] = pos[(size_t)P.iperm[P.rowval[e]] * nv + P.iperm[j]];
    }
  P.diag_pos.resize(nv);
  for (int k = 0; k < nv; ++k) P.diag_pos[k] = pos[(size_t)k * nv + k];
  if (P.lu_nnz + 64 > 65535) return "LU fill exceeds 65471 entries per cell";
  build_tri_program(P, F, pos);
  // (from here on the positions are those the solve reads: Program::lu_at)
  for (int& q : pos)
    if (q >= 0) q = P.lu_at[q];
  // the elimination's products LU[dst] -= LU[l] * LU[u], in pivot order
  std::vector<LuProduct> products;
  products.reserve((size_t)4 * P.lu_nnz);
  std::vector<int> u;
  for (int k = 0; k < nv; ++k) {
    u.clear();
    for (int j = k + 1; j < nv; ++j)
      if (pos[(size_t)k * nv + j] >= 0) u.push_back(j);
    for (int i = k + 1; i < nv; ++i) {
      const int* pi = &pos[(size_t)i * nv];
      if (pi[k] < 0) continue;
      ++P.n_lower;
      for (int j : u)
        products.push_back({(uint16_t)pi[j], (uint16_t)pi[k], (uint16_t)pos[(size_t)k * nv + j]});
    }
  }
  P.n_updates = (long)products.size();
  // The block's size by what a factorisation then costs: the tasks' groups
  // (about 600 cycles each) against the block's pivots, whose cost grows with
  // its size (350 to 850 cycles, measured).  CB05cl_ae5, two thirds of whose
  // last 40 x 40 are zeros, takes 16 (42k -> 21k cycles), the CB05-scale
  // mechanism 32 (55k -> 49k).  Large factors end in a dense block: all 40.
  const LuTasks tasks(P, products, pos);
  std::vector<LuSlot> slots, trial;
  int best = kLuTail, n_groups = 0;
  double best_cost = 0.0;
  // (from the largest down, as long as the cost falls: the schedule's chain grows
  // with every pivot outside the block)
  for (int d = std::max(8, std::min(kLuTail, (nv + 7) / 8 * 8)); d >= 8; d -= 8) {
    const double block = std::min(d, nv) * (230.0 + 125.0 * (d / 8));
    const int most = best_cost > 0.0 ? (int)std::max(0.0, (best_cost - block) / 600.0) + 1
                                     : std::numeric_limits<int>::max();
    const int n = schedule_lu(tasks, d, most, trial);
    const double cost = 600.0 * n + block;
    if (best_cost > 0.0 && cost >= best_cost) break;
    best = d;
    best_cost = cost;
    n_groups = n;
    std::swap(slots, trial);
    if (P.lu_nnz > 4096) break;
  }
  build_lu_program(P, tasks, best, n_groups, slots);
  initialized = true;
  // the f gather's final pass in slot order: {species, first partial, count}
  // (at least one pass: f loads the first one ahead)
  P.es_fin.clear();
  for (int slot = 0; slot < std::max((nv + 63) / 64, 1) * 64; ++slot) {
    const int i = slot < nv ? P.fs_species[slot] : -1;
    P.es_fin.insert(P.es_fin.end(), {i, i < 0 ? 0 : P.fb_fin[2 * i], i < 0 ? -1 : P.fb_fin[2 * i + 1], 0});
  }
  return std::string();
}

// ---------------------------------------------------------------------------
// Multi-phase kernel tables: aerosol phase instances, ZSR items, SIMPOL and
// aqueous-equilibrium instances with their f-contribution slots, the special
// Jacobian records of those instances per reaction-pattern element, and the
// J_rxn * J_params map per solver element (camp_solver.c:1100-1106).
// ---------------------------------------------------------------------------
std::string Model::compile_multiphase(std::vector<std::vector<int>>& f_slots) {
  Program& P = prog;
  P.mp = true;
  P.rnnz = rjac.nnz();
  P.pnnz = pjac.nnz();
  P.pm_ptr.assign(1, 0);
  for (int p = 0; p < n_phase; ++p) {
    PhaseView v{&ph_int[ph_int_idx[p]], &ph_flt[ph_flt_idx[p]]};
    for (int i = 0; i < v.n(); ++i) {
      P.pm_counted.push_back(v.counted(i) ? 1 : 0);
      P.pm_mw.push_back(v.mw(i));
      P.pm_dens.push_back(v.density(i));
    }
    P.pm_ptr.push_back((int)P.pm_counted.size());
  }
  // phase instances in the representation's phase-index order
  std::vector<int> rep_pi_base(n_rep, 0);
  std::vector<double> pi_radius;
  for (int r = 0; r < n_rep; ++r) {
    if (rep_int[rep_int_idx[r]] != kAeroRepModalBinnedMass)
      return "unsupported aerosol representation type";
    rep_pi_base[r] = (int)P.pi_start.size();
    BinnedRepView v = rep_view(*this, r);
    for (int s = 0; s < v.nsec(); ++s) {
      if (v.type(s) != kBinned) return "MODAL sections are not supported by the multi-phase kernels";
      if (v.nph(s) != 1) return "bins holding more than one phase are not supported by the multi-phase kernels";
      for (int b = 0; b < v.nbin(s); ++b) {
        P.pi_start.push_back(v.phase_state(s, 0, b));
        P.pi_model.push_back(v.phase_model(s, 0, b));
        P.pi_dp.push_back(v.bin_dp(s, b));
        pi_radius.push_back(v.radius(s, b));
      }
    }
  }
  P.pit_ptr.assign(1, 0);
  for (size_t i = 0; i < P.pi_start.size(); ++i) {
    const int pm = P.pi_model[i];
    for (int q = P.pm_ptr[pm]; q < P.pm_ptr[pm + 1]; ++q) {
      if (!P.pm_counted[q]) continue;
      P.pit_state.push_back(P.pi_start[i] + q - P.pm_ptr[pm]);
      P.pit_pi.push_back((int)i);
      P.pit_mw.push_back(P.pm_mw[q]);
      P.pit_dens.push_back(P.pm_dens[q]);
    }
    P.pit_ptr.push_back((int)P.pit_state.size());
  }
  // ZSR items
  P.zi_pair_ptr.assign(1, 0);
  for (int k = 0; k < n_sub; ++k) {
    ZsrView z{&sub_int[sub_int_idx[k]] + 1, &sub_flt[sub_flt_idx[k]]};
    for (int p = 0; p < z.nph(); ++p) {
      P.zi_water.push_back(z.phase(p));
      P.zi_gw.push_back(z.gas_water());
      P.zi_sub.push_back(k);
      for (int x = 0; x < z.npair(); ++x) {
        if (z.ny(x) > 8) return "ZSR molality polynomials of more than 8 terms";
        P.zp_zi.push_back((int)P.zi_water.size() - 1);
        P.zp_cat.push_back(z.phase(p) + z.cation(x));
        P.zp_an.push_back(z.phase(p) + z.anion(x));
        P.zp_ncat.push_back(z.n_cation(x));
        P.zp_nan.push_back(z.n_anion(x));
        P.zp_ny.push_back(z.ny(x));
        P.zp_jgw.push_back(z.gw_jac(p, x));
        P.zp_jcat.push_back(z.cation_jac(p, x));
        P.zp_jan.push_back(z.anion_jac(p, x));
        P.zp_catmw.push_back(z.cation_mw(x));
        P.zp_anmw.push_back(z.anion_mw(x));
        P.zp_lowrh.push_back(z.low_rh(x));
        for (int q = 0; q < 8; ++q) P.zp_y.push_back(q < z.ny(x) ? z.y(x, q) : 0.0);
      }
      P.zi_pair_ptr.push_back((int)P.zp_cat.size());
    }
  }
  P.n_sub_env = n_sub;

  std::vector<std::vector<int>> ja(rjac.nnz());
  std::vector<std::vector<double>> jc(rjac.nnz());
  auto addj = [&](int e, int kind, int inst, int p1, int p2, double c) {
    if (e < 0) return;
    ja[e].insert(ja[e].end(), {kind, inst, p1, p2});
    jc[e].push_back(c);
  };
  int slot = 0;
  for (int r = 0; r < n_rxn; ++r) {
    int* id = rint(r);
    int t = id[0];
    if (t == kRxnSimpolPhaseTransfer) {
      SimpolView v{id + 1, rflt(r)};
      for (int i = 0; i < v.n(); ++i) {
        if (v.act(i) > -1) return "SIMPOL activity coefficients are not supported by the multi-phase kernels";
        if (v.rep(i) < 0 || v.rep(i) >= n_rep) return "SIMPOL: bad aerosol representation id";
        int inst = (int)P.sp_gas.size();
        int pi = rep_pi_base[v.rep(i)] + v.phase(i);
        P.sp_gas.push_back(v.gas());
        P.sp_aero.push_back(v.aero(i));
        P.sp_dgas.push_back(v.deriv_id(0));
        P.sp_daero.push_back(v.deriv_id(1 + i));
        P.sp_pi.push_back(pi);
        P.sp_env.push_back(rxn_env_idx[r]);
        P.sp_flt.push_back(rxn_float_idx[r]);
        P.sp_radius.push_back(pi_radius[pi]);
        P.sp_slot.push_back(slot);
        // rxn_SIMPOL_phase_transfer.c:355-399 (total particle mass): gas
        // +N evap, -N cond; aerosol -N evap/kp, +N cond/kp
        if (v.deriv_id(0) >= 0) {
          f_slots[v.deriv_id(0)].push_back(slot);
          f_slots[v.deriv_id(0)].push_back(slot + 1);
        }
        if (v.deriv_id(1 + i) >= 0) {
          f_slots[v.deriv_id(1 + i)].push_back(slot + 2);
          f_slots[v.deriv_id(1 + i)].push_back(slot + 3);
        }
        slot += 4;
        addj(v.jac_id(0), kJsSimpolGG, inst, 0, 0, 0.0);
        addj(v.jac_id(1 + 3 * i), kJsSimpolAG, inst, 0, 0, 0.0);
        addj(v.jac_id(1 + 3 * i + 1), kJsSimpolGA, inst, 0, 0, 0.0);
        addj(v.jac_id(1 + 3 * i + 2), kJsSimpolAA, inst, 0, 0, 0.0);
        // phase element k = k-th counted species of the bin's phase
        int pm = P.pi_model[pi], k = 0;
        for (int q = P.pm_ptr[pm]; q < P.pm_ptr[pm + 1]; ++q) {
          if (!P.pm_counted[q]) continue;
          if (k < v.njac(i)) {
            if (v.phase_jac(i, 0, k) > 0) addj(v.phase_jac(i, 0, k), kJsSimpolGP, inst, q, P.pit_ptr[pi] + k, 0.0);
            if (v.phase_jac(i, 1, k) > 0) addj(v.phase_jac(i, 1, k), kJsSimpolAP, inst, q, P.pit_ptr[pi] + k, 0.0);
          }
          ++k;
        }
      }
    } else if (t == kRxnAqueousEquilibrium) {
      AqEqView v{id + 1, rflt(r)};
      int nr = v.nr(), np = v.np();
      if (nr > 3 || np > 3) return "aqueous equilibria with more than 3 reactants or products";
      for (int p = 0; p < v.nph(); ++p) {
        if (v.act(p) >= 0) return "aqueous-equilibrium activity coefficients are not supported by the multi-phase kernels";
        int inst = (int)P.aq_nr.size();
        P.aq_nr.push_back(nr);
        P.aq_np.push_back(np);
        for (int q = 0; q < 3; ++q) P.aq_sp.push_back(q < nr ? v.react(p * nr + q) : -1);
        for (int q = 0; q < 3; ++q) P.aq_sp.push_back(q < np ? v.prod(p * np + q) : -1);
        P.aq_water.push_back(v.water(p));
        P.aq_env.push_back(rxn_env_idx[r]);
        P.aq_flt.push_back(rxn_float_idx[r]);
        P.aq_small_water.push_back(v.small_water(p));
        P.aq_slot.push_back(slot);
        int d0 = p * (nr + np);
        for (int q = 0; q < 6; ++q) P.aq_deriv.push_back(q < nr + np ? v.deriv_id(d0 + q) : -1);
        // rxn_aqueous_equilibrium.c:362-386: -rf/m, +rr/m per reactant;
        // +rf/m, -rr/m per product
        for (int q = 0; q < nr + np; ++q)
          if (v.deriv_id(d0 + q) >= 0) {
            f_slots[v.deriv_id(d0 + q)].push_back(slot + 2 * q);
            f_slots[v.deriv_id(d0 + q)].push_back(slot + 2 * q + 1);
          }
        slot += 2 * (nr + np);
        // Jacobian ids in the reference's order (rxn_aqueous_equilibrium.c:418-545)
        int j = p * (nr + np) * (nr + np + 2);
        for (int ri = 0; ri < nr; ++ri) {
          for (int rd = 0; rd < nr; ++rd) addj(v.jac_id(j++), kJsAqRR, inst, ri, rd, v.mftm(rd));
          for (int pd = 0; pd < np; ++pd)
            addj(v.jac_id(j++), kJsAqRP, inst, ri, nr + pd, v.mftm(nr + pd));
        }
        for (int pj = 0; pj < np; ++pj) {
          for (int rd = 0; rd < nr; ++rd) addj(v.jac_id(j++), kJsAqPR, inst, 3 + pj, rd, v.mftm(rd));
          for (int pd = 0; pd < np; ++pd)
            addj(v.jac_id(j++), kJsAqPP, inst, 3 + pj, nr + pd, v.mftm(nr + pd));
        }
        for (int rd = 0; rd < nr; ++rd) addj(v.jac_id(j++), kJsAqRW, inst, 0, rd, v.mftm(rd));
        for (int pd = 0; pd < np; ++pd)
          addj(v.jac_id(j++), kJsAqPW, inst, 0, nr + pd, v.mftm(nr + pd));
      }
    }
  }
  P.n_slots = slot;
  P.n_pi = (int)P.pi_start.size();
  P.n_zi = (int)P.zi_water.size();
  P.n_sp = (int)P.sp_gas.size();
  P.n_aq = (int)P.aq_nr.size();
  P.js_ptr.assign(1, 0);
  for (int e = 0; e < rjac.nnz(); ++e) {
    P.js_a.insert(P.js_a.end(), ja[e].begin(), ja[e].end());
    P.js_c.insert(P.js_c.end(), jc[e].begin(), jc[e].end());
    P.js_ptr.push_back((int)P.js_c.size());
  }
  if (P.js_c.empty()) {
    P.js_a.assign(4, 0);
    P.js_c.push_back(0.0);
  }
  // solver element <- (reaction element, parameter element) in map order
  std::vector<std::vector<int>> mr(P.nnz), mpar(P.nnz);
  for (size_t m = 0; m < map_solver.size(); ++m) {
    mr[map_solver[m]].push_back(map_rxn[m]);
    mpar[map_solver[m]].push_back(map_param[m]);
  }
  P.jm_ptr.assign(1, 0);
  for (int e = 0; e < P.nnz; ++e) {
    P.jm_rxn.insert(P.jm_rxn.end(), mr[e].begin(), mr[e].end());
    P.jm_param.insert(P.jm_param.end(), mpar[e].begin(), mpar[e].end());
    P.jm_ptr.push_back((int)P.jm_rxn.size());
  }
  for (auto* v : {&P.pi_start, &P.pi_model, &P.zi_water, &P.zi_gw, &P.zi_sub, &P.zp_cat, &P.zp_an,
                  &P.zp_ncat, &P.zp_nan, &P.zp_ny, &P.zp_jgw, &P.zp_jcat, &P.zp_jan, &P.sp_gas,
                  &P.sp_aero, &P.sp_dgas, &P.sp_daero, &P.sp_pi, &P.sp_env, &P.sp_flt, &P.sp_slot,
                  &P.aq_nr, &P.aq_np, &P.aq_sp, &P.aq_water, &P.aq_env, &P.aq_flt, &P.aq_deriv,
                  &P.aq_slot, &P.jm_rxn, &P.jm_param, &P.pm_counted})
    if (v->empty()) v->push_back(0);
  for (auto* v : {&P.pi_dp, &P.pm_mw, &P.pm_dens, &P.zp_catmw, &P.zp_anmw, &P.zp_lowrh, &P.zp_y,
                  &P.sp_radius, &P.aq_small_water})
    if (v->empty()) v->push_back(0.0);
  return std::string();
}

}  // namespace camp
