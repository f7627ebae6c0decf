// Chains of small products as one kernel (included by smallk.hip, inside its anonymous namespace).
//
// The steps of an unrolled recurrence, `h_t = f (W x_t + V h_(t-1) + b)` and its transposition, are products that
// read one another's results, so each level of the held-back queue has to wait for the one before.  But column p of a
// step's result depends on column p of the earlier results only: a block that owns a few columns can walk all levels
// without hearing from any other block.  One launch replaces a launch per level (4.5 us each in a recorded graph,
// however small), and the factors that every level multiplies by, the weights, are read once.
//
// The kernel (512 threads = 8 wavefronts, 4 * NC columns of P per block):
//   * Rows of the results in groups of 16.  A level's products are shared out between the wavefronts by the weights
//     they use (roles): the two layers of a recurrence get four wavefronts each, which own every fourth row group, so
//     that a SIMD has one wavefront of either and the program of one runs beside the multiplications of the other.
//   * The weights stay where the lanes need them, in registers as far as those go and in LDS beyond: fragment f of a
//     lane is W[16 rg + lane % 16][k], k = 4 VK (f / VK) + VK (lane / 16) + f % VK (VK = 4 in fp32, 2 in fp64).
//   * The columns sit in LDS as [group of 4 columns][k][4], so a wavefront reads 64 neighbouring elements.  The results
//     of a level go to LDS for the next one (two halves, one written while the other is read; one barrier a level) and
//     from there to memory while the next level runs; operands from outside the chain are fetched a level ahead.
//   * fp32: v_mfma_f32_4x4x1 with the columns as the A operand, one of four blocks of four lanes broadcast to its group
//     (cbsz 2): 16 rows x 4 columns x 4 k an instruction, every group of 16 lanes a quarter of k; the quarters meet by
//     two lane swaps.  fp64, and fp32 products whose sums are fp64 (smallk.hip): v_mfma_f64_4x4x4 with the weights as the A
//     operand.  Tiles of four columns cost the same
//     per product as the large ones (probe, 250 CUs, all operands resident: fp32 103 TFLOP/s with NC up to 3, 123 from
//     4 on; fp64 59-64) and let 5000 columns be 250 blocks of 20.
//   * fp64 with up to two columns for every CU: lone columns on vector instructions, whose rate is that of the matrix ones and which
//     need no four columns to be filled (lone_products): 150 columns are 150 blocks instead of 38, and a level multiplies for 0.4
//     instead of 1.4 us.  A lane's program serves one row, not one of four columns, so a wavefront's two row groups share a pass of it.
//
// What bounds it: in fp32 with 20 columns a block the matrix cores, 4.3 of the 5.6 us a level (two layers 128 wide; a level
// by itself 10.6), the rest LDS latency after the barrier and the program; with 4 columns the chain LDS read, multiply,
// program, LDS write, barrier: 1.3-1.6 us in fp32, in fp64 2.5 without and 3.3 with a tanh (a level by itself 4.7); in fp64 with one column
// 2.0, of which the barrier with the loads and stores around it about 1.  29 levels of two layers 128 wide, 150 columns of fp64: 99.7 us in groups of four
// (44 of them the multiplications, 22 the tanh), 58.7 alone.
// Gradients of two layers 128 wide over 28 steps, before / so: fp32 batch 5000 844 / 629 us.
// Taken back: nontemporal stores of the results (no gain beside the movers' priority), all wavefronts on all layers (fp32
// the same, fp64 forward 111 us for 100; still the form where one layer's weights do not fit its wavefronts).

constexpr int kChainMaxPtrs = 448;      // pointers in the kernel's arguments (3.5 KB)
constexpr int kChainMaxSections = 12;
// Levels from which a chain is looked for at all.  (What it costs, reading the weights once, is 5 to 10 us, and a level saves about
// 3 of the 4.5 us of its launch, so that fewer would do where pays() says so: not measured, recurrences of up to seven steps
// keep a launch a level.)
constexpr int kChainMinLevels = 8;
constexpr int kChainMaxWidth = 4;       // products of one level
constexpr int kChainLds = 160 * 1024;

constexpr int kChainMaxUnits = 8;
constexpr int kChainMaxLone = 2;        // lone columns of a block

struct ChainMat {                // a weights factor, W[q][k]
  const void* ptr;
  int64_t Q, K, sq, sk;
  int uses = 0;                  // levels that multiply by it
  int nf = 0;                    // fragments of a lane and row group (K padded to whole tiles, a quarter)
  int role = 0, w0 = 0, nw = 8;  // the wavefronts that multiply by it
  int units = 0;                 // row groups of a wavefront
  int reg[kChainMaxUnits] = {0}; // fragments kept in registers, per row group
  int lds[kChainMaxUnits] = {0}; // LDS element of the others
  int groups() const { return (int)((Q + 15) / 16); }
  int waves(int u) const { return std::min(nw, groups() - nw * u); }
  bool kept() const { return uses > 1; }      // (one level's weights are read when it runs)
};
struct ChainX { int mat; int kind; int off, rows; int64_t K, sxp, sxk; int ptr; };                 // columns factor of a term: 0 an array, 1 a result of the level before, 2 one element
struct ChainIn { int kind; int dtype; int off, rows; int64_t sp, sq; int ptr; };                   // 0: the sum, 1: one value per row, 2: a result of the level before, 3: an array, by lanes, 4: an array that comes through LDS
struct ChainOut { int slot; bool staged; int dtype; int off; int ptr; };                           // staged: goes through LDS
struct ChainItem {
  const Known* kn;
  int64_t Q;
  int rows, role = 0;
  bool wide() const { return kn->spec.wide; }      // fp32 elements, sums in fp64
  std::vector<ChainX> x;
  std::vector<ChainIn> in;
  std::vector<ChainOut> out;
};
struct ChainSection {            // levels that do the same with other arrays
  std::vector<ChainItem> items;
  int n_ptr = 0;                 // pointers per level
  int n_levels = 0;
  int out_elems = 0, ext_elems = 0;
};
struct ChainPlan {
  bool f64 = false;
  bool lone = false;             // columns one by one on vector instructions (NC of them a block) instead of groups of four
  int64_t P = 0;
  int NC = 1, roles = 1;
  std::vector<ChainMat> mats;
  std::vector<ChainSection> sections;
  int n_const = 0;               // pointers before the first level's: weights, then what stands still over a section
  int out_elems = 0, ext_elems = 0, lds_elems = 0;
  std::vector<const void*> ptrs;
  double flops = 0, bytes = 0;
  int n_items = 0, n_levels = 0;
};

// Everything chain_source reads.
Key chain_key(const ChainPlan& c) {
  Key k;
  k.put(c.f64).put(c.lone).put(c.P).put(c.NC).put(c.roles).put(c.out_elems).put(c.ext_elems).put(c.lds_elems).put(c.n_const).put(c.mats.size());
  for (auto& m : c.mats) {
    k.put(m.Q).put(m.K).put(m.sq).put(m.sk).put(m.kept()).put(m.role).put(m.w0).put(m.nw).put(m.units);
    for (int u = 0; u < m.units; ++u) k.put(m.reg[u]).put(m.lds[u]);
  }
  k.put(c.sections.size());
  for (auto& s : c.sections) {
    k.put(s.n_ptr).put(s.items.size());
    for (auto& it : s.items) {
      k.put(it.kn->id).put(it.Q).put(it.rows).put(it.role).put(it.x.size()).put(it.in.size()).put(it.out.size());      // (the id stands for the program)
      for (auto& x : it.x) k.put(x.mat).put(x.kind).put(x.off).put(x.rows).put(x.K).put(x.sxp).put(x.sxk).put(x.ptr);
      for (auto& i : it.in) k.put(i.kind).put(i.dtype).put(i.off).put(i.rows).put(i.sp).put(i.sq).put(i.ptr);
      for (auto& o : it.out) k.put(o.slot).put(o.staged).put(o.dtype).put(o.off).put(o.ptr);
    }
  }
  return k;
}

int chain_vk(bool f64) { return f64 ? 2 : 4; }
int chain_kp(bool f64, int64_t K) { const int kt = 4 * chain_vk(f64); return (int)((K + kt - 1) / kt * kt); }
// LDS elements of `rows` x 4 NC columns; a group of four columns is followed by four elements that keep the groups in different banks
int chain_pitch(const ChainPlan& c, int rows) { return c.lone ? rows : rows * 4 + 4; }
int chain_region(const ChainPlan& c, int rows) { return c.NC * chain_pitch(c, rows); }

int chain_columns(const ChainPlan& c) { return c.lone ? c.NC : 4 * c.NC; }      // of a block
int64_t chain_blocks(const ChainPlan& c) { return (c.P + chain_columns(c) - 1) / chain_columns(c); }
// The wavefronts of a role end where the next one's begin.
int role_end(const ChainPlan& c, int role) {
  for (auto& m : c.mats)
    if (m.role == role) return m.w0 + m.nw;
  return 8;
}

// What the wavefronts of one role do.  All roles meet at every barrier and share the work of moving operands and results.
void chain_role(Src& s, const ChainPlan& c, int role) {
  const int NC = c.NC, VK = chain_vk(c.f64);
  const int half = c.out_elems + c.ext_elems;
  const bool whole4 = c.P % 4 == 0;
  auto str = [](long long v) { return std::to_string(v); };
  // Operands and results are moved by the role with the fewest multiplications
  const bool mover = role == c.roles - 1;
  const int mw = c.roles > 1 ? role_end(c, c.roles - 2) : 0, movers = 64 * (8 - mw);      // its first wavefront, its threads
  const std::string mtid = "(tid - " + str(64 * mw) + ")";
  auto targs = [&](const ChainMat& m) { return str(m.Q) + "LL, " + str(m.K) + "LL, " + str(m.sq) + "LL, " + str(m.sk) + "LL, "; };
  auto row_of = [&](const ChainMat& m, int u) { return "(w + " + str(m.nw * u - m.w0) + ") * 16"; };      // first row of the wavefront's u-th group
  // lone columns: this lane's row of groups 2 v and 2 v + 1, which the halves of the wavefront hold (all of it the first where there is no other)
  auto pair_row = [&](const ChainMat& m, int v, int units) {
    return "(w + " + str(2 * m.nw * v - m.w0) + (2 * v + 1 < units ? " + (lane >> 5) * " + str(m.nw) : std::string()) + ") * 16 + (lane & 15)";
  };
  // the weights that several levels multiply by
  for (size_t m = 0; m < c.mats.size(); ++m) {
    const ChainMat& mt = c.mats[m];
    if (!mt.kept() || mt.role != role) continue;
    for (int u = 0; u < mt.units; ++u) {
      const std::string wn = "w" + str((long long)m) + "_" + str(u);
      if (mt.reg[u]) s << "  T " << wn << "[" << mt.reg[u] << "] = {};\n";
      s << "  " << (mt.waves(u) < mt.nw ? "if (w < " + str(mt.w0 + mt.waves(u)) + ") " : std::string()) << "{\n    const T* y = (const T*)ar.p[" << m << "];\n";
      if (mt.reg[u]) s << "    frags<" << targs(mt) << mt.reg[u] << ", false>(y, " << wn << ", 0, 0, " << row_of(mt, u) << " + (lane & 15), g);\n";
      if (mt.reg[u] < mt.nf)
        s << "    frags<" << targs(mt) << mt.nf - mt.reg[u] << ", true>(y, lds + " << mt.lds[u] - 64 * mt.w0 << " + tid, " << 64 * mt.waves(u) << ", " << mt.reg[u] << ", " << row_of(mt, u)
          << " + (lane & 15), g);\n";
      s << "  }\n";
      if (mt.reg[u]) s << "#pragma unroll\n  for (int f = 0; f < " << mt.reg[u] << "; ++f) landed(" << wn << "[f]);\n";
    }
  }
  s << "  T *cur = lds, *prv = lds + " << half << ";\n  int at = " << c.n_const << ";\n";
  for (size_t k = 0; k < c.sections.size(); ++k) {
    const ChainSection& sec = c.sections[k];
    s << "  {\n";
    // names: x<j>_<t> / z<j>_<i> columns and inputs on their way to LDS (y..., for the next level), b<j>_<i>_<u> one value
    // per row, e<j>_<i>_<u> inputs by lanes (f..., of the next level)
    struct Staged { int rows, off, ptr; int64_t K, sp, sk; std::string nm; };
    std::vector<Staged> staged;
    for (size_t j = 0; j < sec.items.size(); ++j) {
      const ChainItem& it = sec.items[j];
      for (size_t t = 0; t < it.x.size(); ++t)
        if (it.x[t].kind == 0) staged.push_back({it.x[t].rows, it.x[t].off, it.x[t].ptr, it.x[t].K, it.x[t].sxp, it.x[t].sxk, str((long long)j) + "_x" + str((long long)t)});
      for (size_t i = 0; i < it.in.size(); ++i)
        if (it.in[i].kind == 4) staged.push_back({it.rows, it.in[i].off, it.in[i].ptr, it.Q, it.in[i].sp, it.in[i].sq, str((long long)j) + "_i" + str((long long)i)});
    }
    auto each_in = [&](int kind, auto&& fn) {
      for (size_t j = 0; j < sec.items.size(); ++j) {
        const ChainItem& it = sec.items[j];
        if (it.role != role) continue;
        const ChainMat& mt = c.mats[(size_t)it.x[0].mat];
        for (size_t i = 0; i < it.in.size(); ++i)
          if (it.in[i].kind == kind)
            for (int u = 0; u < (c.lone ? (mt.units + 1) / 2 : mt.units); ++u) {
              const std::string row = c.lone ? pair_row(mt, u, mt.units) : row_of(mt, u) + (it.wide() ? " + qw" : " + ql");
              fn(it, it.in[i], row + " < " + str(it.Q) + " ? " + row + " : " + str(it.Q - 1), str((long long)j) + "_" + str((long long)i) + "_" + str(u));
            }
      }
    };
    auto load_staged = [&](const char* base, const char* pre) {
      if (!mover) return;
      for (auto& x : staged) {
        const int ns = (x.rows * NC + movers - 1) / movers;
        s << "      " << (c.lone ? "T " : "A4 ") << pre << x.nm << "[" << ns << "];\n      {\n        const T* a = (const T*)ar.p[" << base << " + " << x.ptr << "];\n#pragma unroll\n";
        s << "        for (int i = 0; i < " << ns << "; ++i) {\n          const int sl = " << mtid << " + " << movers << " * i, kk = sl / NC, cc = sl % NC;\n";
        if (c.lone) s << "          const i64 p = p0 + cc;\n          " << pre << x.nm << "[i] = a[(i64)(kk < " << x.K << " ? kk : " << x.K - 1 << ") * " << x.sk << "LL + (p < P ? p : P - 1) * " << x.sp << "LL];\n        }\n      }\n";
        else s << "          " << pre << x.nm << "[i] = cols<" << x.sp << "LL>(a + (i64)(kk < " << x.K << " ? kk : " << x.K - 1 << ") * " << x.sk << "LL, p0 + 4 * cc);\n        }\n      }\n";
      }
    };
    auto put_staged = [&](const char* buf, const char* pre) {
      if (!mover) return;
      for (auto& x : staged) {
        const int ns = (x.rows * NC + movers - 1) / movers;
        s << "#pragma unroll\n      for (int i = 0; i < " << ns << "; ++i) {\n        const int sl = " << mtid << " + " << movers << " * i, kk = sl / NC, cc = sl % NC;\n";
        if (c.lone) s << "        if (sl < " << x.rows * NC << ") " << buf << "[" << x.off << " + cc * " << x.rows << " + kk] = kk < " << x.K << " ? " << pre << x.nm << "[i] : T(0);\n      }\n";
        else s << "        if (sl < " << x.rows * NC << ") *reinterpret_cast<A4*>(" << buf << " + " << x.off << " + cc * " << x.rows * 4 + 4 << " + kk * 4) = kk < " << x.K << " ? " << pre << x.nm
          << "[i] : A4{0, 0, 0, 0};\n      }\n";
      }
    };
    auto load_lanes = [&](const char* base, const char* pre) {
      each_in(3, [&](const ChainItem& it, const ChainIn& in, const std::string& row, const std::string& nm) {
        s << "    " << ctype(in.dtype) << " " << pre << nm << "[NC];\n    {\n      const " << ctype(in.dtype) << "* a = (const " << ctype(in.dtype) << "*)ar.p[" << base << " + " << in.ptr
          << "] + (i64)(" << row << ") * " << in.sq << "LL;\n";
        s << "#pragma unroll\n      for (int cc = 0; cc < NC; ++cc) {\n        const i64 p = p0 + " << (c.lone ? "cc" : it.wide() ? "4 * cc + pw" : "4 * cc + pl") << ";\n        " << pre << nm << "[cc] = a[(p < P ? p : P - 1) * " << in.sp << "LL];\n      }\n    }\n";
      });
    };
    auto landed_lanes = [&](const char* pre) {
      each_in(3, [&](const ChainItem&, const ChainIn& in, const std::string&, const std::string& nm) {
        if (dtype_size(in.dtype) >= 4) s << "#pragma unroll\n    for (int cc = 0; cc < NC; ++cc) landed(" << pre << nm << "[cc]);\n";
      });
    };
    auto write_out = [&](const std::string& base) {
      if (!mover) return;
      for (auto& it : sec.items)
        for (auto& o : it.out) {
          if (!o.staged) continue;
          const int64_t n = it.Q * NC;
          s << "      {\n        T* a = (T*)ar.p[" << base << " + " << o.ptr << "];\n#pragma unroll\n";
          s << "        for (int i = 0; i < " << (n + movers - 1) / movers << "; ++i) {\n          const int sl = " << mtid << " + " << movers << " * i, qq = sl / NC, cc = sl % NC;\n          const i64 p = p0 + " << (c.lone ? "" : "4 * ") << "cc;\n";
          if (c.lone) {
            s << "          if (sl < " << n << " && p < P) a[(i64)qq * P + p] = prv[" << o.off << " + cc * " << it.rows << " + qq];\n        }\n      }\n";
            continue;
          }
          s << "          if (sl < " << n << " && p < P) {\n            const A4 v = *reinterpret_cast<const A4*>(prv + " << o.off << " + cc * " << it.rows * 4 + 4 << " + qq * 4);\n";
          if (!whole4) s << "            if (p + 3 >= P) {\n#pragma unroll\n              for (int e = 0; e < 3; ++e)\n                if (p + e < P) a[(i64)qq * P + p + e] = v[e];\n            } else\n";
          s << "            *reinterpret_cast<V4*>(a + (i64)qq * P + p) = V4{v[0], v[1], v[2], v[3]};\n          }\n        }\n      }\n";
        }
    };
    each_in(1, [&](const ChainItem&, const ChainIn& in, const std::string& row, const std::string& nm) {
      s << "    const " << ctype(in.dtype) << " b" << nm << " = ((const " << ctype(in.dtype) << "*)ar.p[" << in.ptr << "])[(i64)(" << row << ") * " << in.sq << "LL];\n";
    });
    s << "    {\n";
    load_staged("at", "x");
    put_staged("cur", "x");
    s << "    }\n";
    load_lanes("at", "e");
    landed_lanes("e");
    s << "    __syncthreads();\n    const int n = ar.n[" << k << "];\n    for (int it = 0; it < n; ++it) {\n      const bool more = it + 1 < n;\n";
    s << "      if (it) {\n";
    write_out("at - " + str(sec.n_ptr));
    s << "      }\n";
    // fp32: what moves operands goes first, so that its program runs beside the others' multiplications (128 wide, 28 steps:
    // 5000 columns 173 -> 166 us forward, 178 -> 167 backward, 150 columns 43 -> 38 backward); fp64 loses 10 %
    if (!c.f64 && mover && c.roles > 1) s << "      __builtin_amdgcn_s_setprio(2);\n";
    s << "      const int to = more ? at + " << sec.n_ptr << " : at;      // (always, so that what is waited for does not depend on it)\n";
    load_staged("to", "y");
    load_lanes("to", "f");
    s << "      __builtin_amdgcn_sched_barrier(0);\n";      // (the loads stay here, a level's products before their use)
    // the role's products of this level, then their programs side by side (a lone program of fp64 is one long chain of
    // dependent instructions)
    auto products = [&](const std::vector<size_t>& js, int U) {
      int NA = 1;                  // accumulators taken in turn, so that four sums are under way
      while (U * NC * NA < 4 && NA < VK) NA *= 2;
      s << "        constexpr int NA = " << NA << ", U = " << U << ";\n";
      for (size_t j : js) {
        const ChainItem& it = sec.items[j];
        const std::string acc = "acc" + str((long long)j);
        const bool d64 = c.f64 || it.wide();      // on the fp64 instruction
        s << "        " << (it.wide() ? "double " : "Acc ") << acc << "[U][NC][NA];\n#pragma unroll\n        for (int u = 0; u < U; ++u)\n#pragma unroll\n          for (int cc = 0; cc < NC; ++cc)\n"
             "#pragma unroll\n            for (int a = 0; a < NA; ++a) " << acc << "[u][cc][a] = " << (it.wide() ? "0.0" : c.f64 ? "T(0)" : "Acc{0, 0, 0, 0}") << ";\n";
        for (auto& x : it.x) {
          const ChainMat& mt = c.mats[(size_t)x.mat];
          if (x.kind == 2) s << "        {\n          const T xv = *(const T*)ar.p[at + " << x.ptr << "];\n";
          else s << "        {\n          const T* xb = " << (x.kind == 1 ? "prv" : "cur") << " + " << x.off << (it.wide() ? " + g * 16 + (lane & 3)" : c.f64 ? " + g * 8 + (lane & 3)" : " + lane") << ";\n";
          // fragment of the columns (tile t, for fp64 of its half e)
          const std::string frag = x.kind != 2 ? "xb[cc * " + str(x.rows * 4 + 4) + (it.wide() ? " + 64 * t + 4 * e]" : c.f64 ? " + 32 * t + 4 * e]" : " + 64 * t]")
                                               : std::string(it.wide() ? "16 * t + 4 * g + e" : c.f64 ? "8 * t + 2 * g + e" : "16 * t + (lane >> 2)") + " < " + str(x.K) + " ? xv : T(0)";
          int in_regs[kChainMaxUnits];
          std::vector<int> cuts{0, mt.nf / VK};
          for (int u = 0; u < U; ++u) {
            in_regs[u] = mt.kept() ? mt.reg[u] : mt.nf;
            cuts.push_back(in_regs[u] / VK);
            if (!mt.kept())
              s << "          T ws" << u << "[" << mt.nf << "];\n          frags<" << targs(mt) << mt.nf << ", false>((const T*)ar.p[" << x.mat << "], ws" << u << ", 0, 0, " << row_of(mt, u) << " + (lane & 15), g);\n";
          }
          std::sort(cuts.begin(), cuts.end());
          for (size_t q = 0; q + 1 < cuts.size(); ++q) {
            if (cuts[q] == cuts[q + 1]) continue;
            s << "#pragma unroll\n          for (int t = " << cuts[q] << "; t < " << cuts[q + 1] << "; ++t) {\n";
            if (!d64) s << "            T a[NC];\n#pragma unroll\n            for (int cc = 0; cc < NC; ++cc) a[cc] = " << frag << ";\n";
            else s << "            " << (it.wide() ? "double" : "T") << " a[VK][NC];\n#pragma unroll\n            for (int e = 0; e < VK; ++e)\n#pragma unroll\n              for (int cc = 0; cc < NC; ++cc) a[e][cc] = " << frag << ";\n";
            for (int e = 0; e < VK; ++e)
              for (int u = 0; u < U; ++u) {
                s << "            { const T wv = ";
                if (cuts[q] < in_regs[u] / VK) s << (mt.kept() ? "w" + str(x.mat) + "_" + str(u) : "ws" + str(u)) << "[" << VK << " * t + " << e << "];\n";
                else s << "lds[" << mt.lds[u] - 64 * mt.w0 << " + tid + (" << VK << " * t + " << e - in_regs[u] << ") * " << 64 * mt.waves(u) << "];\n";
                s << "#pragma unroll\n              for (int cc = 0; cc < NC; ++cc) " << acc << "[" << u << "][cc][" << e % NA << "] = ";
                if (!d64) s << "mm<" << e << ">(a[cc], wv, " << acc << "[" << u << "][cc][" << e % NA << "]); }\n";
                else s << "__builtin_amdgcn_mfma_f64_4x4x4f64((double)wv, a[" << e << "][cc], " << acc << "[" << u << "][cc][" << e % NA << "], 0, 0, 0); }\n";
              }
            s << "          }\n";
          }
          s << "        }\n";
        }
      }
      s << "#pragma unroll\n        for (int cc = 0; cc < NC; ++cc) {\n";
      for (size_t j : js) {
        const ChainItem& it = sec.items[j];
        const Spec& sp = it.kn->spec;
        const ChainMat& m0 = c.mats[(size_t)it.x[0].mat];
        for (int u = 0; u < U; ++u) {
          const std::string sfx = "_" + str((long long)j) + "_" + str(u), acc = "acc" + str((long long)j) + "[" + str(u) + "][cc]";
          s << "          const int q" << sfx << " = " << row_of(m0, u) << (it.wide() ? " + qw" : " + ql") << ";\n#pragma unroll\n          for (int a = 1; a < NA; ++a) " << acc << "[0] += " << acc << "[a];\n";
          for (size_t i = 0; i < it.in.size(); ++i) {
            const ChainIn& in = it.in[i];
            s << "          const " << ctype(in.dtype) << " v" << i << sfx << " = ";
            if (in.kind == 0) s << (it.wide() ? "(T)" + acc + "[0]" : c.f64 ? acc + "[0]" : "meet(" + acc + "[0])") << ";\n";
            else if (in.kind == 1) s << "b" << j << "_" << i << "_" << u << ";\n";
            else if (in.kind == 3) s << "e" << j << "_" << i << "_" << u << "[cc];\n";
            else s << (in.kind == 2 ? "prv[" : "cur[") << in.off << " + cc * " << it.rows * 4 + 4 << " + q" << sfx << " * 4 + " << (it.wide() ? "pw" : "pl") << "];\n";
          }
          emit_program(s, sp.n_in, sp.n_instr, sp.prog, sp.dt, "          ", sfx);
        }
      }
      for (size_t j : js) {
        const ChainItem& it = sec.items[j];
        for (int u = 0; u < U; ++u) {
          const std::string sfx = "_" + str((long long)j) + "_" + str(u);
          bool direct = false;
          for (auto& o : it.out) {
            if (o.staged) s << "          cur[" << o.off << " + cc * " << it.rows * 4 + 4 << " + q" << sfx << " * 4 + " << (it.wide() ? "pw" : "pl") << "] = q" << sfx << " < " << it.Q << " ? v" << o.slot << sfx << " : T(0);\n";
            else direct = true;
          }
          if (!direct) continue;
          s << "          {\n            const i64 p = p0 + 4 * cc + " << (it.wide() ? "pw" : "pl") << ";\n            if (q" << sfx << " < " << it.Q << " && p < P) {\n";
          for (auto& o : it.out)
            if (!o.staged) s << "              ((" << ctype(o.dtype) << "*)ar.p[at + " << o.ptr << "])[(i64)q" << sfx << " * P + p] = v" << o.slot << sfx << ";\n";
          s << "            }\n          }\n";
        }
      }
      s << "        }\n";
    };
    // Lone columns: a group of sixteen lanes has a quarter of k, an element a lane, and every lane its row's weights of that
    // quarter; an element reaches its group as the broadcast operand of the multiplication (row_newbcast).  Two row groups side by side; their
    // quarters meet by lane swaps, which leave the first group's sums in the lower half of the wavefront and the second's in the upper.
    auto lone_products = [&](const std::vector<size_t>& js, int U) {
      for (size_t j : js) {
        const ChainItem& it = sec.items[j];
        const std::string acc = "acc" + str((long long)j);
        s << "        T " << acc << "[NC][" << 2 * ((U + 1) / 2) << "] = {};\n";
        for (auto& x : it.x) {
          const ChainMat& mt = c.mats[(size_t)x.mat];
          const int nx = (mt.nf + 15) / 16;
          s << "        {\n          T xr[NC][" << nx << "];\n";
          if (x.kind == 2) s << "          const T xv = *(const T*)ar.p[at + " << x.ptr << "];\n";
          else s << "          const T* xb = " << (x.kind == 1 ? "prv" : "cur") << " + " << x.off << " + kl;\n";
          s << "#pragma unroll\n          for (int cc = 0; cc < NC; ++cc)\n#pragma unroll\n            for (int i = 0; i < " << nx << "; ++i) xr[cc][i] = ";
          if (x.kind == 2) s << "64 * i + kl < " << x.K << " ? xv : T(0);\n";
          else s << "xb[cc * " << x.rows << " + 64 * i];\n";
          if (!mt.kept())
            for (int u = 0; u < U; ++u)
              s << "          T ws" << u << "[" << mt.nf << "];\n          frags<" << targs(mt) << mt.nf << ", false>((const T*)ar.p[" << x.mat << "], ws" << u << ", 0, 0, " << row_of(mt, u) << " + (lane & 15), g);\n";
          auto weight = [&](int u, int f) {
            if (!mt.kept()) return "ws" + str(u) + "[" + str(f) + "]";
            if (f < mt.reg[u]) return "w" + str(x.mat) + "_" + str(u) + "[" + str(f) + "]";
            return "lds[" + str(mt.lds[u] - 64 * mt.w0 + (f - mt.reg[u]) * 64 * mt.waves(u)) + " + tid]";
          };
          for (int f = 0; f < mt.nf; f += 8) {
            const int n = std::min(8, mt.nf - f);
            for (int u = 0; u < U; u += 2) {
              const bool two = u + 1 < U;      // (a lone row group: two sums in turn, one after the other they would wait for each other)
              for (int cc = 0; cc < NC; ++cc) {
                s << "          asm(\"s_nop 1\\n\"\n";       // (two states between another write of the broadcast operand and its use, which the compiler does not see)
                for (int e = 0; e < n; ++e)
                  for (int a = 0; a < (two ? 2 : 1); ++a)
                    s << "              \"v_fmac_f64_dpp %" << (two ? a : e & 1) << ", %2, %" << 3 + a * n + e << " row_newbcast:" << (f + e) % 16 << " row_mask:0xf bank_mask:0xf\\n\"\n";
                s << "              \"s_nop 1\" : \"+v\"(" << acc << "[" << cc << "][" << u << "]), \"+v\"(" << acc << "[" << cc << "][" << u + 1 << "]) : \"v\"(xr[" << cc << "][" << f / 16 << "])";
                for (int a = 0; a < (two ? 2 : 1); ++a)
                  for (int e = 0; e < n; ++e) s << ", \"v\"(" << weight(u + a, f + e) << ")";
                s << ");\n";
              }
            }
          }
          s << "        }\n";
        }
      }
      s << "#pragma unroll\n        for (int cc = 0; cc < NC; ++cc) {\n          const i64 p = p0 + cc;\n";
      for (size_t j : js) {
        const ChainItem& it = sec.items[j];
        const Spec& sp = it.kn->spec;
        const ChainMat& m0 = c.mats[(size_t)it.x[0].mat];
        for (int v = 0; 2 * v < U; ++v) {
          const bool two = 2 * v + 1 < U;
          const std::string sfx = "_" + str((long long)j) + "_" + str(v), acc = "acc" + str((long long)j) + "[cc][";
          s << "          const int q" << sfx << " = " << pair_row(m0, v, U) << ";\n";
          for (size_t i = 0; i < it.in.size(); ++i) {
            const ChainIn& in = it.in[i];
            s << "          const " << ctype(in.dtype) << " v" << i << sfx << " = ";
            if (in.kind == 0) {
              if (two) s << "meet(" << acc << 2 * v << "], " << acc << 2 * v + 1 << "]);\n";
              else s << "meet(" << acc << 2 * v << "] + " << acc << 2 * v + 1 << "], " << acc << 2 * v << "] + " << acc << 2 * v + 1 << "]);\n";
            } else if (in.kind == 1) s << "b" << j << "_" << i << "_" << v << ";\n";
            else if (in.kind == 3) s << "e" << j << "_" << i << "_" << v << "[cc];\n";
            else s << (in.kind == 2 ? "prv[" : "cur[") << in.off << " + cc * " << it.rows << " + q" << sfx << "];\n";
          }
          emit_program(s, sp.n_in, sp.n_instr, sp.prog, sp.dt, "          ", sfx);
          // (a wavefront without the second group computes the first one's rows in both halves, the upper with that group's operands)
          const std::string mine = two ? "" : "lane < 32 && ";
          for (auto& o : it.out) {
            if (o.staged) {
              if (!two) s << "          if (lane < 32) ";
              else s << "          ";
              s << "cur[" << o.off << " + cc * " << it.rows << " + q" << sfx << "] = q" << sfx << " < " << it.Q << " ? v" << o.slot << sfx << " : T(0);\n";
            } else {
              s << "          if (" << mine << "q" << sfx << " < " << it.Q << " && p < P) ((" << ctype(o.dtype) << "*)ar.p[at + " << o.ptr << "])[(i64)q" << sfx << " * P + p] = v" << o.slot << sfx << ";\n";
            }
          }
        }
      }
      s << "        }\n";
    };
    std::vector<char> taken(sec.items.size(), 0);
    for (size_t j = 0; j < sec.items.size(); ++j) {
      if (sec.items[j].role != role || taken[j]) continue;
      const ChainMat& m0 = c.mats[(size_t)sec.items[j].x[0].mat];
      std::vector<size_t> js;      // those with as many row groups
      for (size_t i = j; i < sec.items.size(); ++i)
        if (sec.items[i].role == role && c.mats[(size_t)sec.items[i].x[0].mat].groups() == m0.groups()) { js.push_back(i); taken[i] = 1; }
      const int rem = m0.waves(m0.units - 1);      // wavefronts with all the row groups; the others have one less
      s << "      ";
      if (rem < m0.nw) s << "if (w < " << m0.w0 + rem << ") ";
      s << "{\n";
      c.lone ? lone_products(js, m0.units) : products(js, m0.units);
      s << "      }\n";
      if (rem < m0.nw && m0.units > 1) {
        s << "      else {\n";
        c.lone ? lone_products(js, m0.units - 1) : products(js, m0.units - 1);
        s << "      }\n";
      }
    }
    landed_lanes("f");
    s << "      if (more) {\n";
    put_staged("prv", "y");
    each_in(3, [&](const ChainItem&, const ChainIn&, const std::string&, const std::string& nm) { s << "#pragma unroll\n        for (int cc = 0; cc < NC; ++cc) e" << nm << "[cc] = f" << nm << "[cc];\n"; });
    s << "      }\n      __syncthreads();\n      at += " << sec.n_ptr << ";\n      T* const z = cur;\n      cur = prv;\n      prv = z;\n    }\n";
    write_out("at - " + str(sec.n_ptr));
    s << "  }\n";
  }
}

std::string chain_source(const ChainPlan& c, const std::string& kname) {
  Src s;
  const int NC = c.NC, VK = chain_vk(c.f64);
  const bool whole4 = c.P % 4 == 0;      // a group of four columns is inside the array or outside
  s << kPrelude;
  s << "typedef " << (c.f64 ? "double" : "float") << " T;\n";
  s << "typedef T V2 __attribute__((ext_vector_type(2), aligned(" << (c.f64 ? 8 : 4) << ")));\ntypedef T V4 __attribute__((ext_vector_type(4), aligned(" << (c.f64 ? 8 : 4) << ")));\n";
  s << "typedef T A4 __attribute__((ext_vector_type(4), aligned(16)));\n";
  // The value is here, not on its way: without this the waits for loads from before a loop stand at the uses inside it,
  // where they also wait for everything issued since (a level's stores and the next one's operands)
  s << "template <typename E> __device__ __forceinline__ void landed(E& v) { asm volatile(\"\" : \"+v\"(v)); }\n";
  s << "constexpr int NC = " << NC << ", VK = " << VK << ";\nconstexpr i64 P = " << c.P << "LL;\n";
  s << "struct Args { const void* p[" << kChainMaxPtrs << "]; int n[" << kChainMaxSections << "]; };\n";
  // fragments [f0, f0 + n) of row q of a weights factor, zero past its end
  s << "template <i64 Q, i64 K, i64 SQ, i64 SK, int N, bool PUT> __device__ __forceinline__ void frags(const T* __restrict__ y, T* to, int pitch, int f0, int q, int g) {\n"
       "  const i64 qq = q < Q ? q : Q - 1;\n"
       "#pragma unroll\n  for (int f = 0; f < N; f += VK) {\n    const int k = 4 * VK * ((f0 + f) / VK) + VK * g;\n    T v[VK];\n"
       "    if constexpr (SK == 1 && K % VK == 0) {\n      const T* a = y + qq * SQ + (k < K ? k : K - VK);\n";
  if (c.f64) s << "      const V2 z = *reinterpret_cast<const V2*>(a);\n";
  else s << "      const V4 z = *reinterpret_cast<const V4*>(a);\n";
  s << "#pragma unroll\n      for (int e = 0; e < VK; ++e) v[e] = z[e];\n    } else {\n"
       "#pragma unroll\n      for (int e = 0; e < VK; ++e) v[e] = y[qq * SQ + (k + e < K ? k + e : K - 1) * SK];\n    }\n"
       "#pragma unroll\n    for (int e = 0; e < VK; ++e) {\n      const T z = q < Q && k + e < K ? v[e] : T(0);\n      if constexpr (PUT) to[(f + e) * pitch] = z;\n      else to[f + e] = z;\n    }\n  }\n}\n";
  if (!c.f64) {
    s << "typedef T Acc __attribute__((ext_vector_type(4)));\n";
    s << "template <int E> __device__ __forceinline__ Acc mm(T x, T w, Acc a) { return __builtin_amdgcn_mfma_f32_4x4x1f32(x, w, a, 2, E, 0); }\n";
    // the quarters of k: afterwards the lanes of group g hold column g of the row lane % 16
    s << "__device__ __forceinline__ T meet(Acc a) {\n"
         "  auto r0 = __builtin_amdgcn_permlane32_swap(__float_as_uint(a[0]), __float_as_uint(a[2]), false, false);\n"
         "  auto r1 = __builtin_amdgcn_permlane32_swap(__float_as_uint(a[1]), __float_as_uint(a[3]), false, false);\n"
         "  const T s0 = __uint_as_float(r0[0]) + __uint_as_float(r0[1]), s1 = __uint_as_float(r1[0]) + __uint_as_float(r1[1]);\n"
         "  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(s0), __float_as_uint(s1), false, false);\n"
         "  return __uint_as_float(r[0]) + __uint_as_float(r[1]);\n}\n";
  } else {
    s << "typedef T Acc;\n";
  }
  if (c.lone) {
    // The quarters of k, by groups of sixteen lanes: afterwards the lower half of the lanes holds the sums of a, the upper those of b.
    s << "__device__ __forceinline__ T halves(T a, T b, bool far) {\n"
         "  const unsigned long long x = __double_as_longlong(a), y = __double_as_longlong(b);\n"
         "  auto lo = far ? __builtin_amdgcn_permlane32_swap((unsigned)x, (unsigned)y, false, false) : __builtin_amdgcn_permlane16_swap((unsigned)x, (unsigned)y, false, false);\n"
         "  auto hi = far ? __builtin_amdgcn_permlane32_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false) : __builtin_amdgcn_permlane16_swap((unsigned)(x >> 32), (unsigned)(y >> 32), false, false);\n"
         "  return __longlong_as_double((unsigned long long)hi[0] << 32 | lo[0]) + __longlong_as_double((unsigned long long)hi[1] << 32 | lo[1]);\n}\n"
         "__device__ __forceinline__ T meet(T a, T b) {\n  const T s = halves(a, b, true);\n  return halves(s, s, false);\n}\n";
  }
  // Four neighbouring columns from p on of a row that starts at a; past the end the last column (never stored)
  s << "template <i64 SP> __device__ __forceinline__ A4 cols(const T* __restrict__ a, i64 p) {\n  A4 v;\n";
  if (whole4) s << "  if constexpr (SP == 1) {\n    const V4 z = *reinterpret_cast<const V4*>(a + (p < P ? p : P - 4));\n    v = A4{z[0], z[1], z[2], z[3]};\n    return v;\n  }\n";
  s << "#pragma unroll\n  for (int e = 0; e < 4; ++e) v[e] = a[(p + e < P ? p + e : P - 1) * SP];\n  return v;\n}\n";
  s << "extern \"C\" __global__ void __launch_bounds__(512) " << kname << "(Args ar) {\n";
  s << "  __shared__ __attribute__((aligned(16))) T lds[" << c.lds_elems << "];\n";
  s << "  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, w = __builtin_amdgcn_readfirstlane(tid >> 6);\n";
  if (c.lone) s << "  const int kl = 8 * ((lane & 15) >> 1) + 2 * g + (lane & 1);      // which of 64 k this lane holds for its group\n";
  else if (c.f64) s << "  const int ql = 4 * ((lane >> 2) & 3) + g, pl = lane & 3;      // row and column of this lane's result\n";
  else s << "  const int ql = lane & 15, pl = g, qw = 4 * ((lane >> 2) & 3) + g, pw = lane & 3;      // (w: where sums are fp64)\n";
  // consecutive blocks go round the eight XCDs: neighbouring columns, whose lines of memory overlap, belong to one XCD
  const int64_t nblk = chain_blocks(c), per_xcd = (nblk + 7) / 8;
  s << "  const int blk = (int)(blockIdx.x % 8) * " << per_xcd << " + (int)(blockIdx.x / 8);\n  if (blk >= " << nblk << ") return;\n";
  s << "  const i64 p0 = (i64)blk * (" << (c.lone ? "" : "4 * ") << "NC);\n";
  for (int role = 0; role < c.roles; ++role) {
    s << "  // ---- role " << role << "\n  ";
    if (role + 1 < c.roles) s << "if (w < " << role_end(c, role) << ") ";
    s << "{\n";
    chain_role(s, c, role);
    s << "  return;\n  }\n";
  }
  s << "}\n";
  return s.str();
}

struct ChainLink { int item = -1, out = -1; };     // the queue item, and which of its results
struct ChainCand {
  const Deferred* d = nullptr;
  bool in = false, linked = false;
  int level = 0;
  std::vector<ChainLink> x, inp;      // per term, per input
};

// Where an operand's pointer sits in a Deferred's arguments.
size_t arg_of_input(const Spec& sp, int i) { return 2 * sp.terms.size() + (size_t)(i < sp.c_slot ? i : i - 1); }
size_t arg_of_out(const Spec& sp, int o) { return 2 * sp.terms.size() + (size_t)(sp.n_in - 1) + (size_t)o; }

// The held-back products that form a chain: those with P columns of one type that read one another's results column
// by column (a whole result as the columns factor of a term, or as an input of the program), and nothing else that is
// held back.  Returns the number of levels, 0 when there is none, or when one of them reads a result from further back than the
// level before, or a level has more than kChainMaxWidth of them.
int find_chain(const std::vector<Deferred>& items, std::vector<ChainCand>& cand) {
  int n_small = 0;
  for (auto& d : items) n_small += d.kn != nullptr;
  if (n_small < kChainMinLevels) return 0;
  std::map<std::pair<int64_t, bool>, int> count;
  std::map<const hgpu_buffer*, int> writer;
  for (size_t i = 0; i < items.size(); ++i) {
    for (auto* b : items[i].writes) writer[b] = (int)i;
    if (items[i].kn) ++count[{items[i].kn->spec.P, items[i].kn->spec.f64}];
  }
  std::pair<int64_t, bool> which{0, false};
  int most = 0;
  for (auto& c : count)
    if (c.second > most) { most = c.second; which = c.first; }
  if (most < kChainMinLevels) return 0;
  cand.assign(items.size(), ChainCand());
  for (size_t i = 0; i < items.size(); ++i) {
    if (!items[i].kn) continue;
    const Spec& sp = items[i].kn->spec;
    cand[i].d = &items[i];
    cand[i].in = sp.P == which.first && sp.f64 == which.second && sp.splits == 1 && sp.Q <= 256;
    cand[i].x.resize(sp.terms.size());
    cand[i].inp.resize((size_t)sp.n_in);
  }
  const int own = which.second ? HGPU_F64 : HGPU_F32;
  for (bool again = true; again;) {
    again = false;
    for (size_t i = 0; i < items.size(); ++i) {
      ChainCand& c = cand[i];
      if (!c.in) continue;
      const Spec& sp = items[i].kn->spec;
      bool ok = true;
      for (auto* b : items[i].reads) {
        auto it = writer.find(b);
        if (it == writer.end()) continue;
        const ChainCand& from = cand[(size_t)it->second];
        if (it->second >= (int)i || !from.in) { ok = false; break; }
        const Spec& fs = items[(size_t)it->second].kn->spec;
        int out = -1;
        for (int o = 0; o < (int)fs.out_slots.size(); ++o)
          if (items[(size_t)it->second].writes[(size_t)o] == b) out = o;
        if (out < 0 || fs.dt[(size_t)fs.out_slots[(size_t)out]] != own) { ok = false; break; }
        const char *lo = (const char*)b->ptr, *hi = lo + b->bytes;
        const void* whole = items[(size_t)it->second].args[arg_of_out(fs, out)];
        auto inside = [&](const void* p) { return (const char*)p >= lo && (const char*)p < hi; };
        for (size_t t = 0; t < sp.terms.size(); ++t) {
          const void *x = items[i].args[2 * t], *y = items[i].args[2 * t + 1];
          if (inside(y)) ok = false;
          if (!inside(x)) continue;
          const Term& tm = sp.terms[t];
          if (x != whole || tm.sxp != 1 || tm.sxk != sp.P || tm.K != fs.Q) ok = false;
          c.x[t] = ChainLink{it->second, out};
        }
        for (int k = 0; k < sp.n_in; ++k) {
          if (k == sp.c_slot) continue;
          const void* p = items[i].args[arg_of_input(sp, k)];
          if (!inside(p)) continue;
          if (p != whole || sp.in_sp[(size_t)k] != 1 || sp.in_sq[(size_t)k] != sp.P || fs.Q != sp.Q || sp.dt[(size_t)k] != own) ok = false;
          c.inp[(size_t)k] = ChainLink{it->second, out};
        }
        if (!ok) break;
      }
      if (!ok) { c.in = false; again = true; }
    }
  }
  int top = -1;
  for (size_t i = 0; i < items.size(); ++i) {
    ChainCand& c = cand[i];
    if (!c.in) continue;
    c.level = 0;
    for (auto* v : {&c.x, &c.inp})
      for (auto& l : *v)
        if (l.item >= 0) {
          c.level = std::max(c.level, cand[(size_t)l.item].level + 1);
          c.linked = cand[(size_t)l.item].linked = true;
        }
  }
  std::vector<int> width;
  for (auto& c : cand) {
    if (!c.linked) { c.in = false; continue; }
    top = std::max(top, c.level);
    width.resize((size_t)top + 1, 0);
    if (++width[(size_t)c.level] > kChainMaxWidth) return 0;
    for (auto* v : {&c.x, &c.inp})
      for (auto& l : *v)
        if (l.item >= 0 && cand[(size_t)l.item].level != c.level - 1) return 0;
  }
  return top + 1 >= kChainMinLevels ? top + 1 : 0;
}

// Gives every role its wavefronts; false: some would have too many row groups.
bool share_wavefronts(ChainPlan& c, bool apart) {
  static const int from[5][5] = {{0, 8}, {0, 8}, {0, 4, 8}, {0, 4, 6, 8}, {0, 2, 4, 6, 8}};
  if (!apart) c.roles = 1;
  for (auto& m : c.mats) {
    if (!apart) m.role = 0;
    m.w0 = from[c.roles][m.role];
    m.nw = from[c.roles][m.role + 1] - m.w0;
    m.units = (m.groups() + m.nw - 1) / m.nw;
    if (m.units > kChainMaxUnits) return false;
  }
  for (auto& s : c.sections)
    for (auto& it : s.items) it.role = c.mats[(size_t)it.x[0].mat].role;
  return true;
}

// Which fragments of the weights wait in registers and which in LDS; false: they do not fit.
bool place_weights(ChainPlan& c, int slack) {
  const int es = c.f64 ? 8 : 4, regs_per = es / 4, vk = chain_vk(c.f64);
  c.out_elems = c.ext_elems = 0;
  for (auto& s : c.sections) {
    int out = 0, ext = 0;
    for (auto& it : s.items) {
      for (auto& o : it.out)
        if (o.staged) { o.off = out; out += chain_region(c, it.rows); }
      for (auto& x : it.x)
        if (x.kind == 0) { x.off = ext; ext += chain_region(c, x.rows); }
      for (auto& in : it.in)
        if (in.kind == 4) { in.off = ext; ext += chain_region(c, it.rows); }
    }
    c.out_elems = std::max(c.out_elems, out);
    c.ext_elems = std::max(c.ext_elems, ext);
  }
  // operands from outside the chain come after the results; operands from inside are where the level before put them
  for (auto& s : c.sections)
    for (auto& it : s.items) {
      for (auto& x : it.x)
        if (x.kind == 0) x.off += c.out_elems;
      for (auto& in : it.in)
        if (in.kind == 4) in.off += c.out_elems;
    }
  int at = 2 * (c.out_elems + c.ext_elems);
  const int room = kChainLds / es - 64;
  if (at > room) return false;
  for (int role = 0; role < c.roles; ++role) {
    // 256 registers a lane (two wavefronts per SIMD), less accumulators, what is fetched a level ahead, and the program's own
    int most = 0;
    const int movers = role == c.roles - 1 ? 64 * (c.roles > 1 ? 8 - role_end(c, role - 1) : 8) : 0;
    for (auto& s : c.sections) {
      int ahead = 0, mine = 0, consts = 0, wide = 0;
      for (auto& it : s.items) {
        for (auto& x : it.x)
          if (x.kind == 0 && movers) ahead += (x.rows * c.NC + movers - 1) / movers * (c.lone ? 1 : 4);
        for (auto& in : it.in)
          if (in.kind == 4 && movers) ahead += (it.rows * c.NC + movers - 1) / movers * (c.lone ? 1 : 4);
        if (it.role != role) continue;
        const int units = c.mats[(size_t)it.x[0].mat].units;
        mine += units * c.NC * (c.f64 ? 1 : it.wide() ? 2 : 4);
        if (it.wide()) wide = 44 + 8 * c.NC;      // (an fp64 program's overhead, columns as doubles)
        for (auto& in : it.in) {
          if (in.kind == 3) ahead += 2 * c.NC * units;
          if (in.kind == 1) consts += units;
        }
      }
      // (with many accumulators the compiler keeps about as many other values)
      most = std::max(most, ahead + mine + consts + wide + 2 * c.NC + (c.f64 ? 0 : 2 * std::max(0, mine - 40)));
    }
    int regs = std::max(0, (256 - regs_per * most - (c.f64 ? 84 : 40) - slack) / regs_per / vk * vk);
    for (int u = 0; u < kChainMaxUnits; ++u)
      for (auto& m : c.mats) {
        if (!m.kept() || m.role != role || u >= m.units) continue;
        m.reg[u] = std::min(regs, m.nf);
        regs -= m.reg[u];
        m.lds[u] = at;
        at += (m.nf - m.reg[u]) * 64 * m.waves(u);
        if (at > room) return false;
      }
  }
  c.lds_elems = at + (c.lone ? 64 : 16);      // (lone columns are read 64 k at a time)
  return true;
}

// Whether the chain is faster than its levels one after another.  A level of the chain: the multiplications at the rate of
// the small instructions on the CU's columns (fp32 246, fp64 122 billion a second) and 15 % on top, and what follows one
// after another in it; a level by itself: a launch, or the rate that products of this size reach (fp32 49, fp64 33 TFLOP/s).
// Measured (two layers of 12 steps, gradient, us, levels / chain): fp64 1000 x 128 301 / 263, 2000 x 128 390 / 376, 5000 x
// 128 (five rounds of four columns a block) 714 / 736; fp32 5000 x 128 420 / 355, 150 x 128 191 / 156.
bool pays(const ChainPlan& c, int num_cu) {
  const double rounds = (double)((chain_blocks(c) + num_cu - 1) / num_cu);
  double chain = 0, levels = 0;
  for (auto& s : c.sections) {
    double mul = 0, flops = 0, after = 0.9e-6;      // mul, flops: seconds
    for (auto& it : s.items) {
      const bool d64 = c.f64 || it.wide();
      if (d64) after = 1.2e-6;
      for (auto& x : it.x) {
        mul += (double)it.rows * x.rows * chain_columns(c) / (c.lone ? 102e9 : d64 ? 122e9 : 246e9);
        flops += 2.0 * (double)it.Q * (double)x.K * (double)c.P / (d64 ? 33e12 : 49e12);
      }
    }
    chain += s.n_levels * rounds * (mul * 1.15 + after);
    levels += s.n_levels * std::max(4.7e-6, flops);
  }
  return chain + 5e-6 * rounds < levels;
}

// The plan of levels [l0, ...) as far as the kernel's arguments hold their pointers; *l1 is the first level left out.
bool plan_chain(const std::vector<ChainCand>& cand, const std::vector<std::vector<int>>& levels, int num_cu, int slack, bool lone, int l0, int* l1, ChainPlan* plan) {
  ChainPlan& c = *plan;
  const Spec& first = cand[(size_t)levels[(size_t)l0][0]].d->kn->spec;
  c.f64 = first.f64;
  c.P = first.P;
  std::map<std::tuple<const void*, int64_t, int64_t, int64_t, int64_t>, int> mat_ids;
  struct Level { std::vector<ChainItem> items; std::vector<std::vector<const void*>> consts; std::vector<const void*> ptrs; };
  std::vector<Level> lv;
  size_t n_ptrs = 64;            // (room for weights and constants)
  int l = l0;
  std::map<int, std::pair<int, int>> place;     // queue item -> level, position in it
  for (; l < (int)levels.size(); ++l) {
    Level L;
    for (size_t j = 0; j < levels[(size_t)l].size(); ++j) {
      const int id = levels[(size_t)l][j];
      const ChainCand& cd = cand[(size_t)id];
      const Deferred& d = *cd.d;
      const Spec& sp = d.kn->spec;
      ChainItem it;
      it.kn = d.kn;
      it.Q = sp.Q;
      it.rows = (int)((sp.Q + 15) / 16 * 16);
      for (size_t t = 0; t < sp.terms.size(); ++t) {
        const Term& tm = sp.terms[t];
        auto key = std::make_tuple(d.args[2 * t + 1], sp.Q, tm.K, tm.syq, tm.syk);
        auto m = mat_ids.find(key);
        if (m == mat_ids.end()) {
          m = mat_ids.emplace(key, (int)c.mats.size()).first;
          ChainMat mt;
          mt.ptr = d.args[2 * t + 1];
          mt.Q = sp.Q; mt.K = tm.K; mt.sq = tm.syq; mt.sk = tm.syk;
          mt.nf = chain_kp(c.f64, tm.K) / 4;
          c.mats.push_back(mt);
        }
        ++c.mats[(size_t)m->second].uses;
        ChainX x{m->second, 0, 0, chain_kp(c.f64, tm.K), tm.K, tm.sxp, tm.sxk, 0};
        const ChainLink& ln = cd.x[t];
        if (ln.item >= 0 && place.count(ln.item)) {
          x.kind = 1;
          x.off = -1 - (place[ln.item].second * 8 + ln.out);      // resolved below
          x.rows = (int)((tm.K + 15) / 16 * 16);
          x.sxp = x.sxk = 0;
        } else {
          if (tm.sxp == 0 && tm.sxk == 0) x.kind = 2;       // (the state that a recurrence starts from)
          x.ptr = (int)L.ptrs.size();
          L.ptrs.push_back(d.args[2 * t]);
        }
        it.x.push_back(x);
      }
      std::vector<const void*> consts;
      for (int i = 0; i < sp.n_in; ++i) {
        ChainIn in{0, sp.dt[(size_t)i], 0, 0, sp.in_sp[(size_t)i], sp.in_sq[(size_t)i], 0};
        if (i != sp.c_slot) {
          const ChainLink& ln = cd.inp[(size_t)i];
          const void* p = d.args[arg_of_input(sp, i)];
          if (ln.item >= 0 && place.count(ln.item)) {
            in.kind = 2;
            in.off = -1 - (place[ln.item].second * 8 + ln.out);
            in.rows = it.rows;
          } else if (in.sp == 0) {
            in.kind = 1;
            consts.push_back(p);
          } else {
            in.kind = in.sp == 1 && in.dtype == (c.f64 ? HGPU_F64 : HGPU_F32) ? 4 : 3;
            in.ptr = (int)L.ptrs.size();
            L.ptrs.push_back(p);
          }
        }
        it.in.push_back(in);
      }
      for (int o = 0; o < (int)sp.out_slots.size(); ++o) {
        const int dt = sp.dt[(size_t)sp.out_slots[(size_t)o]];
        ChainOut out{sp.out_slots[(size_t)o], dt == (c.f64 ? HGPU_F64 : HGPU_F32), dt, 0, (int)L.ptrs.size()};
        L.ptrs.push_back(d.args[arg_of_out(sp, o)]);
        it.out.push_back(out);
      }
      L.items.push_back(std::move(it));
      L.consts.push_back(std::move(consts));
    }
    if (n_ptrs + L.ptrs.size() > (size_t)kChainMaxPtrs) break;
    n_ptrs += L.ptrs.size();
    lv.push_back(std::move(L));
    for (size_t j = 0; j < levels[(size_t)l].size(); ++j) {
      place[levels[(size_t)l][j]] = {l, (int)j};
      c.flops += cand[(size_t)levels[(size_t)l][j]].d->flops;
      c.bytes += cand[(size_t)levels[(size_t)l][j]].d->bytes;
      ++c.n_items;
    }
    // only the level before is at hand in LDS: links to it are the only ones there are (find_chain)
  }
  *l1 = l;
  c.n_levels = l - l0;
  if (c.n_levels < 2) return false;
  // sections: consecutive levels with the same items on the same weights and constants
  auto same = [](const ChainItem& a, const ChainItem& b) {
    if (a.kn != b.kn || a.x.size() != b.x.size()) return false;
    for (size_t t = 0; t < a.x.size(); ++t)
      if (a.x[t].mat != b.x[t].mat || a.x[t].kind != b.x[t].kind || a.x[t].off != b.x[t].off) return false;
    for (size_t i = 0; i < a.in.size(); ++i)
      if (a.in[i].kind != b.in[i].kind || a.in[i].off != b.in[i].off) return false;
    return true;
  };
  std::vector<size_t> first_of;
  for (size_t k = 0; k < lv.size(); ++k) {
    bool join = k > 0 && lv[k].items.size() == lv[k - 1].items.size() && lv[k].consts == lv[k - 1].consts;
    for (size_t j = 0; join && j < lv[k].items.size(); ++j) join = same(lv[k].items[j], lv[k - 1].items[j]);
    // (what the level before put where has to be the same too: at the first of several like levels it may not be)
    if (join && first_of.back() == k - 1 && k >= 2) {
      join = lv[k - 2].items.size() == lv[k - 1].items.size();
      for (size_t j = 0; join && j < lv[k - 1].items.size(); ++j) {
        const ChainItem &a = lv[k - 2].items[j], &b = lv[k - 1].items[j];
        join = a.Q == b.Q && a.out.size() == b.out.size();
        for (size_t o = 0; join && o < a.out.size(); ++o) join = a.out[o].staged == b.out[o].staged;
      }
    }
    if (!join) {
      if (first_of.size() >= (size_t)kChainMaxSections) return false;
      first_of.push_back(k);
      ChainSection s;
      s.items = lv[k].items;
      s.n_ptr = (int)lv[k].ptrs.size();
      c.sections.push_back(std::move(s));
    }
    ++c.sections.back().n_levels;
  }
  for (auto& m : c.mats) c.ptrs.push_back(m.ptr);
  for (size_t k = 0; k < c.sections.size(); ++k) {
    auto& s = c.sections[k];
    for (size_t j = 0; j < s.items.size(); ++j) {
      size_t n = 0;
      for (auto& in : s.items[j].in)
        if (in.kind == 1) { in.ptr = (int)c.ptrs.size(); c.ptrs.push_back(lv[first_of[k]].consts[j][n++]); }
    }
  }
  c.n_const = (int)c.ptrs.size();
  for (auto& L : lv) c.ptrs.insert(c.ptrs.end(), L.ptrs.begin(), L.ptrs.end());
  if (c.ptrs.size() > (size_t)kChainMaxPtrs) return false;
  // Roles: the weights that one product multiplies by belong together; those of the section that most levels are in get
  // wavefronts of their own, all others come with the first.
  {
    std::vector<int> family(c.mats.size());
    for (size_t m = 0; m < c.mats.size(); ++m) family[m] = (int)m;
    auto root = [&](int m) {
      while (family[(size_t)m] != m) m = family[(size_t)m];
      return m;
    };
    for (auto& s : c.sections)
      for (auto& it : s.items)
        for (auto& x : it.x) family[(size_t)root(x.mat)] = root(it.x[0].mat);
    const ChainSection* steady = &c.sections[0];
    for (auto& s : c.sections)
      if (s.n_levels > steady->n_levels) steady = &s;
    std::vector<std::pair<int64_t, int>> load;      // work of a family in that section
    for (auto& it : steady->items) {
      int64_t k = 0;
      for (auto& x : it.x) k += c.mats[(size_t)x.mat].K;
      size_t at = 0;
      while (at < load.size() && load[at].second != root(it.x[0].mat)) ++at;
      if (at == load.size()) load.push_back({0, root(it.x[0].mat)});
      load[at].first -= k * it.Q;
    }
    std::stable_sort(load.begin(), load.end());
    for (size_t m = 0; m < c.mats.size(); ++m)
      for (size_t r = 0; r < load.size(); ++r)
        if (load[r].second == root((int)m)) c.mats[m].role = (int)r;
    c.roles = (int)load.size();
  }
  // Columns per block: the fewest that let all blocks run at once, fewer when LDS or registers do not hold that many.  fp64 by lone
  // columns where one or two to a block are enough, two only where a wavefront has two row groups (with one, each column's program
  // leaves half of the lanes idle).  Gradients of two layers over 28 steps, groups of four / lone, us: 128 wide, batch 40 250 / 166, 150 244 / 156, 256
  // 255 / 164, 300 257 / 204, 500 275 / 225; 64 wide, batch 150 134 / 112, 512 149 / 158; 160 wide, 12 steps, batch 150 288 / 280.
  const int64_t groups = (c.P + 3) / 4;
  const int64_t rounds = (groups + 8 * (int64_t)num_cu - 1) / (8 * (int64_t)num_cu);
  // With a wavefront's registers and LDS too few for the weights of its own layer, every wavefront takes all layers.
  struct Form { bool lone; int nc, apart; };
  std::vector<Form> forms;
  if (c.f64 && lone)
    for (int nc = (int)((c.P + num_cu - 1) / num_cu); nc <= kChainMaxLone; ++nc)
      for (int apart = 1; apart >= 0; --apart) forms.push_back({true, nc, apart});
  for (int nc = (int)((groups + num_cu * rounds - 1) / (num_cu * rounds)); nc >= 1; --nc)
    for (int apart = 1; apart >= 0; --apart) forms.push_back({false, nc, apart});
  for (const Form& f : forms) {
    const bool apart = f.apart != 0;
    if (apart && c.roles == 1) continue;
    ChainPlan t = c;
    t.lone = f.lone;
    t.NC = f.nc;
    if (!share_wavefronts(t, apart)) continue;
    if (t.lone && t.NC > 1 && std::any_of(t.mats.begin(), t.mats.end(), [](const ChainMat& m) { return m.kept() && m.units < 2; })) continue;
    if (!place_weights(t, slack) || !pays(t, num_cu)) continue;
    // operands from inside the chain: where the level before put that result
    for (size_t k = 0; k < t.sections.size(); ++k) {
      // (the level before the section's first one, and within the section the section itself, which has the same layout)
      const ChainSection* before = k > 0 ? &t.sections[k - 1] : nullptr;
      for (auto& it : t.sections[k].items) {
        auto resolve = [&](int& off) {
          const int code = -1 - off;
          off = before->items[(size_t)(code / 8)].out[(size_t)(code % 8)].off;
        };
        for (auto& x : it.x) if (x.kind == 1) resolve(x.off);
        for (auto& in : it.in) if (in.kind == 2) resolve(in.off);
      }
    }
    c = std::move(t);
    return true;
  }
  return false;
}

// The chain's kernel, compiled once per key; nullptr when the compiler refuses it or keeps more than a few values in scratch
// memory (20 bytes a lane: 72.7 us for 71.4).
hipFunction_t chain_kernel(hgpu_ctx* ctx, const ChainPlan& plan) {
  auto& chains = known_of(ctx).chains;
  const Key key = chain_key(plan);
  char kname[80];
  snprintf(kname, sizeof kname, "smallk_chain_%s_p%lld_t%d_s%d", plan.f64 ? "f64" : "f32", (long long)plan.P, chain_columns(plan), (int)plan.sections.size());
  auto it = chains.find(key.bytes);
  if (it != chains.end()) {
    if (check_keys() && it->second.src != chain_source(plan, kname)) {
      fprintf(stderr, "hordead_gpu: two different kernels under one key (%s)\n", kname);
      if (!ctx->deferred_rc) ctx->deferred_rc = HGPU_ERR_DEVICE;
    }
    return it->second.fn;
  }
  KnownChain k;
  k.src = chain_source(plan, kname);
  std::vector<char> code;
  int rc = rtc_compile(ctx, k.src, "chain of small products", &code);
  const bool debug = getenv("HORDEAD_GPU_DEBUG") != nullptr;
  if (rc && debug) fprintf(stderr, "hordead_gpu: %s rejected: %s\n", kname, hgpu_last_error(ctx));
  if (!rc) {
    hipModule_t mod;
    int scratch = 0;
    hipError_t e = hipModuleLoadData(&mod, code.data());
    if (e == hipSuccess) e = hipModuleGetFunction(&k.fn, mod, kname);
    if (e == hipSuccess) e = hipFuncGetAttribute(&scratch, HIP_FUNC_ATTRIBUTE_LOCAL_SIZE_BYTES, k.fn);
    if (debug) fprintf(stderr, "hordead_gpu: %s: %d bytes of scratch memory\n", kname, scratch);
    if (e != hipSuccess || scratch > 64) k.fn = nullptr;
  }
  return chains.emplace(key.bytes, std::move(k)).first->second.fn;
}
