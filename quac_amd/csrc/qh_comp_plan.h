// qh_comp_plan.h -- the host-side choices of a closed-set plan (qh_comp.hip): which
// bins are stepped by which kernel.  Plain C++, without HIP.
#ifndef QH_COMP_PLAN_H
#define QH_COMP_PLAN_H
#include <algorithm>
#include <cstdint>
#include <vector>

const int CP_REG_ROWS = 2048;  // largest bin with its entries in registers (1024 threads, two rows each)
// largest bin: two buffers of rows + 1 entries (complex128, or complex64 for an FP32
// state) and the table in 160 KB of LDS, 6 or 8 rows a thread
const int CP_MAX_ROWS64 = 4800, CP_MAX_ROWS32 = 8128;
const int CP_DICT = 1024;  // values of a bin's table, zero among them

// the kernels k_comp_rk4<S, W, SKIP> that are built
#define CP_REG_KERNELS(X)                                                                        \
  X(1, 4, false) X(1, 8, false) X(1, 10, false) X(1, 12, false) X(1, 16, false) X(1, 24, false)  \
  X(1, 32, false) X(2, 4, false) X(2, 8, false) X(2, 10, false) X(2, 12, false)                  \
  X(1, 4, true) X(1, 8, true) X(1, 12, true) X(1, 16, true) X(1, 24, true) X(1, 32, true)        \
  X(2, 4, true) X(2, 8, true) X(2, 12, true)

// time of a stage in clocks of a CU: a slot of a slice is 64 LDS reads of 16 B (8
// clocks at 128 B a clock, 10 measured), as words 64 reads of the vector and of the
// table
const double CP_CLK_REG = 10.0, CP_CLK_WORD = 24.0, CP_CLK_FIXED = 500.0;

// Whether a stage of the plan (the largest bin's clocks, and all bins') beats the
// sliced stage kernels: 2.5 us a launch, and 11 us a million rows.
// Measured us a stage, here / there: Jaynes-Cummings 2 x 24 0.30 / 2.6, Tavis-Cummings
// 2^2 x 23 0.44 / 2.7, 2^3 x 17 1.00 / 3.5, 2^3 x 30 1.49 / 4.3, decay and dephasing of
// 7 qubits 0.34 / 2.8, 10 5.1 / 13.2, 12 46.7 / 243.  Refused: 2^4 x 8 (bins of 1768
// rows whose entries do not fit the registers) 5.0 / 3.3, 2^4 x 19 10.5 / 5.4, 6-qubit
// chain (one bin of 4096 rows) 10.9 / 3.0.
inline bool cp_worth(double most, double all, int64_t n, int cus) {
  const double comp_us = std::max(most, all / (double)cus + CP_CLK_FIXED) / 2400.0;
  return comp_us <= 0.9 * (2.5 + 1.1e-5 * (double)n);
}

// slots that a row holds for a slice of w slots: the kernels that pass over unfilled
// slots (many bins, or bins of several shapes) have no width of 10
inline int cp_width_class(int w, bool skip) {
  for (int u : {4, 8, 10, 12, 16, 24, 32})
    if (w <= u && !(skip && u == 10)) return u;
  return 0;
}

inline int cp_threads(int rows) {
  return rows <= 64 ? 64 : rows <= 128 ? 128 : rows <= 256 ? 256 : rows <= 512 ? 512 : 1024;
}

// two rows a thread: up to 12 slots each fit the 128 registers
inline bool cp_fits_registers(int rows, int W) { return W && (rows <= 1024 || (rows <= CP_REG_ROWS && W <= 12)); }

// clocks of a stage of a bin of so many rows at the least: w, the entries off the
// diagonal of a row on average
inline double cp_least(int64_t rows, double w) {
  return (rows <= CP_REG_ROWS ? CP_CLK_REG : CP_CLK_WORD) * std::max(0.0, w) * (double)rows / 64.0 + CP_CLK_FIXED;
}

// one launch: bins of one shape
struct CpClass {
  int threads, S, W;  // W 0: entries read as words
  bool skip, side;    // side: few blocks, launched beside the others
  int first, count;   // range of the plan's bin list
  int cells;          // entries of one LDS buffer
};

inline bool cp_has_kernel(const CpClass &c) {
#define CP_HAS(SS, WW, SK) || (c.S == SS && c.W == WW && c.skip == SK)
  return c.W == 0 CP_REG_KERNELS(CP_HAS);
#undef CP_HAS
}

// a bin: its rows in whole slices of 64, the slots of its widest slice and of all
struct CpBin {
  int rows, width;
  int64_t slots;
};

// what the bins are stepped by
struct CpShapes {
  std::vector<uint8_t> words;         // per bin: entries read as words
  std::vector<CpClass> classes;       // the launches, the one of words first
  std::vector<int32_t> bins;          // all bins in the order of the launches
  double most = 0.0, all = 0.0;       // clocks of a stage: the largest bin, all bins
  bool runnable = true;               // every launch has a kernel
  // the launches of a call of up to brief_steps steps: words, and all other bins in one
  std::vector<CpClass> brief;
  int64_t brief_steps = 0;
};

// wavefronts that a CU holds of a class's kernel (its registers), as workgroups
inline double cp_resident(const CpClass &c) {
  const int waves = c.W == 0 || c.S > 1 || c.W > 12 ? 16 : c.W > 8 ? 20 : 32;
  return (double)waves * 64.0 / c.threads;
}

// Bins of several shapes each have their launch, and launches run one after the other or
// wait for a stream beside: 6 to 8 us each, whatever the steps.  In one launch of the
// largest shape small bins hold more wavefronts than they need, and fewer bins run at a
// time.  The line lies where that costs as much as 3 us a launch saved (half of what a
// launch costs, so that a call of more steps is not slowed down where the estimate is off).
// Measured us a call, several launches / one, for 1, 5 and 20 steps: decay and dephasing of
// 8 qubits 45 / 8, 50 / 13, 94 / 30; 9 qubits 58 / 24, 62 / 47, 122 / 132; 10 qubits 80 / 42,
// 124 / 85, 315 / 250; 11 qubits 180 / 192, 263 / 371, 764 / 1082 (several always).
inline void cp_brief(CpShapes &s, const std::vector<CpBin> &bin, int cus) {
  CpClass one{0, 0, 0, true, false, -1, 0, 0};
  double apart = 0.0, together = 0.0, reads = 0.0;  // clocks of a stage of all CUs
  for (const CpClass &k : s.classes) {
    if (k.W == 0) {
      s.brief.push_back(k);
      s.brief.back().side = false;
      continue;
    }
    if (one.first < 0) one.first = k.first;
    one.threads = std::max(one.threads, k.threads);
    one.S = std::max(one.S, k.S);
    one.W = std::max(one.W, k.W);
    one.cells = std::max(one.cells, k.cells);
    one.count += k.count;
  }
  if (one.count == 0 || !cp_has_kernel(one) || s.brief.size() + 1 >= s.classes.size()) {
    s.brief.clear();
    return;
  }
  for (const CpClass &k : s.classes) {
    if (k.W == 0) continue;
    for (int i = 0; i < k.count; i++) {
      const double clk = CP_CLK_REG * (double)bin[s.bins[k.first + i]].slots;
      reads += clk;
      apart += (clk + CP_CLK_FIXED) / cp_resident(k);
      together += (clk + CP_CLK_FIXED) / cp_resident(one);
    }
  }
  const double more_us = 4.0 * (std::max(together, reads) - std::max(apart, reads)) / cus / 2400.0;
  const double saved_us = 3.0 * (double)(s.classes.size() - s.brief.size() - 1);
  s.brief.push_back(one);
  s.brief_steps = more_us <= 0.0 ? INT64_MAX : (int64_t)std::min(1e9, saved_us / more_us);
}

inline CpShapes cp_shapes(const std::vector<CpBin> &bin, bool f32, int cus) {
  CpShapes out;
  const int n = (int)bin.size();
  // Where the chip is not full, all bins that fit registers go into one launch, so that
  // nothing waits for a launch before it; a large bin beside a wide one has no kernel in
  // common with it, and then each shape has its launch as where there are many bins.
  bool merge = n <= 2 * cus;
  int few_rows = 0, few_w = 0;
  if (merge) {
    for (const CpBin &b : bin) {
      const int W = cp_width_class(b.width, false);
      if (!cp_fits_registers(b.rows, W)) continue;
      few_rows = std::max(few_rows, b.rows <= 1024 ? cp_threads(b.rows) : b.rows);
      few_w = std::max(few_w, W);
    }
    merge = cp_fits_registers(few_rows, few_w) || few_w == 0;
  }
  struct Shape {
    int words, rows, W;
    int32_t bin;
  };
  std::vector<Shape> sh(n);
  out.words.resize(n);
  for (int b = 0; b < n; b++) {
    int W = cp_width_class(bin[b].width, !merge);
    const bool reg = cp_fits_registers(bin[b].rows, W);
    const double clk = reg ? CP_CLK_REG * W * (bin[b].rows / 64) : CP_CLK_WORD * (double)bin[b].slots;
    out.most = std::max(out.most, clk + CP_CLK_FIXED);
    out.all += clk;
    out.words[b] = !reg;
    int rows = bin[b].rows <= 1024 ? cp_threads(bin[b].rows) : bin[b].rows;
    if (reg && merge) {
      rows = few_rows;
      W = few_w;
    }
    sh[b] = Shape{!reg, rows, W, b};
  }
  std::stable_sort(sh.begin(), sh.end(), [](const Shape &p, const Shape &q) {
    if (p.words != q.words) return p.words > q.words;
    const int pr = p.words || p.rows > 1024 ? 1 << 20 : p.rows, qr = q.words || q.rows > 1024 ? 1 << 20 : q.rows;
    if (pr != qr) return pr > qr;
    return !p.words && p.W > q.W;
  });
  out.bins.resize(n);
  for (int i = 0; i < n; i++) {
    const Shape &q = sh[i];
    out.bins[i] = q.bin;
    const int S = q.words ? (f32 ? 8 : 6) : q.rows > 1024 ? 2 : 1, threads = q.words || S == 2 ? 1024 : q.rows;
    const int W = q.words ? 0 : q.W;
    if (out.classes.empty() || out.classes.back().threads != threads || out.classes.back().S != S ||
        out.classes.back().W != W)
      out.classes.push_back(CpClass{threads, S, W, !merge, false, i, 0, 0});
    CpClass &k = out.classes.back();
    k.count++;
    k.cells = std::max(k.cells, bin[q.bin].rows + 1);
  }
  for (CpClass &k : out.classes) {
    if (out.classes.size() > 1 && k.count < cus && k.first + k.count < n) k.side = true;
    if (!cp_has_kernel(k)) out.runnable = false;
  }
  cp_brief(out, bin, cus);
  return out;
}

// Time in us that a plan of a matrix of n rows takes to form (one workgroup up to
// 16 384 rows): measured 55 at 1296 rows, 78 at 4096, 140 at 8464, 200 at 16 384, 258 at
// 18 496, 370 at 65 536, 1350 at 1 M, 3300 at 4 M; a refused one costs up to that.
inline double cp_plan_us(int64_t n) {
  const double r = (double)n;
  if (n <= 16384) return 45.0 + 0.0105 * r;
  return 230.0 + 0.0023 * std::min(r, 65536.0) + 0.0008 * std::max(0.0, r - 65536.0);
}

// Whether a call of nsteps steps forms the plan, seen steps of the matrix having run on
// the stage kernels: where these steps there would take as long (their part that the
// plan saves, the captured graph of a call of graph_len steps or more, and the sliced
// layout where it is still to be built).  So a matrix that is stepped a few times never
// waits for a plan, and one that is stepped often waits at most twice as long as it must.
// First call, plan / stage kernels once their variant is known, for 1, 5 and 20 steps:
// Tavis-Cummings 2^2 x 23 151 / 41, 150 / 90, 166 / 393 us; 2^3 x 17 268 / 51, 283 / 110,
// 312 / 475 us.
inline bool cp_pays(int64_t n, int64_t seen, int64_t nsteps, int graph_len, bool layout) {
  const double step_us = 4.0 * (2.5 + 1.1e-5 * (double)n);
  const double stage_us = 0.75 * step_us * ((double)seen + (double)nsteps) + (nsteps >= graph_len ? 250.0 : 0.0) +
                          (layout ? 0.0 : 100.0 + 0.0012 * (double)n);
  return stage_us >= cp_plan_us(n);
}

// All launches of a plan: fork() before the first where some run on the side stream,
// launch(class) each, and join() after them, also when a launch fails: the caller's
// stream never goes on while the side stream still writes the state.
template <typename Launch, typename Fork, typename Join>
int cp_run(const std::vector<CpClass> &classes, Launch &&launch, Fork &&fork, Join &&join) {
  bool side = false;
  int rc = 0;
  for (const CpClass &k : classes) side = side || k.side;
  if (side && (rc = fork())) return rc;
  for (const CpClass &k : classes)
    if ((rc = launch(k))) break;
  const int jrc = side ? join() : 0;
  return rc ? rc : jrc;
}

#endif
