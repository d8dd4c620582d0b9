#include "tc/core/mapper/mapper.h"
#include "tc/core/mapper/sync_placement.h"

#include <limits>
#include <algorithm>
#include <cctype>
#include <cmath>
#include <cstdio>
#include <functional>
#include <set>
#include <sstream>

#include "tc/core/check.h"
#include "tc/core/hip/hip_column_sums.h"
#include "tc/core/hip/hip_libraries.h"
#include "tc/core/hip/hip_split_products.h"

namespace tc {
namespace mapper {
namespace {

using ir::Affine;
using ir::Expr;
using ir::ExprRef;
using ir::ReduceOp;
using ir::ScalarType;

// ------------------------------------------------------------------------------------------
// expression helpers
// ------------------------------------------------------------------------------------------
ExprRef mkExpr(Expr::Kind k, ScalarType t, std::string name, std::vector<ExprRef> args) {
  auto e = std::make_shared<Expr>();
  e->kind = k;
  e->type = t;
  e->name = std::move(name);
  e->args = std::move(args);
  return e;
}
ExprRef mkInt(int64_t v) {
  auto e = std::make_shared<Expr>();
  e->kind = Expr::IntImm;
  e->type = ScalarType{ScalarType::Int, 32};
  e->ival = v;
  return e;
}
ExprRef mkVar(const std::string& n) {
  return mkExpr(Expr::Var, ScalarType{ScalarType::Int, 32}, n, {});
}
ExprRef mkBin(const std::string& op, ExprRef a, ExprRef b) {
  return mkExpr(Expr::Binary, ScalarType{ScalarType::Int, 32}, op, {std::move(a), std::move(b)});
}

// Rebuilds `e` bottom-up; `fn` may return a replacement for a node (after its children were
// rewritten) or nullptr to keep it.
ExprRef rewrite(const ExprRef& e, const std::function<ExprRef(const ExprRef&)>& fn) {
  std::vector<ExprRef> args;
  bool changed = false;
  for (const auto& a : e->args) {
    ExprRef n = rewrite(a, fn);
    changed |= n != a;
    args.push_back(n);
  }
  ExprRef cur = e;
  if (changed) {
    auto c = std::make_shared<Expr>(*e);
    c->args = std::move(args);
    cur = c;
  }
  ExprRef r = fn(cur);
  return r ? r : cur;
}

void visit(const ExprRef& e, const std::function<void(const ExprRef&)>& fn) {
  fn(e);
  for (const auto& a : e->args) {
    visit(a, fn);
  }
}

// Visits only what every evaluation of `e` evaluates: not the branches of a select and not the
// right-hand side of a short-circuit operator.  A load found this way may be issued ahead of the
// expression; one guarded by a condition may address outside its tensor when the guard is false.
void visitUnconditional(const ExprRef& e, const std::function<void(const ExprRef&)>& fn) {
  fn(e);
  size_t n = e->args.size();
  if (e->kind == Expr::Select) n = 1;
  if (e->kind == Expr::Binary && (e->name == "&&" || e->name == "||")) n = 1;
  for (size_t i = 0; i < n; ++i) {
    visitUnconditional(e->args[i], fn);
  }
}

bool sameExpr(const ExprRef& a, const ExprRef& b) {
  if (a->kind != b->kind || a->name != b->name || a->ival != b->ival || a->fval != b->fval ||
      a->args.size() != b->args.size() || a->type != b->type) {
    return false;
  }
  for (size_t i = 0; i < a->args.size(); ++i) {
    if (!sameExpr(a->args[i], b->args[i])) {
      return false;
    }
  }
  return true;
}

ScalarType matchType(const ScalarType& a, const ScalarType& b) {
  if (a == b) return a;
  if (!a.isFloat() && b.isFloat()) return b;
  if (a.isFloat() && !b.isFloat()) return a;
  if (a.isFloat() && b.isFloat()) return a.bits > b.bits ? a : b;
  if (a.code == ScalarType::UInt && b.code == ScalarType::UInt) return a.bits > b.bits ? a : b;
  return ScalarType{ScalarType::Int, std::max(a.bits, b.bits)};
}

std::string floatLiteral(double v, const ScalarType& t) {
  char buf[64];
  std::snprintf(buf, sizeof(buf), t.bits == 64 ? "%.17g" : "%.9g", v);
  std::string s = buf;
  if (s.find_first_of(".en") == std::string::npos) {
    s += ".0";
  }
  if (s.find("inf") != std::string::npos || s.find("nan") != std::string::npos) {
    return v > 0 ? "(1.0f/0.0f)" : "(-1.0f/0.0f)";
  }
  return t.bits == 64 ? s : t.bits == 16 ? "((_Float16)" + s + "f)" : s + "f";
}

int64_t ceilDiv(int64_t a, int64_t b) {
  return (a + b - 1) / b;
}

const char* axisName(int a) {
  return a == 0 ? "x" : a == 1 ? "y" : "z";
}

#include "tc/core/mapper/stage_builder.h"
#include "tc/core/mapper/stage_codegen.h"

// ------------------------------------------------------------------------------------------
// mapping of one kernel
// ------------------------------------------------------------------------------------------
// Whether a tile of reduction variable `k` may reach past its extent: in both operands of the
// contraction `k` alone moves one subscript, in steps of one, so that the surplus points of the last
// tile are whole rows or columns of the footprint, which the staging copies fill with zeros.
bool reductionMayEndInMidTile(const StagePlan& st, const std::string& k) {
  // A tile of whole matrix-core steps, four points of the flattened reduction each, and at least four
  // steps deep: every tile costs a barrier and a round through LDS, which two steps do not repay
  // (a 1x1 convolution over 52 channels in tiles of 8: 6.2 us, untiled 3.9; a product of depth 249
  // in tiles of 32: 4.4 us, untiled 12.5).
  int64_t depth = 1;
  for (size_t i = 0; i < st.mfmaK.size(); ++i) {
    for (const auto& v : st.vars) {
      if (v.name == st.mfmaK[i]) depth *= i == 0 ? v.tile : v.extent;
    }
  }
  if (depth % 4 != 0 || depth < 16) return false;
  for (const auto& operand : st.stmts[0].rhs->args) {
    const ExprRef load = contractionOperand(operand);
    int found = 0;
    for (const auto& sub : load->args) {
      Affine a = ir::toAffine(sub);
      if (a.coefOf(k) == 0) continue;
      ++found;
      if (a.coefOf(k) != 1) return false;
      for (const auto& c : a.coef) {
        if (c.first == k || c.second == 0) continue;
        // (another variable moves the origin of the footprint, not its extent, only when a block
        // holds one point of it)
        for (const auto& v : st.vars) {
          if (v.name == c.first && (v.reduction || v.tile != 1)) return false;
        }
      }
    }
    if (found != 1) return false;
  }
  return true;
}

// Products of halves are multiplied 32 points of the reduction an instruction (eight per lane), and
// the rotated pipeline cuts a tile in two: tiles of 32 points are made 64 deep where both operands
// still fit in LDS twice, two tiles at least and every wavefront with an output tile of its own.  Rows
// of a copy are then 128 bytes, and the tile is not left on the instruction of half the rate
// (4096^3, 128x256x32, second operand transposed 211 -> 157 us and plain 253 -> 158; 512x2048x768,
// 64x64x32: 14.1 -> 11.5 and 20.8 -> 11.5).  Not where the deeper tiles multiply an eighth more
// points than the given ones and a block holds more than 64x64 outputs, which a deeper tile serves
// least (1024x1024, 128x128x32, second operand transposed: depth 224 as 4 tiles of 64 5.8 us, as 7 of
// 32 5.2; depth 288 6.2 and 5.9, before 6.9; 64x64x32 of depth 224 3.6 and 3.5).  The planning of the
// copies returns to the given tile when they turn out not to fit twice.
void deepenHalfTile(StagePlan& st, LoopVar& v, const HipMappingOptions& o, int64_t waves, const DeviceLimits& limits) {
  if (!o.prefetchSharedValue || !o.useSharedMemoryValue || st.mfmaK.size() != 1 || !st.mfmaBatch.empty()) return;
  for (const auto& operand : st.stmts[0].rhs->args) {
    if (st.views.at(contractionOperand(operand)->name).type.bits != 16) return;
  }
  const int64_t depth = 64, given = v.tile;
  if (given != depth / 2 || v.extent < 2 * depth) return;
  int64_t rows = 1, columns = 1;
  for (const auto& w : st.vars) {
    for (const auto& n : st.mfmaM) rows *= w.name == n ? w.tile : 1;
    for (const auto& n : st.mfmaN) columns *= w.name == n ? w.tile : 1;
  }
  int64_t lds = limits.ldsBytesPerBlock;
  if (o.hasMaxSharedMemory) lds = std::min<int64_t>(lds, o.maxSharedMemoryValue);
  if (rows * columns < 256 * waves || 2 * 2 * (rows + columns) * (depth + 8) > lds) return;
  if (rows * columns > 64 * 64 && 8 * depth * ceilDiv(v.extent, depth) > 9 * given * ceilDiv(v.extent, given)) return;
  v.tile = depth;
  v.numTiles = ceilDiv(v.extent, depth);
  st.givenReductionTile = given;
  if (v.extent % depth != 0 && !reductionMayEndInMidTile(st, v.name)) {
    v.tile = given;
    v.numTiles = ceilDiv(v.extent, given);
    st.givenReductionTile = 0;
  }
}

// Blocks that the options allow a variable on block axis `axis`.  A variable with a single tile uses up no axis, so the ones
// behind it move up; a variable's size is the one of its place among the options' sizes (`position`, among the
// parallel variables of the kernel, lanes of a vector left out) as well as that of the axis it moves up to (one image of 11
// groups under mapToBlocks=1,11: on one block 115 us, on eleven 11.5).  The size of a place counts up to 65535: on the second
// and third axis, which any variable may end up on, a launch takes no more.
int64_t allowedBlocks(const HipMappingOptions& o, int axis, int position) {
  constexpr uint64_t kMostAcross = 65535;
  uint64_t blocks = o.grid[axis];
  if (position < static_cast<int>(o.grid.size())) blocks = std::max<uint64_t>(blocks, std::min<uint64_t>(o.grid[position], kMostAcross));
  return static_cast<int64_t>(std::min<uint64_t>(blocks, std::numeric_limits<int32_t>::max()));
}

// A matrix-core stage whose blocks leave compute units idle: a block-mapped variable gets the smaller tile
// that shortens the longest-running compute unit by a quarter or more, if there is one, and then another one (compute units
// are those of the device, or of its partition).  A compute unit's time is its rounds of blocks times the output tiles
// of the busiest wavefront, or its share of one where wavefronts divide the reduction, and about two more for a block's staging.
//   Convolutions: any smaller number of rows, whole sixteens of filters (3x3 of 16x64x57x57, 64 filters: 160 blocks of 10
// tiles a wavefront 55.5 us, 256 of 7 46.0, 320 of 6 in two rounds 63.9; 13x83x7x38, 38 filters: 26 blocks of 32 filters x 5 rows
// 28.0 us, 130 of one row 12.0; 1x1 of 4x118x30x38, 21 filters: 8 blocks of 15 rows 20.0, 120 of one 4.2).  Floats only.
//   Products of eight reduction tiles and more: sides of half the length and more whose output tiles divide into rectangles for the
// wavefronts (halves: of half the length), already for a fifth (881x655x2389: 133 blocks of 128x128 47.8 us, 210 of 128x80 38.3, 228 of 80x128
// 35.9; 1500x800x1700: 168 blocks 56.8, 224 of 96x128 46.8; 215x1188x1305: 84 blocks of 64x64 24.2 us, 164 of 64x32 14.8, 287 of 32x32 21.9; 430x1367x1095 27.2 and 18.1; halves
// 322x2061x993 17.9 and 13.6; where the halves make two rounds there is nothing to gain: 691x1840x792, 143 blocks, 35.7, 36.1).
//   Products whose blocks make a second round for a few: a side up to half as long again under which there is one, where the
// estimate says 13 / 20 of the time or less (2100x900x2100: 289 blocks of 128x128 117.7 us, 255 of 144x128 85.2; 1100x2000x1100: 324 of 64x64 72.6,
// 216 of 96x64 61.7; 1400x600x1100, three quarters: 396 of 64x64 25.8, 198 of 128x64 26.9).
//   Products whose wavefronts share the reduction of a tile, on half the compute units or fewer: half the longer side, as the
// staging of a block is what takes the time (116x2960x204: 56 blocks of 16x32 14.6 us, 104 of 16x16 9.5; 108x1643x127 7.8 and 6.1;
// 128x1000x1024, 256 blocks, 6.1 and 9.9).
//   Of a product's two sides that come out alike the second is taken, a long one unless it makes clearly fewer blocks.  Measured
// on 70 products that leave the choice: tiles of 64x64 and of halves are as fast either way (3 % at most, the mean the same);
// in tiles of 128x128 the first side was 2 to 11 % faster in all eight (1789x2010x1391: 252 blocks of 128x80 104.5 us, 253 of
// 80x128 93.2; 1883x157x1271, 240 blocks either way, 16.9 and 15.3).
// mapToBlocks sizes that hold exactly the given tiles keep those tiles, as maxSharedMemory keeps those of products.
void fillComputeUnits(const KernelPlan& k, StagePlan& st, const HipMappingOptions& o, int64_t waves, int64_t computeUnits) {
  constexpr int64_t kStaging = 2, kLongReduction = 8, kLongSidesLds = 64 << 10;
  if (k.stages.size() != 1 || !o.prefetchSharedValue || !o.useSharedMemoryValue || !st.mfmaBatch.empty()) return;
  const bool product = st.mfmaM.size() + st.mfmaN.size() == 2;
  bool halves = false;
  for (const auto& operand : st.stmts[0].rhs->args) halves |= st.views.at(contractionOperand(operand)->name).type.bits != 32;
  if (product ? o.hasMaxSharedMemory : halves) return;
  int64_t points = 1; // of a reduction tile
  int position = 0;
  for (const auto& v : st.vars) {
    if (v.reduction && v.name == st.mfmaK[0]) {
      // (a reduction the options do not tile has its operands staged whole)
      const bool given = o.generic.hasTiling && position < static_cast<int>(o.generic.tiling.size()) && o.generic.tiling[position] > 0;
      if (!given) return;
      const bool tiled = v.numTiles > 1 && (v.extent % v.tile == 0 || reductionMayEndInMidTile(st, v.name));
      if (product && (!tiled || v.numTiles < kLongReduction)) return;
      points *= tiled ? v.tile : v.extent;
    } else if (v.reduction) {
      points *= v.extent;
    }
    if (!v.vectorLane) ++position;
  }
  auto mayBeSplit = [&](int i) { return i < k.sharedDepth && !st.vars[i].vectorLane; };
  auto inRectangles = [&](int64_t rowTiles, int64_t columnTiles) {
    for (int64_t wm = 1; wm <= waves; ++wm) {
      if (waves % wm == 0 && rowTiles % wm == 0 && columnTiles % (waves / wm) == 0) return true;
    }
    return false;
  };
  // in units of 1 / waves of an output tile; 0: not a form this speaks of
  bool byAxis = true; // (sizes that hold the given tiles axis by axis are those of the axes)
  bool onGrid = false, fewTiles = false; // (every tile has a block; fewer output tiles than wavefronts)
  auto cost = [&](int64_t& blocks) -> int64_t {
    blocks = 1;
    onGrid = fewTiles = false;
    int axis = 0, position = -1;
    for (int i = 0; i < st.numParallel; ++i) {
      if (!st.vars[i].vectorLane) ++position;
      if (st.vars[i].numTiles == 1) continue;
      if (!mayBeSplit(i) || axis >= static_cast<int>(o.grid.size())) return 0;
      if (st.vars[i].numTiles > (byAxis ? allowedBlocks(o, axis, axis) : allowedBlocks(o, axis, position))) return 0;
      blocks *= st.vars[i].numTiles;
      ++axis;
    }
    int64_t rows = 1, columns = 1;
    for (const auto& w : st.vars) {
      for (const auto& n : st.mfmaM) rows *= w.name == n ? w.tile : 1;
      for (const auto& n : st.mfmaN) columns *= w.name == n ? w.tile : 1;
    }
    const int64_t tiles = ceilDiv(rows, 16) * ceilDiv(columns, 16);
    onGrid = true;
    fewTiles = tiles < waves;
    if (product && (tiles < waves || !inRectangles(ceilDiv(rows, 16), ceilDiv(columns, 16)))) return 0;
    const int64_t shared = std::max<int64_t>(1, std::min(waves / tiles, points / 4 / StageCodegen::kMinStepsPerSplit));
    const int64_t work = tiles >= waves ? waves * ceilDiv(tiles, waves) : ceilDiv(waves, shared);
    return ceilDiv(blocks, computeUnits) * (work + kStaging * waves);
  };
  auto setTile = [&](LoopVar& v, int64_t tile) {
    v.tile = tile;
    v.numTiles = ceilDiv(v.extent, tile);
  };
  int64_t blocks = 0;
  cost(blocks);
  byAxis = onGrid;
  const int64_t given = cost(blocks);
  if (product && !halves && fewTiles && 2 * blocks <= computeUnits) {
    LoopVar* longer = nullptr;
    for (int i = 0; i < st.numParallel; ++i) {
      LoopVar& v = st.vars[i];
      if (mayBeSplit(i) && v.tile % 32 == 0 && (!longer || v.tile >= longer->tile)) longer = &v;
    }
    if (!longer) return;
    const int64_t tile = longer->tile;
    setTile(*longer, tile / 2);
    cost(blocks);
    if (blocks > computeUnits || !onGrid) setTile(*longer, tile);
    else st.fittedToDevice = true;
    return;
  }
  if (product && !halves && blocks > computeUnits && given > 0) {
    LoopVar* best = nullptr;
    int64_t bestTile = 0, bestCost = given;
    for (int i = 0; i < st.numParallel; ++i) {
      if (!mayBeSplit(i)) continue;
      LoopVar& v = st.vars[i];
      const int64_t tile = v.tile;
      for (int64_t t = tile + 16; tile % 16 == 0 && 2 * t <= 3 * tile; t += 16) {
        setTile(v, t);
        int64_t n = 0, sides = 0;
        const int64_t c = cost(n);
        for (int j = 0; j < st.numParallel; ++j) sides += st.vars[j].tile;
        const bool fits = sides * (points + 4) * 4 * 2 <= kLongSidesLds;
        if (fits && c > 0 && n <= computeUnits && c < bestCost) {
          best = &v;
          bestTile = t;
          bestCost = c;
        }
      }
      setTile(v, tile);
    }
    if (best && 20 * bestCost <= 13 * given) {
      setTile(*best, bestTile);
      st.fittedToDevice = true;
    }
    return;
  }
  for (int round = 0; round < 2; ++round) {
    int64_t blocks = 0;
    const int64_t given = cost(blocks);
    if (given == 0 || blocks >= computeUnits) return;
    int best = -1;
    int64_t bestTile = 0, bestCost = given, bestBlocks = 0;
    for (int i = 0; i < st.numParallel; ++i) {
      if (!mayBeSplit(i)) continue;
      LoopVar& v = st.vars[i];
      const int64_t tile = v.tile, step = product && halves ? tile / 2 : product || tile > 16 ? 16 : 1;
      if (product && tile % (halves ? 32 : 16) != 0) continue;
      for (int64_t t = (tile - 1) / step * step; t > 0 && (!product || 2 * t >= tile); t -= step) {
        setTile(v, t);
        int64_t n = 0;
        const int64_t c = cost(n);
        // (as long, of less work: the smaller tile; of a product's two sides the second, if not a long one of clearly fewer blocks)
        if (c > 0 && (c < bestCost || (c == bestCost && best >= 0 && (best == i || (product && (tile <= 64 || halves || 20 * n >= 19 * bestBlocks)))))) {
          best = i;
          bestTile = t;
          bestCost = c;
          bestBlocks = n;
        }
      }
      setTile(v, tile);
    }
    if (best < 0 || (product && !halves ? 5 * bestCost > 4 * given : 4 * bestCost > 3 * given)) return;
    setTile(st.vars[best], bestTile);
    st.fittedToDevice = true;
  }
}

// Products of float16 matrices O(m, n) +=! A * B whose outputs fill the device in blocks of 256 x 256 go to
// __tc::largeHalfProduct (hip_libraries.h), whichever side of the operands the reduction is on: a block multiplies
// more per value it reads from LDS than one of the given tiles.  Where the blocks leave compute units idle
// the given tiles stay; so they do in other than 8 wavefronts, on other grids than one block a tile, without
// shared memory or prefetchShared, where maxSharedMemory is below the 128 KB of the copies, for rows that are no whole
// number of 16-byte vectors, and for reductions of fewer than 256 points.
// Rounds of blocks x outputs of a block are compared.  Per output the large blocks take 0.5 to 0.7 of the time of
// 128x256 ones and 0.4 to 0.6 of 128x128 ones, so they may compute a third more outputs, and twice as many where they occupy
// 7/16 of the compute units (48 products of 800 to 4096 rows and columns, depths 256 to 4096, given / large: as many 1.3 to
// 1.9, a third more 1.7 and 1.9, twice as many 1.01 to 1.32 from 112 blocks and 0.82 to 0.97 of 80 to 91, four times 0.5 to 0.65).
// Twice as many pay for a deep reduction only, or one that ends inside a tile of 64 points, which costs the given tiles more:
// given / large of 112 to 128 blocks at depth 264 to 360 0.95 to 1.15, 392 to 840 1.02 to 1.30; whole tiles, an even number of them: 256
// 0.88 to 0.99, 384 1.04 to 1.08 where the given blocks leave a seventh of the compute units idle (1808x3688) and 0.92 to 1.02
// where they do not, 512 to 1024 1.02 to 1.27; an odd number, which the given tiles take faster: 320 0.83 to 0.95, 448 to 1088
// 0.86 to 1.02 (only 1808x3688, A * B, 1.01 to 1.15), 1344 0.96 to 1.16, 1984 1.0 to 1.2.  (Operands off 16-byte boundaries
// are not known here: 2 bytes off, twice as many take 0.9 of the given tiles' speed at depths from 768, 0.8 of it at less.)
constexpr int64_t kLargeHalfBlock = 256, kLargeHalfLds = 2 * 2 * 256 * 64 * 2;
void takeLargeHalfProduct(KernelPlan& k, StagePlan& st, const HipMappingOptions& o, int64_t waves, const DeviceLimits& limits, bool wide) {
  if (k.stages.size() != 1 || wide || waves != 8 || !o.prefetchSharedValue || !o.useSharedMemoryValue || st.atomic) return;
  int64_t lds = limits.ldsBytesPerBlock;
  if (o.hasMaxSharedMemory) lds = std::min<int64_t>(lds, o.maxSharedMemoryValue);
  if (lds < kLargeHalfLds || st.stmts.size() != 1 || !st.stmts[0].init || st.vars.size() != 3 || st.numParallel != 2 || st.lhsSubs.size() != 2) return;
  const LoopVar &m = st.vars[0], &n = st.vars[1], &r = st.vars[2];
  for (const auto& v : st.vars) {
    if (v.min != 0) return;
  }
  auto isVar = [](const ExprRef& e, const LoopVar& v) { return e->kind == Expr::Var && e->name == v.name; };
  auto isMatrix = [&](const std::string& tensor, int64_t rows, int64_t columns) {
    const auto& view = st.views.at(tensor);
    return view.extents.size() == 2 && view.extents[0] == rows && view.extents[1] == columns &&
        rows * columns * view.type.bytes() < (int64_t(1) << 31);
  };
  if (!isVar(st.lhsSubs[0], m) || !isVar(st.lhsSubs[1], n) || !isMatrix(st.tensor, m.extent, n.extent)) return;
  std::string tensors[2];  // of the m and of the n side
  bool innermost[2];       // the reduction is the last subscript
  for (const auto& operand : st.stmts[0].rhs->args) {
    const ExprRef load = contractionOperand(operand);
    if (st.views.at(load->name).type.bits != 16 || load->args.size() != 2) return;
    bool found = false;
    for (int side = 0; side < 2; ++side) {
      const LoopVar& v = side == 0 ? m : n;
      for (int last = 0; last < 2; ++last) {
        const LoopVar &outer = last ? v : r, &inner = last ? r : v;
        if (!isVar(load->args[0], outer) || !isVar(load->args[1], inner)) continue;
        if (!isMatrix(load->name, outer.extent, inner.extent) || inner.extent % 8 != 0 || !tensors[side].empty()) return;
        tensors[side] = load->name;
        innermost[side] = last == 1;
        found = true;
      }
    }
    if (!found) return;
  }
  if (r.extent < 256) return;
  const int64_t numTiles[2] = {m.numTiles, n.numTiles};
  int axis = 0;
  for (int position = 0; position < 2; ++position) {
    if (numTiles[position] == 1) continue;
    if (axis >= static_cast<int>(o.grid.size()) || numTiles[position] > allowedBlocks(o, axis, position)) return;
    ++axis;
  }
  const int64_t blocks = ceilDiv(m.extent, kLargeHalfBlock) * ceilDiv(n.extent, kLargeHalfBlock);
  const int64_t tiles = m.numTiles * n.numTiles, rounds = ceilDiv(tiles, limits.computeUnits);
  const int64_t given = rounds * m.tile * n.tile;
  const int64_t large = ceilDiv(blocks, limits.computeUnits) * kLargeHalfBlock * kLargeHalfBlock;
  const bool idle = 7 * tiles <= 6 * rounds * limits.computeUnits; // (a seventh of the given blocks' rounds)
  const bool deep = r.extent % 64 != 0 || (r.extent % 128 == 0 ? r.extent >= (idle ? 384 : 512) : r.extent >= 1344);
  if (3 * large > 4 * given && (large > 2 * given || 16 * blocks < 7 * limits.computeUnits || !deep)) return;
  std::ostringstream ss;
  ss << (innermost[0] ? "true" : "false") << ", " << (innermost[1] ? "true" : "false") << ", " << m.extent << ", " << n.extent << ", " << r.extent
     << ">(p" << st.tensor << ", p" << tensors[0] << ", p" << tensors[1];
  st.largeHalfProduct = ss.str();
  k.grid = {{blocks, 1, 1}};
  k.block = {{64, waves, 1}};
}

// Convolutions of floats O(n, g, f, h, w) +=! I(n, g, c, h + kh, w + kw) * W1(g, f, c, kh, kw), with or without the group and
// a statement that adds a bias B(g, f) behind them, go to __tc::SplitConvolution (hip_split_products.h) where that is the faster
// form.  Both forms are judged by an estimate in microseconds, fitted by least squares of the relative error to measured times of 120 convolutions
// (1 to 64 images, 3 to 128 channels, 4 to 128 filters, planes of 7 x 7 to 64 x 64, windows of 1, 3 and 5; 7 to 16 shapes of the split form
// each): 11 % off on average for the split form, 16 % for the given tiles.
// The shape the estimate takes is 2 % slower than the best one timed on average, a quarter at most.  The split form is taken where it comes
// out 15 % faster, 40 % without groups, and half as fast again where an output has fewer than 48 terms (the results' stores bound such a kernel, and the general
// pipeline has less in front of them).  Without groups and with a window of one point the estimate of the given tiles is too high below 96 channels:
// 12 x 60 x 43 x 22, 60 filters, 4.0 us as given and 5.1 split, 9 x 29 x 31 x 23, 119 filters, 3.9 and 4.9, and they keep them.  With 15 % for all, 12 of 80 drawn
// convolutions without groups were slower (27 x 8 x 46 x 59, 28 filters 3 x 3, 6.0 and 7.9).  Of 125 drawn group convolutions that were taken none is
// slower by more than 1 %, 1.7 to 1.8 times as fast by geometric mean; of 70 without groups the worst 7 % slower, 1.33.  What gains are the
// large ones (16 x 64 x 57 x 57, 64 filters 3 x 3, 42.5 -> 29.6 us; 28 x 65 x 43 x 29, 38 filters, 41 -> 24) and those whose given tiles
// make few blocks (2 images x 8 groups of 15 channels, 25 x 28, 4 filters 3 x 3, 11.4 -> 4.1; 1 x 5 x 18 x 20 x 27, 18 filters
// 5 x 5, 36 -> 6.7).
struct ConvolutionSizes {
  int64_t images, groups, channels, filters, height, width, kernelHeight, kernelWidth;
};
struct SplitConvolutionShape {
  int64_t pixelTiles = 0, filterTiles = 0, channels = 0, filterWaves = 0, pixelWaves = 0, lds = 0, blocks = 0;
  double microseconds = 0;
};
SplitConvolutionShape bestSplitConvolution(const ConvolutionSizes& s, int64_t waves, int64_t ldsBudget, const DeviceLimits& limits) {
  const int64_t rows = s.height - s.kernelHeight + 1, columns = s.width - s.kernelWidth + 1, plane = rows * columns;
  SplitConvolutionShape best;
  for (int64_t chunks = 1, last = 0; chunks <= 16; ++chunks) {
    const int64_t channels = 8 * ceilDiv(ceilDiv(s.channels, chunks), 8);
    if (channels == last) continue;
    last = channels;
    // (byte offsets are 32 bits, also those of channels behind the last one.  16 chunks of what LDS holds are 27 000 terms at most, and
    // isUnsureSum counts on 65536.)
    if (std::max(channels * s.height * s.width, (s.filters * s.channels + channels) * s.kernelHeight * s.kernelWidth) >= (int64_t(1) << 29)) continue;
    const int64_t octets = channels / 8, slots = s.kernelHeight * s.kernelWidth * octets, steps = ceilDiv(slots, 4), turns = ceilDiv(s.channels, channels);
    for (int64_t used = 4; used <= std::min<int64_t>(waves, 8); used *= 2) {
      for (int64_t filterTiles = 1; filterTiles <= std::min<int64_t>(8, ceilDiv(s.filters, 16)); ++filterTiles) {
        for (int64_t filterWaves = 1; filterWaves <= 4; filterWaves *= 2) {
          if (filterTiles % filterWaves != 0) continue;
          const int64_t pixelWaves = used / filterWaves, ft = filterTiles / filterWaves;
          for (int64_t pt = 1; pt <= 8 && ft * pt <= 12; ++pt) {
            if (pt > 1 && (pt - 1) * pixelWaves >= ceilDiv(plane, 16)) break;
            SplitConvolutionShape c;
            c.pixelTiles = pt * pixelWaves;
            const int64_t pixels = (std::min(rows, (16 * c.pixelTiles + columns - 2) / columns + 1) + s.kernelHeight - 1) * s.width;
            c.lds = 3 * 16 * (pixels * (octets | 1) + 16 * filterTiles * ((4 * steps) | 1)) + 16; // (a flag)
            if (c.lds > ldsBudget) continue;
            const int64_t items = ceilDiv(pixels * octets, 64 * used) + ceilDiv(16 * filterTiles * slots, 64 * used);
            const int64_t registers = 10 * items + 8 * ft * pt + 16 * (ft + pt) + steps + pt + 30;
            if (registers > (used == 8 ? 225 : 400)) continue; // (two wavefronts share a SIMD, or one has it; 8 x 4: from 228 on some spill)
            c.blocks = s.images * s.groups * ceilDiv(plane, 16 * c.pixelTiles) * ceilDiv(s.filters, 16 * filterTiles);
            const int64_t rounds = ceilDiv(c.blocks, limits.computeUnits);
            const int64_t resident = std::max<int64_t>(1, std::min<int64_t>({limits.ldsBytesPerBlock / c.lds, (registers > 128 ? 8 : 16) / used, 4}));
            const double multiply = 24.0 * steps * turns * filterTiles * c.pixelTiles; // cycles of the matrix cores
            c.microseconds = 2.05 + rounds * (6.3e-4 * multiply + 0.0368 * turns * items * used) +
                ceilDiv(rounds, resident) * turns * (0.306 * items + 0.005 * steps * ft * pt);
            if (best.blocks != 0 && c.microseconds >= best.microseconds) continue;
            c.channels = channels;
            c.filterTiles = filterTiles;
            c.filterWaves = filterWaves;
            c.pixelWaves = pixelWaves;
            best = c;
          }
        }
      }
    }
  }
  return best;
}
// The general pipeline under the tiles the stage has now.
double givenConvolutionMicroseconds(const StagePlan& st, size_t rank, const ConvolutionSizes& s, int64_t waves, const DeviceLimits& limits) {
  const LoopVar &filter = st.vars[rank - 3], &row = st.vars[rank - 2], &column = st.vars[rank - 1], &channel = st.vars[rank];
  const int64_t places = s.kernelHeight * s.kernelWidth;
  int64_t blocks = 1;
  for (size_t v = 0; v < rank; ++v) blocks *= st.vars[v].numTiles;
  const int64_t tiles = ceilDiv(filter.tile, 16) * ceilDiv(st.vars[0].tile * row.tile * column.tile, 16);
  const int64_t steps = ceilDiv(s.channels * places, 4), lds = 4 * channel.tile *
      (st.vars[0].tile * (row.tile + s.kernelHeight - 1) * (column.tile + s.kernelWidth - 1) + filter.tile * places);
  const int64_t rounds = ceilDiv(blocks, limits.computeUnits);
  const int64_t resident = std::max<int64_t>(1, std::min<int64_t>({limits.ldsBytesPerBlock / lds, 32 / waves, 8}));
  const int64_t inTurn = ceilDiv(rounds, resident);
  const double staged = 1e-5 * lds * channel.numTiles;
  return 0.91 + rounds * (1.618 * tiles * steps * 8 / 2400 + 0.1025 * staged) + inTurn * (1.49 + 1.373 * staged + 0.0925 * channel.numTiles);
}

void takeSplitConvolution(KernelPlan& k, StagePlan& st, const HipMappingOptions& o, int64_t waves, const DeviceLimits& limits, bool wide) {
  // (useReadOnlyCache: options without it keep the given tiles)
  if (k.stages.size() != 1 || wide || waves < 4 || !o.useSharedMemoryValue || !o.useReadOnlyCacheValue || st.atomic || st.stmts.size() > 2 || !st.stmts[0].init) return;
  const size_t rank = st.lhsSubs.size(); // n, (g,) f, h, w
  if ((rank != 4 && rank != 5) || st.numParallel != static_cast<int>(rank) || st.vars.size() != rank + 3) return;
  const size_t f = rank - 3;
  for (const auto& v : st.vars) {
    if (v.min != 0) return;
  }
  auto isVar = [&](const ExprRef& e, size_t v) { return e->kind == Expr::Var && e->name == st.vars[v].name; };
  auto isSum = [&](const ExprRef& e, size_t v, size_t w) {
    const Affine a = ir::toAffine(e);
    if (!a.valid || a.constant != 0) return false;
    for (const auto& c : a.coef) {
      if (c.second != (c.first == st.vars[v].name || c.first == st.vars[w].name ? 1 : 0)) return false;
    }
    return a.coefOf(st.vars[v].name) == 1 && a.coefOf(st.vars[w].name) == 1;
  };
  auto hasExtents = [&](const std::string& tensor, const std::vector<int64_t>& extents) {
    const auto& view = st.views.at(tensor);
    int64_t bytes = 4;
    for (auto e : extents) bytes *= e;
    return view.type == ScalarType{ScalarType::Float, 32} && view.extents == extents && bytes < (int64_t(1) << 31);
  };
  std::vector<int64_t> planes, filters, result;  // extents of the input, the weights and the result
  for (size_t v = 0; v < rank; ++v) {
    if (!isVar(st.lhsSubs[v], v)) return;
    result.push_back(st.vars[v].extent);
  }
  const ConvolutionSizes s{st.vars[0].extent, rank == 5 ? st.vars[1].extent : 1, st.vars[rank].extent, st.vars[f].extent,
                           st.vars[f + 1].extent + st.vars[rank + 1].extent - 1, st.vars[f + 2].extent + st.vars[rank + 2].extent - 1,
                           st.vars[rank + 1].extent, st.vars[rank + 2].extent};
  if (rank == 5) planes = {s.images, s.groups, s.channels, s.height, s.width}, filters = {s.groups, s.filters, s.channels, s.kernelHeight, s.kernelWidth};
  else planes = {s.images, s.channels, s.height, s.width}, filters = {s.filters, s.channels, s.kernelHeight, s.kernelWidth};
  std::string input, weights, bias;
  for (const auto& load : st.stmts[0].rhs->args) {
    if (load->kind != Expr::Load) return;
    bool isInput = load->args.size() == rank, isWeights = isInput;
    for (size_t d = 0; isInput && d < rank; ++d) {
      isInput = d < f ? isVar(load->args[d], d) : d == f ? isVar(load->args[d], rank) : isSum(load->args[d], d, rank + d - f);
    }
    // (the group and the filter in front of the channels)
    for (size_t d = 0; isWeights && d < rank; ++d) isWeights = isVar(load->args[d], d < f ? d + 1 : rank + d - f);
    if (isInput && input.empty() && hasExtents(load->name, planes)) input = load->name;
    else if (isWeights && weights.empty() && hasExtents(load->name, filters)) weights = load->name;
    else return;
  }
  if (!hasExtents(st.tensor, result)) return;
  if (st.stmts.size() == 2) { // O(...) = O(...) + B(g, f)
    const StageStmt& add = st.stmts[1];
    if (add.op != ReduceOp::None || !add.redVars.empty() || add.rhs->kind != Expr::Binary || add.rhs->name != "+") return;
    for (const auto& load : add.rhs->args) {
      if (load->kind != Expr::Load) return;
      bool isResult = load->name == st.tensor && load->args.size() == rank;
      for (size_t d = 0; isResult && d < rank; ++d) isResult = isVar(load->args[d], d);
      if (isResult) continue;
      std::vector<int64_t> extents;
      bool isBias = bias.empty() && load->name != st.tensor && load->args.size() == f;
      for (size_t d = 0; isBias && d < f; ++d) {
        isBias = isVar(load->args[d], d + 1);
        extents.push_back(st.vars[d + 1].extent);
      }
      if (!isBias || !hasExtents(load->name, extents)) return;
      bias = load->name;
    }
    if (bias.empty()) return;
  }
  // a block for every tile, as the options ask for
  int axis = 0;
  for (size_t v = 0; v < rank; ++v) {
    if (st.vars[v].numTiles == 1) continue;
    if (axis >= static_cast<int>(o.grid.size()) || st.vars[v].numTiles > allowedBlocks(o, axis, static_cast<int>(v))) return;
    ++axis;
  }
  int64_t lds = limits.ldsBytesPerBlock;
  if (o.hasMaxSharedMemory) lds = std::min<int64_t>(lds, o.maxSharedMemoryValue);
  const SplitConvolutionShape shape = bestSplitConvolution(s, waves, lds, limits);
  if (s.groups == 1 && s.kernelHeight * s.kernelWidth == 1 && s.channels < 96) return;
  const double margin = s.channels * s.kernelHeight * s.kernelWidth < 48 ? 1.5 : s.groups == 1 ? 1.4 : 1.15;
  if (shape.blocks == 0 || margin * shape.microseconds >= givenConvolutionMicroseconds(st, rank, s, waves, limits)) return;
  std::ostringstream ss;
  ss << (bias.empty() ? "false" : "true");
  for (int64_t x : {s.images, s.groups, s.channels, s.filters, s.height, s.width, s.kernelHeight, s.kernelWidth, shape.pixelTiles, shape.filterTiles,
                    shape.channels, shape.filterWaves, shape.pixelWaves}) ss << ", " << x;
  ss << ">::run(p" << st.tensor << ", p" << input << ", p" << weights << ", " << (bias.empty() ? "nullptr" : "p" + bias);
  st.splitConvolution = ss.str();
  st.splitConvolutionLds = shape.lds;
  k.grid = {{shape.blocks, 1, 1}};
  k.block = {{64, shape.filterWaves * shape.pixelWaves, 1}};
}

// Products of float matrices O(m, n) +=! A * B, whichever side of the operands the reduction is on, with or without a bias
// of the columns added behind them, go to __tc::SlicedProduct (hip_split_products.h) where that is the faster form.
// Both forms are judged by an estimate in microseconds, fitted by least squares of the relative error to the times of 75 products
// (8 to 4096 rows, columns and points, 6e7 to 9e9 multiplications; twelve shapes of the sliced form each): 9 % off on average for the sliced
// form, 11 % for the given tiles; full tiles in four slices took a quarter longer than that fit says in 66 others, and are judged so.
// The sliced form is taken where it comes out 10 % faster (25 % below 320 points, 35 % with the reduction innermost in both operands, which the
// general pipeline copies best: with smaller margins products of 250 to 500 thousand results and some 200 points took up to 1.4 times as long
// as before, 1250 x 208 x 1015 14.6 us for 10.8): 1000^3 22 -> 17 us, 45 x 2516 x 2699 27.1 -> 13.5, 1250 x 1015 x 208 14.5 -> 10.3,
// 2048^3 126 -> 93 (rows, points, columns); 251 products drawn over these ranges and taken: 1.27 times as fast, the worst 6 % slower.
// Tiles that were fitted to the device stay as they are, and are taken where the sliced form has their shape.  The general
// pipeline keeps products of fewer than 1.06e8 multiplications (28 timed down to 2e7: 0.78 to 1.54 times as fast sliced, 0.99 on average, which the
// estimate does not tell apart) or 128 reduction points (19 from 62 on: 0.80 to 1.25, 1.05), and those whose tiles leave two compute units of three
// idle, which the estimate was not fitted to (20 timed since: 1.14 to 2.97 times as fast sliced, 1.65 on average; 138 x 9294 x 128 46 and 22 us).
// Blocks of eight wavefronts and prefetchShared are what the stored options of such products say; others keep the given tiles.
struct SlicedProductShape {
  int64_t rowTiles = 0, columnTiles = 0, rowWaves = 0, columnWaves = 0, slices = 0, lds = 0;
  double microseconds = 0;
};
void takeSlicedProduct(KernelPlan& k, StagePlan& st, const HipMappingOptions& o, int64_t waves, const DeviceLimits& limits, bool wide) {
  if (k.stages.size() != 1 || wide || waves != 8 || !o.prefetchSharedValue || !o.useSharedMemoryValue || st.atomic) return;
  if (st.stmts.size() > 2 || !st.stmts[0].init || st.vars.size() != 3 || st.numParallel != 2 || st.lhsSubs.size() != 2) return;
  LoopVar &m = st.vars[0], &n = st.vars[1];
  const LoopVar& r = st.vars[2];
  for (const auto& v : st.vars) {
    if (v.min != 0) return;
  }
  auto isVar = [](const ExprRef& e, const LoopVar& v) { return e->kind == Expr::Var && e->name == v.name; };
  auto hasExtents = [&](const std::string& tensor, const std::vector<int64_t>& extents) {
    const auto& view = st.views.at(tensor);
    int64_t bytes = 4;
    for (auto e : extents) bytes *= e;
    return view.type == ScalarType{ScalarType::Float, 32} && view.extents == extents && bytes < (int64_t(1) << 31);
  };
  if (!isVar(st.lhsSubs[0], m) || !isVar(st.lhsSubs[1], n) || !hasExtents(st.tensor, {m.extent, n.extent})) return;
  std::string tensors[2], bias;  // of the m and of the n side
  bool innermost[2];             // the reduction is the last subscript
  for (const auto& load : st.stmts[0].rhs->args) {
    if (load->kind != Expr::Load || load->args.size() != 2) return;
    bool found = false;
    for (int side = 0; side < 2; ++side) {
      const LoopVar& v = side == 0 ? m : n;
      for (int last = 0; last < 2; ++last) {
        const LoopVar &outer = last ? v : r, &inner = last ? r : v;
        if (!isVar(load->args[0], outer) || !isVar(load->args[1], inner)) continue;
        if (!hasExtents(load->name, {outer.extent, inner.extent}) || !tensors[side].empty()) return;
        tensors[side] = load->name;
        innermost[side] = last == 1;
        found = true;
      }
    }
    if (!found) return;
  }
  if (st.stmts.size() == 2) { // O(m, n) = O(m, n) + B(n)
    const StageStmt& add = st.stmts[1];
    if (add.op != ReduceOp::None || !add.redVars.empty() || add.rhs->kind != Expr::Binary || add.rhs->name != "+") return;
    for (const auto& load : add.rhs->args) {
      if (load->kind != Expr::Load) return;
      if (load->name == st.tensor && load->args.size() == 2 && isVar(load->args[0], m) && isVar(load->args[1], n)) continue;
      if (!bias.empty() || load->name == st.tensor || load->args.size() != 1 || !isVar(load->args[0], n) || !hasExtents(load->name, {n.extent})) return;
      bias = load->name;
    }
    if (bias.empty()) return;
  }
  const double multiplications = 1.0 * m.extent * n.extent * r.extent;
  if (multiplications < 1.06e8 || r.extent < 128 || r.extent > 65536) return;  // (longer sums are not what isUnsureSum counts on)
  // a block for every tile of these sizes?
  auto isOneBlockATile = [&](int64_t rows, int64_t columns) {
    int axis = 0;
    for (int position = 0; position < 2; ++position) {
      const int64_t tiles = position == 0 ? ceilDiv(m.extent, rows) : ceilDiv(n.extent, columns);
      if (tiles == 1) continue;
      if (axis >= static_cast<int>(o.grid.size()) || tiles > allowedBlocks(o, axis, position)) return false;
      ++axis;
    }
    return true;
  };
  if (!isOneBlockATile(m.tile, n.tile) || 3 * m.numTiles * n.numTiles < limits.computeUnits) return;
  int64_t lds = limits.ldsBytesPerBlock;
  if (o.hasMaxSharedMemory) lds = std::min<int64_t>(lds, o.maxSharedMemoryValue);
  static const int64_t kShapes[][5] = { // tiles of a wavefront, wavefronts along rows and columns, slices
      {1, 1, 1, 1, 8}, {1, 2, 1, 1, 8}, {2, 2, 1, 1, 8}, {2, 4, 1, 1, 8}, {4, 2, 1, 1, 8}, {4, 4, 1, 1, 8}, {2, 2, 1, 1, 4}, {2, 4, 1, 1, 4},
      {4, 4, 1, 1, 4}, {2, 2, 1, 2, 4}, {2, 4, 2, 1, 4}, {4, 2, 1, 2, 4}, {4, 4, 2, 1, 4}, {4, 4, 1, 2, 4}, {2, 2, 2, 2, 2}, {4, 4, 2, 2, 2}};
  SlicedProductShape best;
  for (const auto& s : kShapes) {
    SlicedProductShape c;
    c.rowTiles = s[0], c.columnTiles = s[1], c.rowWaves = s[2], c.columnWaves = s[3], c.slices = s[4];
    const int64_t rows = 16 * c.rowTiles * c.rowWaves, columns = 16 * c.columnTiles * c.columnWaves;
    if (st.fittedToDevice ? rows != m.tile || columns != n.tile : !isOneBlockATile(rows, columns)) continue;
    const int64_t used = c.rowWaves * c.columnWaves * c.slices, area = c.rowTiles * c.columnTiles;
    c.lds = 64 * used * c.rowTiles * (16 * c.columnTiles + 4);
    const int64_t blocks = ceilDiv(m.extent, rows) * ceilDiv(n.extent, columns), rounds = ceilDiv(blocks, limits.computeUnits);
    if (c.lds > lds) continue;
    const int64_t resident = std::max<int64_t>(1, std::min(limits.ldsBytesPerBlock / c.lds, (area <= 4 ? 16 : 8) / used));
    const int64_t steps = ceilDiv(ceilDiv(r.extent, 32), c.slices), inTurn = ceilDiv(rounds, resident);
    c.microseconds = 2.71 + 0.01 * rounds * used * (steps * (0.52 * area + 2.31 * (c.rowTiles + c.columnTiles) +
                                                             0.81 * (innermost[0] * c.rowTiles + innermost[1] * c.columnTiles)) + 0.66 * area) +
        inTurn * (0.1 + 0.267 * steps) + 0.66e-6 * m.extent * n.extent;
    if (area == 16 && c.slices == 4) c.microseconds *= 1.25;
    if (best.slices == 0 || c.microseconds < best.microseconds) best = c;
  }
  if (best.slices == 0) return;
  // the general pipeline under the tiles the stage has now
  const int64_t tiles = ceilDiv(m.tile, 16) * ceilDiv(n.tile, 16), rounds = ceilDiv(m.numTiles * n.numTiles, limits.computeUnits);
  const double points = 1e-3 * (r.numTiles > 1 ? r.numTiles * r.tile : 16 * ceilDiv(r.extent, 16));
  const double given = 1.37 + rounds * (points * (0.89 * tiles + 0.211 * std::sqrt(1.0 * tiles)) + 0.608) + 0.13 * r.numTiles +
      (tiles < 8 ? 1.93 * points : 0) + 1.21e-6 * m.extent * n.extent;
  const double margin = innermost[0] && innermost[1] ? 1.35 : r.extent < 320 ? 1.25 : 1.1;
  if (margin * best.microseconds >= given) return;
  m.tile = 16 * best.rowTiles * best.rowWaves;
  n.tile = 16 * best.columnTiles * best.columnWaves;
  for (LoopVar* v : {&m, &n}) {
    v->tile = std::min(v->tile, v->extent);
    v->numTiles = ceilDiv(v->extent, v->tile);
  }
  std::ostringstream ss;
  ss << (bias.empty() ? "false" : "true") << ", " << (innermost[0] ? "true" : "false") << ", " << (innermost[1] ? "true" : "false");
  for (int64_t x : {m.extent, n.extent, r.extent, best.rowTiles, best.columnTiles, best.rowWaves, best.columnWaves, best.slices}) ss << ", " << x;
  ss << ">::run(p" << st.tensor << ", p" << tensors[0] << ", p" << tensors[1] << ", " << (bias.empty() ? "nullptr" : "p" + bias);
  st.slicedProduct = ss.str();
  st.slicedProductLds = best.lds;
  st.waves = best.rowWaves * best.columnWaves * best.slices;
}

// A batch of float products, a block for every product and tile of it, whose rows or columns take two tiles: one product a block where
// there are two products a compute unit.  Every block copies the operands it needs to LDS behind one barrier, so the second tile of rows
// copies the whole other operand again, often for a few rows: 1024 products 65x128x65 (rows, points, columns) 52 -> 27 us, 768 of 80x80x80 28.9 -> 16.0,
// 512 of 100x100x100 32.5 -> 23.2, 654 of 68x108x45 19.8 -> 12.5.
// The tiles stay where the second is nearly full or one product takes more than half of the LDS, with one block of four wavefronts a compute unit
// then (600 of 128x128x128 34.8 us in tiles, 51 whole; 1314 of 98x128x98 80 and 100; 600 of 128x32x128 12.7 and 15.4), where the
// rows alone have two tiles and are more than 96 (700 of 128x64x64 13.5 and 14.4; 643 of 101x127x40 21.5 and 23.6) or the blocks are too few without them
// (716 of 79x12x8 2.9 and 3.8; 586 of 81x18x37 5.5 and 6.1), and of fewer products (140 of 111x67x83 9.4 and 11.0).
// They stay too where the blocks have fewer than eight wavefronts a compute unit between them (blocks of two: 998 of 60x9x114 9.4 and 11.2, 694 of 79x2x82
// 7.2 and 8.5; 1507 of 119x7x67 goes, 17.6 -> 16.7), with reductions of less than four points (1982 of 108x1x102 19.8 and 23.7), which leave little to
// copy twice, and with 5 to 8 columns on four wavefronts (2233 of 85x7x5 4.4 and 6.8, nine of nine such; eight wavefronts 14.2 -> 8.3 for 1830 of 88x47x5).  Of
// 231 others drawn with up to 48 points one is 14 % slower (861 of 95x7x104, 10.4 and 12.0) and none of the rest more than 3 %, 1.24 times as fast by geometric mean.
void takeProductsWhole(const KernelPlan& k, StagePlan& st, const HipMappingOptions& o, int64_t waves, const DeviceLimits& limits) {
  constexpr int64_t kMostTiles = 49, kMostRows = 120, kMostRowsAlone = 96;
  if (k.stages.size() != 1 || st.mfmaBatch.size() != 1 || st.stmts.size() != 1 || !o.useSharedMemoryValue || o.prefetchSharedValue || st.atomic) return;
  if (st.vars.size() != 4 || st.numParallel != 3 || k.sharedDepth < 3) return;
  for (const auto& load : st.stmts[0].rhs->args) {
    if (load->kind != Expr::Load || st.views.at(load->name).type != ScalarType{ScalarType::Float, 32}) return;
  }
  const LoopVar &b = st.vars[0], &r = st.vars[3];
  LoopVar &m = st.vars[1], &n = st.vars[2];
  if (b.name != st.mfmaBatch[0] || b.tile != 1 || r.numTiles != 1 || b.extent < 2 * limits.computeUnits) return;
  if (b.numTiles > allowedBlocks(o, 0, 0)) return;
  if (m.numTiles > 2 || n.numTiles > 2 || m.numTiles * n.numTiles == 1) return;
  if (ceilDiv(m.extent, 16) * ceilDiv(n.extent, 16) > kMostTiles || m.extent > kMostRows) return;
  if (r.extent < 4 || b.extent * waves < 8 * limits.computeUnits) return;
  if (n.numTiles == 1 && (m.extent > kMostRowsAlone || b.extent < 3 * limits.computeUnits)) return;
  if (n.numTiles == 1 && waves == 4 && n.extent > 4 && n.extent <= 8) return;
  int64_t lds = limits.ldsBytesPerBlock / 2;
  if (o.hasMaxSharedMemory) lds = std::min<int64_t>(lds, o.maxSharedMemoryValue);
  if (4 * r.extent * (m.extent + n.extent + 8) > lds) return;
  for (LoopVar* v : {&m, &n}) {
    v->tile = v->extent;
    v->numTiles = 1;
  }
}

// Sums of the columns of a float matrix, O(n) +=! A(r, n), whose threads keep whole sums, under tiles that leave three quarters of the
// device's wavefronts out, go to __tc::columnSums (hip_column_sums.h): rows on other threads as well, whatever the options say about
// unrolling.  (One axis of threads, one block a tile, no matchLibraryCalls, which has the rows on threads as it is.)
// Beyond half as many tiles as compute units (8192 columns) one thread a column has the device half full, and two blocks of 16 columns, on different
// XCDs, read every line of 128 bytes twice.  Of 200 sizes timed there these were slower and stay: few rows (64 x 12288 2.2 -> 2.4 us, 100 x 15360 2.6 -> 2.7),
// whole tiles of a matrix that is more than half of the L2 caches but fits them (320 x 14336 5.0 -> 6.7, 512 x 12288 7.3 -> 8.6; 200 x 14336 4.0 -> 2.9 and
// 1024 x 9216 20 -> 13.5 go), and other tiles on nearly all compute units (200 x 16001 5.8 -> 6.5; 200 x 15001 6.5 -> 4.9).
constexpr int64_t kColumnSumWaves = 16;
void takeColumnSums(KernelPlan& k, StagePlan& st, const HipMappingOptions& o, const DeviceLimits& limits, bool wide) {
  if (k.stages.size() != 1 || wide || st.atomic || o.generic.matchLibraryCallsValue || o.block.size() != 1 || !o.generic.hasTiling) return;
  if (st.stmts.size() != 1 || !st.stmts[0].init || st.stmts[0].op != ReduceOp::Plus || st.vars.size() != 2 || st.numParallel != 1) return;
  const LoopVar &n = st.vars[0], &r = st.vars[1];
  if (n.min != 0 || r.min != 0 || !r.reduction || st.lhsSubs.size() != 1) return;
  auto isVar = [](const ExprRef& e, const LoopVar& v) { return e->kind == Expr::Var && e->name == v.name; };
  const ExprRef& load = st.stmts[0].rhs;
  const ScalarType f32{ScalarType::Float, 32};
  if (load->kind != Expr::Load || load->args.size() != 2 || !isVar(load->args[0], r) || !isVar(load->args[1], n) || !isVar(st.lhsSubs[0], n)) return;
  const auto &a = st.views.at(load->name), &out = st.views.at(st.tensor);
  if (a.type != f32 || out.type != f32 || a.extents != std::vector<int64_t>{r.extent, n.extent} || out.extents != std::vector<int64_t>{n.extent}) return;
  const int64_t waves = n.numTiles * ceilDiv(std::min<int64_t>(static_cast<int64_t>(o.block[0]), n.tile), limits.wavefront);
  if (n.numTiles > allowedBlocks(o, 0, 0) || waves >= limits.computeUnits || r.extent < 4 * kColumnSumWaves || r.extent * n.extent >= (int64_t(1) << 29)) return;
  if (2 * waves > limits.computeUnits) {
    const bool whole = n.extent % n.tile == 0;
    const int64_t mebibytes = r.extent * n.extent >> 18;
    if (r.extent < (whole ? 128 : 80) || (whole ? mebibytes >= 16 && mebibytes < 36 : 16 * waves > 15 * limits.computeUnits)) return;
  }
  if (limits.maxThreadsPerBlock < 64 * kColumnSumWaves) return;
  if (o.hasMaxSharedMemory && static_cast<int64_t>(o.maxSharedMemoryValue) < 4 * 64 * kColumnSumWaves) return;
  std::ostringstream ss;
  ss << r.extent << ", " << n.extent << ", " << kColumnSumWaves << ">(p" << st.tensor << ", p" << load->name;
  st.columnSums = ss.str();
  k.grid = {{ceilDiv(n.extent, 16), 1, 1}};
  k.block = {{64, kColumnSumWaves, 1}};
}

// A contraction whose threads keep whole sums (no matrix cores, no LDS, one axis of threads) under tile sizes that were made
// for other extents.  Returns the innermost variable where it takes a block axis behind those of the options.
//   A variable without a block axis is not walked tile by tile where all its points fit the registers under the tiles given
// to the others: every walk reads the operands that do not depend on it again (tensordot of 7x404x9x4x9x21 in tiles of two of
// the 4: 12.6 -> 5.7 us).  Where they would fit only once the tiles of others are halved the walk stays: 90 such tensordots
// took 0.5 to 1.5 times as long with the variable whole, as often longer as shorter.
//   Blocks with fewer than six wavefronts a compute unit get less work each, until there are sixteen: a block's loads wait for
// each other and there is nobody to fill in.  First the points a thread takes of the innermost variable go to blocks
// of their own, then the largest tile of the others is halved; more blocks along a variable than the options allow
// it there are not, and no variable loses its block axis to one in front of it, unless all its points fit the registers: it
// would be walked in every block (3x7x15x79x14x13, c1 on the axis of 40 tiles of c3: 33.2 us, 12.4 as given;
// 2x84x12x3x49x37 in tiles of four of c3 under mapToBlocks=32,64,8: 17.2 and 8.1) (tensordot 4x17x8x4x47x25, 12 blocks of 256 threads and 80 sums each, 29.7 us; 180 blocks of 8 sums
// 3.9; 10x285x12x2x29x31, 360 blocks 45.7, 1440 32.3; 7x33x12x2x39x56 83.6 and 7.7).  Beyond that there is nothing to gain:
// 16x286x3x2x25x30, 576 blocks of nine wavefronts a unit, 16.1 us, in 1728 shorter pieces of its rows 20.6.
const LoopVar* spreadContraction(const KernelPlan& k, StagePlan& st, const HipMappingOptions& o, const DeviceLimits& limits) {
  constexpr int64_t kFewWaves = 6, kWavesPerUnit = 16, kMostSums = 64;
  if (k.stages.size() != 1 || st.mfma || st.atomic || o.useSharedMemoryValue || !o.generic.hasTiling || k.sharedDepth < st.numParallel) return nullptr;
  if (st.stmts.empty() || st.stmts[0].redVars.empty() || o.generic.matchLibraryCallsValue) return nullptr;
  for (size_t a = 1; a < o.block.size(); ++a) {
    if (o.block[a] != 1) return nullptr;
  }
  std::vector<LoopVar*> vars; // parallel, the lanes of a vector left out
  int64_t lanes = 1;
  for (int i = 0; i < st.numParallel; ++i) {
    if (st.vars[i].vectorLane) lanes *= st.vars[i].extent;
    else vars.push_back(&st.vars[i]);
  }
  if (vars.size() < 2) return nullptr;
  LoopVar& inner = *vars.back();
  const int64_t mostSums = std::min<int64_t>(kMostSums, o.generic.hasUnroll ? static_cast<int64_t>(o.generic.unrollValue) : 1);
  const int64_t threads = std::min<int64_t>(static_cast<int64_t>(o.block[0]), inner.tile);
  auto setTile = [](LoopVar& v, int64_t tile) {
    v.tile = tile;
    v.numTiles = ceilDiv(v.extent, tile);
  };
  // the block axis a variable takes (as mapKernel gives them out), -1: none
  const bool hadTiles = inner.numTiles > 1;
  auto axisOf = [&](const LoopVar& v) -> int {
    int axis = 0;
    for (const LoopVar* w : vars) {
      const bool takes = w->numTiles > 1 && (axis < static_cast<int>(o.grid.size()) || (w == &inner && !hadTiles && axis < 3));
      if (w == &v) return takes ? axis : -1;
      if (takes) ++axis;
    }
    return -1;
  };
  auto isDistributed = [&](const LoopVar& v) { return axisOf(v) >= 0; };
  // 0: more tiles than blocks, which are then the ones asked for
  auto blocks = [&]() -> int64_t {
    int64_t n = 1;
    for (size_t i = 0; i < vars.size(); ++i) {
      const int axis = axisOf(*vars[i]);
      if (axis < 0) continue;
      if (axis < static_cast<int>(o.grid.size()) && vars[i]->numTiles > allowedBlocks(o, axis, static_cast<int>(i))) return 0;
      n *= vars[i]->numTiles;
    }
    return n;
  };
  auto sums = [&]() {
    int64_t n = lanes * ceilDiv(inner.tile, threads);
    for (const LoopVar* v : vars) n *= v == &inner ? 1 : v->tile;
    return n;
  };
  if (blocks() == 0) return nullptr;
  auto waves = [&]() { return blocks() * ceilDiv(threads, limits.wavefront); };
  const bool isShort = waves() < kFewWaves * limits.computeUnits;
  std::set<const LoopVar*> whole; // whose tiles stay, as others would lose their axis
  auto largestOuter = [&]() {
    LoopVar* best = nullptr;
    for (LoopVar* v : vars) {
      if (v != &inner && !whole.count(v) && v->tile > 1 && (v->numTiles == 1 ? v->tile > 2 : isDistributed(*v)) && (!best || v->tile > best->tile)) best = v;
    }
    return best;
  };
  if (isShort && (!hadTiles || isDistributed(inner))) {
    const int64_t given = inner.tile, most = ceilDiv(given, threads);
    const int64_t per = std::max<int64_t>(1, most / ceilDiv(kWavesPerUnit * limits.computeUnits, waves()));
    if (per < most) {
      setTile(inner, per * threads);
      if (blocks() == 0 || !isDistributed(inner)) setTile(inner, given);
    }
  }
  for (LoopVar* v : vars) {
    if (v == &inner || v->numTiles == 1 || isDistributed(*v)) continue;
    const int64_t tile = v->tile;
    setTile(*v, v->extent);
    if (sums() > mostSums) setTile(*v, tile);
  }
  while (isShort && waves() < kWavesPerUnit * limits.computeUnits) {
    LoopVar* v = largestOuter();
    if (!v) break;
    std::vector<LoopVar*> distributed;
    for (LoopVar* w : vars) {
      if (isDistributed(*w)) distributed.push_back(w);
    }
    const int64_t before = blocks();
    const int64_t tile = v->tile, numTiles = v->numTiles;
    setTile(*v, ceilDiv(v->tile, 2));
    if (blocks() == 0 || (numTiles == 1 && !isDistributed(*v))) {
      setTile(*v, tile);
      break;
    }
    // a variable that loses its axis to this one is taken whole where its sums fit, else this one stays as it was
    for (LoopVar* w : distributed) {
      if (isDistributed(*w)) continue;
      const int64_t given = w->tile;
      if (w != &inner) setTile(*w, w->extent);
      if (w != &inner && sums() <= mostSums && blocks() >= before) continue;
      setTile(*w, given);
      setTile(*v, tile);
      whole.insert(v);
      break;
    }
  }
  return inner.numTiles > 1 && !hadTiles ? &inner : nullptr;
}

void mapKernel(KernelCtx& kc, const DeviceLimits& limits) {
  const HipMappingOptions& o = kc.opts;
  KernelPlan& k = kc.k;
  TC_CHECK(!o.generic.hasTiling || !o.generic.tiling.empty()) << "tiling must hold at least one size";
  for (size_t a = 0; a < 3; ++a) {
    TC_CHECK_GT(o.grid[a], 0u) << "NYI: mapping to 0 blocks";
    TC_CHECK_GT(o.block[a], 0u) << "NYI: mapping to 0 threads";
  }
  std::array<int64_t, 3> blockUse{{1, 1, 1}}, gridUse{{1, 1, 1}};
  // Threads the stages may spread over.  A matrix-core stage addresses its lanes as
  // (threadIdx.x = lane of a wavefront, threadIdx.y = wavefront), so a kernel that holds one runs
  // 64 x waves threads and its other stages map onto that shape.
  std::array<int64_t, 3> blk{{static_cast<int64_t>(o.block[0]), static_cast<int64_t>(o.block[1]),
                              static_cast<int64_t>(o.block[2])}};
  int nb = static_cast<int>(o.block.size());
  int64_t waves = std::max<int64_t>(1, std::min<int64_t>(16, blk[0] * blk[1] * blk[2] / 64));
  for (const auto& st : k.stages) {
    if (st.mfma) {
      blk = {{64, waves, 1}};
      nb = 2;
    }
  }
  for (auto& st : k.stages) {
    // tile sizes by band position (lanes do not take a position)
    int pos = 0;
    for (auto& v : st.vars) {
      TC_CHECK_GT(v.extent, 0) << "loop variable " << v.name << " has no points";
      if (v.vectorLane) {
        v.tile = v.extent;
        v.numTiles = 1;
        continue;
      }
      int64_t t = 0;
      if (o.generic.hasTiling && pos < static_cast<int>(o.generic.tiling.size())) {
        t = static_cast<int64_t>(o.generic.tiling[pos]);
      }
      ++pos;
      // a lane-split variable is tiled in units of whole lane groups
      const LoopVar* next = (&v + 1 < &st.vars[0] + st.vars.size()) ? &v + 1 : nullptr;
      if (next && next->vectorLane && t > 0) t = std::max<int64_t>(1, t / next->extent);
      v.tile = (t <= 0 || t > v.extent) ? v.extent : t;
      v.numTiles = ceilDiv(v.extent, v.tile);
    }
    if (st.mfma) takeLargeHalfProduct(k, st, o, waves, limits, kc.wide);
    if (!st.largeHalfProduct.empty()) return;
    if (st.mfma) fillComputeUnits(k, st, o, waves, limits.computeUnits);
    if (st.mfma) takeProductsWhole(k, st, o, waves, limits);
    if (st.mfma) takeSlicedProduct(k, st, o, waves, limits, kc.wide);
    if (st.mfma) takeSplitConvolution(k, st, o, waves, limits, kc.wide);
    if (!st.splitConvolution.empty()) return;
    takeColumnSums(k, st, o, limits, kc.wide);
    if (!st.columnSums.empty()) return;
    const LoopVar* spread = spreadContraction(k, st, o, limits);
    // blocks: outermost shared parallel variables, x first
    int axis = 0, position = -1;
    for (int i = 0; i < st.numParallel && i < k.sharedDepth && axis < 3; ++i) {
      LoopVar& v = st.vars[i];
      // a variable with a single tile has nothing to distribute and does not use up an axis
      if (!v.vectorLane) ++position;
      if (v.vectorLane || v.numTiles == 1) continue;
      if (axis >= static_cast<int>(o.grid.size())) {
        if (&v != spread) continue;
        v.blockAxis = axis;
        v.gridExtent = v.numTiles;
        gridUse[axis] = std::max(gridUse[axis], v.gridExtent);
        break;
      }
      v.blockAxis = axis;
      v.gridExtent = std::min<int64_t>(allowedBlocks(o, axis, position), v.numTiles);
      gridUse[axis] = std::max(gridUse[axis], v.gridExtent);
      ++axis;
    }
    if (!st.slicedProduct.empty()) {
      blockUse = {{64, st.waves, 1}};
      continue;
    }
    if (st.mfma) {
      // one wavefront per 16x16 output tile; the block holds as many wavefronts as the block
      // option has threads.  Only the outermost reduction variable may be tiled (a tile that does
      // not divide the extent needs operands whose surplus points can be told apart, and is kept
      // where it pays, which the planning of the copies decides): operands are then staged in LDS
      // one reduction tile at a time while the accumulators of a wavefront's output tiles stay in
      // registers.
      bool firstReduction = true;
      for (auto& v : st.vars) {
        if (!v.reduction) continue;
        if (firstReduction) deepenHalfTile(st, v, o, waves, limits);
        bool keep = firstReduction && v.numTiles > 1 && (v.extent % v.tile == 0 || reductionMayEndInMidTile(st, v.name));
        firstReduction = false;
        if (!keep) {
          v.tile = v.extent;
          v.numTiles = 1;
        }
      }
      st.waves = waves;
      blockUse[0] = std::max<int64_t>(blockUse[0], 64);
      blockUse[1] = std::max<int64_t>(blockUse[1], st.waves);
      continue;
    }
    // threads: innermost variables, x first
    bool hasReduction = false;
    for (const auto& s : st.stmts) hasReduction |= !s.redVars.empty();
    st.threadReduction = o.generic.matchLibraryCallsValue && hasReduction && blk[0] > 1 && o.block[0] > 1;
    int taxis = 0;
    if (st.threadReduction) {
      for (int i = static_cast<int>(st.vars.size()) - 1; i >= st.numParallel; --i) {
        if (!st.vars[i].vectorLane) {
          st.vars[i].threadAxis = 0;
          break;
        }
      }
      taxis = 1;
    }
    for (int i = st.numParallel - 1; i >= 0 && taxis < nb; --i) {
      if (st.vars[i].vectorLane) continue;
      st.vars[i].threadAxis = taxis++;
    }
    for (auto& v : st.vars) {
      if (v.threadAxis >= 0) {
        int64_t want = v.tile;
        if (st.threadReduction && v.reduction) {
          // the reduction library is fastest on rows that are lane groups of a wavefront or
          // whole wavefronts: tighten to the next such width when the option allows it
          if (want <= 64) {
            while (want & (want - 1)) ++want;
          } else {
            want = ceilDiv(want, 64) * 64;
          }
          if (want > blk[v.threadAxis]) want = v.tile;
        }
        blockUse[v.threadAxis] = std::max(blockUse[v.threadAxis], std::min<int64_t>(blk[v.threadAxis], want));
      }
    }
  }
  // XCD-aware block order.  Consecutive linear block ids go round-robin to the 8 XCDs, each
  // with its own L2: blocks that differ only in the x-mapped tile index end up on different XCDs.
  // Operands that do not depend on a block-mapped variable are shared by the blocks along it, so
  // the variable with the least shared bytes takes blockIdx.x and the one with the most the
  // slowest axis (its blocks then meet in one L2 when the faster extents are multiples of 8).
  {
    const StagePlan& s0 = k.stages.front();
    std::vector<int> positions;
    for (int i = 0; i < s0.numParallel && i < k.sharedDepth; ++i) {
      if (s0.vars[i].blockAxis >= 0) positions.push_back(i);
    }
    if (positions.size() >= 2) {
      std::vector<double> shared(positions.size(), 0.0);
      for (const auto& st : k.stages) {
        std::map<std::string, std::set<std::string>> uses; // tensor -> variables in its subscripts
        for (const auto& stmt : st.stmts) {
          visit(stmt.rhs, [&](const ExprRef& e) {
            if (e->kind != Expr::Load) return;
            auto& u = uses[e->name];
            for (const auto& a : e->args) {
              Affine x = ir::toAffine(a);
              if (!x.valid) {
                for (const auto& v : st.vars) u.insert(v.name); // unknown: assume it depends on all
                continue;
              }
              for (const auto& c : x.coef) {
                if (c.second != 0) u.insert(c.first);
              }
            }
          });
        }
        for (const auto& t : uses) {
          const TensorView& view = st.views.at(t.first);
          double bytes = view.type.bytes();
          for (auto e : view.extents) bytes *= static_cast<double>(e);
          for (int pos : positions) {
            if (t.second.count(st.vars[pos].name)) bytes /= static_cast<double>(st.vars[pos].numTiles);
          }
          for (size_t r = 0; r < positions.size(); ++r) {
            if (!t.second.count(st.vars[positions[r]].name)) shared[r] += bytes;
          }
        }
      }
      std::vector<size_t> order(positions.size());
      for (size_t r = 0; r < order.size(); ++r) order[r] = r;
      std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t b) { return shared[a] < shared[b]; });
      bool changes = false;
      for (size_t r = 0; r < order.size(); ++r) changes |= order[r] != r;
      // every stage must distribute the same positions over the same extents
      bool uniform = true;
      for (const auto& st : k.stages) {
        int mapped = 0;
        for (int i = 0; i < st.numParallel; ++i) mapped += st.vars[i].blockAxis >= 0;
        uniform &= mapped == static_cast<int>(positions.size());
        for (int pos : positions) {
          uniform &= pos < st.numParallel && st.vars[pos].blockAxis == s0.vars[pos].blockAxis &&
              st.vars[pos].gridExtent == s0.vars[pos].gridExtent;
        }
      }
      if (changes && uniform && s0.vars[positions[order[0]]].gridExtent % 8 == 0) {
        gridUse = {{1, 1, 1}};
        for (auto& st : k.stages) {
          for (size_t r = 0; r < order.size(); ++r) {
            LoopVar& v = st.vars[positions[order[r]]];
            v.blockAxis = static_cast<int>(r);
            gridUse[r] = std::max(gridUse[r], v.gridExtent);
          }
        }
      }
    }
  }
  k.block = blockUse;
  k.grid = gridUse;
  TC_CHECK_LE(k.block[0] * k.block[1] * k.block[2], limits.maxThreadsPerBlock)
      << "thread block of " << k.block[0] << "x" << k.block[1] << "x" << k.block[2] << " exceeds the device limit";
  int64_t budget = o.generic.hasUnroll ? static_cast<int64_t>(o.generic.unrollValue) : 1;
  for (auto& st : k.stages) {
    for (auto& v : st.vars) {
      v.perThread = v.threadAxis >= 0 ? ceilDiv(v.tile, k.block[v.threadAxis]) : v.tile;
    }
    if (st.mfma) {
      st.accCount = 1;
      continue;
    }
    // register tile: innermost parallel variables first, while the tile fits the budget
    int64_t prod = 1;
    for (int i = st.numParallel - 1; i >= 0; --i) {
      LoopVar& v = st.vars[i];
      if (v.vectorLane || prod * v.perThread <= std::max<int64_t>(budget, 1) || v.perThread == 1) {
        // bound on fully unrolled code: every accumulator of a thread-mapped reduction also
        // unrolls one block reduction (compile time of hipRTC grows steeply beyond this)
        if (prod * v.perThread > (st.threadReduction ? 32 : 256)) break;
        v.unrolled = true;
        prod *= v.perThread;
      } else {
        break;
      }
    }
    st.accCount = prod;
  }
}

std::string kernelSignature(const ir::Function& f, const std::string& name, int64_t nt) {
  std::ostringstream ss;
  ss << "extern \"C\" __global__ void __launch_bounds__(" << nt << ") " << name << "(";
  bool first = true;
  for (const auto& p : f.params) {
    ss << (first ? "" : ", ") << "int " << p.first;
    first = false;
  }
  for (const auto& t : f.outputs) {
    ss << (first ? "" : ", ") << t.type.cName() << "* __restrict__ p" << t.name;
    first = false;
  }
  for (const auto& t : f.inputs) {
    ss << (first ? "" : ", ") << "const " << t.type.cName() << "* __restrict__ p" << t.name;
    first = false;
  }
  ss << ")";
  return ss.str();
}

void emitKernel(KernelCtx& kc, const DeviceLimits& limits, Emitter& em) {
  KernelPlan& k = kc.k;
  if (!k.stages[0].largeHalfProduct.empty()) {
    em.open(kernelSignature(kc.f, k.name, kc.NT()));
    for (const auto& p : kc.f.params) em.line("(void)" + p.first + ";");
    em.line("__shared__ __attribute__((aligned(1024))) char tiles_[" + std::to_string(kLargeHalfLds) + "];");
    em.line("__tc::largeHalfProduct<" + k.stages[0].largeHalfProduct + ", (__tc::ldschar*)tiles_);");
    em.close();
    k.ldsBytes = kLargeHalfLds;
    return;
  }
  if (!k.stages[0].columnSums.empty()) {
    em.open(kernelSignature(kc.f, k.name, kc.NT()));
    for (const auto& p : kc.f.params) em.line("(void)" + p.first + ";");
    em.line("__shared__ float sums_[" + std::to_string(64 * kColumnSumWaves) + "];");
    em.line("__tc::columnSums<" + k.stages[0].columnSums + ", sums_);");
    em.close();
    k.ldsBytes = 4 * 64 * kColumnSumWaves;
    return;
  }
  if (!k.stages[0].slicedProduct.empty()) {
    em.open(kernelSignature(kc.f, k.name, kc.NT()));
    for (const auto& p : kc.f.params) em.line("(void)" + p.first + ";");
    em.line("// matrix cores: the bf16 parts of floats, each wavefront a slice of the reduction");
    em.line("__shared__ __attribute__((aligned(16))) char sums_[" + std::to_string(k.stages[0].slicedProductLds) + "];");
    em.line("__tc::SlicedProduct<" + k.stages[0].slicedProduct + ", (__tc::ldschar*)sums_);");
    em.close();
    k.ldsBytes = k.stages[0].slicedProductLds;
    return;
  }
  if (!k.stages[0].splitConvolution.empty()) {
    em.open(kernelSignature(kc.f, k.name, kc.NT()));
    for (const auto& p : kc.f.params) em.line("(void)" + p.first + ";");
    em.line("// matrix cores: the bf16 parts of floats, a window of the input and the filters above it in LDS");
    em.line("__shared__ __attribute__((aligned(16))) char window_[" + std::to_string(k.stages[0].splitConvolutionLds) + "];");
    em.line("__tc::SplitConvolution<" + k.stages[0].splitConvolution + ", (__tc::ldschar*)window_);");
    em.close();
    k.ldsBytes = k.stages[0].splitConvolutionLds;
    return;
  }
  std::vector<StageCodegen> gens;
  gens.reserve(k.stages.size());
  int64_t ldsBudget = limits.ldsBytesPerBlock;
  if (kc.opts.hasMaxSharedMemory) ldsBudget = std::min<int64_t>(ldsBudget, kc.opts.maxSharedMemoryValue);
  int64_t scratchElems = 0;
  ScalarType scratchType;
  for (auto& st : k.stages) {
    if (st.threadReduction) {
      int64_t bx = k.block[0], rows = k.block[1] * k.block[2];
      int64_t e = ((bx & (bx - 1)) == 0 && bx <= 64) ? 1 : (bx % 64 == 0 ? (bx / 64) * rows : bx * rows);
      scratchElems = std::max(scratchElems, e);
      ScalarType t = st.views.at(st.tensor).type;
      if (t.bytes() > scratchType.bytes() || scratchElems == e) scratchType = t;
    }
  }
  ldsBudget -= scratchElems * 8;
  int64_t before = ldsBudget;
  for (size_t i = 0; i < k.stages.size(); ++i) {
    gens.emplace_back(kc, k.stages[i], static_cast<int>(i), em);
    gens.back().plan(ldsBudget);
  }
  // One copy per kernel: a later stage whose footprint of a tensor is the one an earlier stage has
  // staged (same box, same origin, fixed for the whole kernel-level iteration) reads the earlier
  // stage's array.  Staged tensors are inputs of the TC, so nothing in the kernel changes them.
  {
    std::map<std::string, std::string> staged; // footprint key -> LDS array of the first stage that stages it
    for (size_t i = 0; i < gens.size(); ++i) {
      for (auto& p : gens[i].mutablePromotions()) {
        if (!gens[i].footprintFixedPerKernelIteration(p)) continue;
        std::string key = gens[i].footprintKey(p);
        auto found = staged.find(key);
        if (found == staged.end()) {
          staged.emplace(key, p.ldsName);
        } else {
          p.sharedWithEarlierStage = true;
          p.ldsName = found->second;
          ldsBudget += p.elems * k.stages[i].views.at(p.tensor).type.bytes();
        }
      }
    }
  }
  // Producer -> consumer through a register (usePrivateMemory): a block-wide reduction along
  // threadIdx.x leaves its result in every thread of the row.  When the element a thread has just
  // finished is the very element every later read of that tensor in the kernel asks of it, the
  // readers use the register (the reference promotes such written scalars to registers,
  // memory_promotion_heuristic.cc:581-616).  That holds when each subscript, on both sides, is one
  // parallel variable that the two stages tile alike at kernel level and spread alike over the
  // blocks and over threadIdx.y/z with one point per thread.
  std::vector<std::string> forwardDecls;
  if (kc.opts.usePrivateMemoryValue) {
    auto findVar = [](const StagePlan& st, const std::string& name, int* pos) -> const LoopVar* {
      for (size_t v = 0; v < st.vars.size(); ++v) {
        if (st.vars[v].name == name) {
          *pos = static_cast<int>(v);
          return &st.vars[v];
        }
      }
      return nullptr;
    };
    // the single variable of a subscript `v + c`; null otherwise
    auto plainVar = [&](const StagePlan& st, const ExprRef& e, int* pos, int64_t* constant) -> const LoopVar* {
      Affine a = ir::toAffine(e);
      if (!a.valid) return nullptr;
      const LoopVar* found = nullptr;
      for (const auto& c : a.coef) {
        if (c.second == 0) continue;
        if (c.second != 1 || found) return nullptr;
        found = findVar(st, c.first, pos);
        if (!found) return nullptr;
      }
      *constant = a.constant;
      return found;
    };
    for (size_t i = 0; i + 1 < gens.size(); ++i) {
      const StagePlan& prod = k.stages[i];
      const std::string& t = prod.tensor;
      if (!prod.threadReduction || prod.atomic || prod.mfma || prod.accCount != 1) continue;
      // the first stage that writes the tensor; later ones may update the value in place (below)
      bool first = true;
      for (size_t j = 0; j < i; ++j) first &= k.stages[j].tensor != t;
      // (an epilogue of the producer may re-read the element it is finishing: its running value)
      bool readsOtherElements = false;
      for (const auto& stmt : prod.stmts) {
        visit(stmt.rhs, [&](const ExprRef& e) {
          if (e->kind != Expr::Load || e->name != t) return;
          bool same = e->args.size() == prod.lhsSubs.size();
          for (size_t d = 0; same && d < e->args.size(); ++d) same = sameExpr(e->args[d], prod.lhsSubs[d]);
          readsOtherElements |= !same;
        });
      }
      if (!first || readsOtherElements) continue;
      // the producer's side: one point per thread, rows along threadIdx.y/z only
      std::vector<const LoopVar*> pvars;
      std::vector<int> ppos;
      std::vector<int64_t> pconst;
      bool ok = true;
      bool axisUsed[3] = {false, false, false};
      for (const auto& sub : prod.lhsSubs) {
        int pos = -1;
        int64_t c = 0;
        const LoopVar* v = plainVar(prod, sub, &pos, &c);
        ok = ok && v && !v->reduction && !v->vectorLane && v->perThread == 1 && v->threadAxis != 0 &&
            (pos < k.sharedDepth || v->numTiles == 1);
        if (!ok) break;
        if (v->threadAxis > 0) axisUsed[v->threadAxis] = true;
        pvars.push_back(v);
        ppos.push_back(pos);
        pconst.push_back(c);
      }
      // a row of threads that works on no element of the tensor reduces nothing but identities
      for (int a = 1; a < 3 && ok; ++a) ok = k.block[a] == 1 || axisUsed[a];
      // A later stage addresses the element this thread holds: the same variable of the same
      // tiling in every subscript.  Where the producer's variable is on no thread axis, every
      // thread holds the value of the block's one point along it, and the reader's variable may
      // sit on a thread axis: its threads beyond the point compute on the clamped index.
      auto sameElement = [&](const StagePlan& cons, const std::vector<ExprRef>& subs) {
        bool same = subs.size() == pvars.size();
        for (size_t d = 0; same && d < pvars.size(); ++d) {
          int pos = -1;
          int64_t c = 0;
          const LoopVar* v = plainVar(cons, subs[d], &pos, &c);
          const LoopVar* w = pvars[d];
          same = v && c == pconst[d] && !v->reduction && !v->vectorLane && v->perThread == 1 && v->min == w->min &&
              v->extent == w->extent && v->tile == w->tile && v->numTiles == w->numTiles &&
              v->blockAxis == w->blockAxis && v->gridExtent == w->gridExtent &&
              (v->threadAxis == w->threadAxis || (w->threadAxis < 0 && v->tile == 1)) &&
              (v->numTiles == 1 || (pos == ppos[d] && pos < k.sharedDepth));
        }
        return same;
      };
      bool anyReader = false;
      int lastWriter = static_cast<int>(i);
      for (size_t j = i + 1; j < gens.size() && ok; ++j) {
        const StagePlan& cons = k.stages[j];
        const bool writes = cons.tensor == t;
        if (!writes && !tensorsRead(cons).count(t)) continue;
        anyReader = true;
        ok = cons.views.at(t).extents == prod.views.at(t).extents;
        if (writes) {
          // an update in place of the value the threads hold: pointwise, one element per thread
          bool pointwise = !cons.atomic && !cons.mfma && !cons.threadReduction && cons.accCount == 1;
          for (const auto& stmt : cons.stmts) pointwise &= stmt.redVars.empty();
          ok = ok && pointwise && sameElement(cons, cons.lhsSubs);
          lastWriter = static_cast<int>(j);
        }
        for (const auto& stmt : cons.stmts) {
          visit(stmt.rhs, [&](const ExprRef& e) {
            if (!ok || e->kind != Expr::Load || e->name != t) return;
            ok = sameElement(cons, e->args);
          });
        }
      }
      if (!anyReader || !ok) continue;
      KernelCtx::RegisterForward f;
      f.producer = static_cast<int>(i);
      f.lastWriter = lastWriter;
      f.name = "rfwd" + std::to_string(i) + "_" + t;
      forwardDecls.push_back(prod.views.at(t).type.cName() + " " + f.name + ";");
      kc.registerForwards[t] = f;
    }
  }
  // Producer -> consumer through LDS (useSharedMemory): a tensor exactly one stage of the kernel
  // writes and later stages read, when every reader's box of one kernel-level iteration lies inside
  // the producer's and that box fits what is left of LDS.  Stages see the tensor through views that
  // may merge dimensions differently: only identical views are matched.
  if (kc.opts.useSharedMemoryValue) {
    for (size_t i = 0; i + 1 < gens.size(); ++i) {
      const StagePlan& prod = k.stages[i];
      const std::string& t = prod.tensor;
      bool sole = true;
      for (size_t j = 0; j < k.stages.size(); ++j) sole &= j == i || k.stages[j].tensor != t;
      if (!sole || tensorsRead(prod).count(t) || kc.registerForwards.count(t)) continue;
      auto wbox = gens[i].writeBox();
      if (!wbox.valid) continue;
      bool anyReader = false, ok = true;
      for (size_t j = i + 1; j < gens.size() && ok; ++j) {
        if (!tensorsRead(k.stages[j]).count(t)) continue;
        anyReader = true;
        ok = k.stages[j].views.at(t).extents == prod.views.at(t).extents;
        auto rbox = ok ? gens[j].readBox(t) : StageCodegen::IterationBox();
        ok = ok && rbox.valid && rbox.low.size() == wbox.low.size();
        for (size_t d = 0; ok && d < wbox.low.size(); ++d) {
          int64_t delta = rbox.low[d].constant - wbox.low[d].constant;
          ok = rbox.low[d].coef == wbox.low[d].coef && delta >= 0 && delta + rbox.extents[d] <= wbox.extents[d];
        }
      }
      if (!anyReader || !ok) continue;
      KernelCtx::Forward f;
      f.producer = static_cast<int>(i);
      f.ldsName = "fwd" + std::to_string(i) + "_" + t;
      f.extents = wbox.extents;
      // pitches: one that is a multiple of the 32 banks puts the lanes (or the four lane groups
      // of a matrix-core operand read) that step along its dimension onto the same banks; four
      // elements more spread them and keep rows 16-byte aligned
      f.strides.assign(wbox.extents.size(), 1);
      for (size_t d = wbox.extents.size(); d-- > 1;) {
        f.strides[d - 1] = f.strides[d] * wbox.extents[d];
        if (f.strides[d - 1] % 32 == 0 && wbox.extents[d - 1] > 1) f.strides[d - 1] += 4;
      }
      f.elems = wbox.extents.empty() ? 1 : f.strides[0] * wbox.extents[0];
      int64_t bytes = f.elems * prod.views.at(t).type.bytes();
      if (bytes > ldsBudget) continue;
      ldsBudget -= bytes;
      for (const auto& low : wbox.low) f.lows.push_back(StageCodegen::tileAffineStr(low));
      kc.forwards[t] = f;
    }
  }
  k.ldsBytes = (before - ldsBudget) + scratchElems * 8;

  // Register promotion across stages (usePrivateMemory): an input that several stages read with
  // the same loop structure and addresses is loaded once, by the first of them, into a
  // per-thread register array that lives across the stages of one block iteration.
  std::vector<std::string> cacheDecls;
  if (kc.opts.usePrivateMemoryValue && gens.size() >= 2) {
    std::vector<std::string> sigs(gens.size());
    std::vector<std::vector<std::pair<std::string, std::string>>> loads(gens.size());
    for (size_t i = 0; i < gens.size(); ++i) sigs[i] = gens[i].cacheSignature(loads[i]);
    std::map<std::string, std::string> produced; // canonical load -> cache name
    for (size_t i = 0; i < gens.size(); ++i) {
      if (sigs[i].empty() || sigs[i] != sigs[0]) continue;
      if (gens[i].cacheSlots() > StageCodegen::kMaxCacheSlots) continue;
      for (const auto& l : loads[i]) {
        bool sharedLater = false;
        for (size_t j = 0; j < gens.size(); ++j) {
          if (j == i || sigs[j] != sigs[i]) continue;
          for (const auto& m : loads[j]) sharedLater |= m.first == l.first;
        }
        if (!sharedLater) continue;
        auto it = produced.find(l.first);
        bool producer = it == produced.end();
        if (producer) {
          std::string name = "rcache" + std::to_string(produced.size()) + "_";
          it = produced.emplace(l.first, name).first;
          std::string tensor = l.second.substr(1, l.second.find('[') - 1);
          cacheDecls.push_back(k.stages[i].views.at(tensor).type.cName() + " " + name + "[" +
                               std::to_string(gens[i].cacheSlots()) + "];");
        }
        gens[i].regCaches[l.second] = StageCodegen::RegCache{it->second, producer};
        gens[i].cachedStmt_ = gens[i].firstReduction();
      }
    }
  }

  // The same for a pointwise stage after a reduction over the same elements (normalise after
  // moments, say): when an operand's address forms agree, the reduction's single read of each
  // element fills the cache and the pointwise stage finds it there.
  if (kc.opts.usePrivateMemoryValue && gens.size() >= 2) {
    for (size_t j = 1; j < gens.size(); ++j) {
      const StagePlan& cs = k.stages[j];
      bool pointwise = !cs.mfma && !cs.threadReduction && gens[j].firstReduction() == nullptr;
      if (!pointwise) continue;
      for (const auto& stmt : cs.stmts) {
        if (stmt.op != ReduceOp::None) continue;
        visitUnconditional(stmt.rhs, [&](const ExprRef& e) {
          if (e->kind != Expr::Load || kc.registerForwards.count(e->name)) return; // (already in a register)
          StageCodegen::AddressForm want = gens[j].addressForm(e, nullptr);
          if (!want.valid || want.slots > StageCodegen::kMaxCacheSlots) return;
          std::string mine = "p" + e->name + "[" + gens[j].flatIndex(e->name, e->args, "") + "]";
          if (gens[j].regCaches.count(mine)) return;
          for (size_t i = 0; i < j; ++i) {
            const StageStmt* red = gens[i].firstReduction();
            if (!red || k.stages[i].mfma) continue;
            if (gens[i].cachedStmt_ && gens[i].cachedStmt_ != red) continue;
            std::string found;
            visitUnconditional(red->rhs, [&](const ExprRef& m) {
              if (m->kind != Expr::Load || !found.empty() || kc.registerForwards.count(m->name)) return;
              if (gens[i].addressForm(m, red) == want) {
                found = "p" + m->name + "[" + gens[i].flatIndex(m->name, m->args, "") + "]";
              }
            });
            if (found.empty()) continue;
            auto it = gens[i].regCaches.find(found);
            if (it == gens[i].regCaches.end()) {
              std::string name = "rcache" + std::to_string(cacheDecls.size()) + "_";
              cacheDecls.push_back(cs.views.at(e->name).type.cName() + " " + name + "[" + std::to_string(want.slots) + "];");
              it = gens[i].regCaches.emplace(found, StageCodegen::RegCache{name, true}).first;
              gens[i].cachedStmt_ = red;
            }
            gens[j].regCaches[mine] = StageCodegen::RegCache{it->second.name, false};
            gens[j].cachedPointwise_ = true;
            break;
          }
        });
      }
    }
  }

  em.open(kernelSignature(kc.f, k.name, kc.NT()));
  for (const auto& p : kc.f.params) em.line("(void)" + p.first + ";");
  em.line("const int tid_ = threadIdx.x + " + std::to_string(k.block[0]) + " * (threadIdx.y + " +
          std::to_string(k.block[1]) + " * threadIdx.z);");
  em.line("(void)tid_;");
  {
    // buffer descriptors (base, size in bytes, raw 32-bit data format) of the results that are
    // stored with write-through
    std::set<std::string> through, bounded; // (bounded: of the operands whose copies may pass the end of the tensor)
    for (size_t i = 0; i < gens.size(); ++i) {
      if (gens[i].streamedStore()) through.insert(k.stages[i].tensor);
      for (const auto& t : gens[i].boundedLoads()) {
        if (!bounded.insert(t).second) continue;
        em.line("const __amdgpu_buffer_rsrc_t " + StageCodegen::inputBufferName(t) + " = __builtin_amdgcn_make_buffer_rsrc((void*)p" +
                t + ", 0, " + std::to_string(gens[0].viewBytes(t)) + ", 0x00020000);");
      }
    }
    for (const auto& t : through) {
      em.line("const __amdgpu_buffer_rsrc_t " + StageCodegen::bufferName(t) + " = __builtin_amdgcn_make_buffer_rsrc((void*)p" +
              t + ", 0, " + std::to_string(gens[0].viewBytes(t)) + ", 0x00020000);");
    }
  }
  if (scratchElems > 0) {
    // one scratch area typed per use; sized for the widest element
    em.line("__shared__ double red_scratch_raw_[" + std::to_string(scratchElems) + "];");
  }
  for (auto& g : gens) g.emitLdsDecls();
  for (const auto& fw : kc.forwards) {
    em.line("__shared__ __attribute__((aligned(16))) " + k.stages[fw.second.producer].views.at(fw.first).type.cName() + " " +
            fw.second.ldsName + "[" + std::to_string(fw.second.elems) + "];");
  }
  // kernel-level tile loops over the shared parallel variables (taken from the first stage):
  // first the tile indices that are plain block ids, then the loops, outermost first
  int opened = 0;
  const StagePlan& s0 = k.stages.front();
  std::vector<const LoopVar*> loops;
  for (int i = 0; i < k.sharedDepth && i < s0.numParallel; ++i) {
    const LoopVar& v = s0.vars[i];
    if (v.vectorLane || v.numTiles == 1) continue;
    if (v.blockAxis >= 0 && v.gridExtent == v.numTiles) {
      em.line("const int t_" + v.name + " = blockIdx." + axisName(v.blockAxis) + ";");
    } else {
      loops.push_back(&v);
    }
  }
  kc.kernelLoops = !loops.empty();
  auto loopHeader = [&](const LoopVar& v, std::string& start, std::string& step) {
    start = v.blockAxis >= 0 ? std::string("blockIdx.") + axisName(v.blockAxis) : "0";
    step = v.blockAxis >= 0 ? std::to_string(v.gridExtent) : "1";
    std::string t = "t_" + v.name;
    return "for (int " + t + " = " + start + "; " + t + " < " + std::to_string(v.numTiles) + "; " + t + " += " + step + ")";
  };
  // Software pipeline over the innermost kernel-level loop (prefetchShared): the global loads of
  // the next tile's LDS footprints are issued before the current tile is computed and land in
  // registers; they are written to LDS after the computation, between two barriers.
  bool pipelined = false;
  if (kc.opts.prefetchSharedValue && k.stages.size() == 1 && !loops.empty() && !gens[0].promotions().empty()) {
    int64_t regs = 0;
    pipelined = true;
    for (const auto& p : gens[0].promotions()) {
      pipelined &= !p.insideReductionTiles;
      regs += gens[0].copyRegisters(p);
    }
    pipelined &= regs <= 96;
  }
  for (size_t li = 0; li < loops.size(); ++li) {
    const LoopVar& v = *loops[li];
    std::string start, step;
    std::string header = loopHeader(v, start, step);
    if (!(pipelined && li + 1 == loops.size())) {
      em.open(header);
      ++opened;
      continue;
    }
    StageCodegen& g = gens[0];
    std::string t = "t_" + v.name;
    em.open("");
    ++opened;
    for (const auto& p : g.promotions()) {
      em.line(g.copyRegisterDecl(p, "pf_" + p.tensor + "_"));
    }
    em.open("");
    em.line("const int " + t + " = " + start + ";");
    for (const auto& p : g.promotions()) {
      g.declareLows(p);
      g.emitCopyLoads(p, "pf_" + p.tensor + "_");
    }
    for (const auto& p : g.promotions()) g.emitCopyStores(p, "pf_" + p.tensor + "_");
    em.close();
    em.open(header);
    ++opened;
    em.line("__syncthreads();");
    em.line("const bool more_ = " + t + " + " + step + " < " + std::to_string(v.numTiles) + ";");
    em.open("if (more_)");
    g.tileOverride[v.name] = "(" + t + " + " + step + ")";
    for (const auto& p : g.promotions()) {
      g.declareLows(p);
      g.emitCopyLoads(p, "pf_" + p.tensor + "_");
    }
    g.tileOverride.clear();
    em.close();
    g.suppressCopy = true;
  }
  for (const auto& d : cacheDecls) em.line(d);
  for (const auto& d : forwardDecls) em.line(d);
  // Barriers between the stages: only where a later stage touches what an earlier one wrote (or
  // overwrites what it read) through different threads, at the weakest sufficient level, placed
  // by the exact search of sync_placement.h.  Every stage writes elements indexed by the
  // kernel-level loop variables and reads other stages' results at the same indices, so nothing
  // is carried from one iteration of those loops to the next.
  std::vector<int> syncAfter(k.stages.size(), 0);
  {
    const int n = static_cast<int>(k.stages.size());
    SyncNeeds need(n, std::vector<int>(n, 0));
    const int level = static_cast<int>(kc.NT() <= limits.wavefront ? SyncLevel::Wave : SyncLevel::Block);
    for (int i = 0; i < n; ++i) {
      for (int j = i + 1; j < n; ++j) {
        const StagePlan& a = k.stages[i];
        const StagePlan& b = k.stages[j];
        // (a result the later stage takes from a register is no dependence through memory)
        // (of its writers the last one alone stores it)
        auto inRegister = [&](const std::string& t) { return kc.registerForwards.count(t) > 0; };
        bool conflict = (a.tensor == b.tensor && !inRegister(a.tensor)) ||
            (tensorsRead(a).count(b.tensor) && !inRegister(b.tensor)) ||
            (tensorsRead(b).count(a.tensor) && !inRegister(a.tensor));
        if (conflict && !gens[j].readsPrivatelyFrom(a)) need[i][j - i] = level;
      }
    }
    for (const auto& sy : findBestSyncs(need, opened > 0)) syncAfter[sy.first] = static_cast<int>(sy.second);
    // a producer's copy in LDS is overwritten by the next kernel-level iteration: not before the
    // readers of this one are done
    if (opened > 0 && !kc.forwards.empty()) syncAfter.back() = std::max(syncAfter.back(), level);
  }
  auto emitSync = [&](int level) {
    if (level == static_cast<int>(SyncLevel::Block)) {
      em.line("__syncthreads();");
    } else if (level == static_cast<int>(SyncLevel::Wave)) {
      // the block is a single wavefront: order its memory operations, no hardware barrier
      em.line("__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, \"wavefront\");");
      em.line("__builtin_amdgcn_wave_barrier();");
    }
  };
  for (size_t i = 0; i < k.stages.size(); ++i) {
    if (i > 0) emitSync(syncAfter[i - 1]);
    if (k.stages[i].threadReduction) {
      em.open("");
      em.line(k.stages[i].views.at(k.stages[i].tensor).type.cName() + "* red_scratch_ = (" +
              k.stages[i].views.at(k.stages[i].tensor).type.cName() + "*)red_scratch_raw_;");
      gens[i].emit();
      em.close();
    } else {
      gens[i].emit();
    }
  }
  if (pipelined) {
    StageCodegen& g = gens[0];
    em.line("__syncthreads();");
    em.open("if (more_)");
    std::string start, step;
    loopHeader(*loops.back(), start, step);
    g.tileOverride[loops.back()->name] = "(t_" + loops.back()->name + " + " + step + ")";
    for (const auto& p : g.promotions()) {
      if (g.copyPlan(p).shifted) g.declareLows(p); // (the shift follows from the place of the tile that was requested)
      g.emitCopyStores(p, "pf_" + p.tensor + "_");
    }
    g.tileOverride.clear();
    em.close();
  }
  emitSync(syncAfter.back());
  for (int i = 0; i < opened; ++i) em.close();
  em.close();
}

} // namespace

namespace {
// e + c with the constant folded into an existing "+ constant"
ExprRef addConstant(const ExprRef& e, int64_t c) {
  if (e->kind == Expr::IntImm) return mkInt(e->ival + c);
  if (e->kind == Expr::Binary && e->name == "+" && e->args[1]->kind == Expr::IntImm) {
    return addConstant(e->args[0], e->args[1]->ival + c);
  }
  return c == 0 ? e : mkBin("+", e, mkInt(c));
}

// The storage of an output starts at its inferred lower bound: element k of dimension d holds
// the point mins[d] + k, the way a Halide buffer with a non-zero min is addressed (the bounds
// are set in tc/core/tc2halide.cc:903).  Rewrites the function to zero-based outputs: an index
// variable that subscripts a shifted dimension on the left-hand side is shifted by the bound
// (range and every use), and every other subscript of such a tensor has the bound subtracted.
ir::Function withZeroBasedOutputs(const ir::Function& in) {
  ir::Function f = in;
  std::map<std::string, std::vector<int64_t>> mins;
  for (auto& t : f.outputs) {
    mins[t.name] = t.mins;
    std::fill(t.mins.begin(), t.mins.end(), 0);
  }
  for (auto& s : f.statements) {
    std::map<std::string, int64_t> shift;
    const auto& m = mins.at(s.tensor);
    for (size_t d = 0; d < s.lhsVars.size(); ++d) {
      auto it = shift.find(s.lhsVars[d]);
      TC_CHECK(it == shift.end() || it->second == m[d])
          << "index " << s.lhsVars[d] << " subscripts two dimensions of " << s.tensor << " with different lower bounds";
      shift[s.lhsVars[d]] = m[d];
    }
    for (const auto& sh : shift) {
      ir::Range& r = s.ranges.at(sh.first);
      r.min -= sh.second;
      r.max -= sh.second;
    }
    s.rhs = rewrite(s.rhs, [&](const ExprRef& e) -> ExprRef {
      if (e->kind == Expr::Var) {
        auto it = shift.find(e->name);
        return it == shift.end() || it->second == 0 ? nullptr : mkBin("+", e, mkInt(it->second));
      }
      if (e->kind == Expr::Load) {
        auto it = mins.find(e->name);
        if (it == mins.end()) return nullptr;
        auto c = std::make_shared<Expr>(*e);
        for (size_t d = 0; d < c->args.size(); ++d) c->args[d] = addConstant(c->args[d], -it->second[d]);
        return c;
      }
      return nullptr;
    });
  }
  return f;
}
// reductionBlocks: a reduction `O(p...) op=(!) rhs` is divided among blocks along its outermost
// reduction index r (extent E, `split` = the largest divisor of E not above `blocks`):
//     O(p...) = identity of op                       only for "op=!", a kernel of its own
//     O(p...) op= rhs[r := r + (E / split) * slice]   slice in 0:split, r in 0:E/split
// where `slice` becomes the outermost parallel variable of the second statement and its partial
// results are combined into O atomically.  Floating-point sums then depend on the order in which the
// blocks arrive (within the rounding of any other summation order); integer sums do not.
// The identity of a reduction operator as an expression of the given 32- or 64-bit type (values
// an integer literal cannot spell are formed by an operation: 0 - 1 for the largest uint64).
ExprRef identityExpr(ReduceOp op, const ScalarType& t) {
  auto imm = [&](double f, int64_t i) {
    auto e = std::make_shared<Expr>();
    e->kind = t.isFloat() ? Expr::FloatImm : Expr::IntImm;
    e->type = t;
    e->fval = f;
    e->ival = i;
    return ExprRef(e);
  };
  auto minus = [&](const ExprRef& a, const ExprRef& b) { return mkExpr(Expr::Binary, t, "-", {a, b}); };
  if (op == ReduceOp::Plus) return imm(0.0, 0);
  if (op == ReduceOp::Times) return imm(1.0, 1);
  const bool largest = op == ReduceOp::Min; // a minimum starts from the largest value of the type
  if (t.isFloat()) {
    double m = t.bits == 64 ? std::numeric_limits<double>::max() : static_cast<double>(std::numeric_limits<float>::max());
    return imm(largest ? m : -m, 0);
  }
  if (t.code == ScalarType::UInt) {
    if (!largest) return imm(0.0, 0);
    return t.bits == 64 ? minus(imm(0.0, 0), imm(0.0, 1)) : imm(0.0, (int64_t(1) << t.bits) - 1);
  }
  const int64_t top = t.bits == 64 ? std::numeric_limits<int64_t>::max() : (int64_t(1) << (t.bits - 1)) - 1;
  return largest ? imm(0.0, top) : minus(imm(0.0, -top), imm(0.0, 1));
}

ir::Function withSplitReductions(const ir::Function& in, int64_t blocks) {
  ir::Function f = in;
  f.statements.clear();
  int counter = 0;
  for (const auto& s : in.statements) {
    const ir::Tensor* t = in.find(s.tensor);
    bool ok = t && s.op != ReduceOp::None && !s.redVars.empty() && accessesTo(s, s.tensor).empty() &&
        (t->type.bits == 32 || t->type.bits == 64);
    int64_t split = 1, extent = 0;
    if (ok) {
      extent = s.ranges.at(s.redVars[0]).extent();
      for (int64_t d = std::min<int64_t>(blocks, extent); d >= 2; --d) {
        if (extent % d == 0) {
          split = d;
          break;
        }
      }
    }
    if (split < 2) {
      f.statements.push_back(s);
      continue;
    }
    std::string slice;
    do {
      slice = "slice" + std::to_string(counter++);
    } while (s.ranges.count(slice));
    if (s.init) {
      ir::Statement zero;
      zero.tensor = s.tensor;
      zero.lhsVars = s.lhsVars;
      zero.zeroing = true;
      for (const auto& v : s.lhsVars) zero.ranges[v] = s.ranges.at(v);
      zero.type = t->type;
      zero.tree = s.tree;
      zero.rhs = identityExpr(s.op, t->type);
      f.statements.push_back(zero);
    }
    ir::Statement part = s;
    part.init = false;
    part.atomic = true;
    part.sliceVar = slice;
    part.lhsVars.insert(part.lhsVars.begin(), part.sliceVar);
    part.ranges[part.sliceVar] = ir::Range{0, split - 1};
    const std::string r = s.redVars[0];
    const int64_t chunk = extent / split;
    ir::Range& rr = part.ranges.at(r);
    rr.max = rr.min + chunk - 1;
    part.rhs = rewrite(s.rhs, [&](const ExprRef& e) -> ExprRef {
      if (e->kind != Expr::Var || e->name != r) return nullptr;
      return mkBin("+", e, mkBin("*", mkVar(part.sliceVar), mkInt(chunk)));
    });
    f.statements.push_back(part);
  }
  return f;
}
} // namespace

namespace {
HipMappingOptions fillMappingOptions(const HipMappingOptions& given) {
  HipMappingOptions o = given;
  o.tile(std::vector<uint64_t>{1024}).unroll(4).matchLibraryCalls(false);
  o.mapToThreads(256).mapToBlocks(1 << 20).useSharedMemory(false).usePrivateMemory(false);
  o.vectorWidth(4).collapseContiguous(true).useMfma(false).prefetchShared(false);
  return o;
}

// A point-wise stage whose dimensions all merged into one, every operand read at the element that
// is written: a stream.
bool isStream(const StagePlan& st) {
  if (st.vars.size() != 1 || st.numParallel != 1 || st.atomic) return false;
  auto alongTheStream = [&](const std::vector<ExprRef>& subs) {
    if (subs.size() != 1) return false;
    Affine a = ir::toAffine(subs[0]);
    return a.valid && a.coefOf(st.vars[0].name) == 1;
  };
  bool ok = alongTheStream(st.lhsSubs);
  for (const auto& s : st.stmts) {
    ok = ok && s.redVars.empty();
    visit(s.rhs, [&](const ExprRef& e) {
      if (e->kind == Expr::Load && !e->args.empty()) ok = ok && alongTheStream(e->args);
    });
  }
  return ok;
}

// Product of thread or block sizes.  Those of a stream are nominal: a product beyond what the device
// takes (64 x 64 threads on two loops) is cut.
uint64_t boundedProduct(const std::array<uint64_t, 3>& sizes, uint64_t most) {
  uint64_t product = 1;
  for (uint64_t s : sizes) product = s == 0 ? 0 : product > most / s ? most : product * s;
  return product;
}
// Options for a stream whose given options leave threads of the block unused: sizes for two or
// three loops say little about the one loop that merging left (tile 32, 64 x 4 threads and 256 x
// 256 blocks put 32 threads in each of 256 blocks, every one of which walks thousands of tiles).  It
// gets all the threads of the block in lanes of four, one lane group each, and as many of the blocks
// as that takes (a residual sum of 6.3 M floats under the naive options: 203 -> 12.5 us; lanes of four
// where the extent is a multiple of four, else the threads step through the tile).  32-bit results
// are stored with write-through (11.4 -> 9.5 us); lanes of one, two or eight bytes would each be a store
// of their own on its way to memory (6.3 M halves 12.9 us against 5.4, doubles 37.7 against 22.0,
// bytes 7.5 against 3.7), so results of other widths keep the given option.
HipMappingOptions streamMappingOptions(const HipMappingOptions& given, const DeviceLimits& limits, bool words) {
  HipMappingOptions o = given;
  const uint64_t threads = boundedProduct({{o.block[0], o.block[1], o.block[2]}}, limits.maxThreadsPerBlock);
  o.tile(std::vector<uint64_t>{4 * threads}).unroll(4).useSharedMemory(false);
  o.mapToThreads(threads).mapToBlocks(boundedProduct({{o.grid[0], o.grid[1], o.grid[2]}}, std::numeric_limits<int32_t>::max()));
  o.vectorWidth(4);
  if (words) o.useReadOnlyCache(true);
  return o;
}
bool leavesThreadsOfAStreamUnused(const HipMappingOptions& o, const StagePlan& st, const DeviceLimits& limits) {
  const uint64_t threads = boundedProduct({{o.block[0], o.block[1], o.block[2]}}, limits.maxThreadsPerBlock);
  uint64_t tile = o.generic.hasTiling && !o.generic.tiling.empty() ? o.generic.tiling[0] : 0;
  if (tile == 0) tile = static_cast<uint64_t>(st.vars[0].extent);
  return threads >= 64 && std::min<uint64_t>(o.block[0], tile / o.vectorWidthValue) < threads;
}
} // namespace

MappedProgram mapToHip(
    const ir::Function& given,
    const HipMappingOptions& optionsIn,
    const std::string& specializedName,
    const DeviceLimits& limits) {
  // Range inference accepts `where i in 8:4` and reports a negative extent, as the reference's does
  // (test/test_inference.cc:498-511: "silently infers a negative size"); nothing can be launched
  // over such a range.
  for (const auto& s : given.statements) {
    for (const auto& r : s.ranges) {
      if (r.second.max < r.second.min) {
        throw lang::errorAt(s.tree) << "Empty range for variable " << r.first << ": " << r.second.min << ":" << r.second.max + 1;
      }
    }
  }
  bool shifted = false;
  for (const auto& t : given.outputs) {
    for (auto m : t.mins) shifted |= m != 0;
  }
  const ir::Function zeroBased = shifted ? withZeroBasedOutputs(given) : ir::Function();
  const bool divided = optionsIn.reductionBlocksValue > 1;
  const ir::Function dividedSums =
      divided ? withSplitReductions(shifted ? zeroBased : given, optionsIn.reductionBlocksValue) : ir::Function();
  const ir::Function& f = divided ? dividedSums : shifted ? zeroBased : given;
  // 1. stages
  std::vector<RawStage> raw;
  bool allowStageFusion = optionsIn.generic.intraTileScheduleOptions.fusionStrategy != FusionStrategy::Min ||
      optionsIn.generic.outerScheduleOptions.fusionStrategy != FusionStrategy::Min;
  for (const auto& s : f.statements) {
    for (const auto& subs : accessesTo(s, s.tensor)) {
      TC_CHECK(isIdentityAccess(subs, s.lhsVars))
          << "statement on " << s.tensor << " reads its own output at other points; not supported";
    }
    bool merged = false;
    if (!raw.empty() && allowStageFusion && sameBox(raw.back().first(), s)) {
      raw.back().stmts.push_back(&s);
      merged = true;
    }
    if (!merged) {
      RawStage r;
      r.stmts.push_back(&s);
      raw.push_back(r);
    }
  }
  // 2. kernels
  struct Group {
    std::vector<size_t> stages;
    int depth;
  };
  std::vector<Group> groups;
  FusionStrategy fs = optionsIn.generic.outerScheduleOptions.fusionStrategy;
  for (size_t i = 0; i < raw.size(); ++i) {
    bool joined = false;
    if (!groups.empty() && fs != FusionStrategy::Min) {
      Group& g = groups.back();
      int d = g.depth;
      for (size_t j : g.stages) {
        d = std::min(d, sharedPrefix(raw[j], raw[i]));
      }
      int need = 1;
      if (fs == FusionStrategy::Preserve3Coincident) {
        size_t rank = raw[i].first().lhsVars.size();
        for (size_t j : g.stages) rank = std::min(rank, raw[j].first().lhsVars.size());
        need = static_cast<int>(std::min<size_t>(3, rank));
      }
      if (d >= need && d >= 1) {
        g.stages.push_back(i);
        g.depth = d;
        joined = true;
      }
    }
    if (!joined) {
      groups.push_back(Group{{i}, static_cast<int>(raw[i].first().lhsVars.size())});
    }
  }
  // 3. plans
  MappedProgram prog;
  for (const auto& p : f.params) {
    prog.paramNames.push_back(p.first);
    prog.paramValues.push_back(p.second);
  }
  // Loop variables and size parameters are 32-bit: every single extent must fit; a tensor as a
  // whole may hold 2^31 elements or more, element offsets are then formed in 64 bits.
  int64_t maxNumel = 0;
  for (const auto* ts : {&f.inputs, &f.outputs}) {
    for (const auto& t : *ts) {
      maxNumel = std::max(maxNumel, t.numel());
      for (auto e : t.extents) {
        TC_CHECK_LT(e, (1LL << 31)) << "tensor " << t.name << " has a dimension of 2^31 or more elements; not supported";
      }
    }
  }
  const bool wide = maxNumel >= (1LL << 31);

  // The fill that precedes a divided sum: all dimensions merged, four elements per thread, 256
  // threads, as many blocks as that takes.
  HipMappingOptions fillOptions = fillMappingOptions(optionsIn);
  const HipMappingOptions streamOptions[2] = {streamMappingOptions(optionsIn, limits, false), streamMappingOptions(optionsIn, limits, true)};
  std::vector<const HipMappingOptions*> kernelOptions;
  bool anyThreadReduction = false;
  std::vector<std::unique_ptr<Emitter>> bodies;
  for (size_t gi = 0; gi < groups.size(); ++gi) {
    const bool fill = groups[gi].stages.size() == 1 && raw[groups[gi].stages[0]].first().zeroing;
    const HipMappingOptions* chosen = fill ? &fillOptions : &optionsIn;
    KernelPlan k;
    k.name = specializedName + (gi == 0 ? "" : "_k" + std::to_string(gi));
    bool single = groups[gi].stages.size() == 1;
    for (size_t si : groups[gi].stages) {
      StageBuilder b(f);
      b.init(raw[si]);
      if (chosen->collapseContiguousValue) b.collapse(single ? 0 : static_cast<size_t>(groups[gi].depth));
      k.stages.push_back(std::move(b.st));
    }
    // (a definition of one dimension is mapped as its options say)
    if (!fill && single && raw[groups[gi].stages[0]].first().lhsVars.size() > 1 && isStream(k.stages[0]) && leavesThreadsOfAStreamUnused(optionsIn, k.stages[0], limits)) {
      chosen = &streamOptions[k.stages[0].views.at(k.stages[0].tensor).type.bits == 32];
    }
    const HipMappingOptions& options = *chosen;
    kernelOptions.push_back(chosen);
    k.sharedDepth = single ? k.stages[0].numParallel : groups[gi].depth;
    // later stages of a fused kernel adopt the first stage's names for the shared variables;
    // their other variables get a stage suffix so nothing can collide
    for (size_t si = 1; si < k.stages.size(); ++si) {
      StagePlan& st = k.stages[si];
      std::map<std::string, std::string> ren;
      for (size_t vi = 0; vi < st.vars.size(); ++vi) {
        ren[st.vars[vi].name] = static_cast<int>(vi) < k.sharedDepth
            ? k.stages[0].vars[vi].name
            : st.vars[vi].name + "_s" + std::to_string(si);
      }
      auto sub = [&](const ExprRef& e) -> ExprRef {
        return e->kind == Expr::Var ? mkVar(ren.at(e->name)) : nullptr;
      };
      for (auto& v : st.vars) v.name = ren.at(v.name);
      for (auto& e : st.lhsSubs) e = rewrite(e, sub);
      for (auto& ss : st.stmts) {
        ss.rhs = rewrite(ss.rhs, sub);
        for (auto& r : ss.redVars) r = ren.at(r);
      }
    }
    if (options.useMfmaValue) {
      for (auto& st : k.stages) classifyContraction(st);
    }
    // vector lanes on the variable that will sit on threadIdx.x
    if (options.vectorWidthValue > 1) {
      for (auto& st : k.stages) {
        if (st.mfma) continue;
        bool hasRed = false;
        for (const auto& s : st.stmts) hasRed |= !s.redVars.empty();
        bool threadRed = options.generic.matchLibraryCallsValue && hasRed && options.block[0] > 1;
        std::string target;
        if (threadRed) {
          target = st.vars.back().name;
        } else if (st.numParallel > 0) {
          target = st.vars[st.numParallel - 1].name;
        }
        // the shared prefix must keep its shape in every stage
        bool inPrefix = !threadRed && !single && st.numParallel - 1 < k.sharedDepth;
        if (!target.empty() && !inPrefix) {
          StageBuilder b(f);
          b.st = std::move(st);
          int before = b.st.numParallel;
          b.splitLanes(target, options.vectorWidthValue);
          if (single) k.sharedDepth += b.st.numParallel - before;
          st = std::move(b.st);
        }
      }
    }
    prog.kernels.push_back(std::move(k));
  }
  std::ostringstream src;
  for (size_t ki = 0; ki < prog.kernels.size(); ++ki) {
    KernelPlan& k = prog.kernels[ki];
    KernelCtx kc{f, *kernelOptions[ki], k};
    kc.wide = wide;
    if (wide) kc.idx = "int64";
    mapKernel(kc, limits);
    for (const auto& st : k.stages) anyThreadReduction |= st.threadReduction || st.atomic;
    bodies.emplace_back(new Emitter());
    emitKernel(kc, limits, *bodies.back());
  }
  src << "// generated by the TC HIP mapper for gfx950; function " << f.name << "\n";
  bool halfProducts = false, largeHalfProducts = false, splitConvolutions = false, slicedProducts = false, columnSums = false;
  for (const auto& b : bodies) {
    halfProducts |= b->out.str().find("__tc::multiplyHalves(") != std::string::npos;
    largeHalfProducts |= b->out.str().find("__tc::largeHalfProduct<") != std::string::npos;
    splitConvolutions |= b->out.str().find("__tc::SplitConvolution<") != std::string::npos;
    slicedProducts |= b->out.str().find("__tc::SlicedProduct<") != std::string::npos;
    columnSums |= b->out.str().find("__tc::columnSums<") != std::string::npos;
  }
  src << hip::deviceLibrary(anyThreadReduction, halfProducts, largeHalfProducts);
  if (splitConvolutions || slicedProducts) src << hip::kDeviceSplitParts;
  if (splitConvolutions) src << hip::kDeviceSplitConvolution;
  if (slicedProducts) src << hip::kDeviceSlicedProduct;
  if (columnSums) src << hip::kDeviceColumnSums;
  for (const auto& b : bodies) src << "\n" << b->out.str();
  prog.source = src.str();
  return prog;
}

} // namespace mapper
} // namespace tc
