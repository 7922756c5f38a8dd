// cuttPlanMeasure on a device whose clock is simulated (no GPU): launches take the time a scenario says, events read
// that clock, everything else is fake_hip_layer.cpp.  Prints the plan that came out.
//   cold      - the first launch of every kernel instance takes 400 us longer (its code has to be loaded); afterwards a
//               Packed plan takes 6 us, all others 10 us
//   plain     - a tensor that the rules give line-aligned stores: 64x64 tiles take 60 us in the planner's own tile order
//               and with its cache policy, 130 us in any other form; line-aligned ones 100 us, Packed plans 90 us
//   lines     - a tensor that the rules give 64x64 tiles: line-aligned stores take 60 us in their own order and with
//               their own cache policy, 130 us in any other form; 64x64 tiles 100 us, Packed plans 90 us
//   accesses  - no timing: the plan cuttPlan makes for two tensors of 4-byte elements off the line grid with short output
//               rows, once as it is and once with the cache policy pinned to non-temporal loads
//   predicted - no timing: prints what cuttPlan expects of its plan for one tensor, with and without row gathering
//   groups    - Tiled plans numbered by address bits, whose XCDs each have a part of their own, 50 us, all others 100 us: prints how
//               often the winner was launched
//   narrow    - wide tiles 100 us, 64x64 tiles in tile order 6 40 us in patches of 2 x 2 and 41 us in others, 60 us in any other order:
//               prints how often one plan in order 6 other than the winner was launched
//   tie98, tie99 - Packed plans: the one cuttPlan makes 100 us, all others 98 or 99.5 us; prints the policy of cuttPlan's plan
//   bits      - PackedSplit plans: work items numbered by address bits 50 us, others 100 us, for a tensor that cuttPlan numbers the other way
//   nobits    - the same for one whose plan cuttPlan numbers by address bits: these 100 us, others in groups of workgroups 50 us, 120 us in chunks
//   drift     - line-aligned Tiled plans 100 us, others 200 us, every launch a little less than the one before
#define cuttHipEventCreate fakeEventCreate
#define cuttHipEventDestroy fakeEventDestroy
#define cuttHipEventRecord fakeEventRecord
#define cuttHipEventElapsedMs fakeEventElapsedMs
#define cuttHipLaunchTiled fakeLaunchTiled
#define cuttHipLaunchTiledCopy fakeLaunchTiledCopy
#define cuttHipLaunchPacked fakeLaunchPacked
#include "fake_hip_layer.cpp"
#undef cuttHipEventCreate
#undef cuttHipEventDestroy
#undef cuttHipEventRecord
#undef cuttHipEventElapsedMs
#undef cuttHipLaunchTiled
#undef cuttHipLaunchTiledCopy
#undef cuttHipLaunchPacked

#include <cstdio>
#include <functional>
#include <map>
#include <set>
#include <string>

#include "cutt.h"
#include "cutt_ext.h"

static double gNow = 0;  // us
static long gLaunches = 0;

// What a launch takes, from its arguments; `instance` names the kernel instance.
static std::function<double(const cuttHipTiledArgs&)> gTiledUs;
static std::function<double(const cuttHipTiledCopyArgs&)> gCopyUs;
static std::function<double(const cuttHipPackedArgs&)> gPackedUs;
static double gColdUs = 0;
static std::set<std::string> gUsed;

static int launched(const std::string& instance, double us) {
  gLaunches++;
  gNow += us + (gUsed.insert(instance).second ? gColdUs : 0.0);
  return 0;
}

extern "C" {
int cuttHipEventCreate(void** event) { *event = new double(0); return 0; }
int cuttHipEventDestroy(void* event) { delete (double*)event; return 0; }
int cuttHipEventRecord(void* event, void*) { *(double*)event = gNow; return 0; }
int cuttHipEventElapsedMs(void* start, void* stop, float* ms) { *ms = (float)((*(double*)stop - *(double*)start) * 1e-3); return 0; }
int cuttHipLaunchTiled(const cuttHipTiledArgs* a, const void*, void*, void*) {
  return launched("tiled " + std::to_string(a->elemSize) + (a->lineWidth ? " lines" : "") + (a->grouped ? " grouped" : "") +
                  (a->rowsK.n > 0 || a->rowsM.n > 0 ? " fused" : "") + " policy " + std::to_string(a->cachePolicy), gTiledUs(*a));
}
int cuttHipLaunchTiledCopy(const cuttHipTiledCopyArgs* a, const void*, void*, void*) {
  return launched((a->rowGather ? "rows " : "copy ") + std::to_string(a->rowGather ? a->rows.cachePolicy : a->tiles.cachePolicy), gCopyUs(*a));
}
int cuttHipLaunchPacked(const cuttHipPackedArgs* a, const void*, void*, void*) {
  return launched("packed " + std::to_string(a->elemSize) + " " + std::to_string(a->elemsPerThread) + " policy " + std::to_string(a->cachePolicy), gPackedUs(*a));
}
}

static bool oneSlab(const cuttHipPackedArgs& a) { return a.split[0].numSplit == 1 && a.split[1].numSplit == 1; }

static int measure(std::vector<int> dim, std::vector<int> perm, int es) {
  char in, out;
  cuttHandle h;
  const cuttResult rc = cuttPlanMeasure(&h, (int)dim.size(), dim.data(), perm.data(), es, 0, &in, &out);
  if (rc != CUTT_SUCCESS) { std::printf("failed %d\n", (int)rc); return 1; }
  cuttPlanInfo i;
  if (cuttGetPlanInfo(h, &i) != CUTT_SUCCESS) return 1;
  std::printf("method %d measured %.2f policy %d order %d super %dx%d lines %d grouped %d launches %ld\n", i.method, i.usMeasured, i.cachePolicy,
              i.tiledOrder, i.superM, i.superK, i.tiledAligned, i.tiledGrouped, gLaunches);
  return cuttDestroy(h) == CUTT_SUCCESS ? 0 : 1;
}

static int cold() {
  gColdUs = 400;
  gTiledUs = [](const cuttHipTiledArgs&) { return 10.0; };
  gCopyUs = [](const cuttHipTiledCopyArgs&) { return 10.0; };
  gPackedUs = [](const cuttHipPackedArgs& a) { return oneSlab(a) ? 6.0 : 10.0; };
  return measure({100, 20, 40, 30}, {2, 1, 3, 0}, 8);
}

// What the planner makes of a Tiled plan with line-aligned stores, or without.
static cuttPlanInfo ownForm(std::vector<int> dim, std::vector<int> perm, int es, bool lines) {
  cuttHandle h;
  cuttPlanInfo i = {};
  setenv("CUTT_TILED_ALIGNED", lines ? "1" : "0", 1);
  cuttSetMethodOverride(CUTT_METHOD_TILED);
  if (cuttPlan(&h, (int)dim.size(), dim.data(), perm.data(), es, 0) != CUTT_SUCCESS || cuttGetPlanInfo(h, &i) != CUTT_SUCCESS) std::exit(1);
  cuttDestroy(h);
  cuttSetMethodOverride(0);
  unsetenv("CUTT_TILED_ALIGNED");
  std::printf("own form: order %d super %dx%d policy %d lines %d\n", i.tiledOrder, i.superM, i.superK, i.cachePolicy, i.tiledAligned);
  return i;
}

static int otherForm(std::vector<int> dim, std::vector<int> perm, int es, bool lines) {
  const cuttPlanInfo own = ownForm(dim, perm, es, lines);
  gTiledUs = [=](const cuttHipTiledArgs& a) {
    if ((a.lineWidth > 0) != lines) return 100.0;
    return a.order == own.tiledOrder && (int)a.superM == own.superM && (int)a.superK == own.superK && a.cachePolicy == own.cachePolicy ? 60.0 : 130.0;
  };
  gPackedUs = [](const cuttHipPackedArgs&) { return 90.0; };
  return measure(dim, perm, es);
}

static int drift() {
  gTiledUs = [](const cuttHipTiledArgs& a) { return (a.lineWidth ? 100.0 : 200.0) * (1.0 - 1e-5 * gLaunches); };
  gPackedUs = [](const cuttHipPackedArgs&) { return 200.0; };
  return measure({1201, 30011}, {1, 0}, 8);
}

static int tie(double othersUs) {
  int dim[4] = {1544, 426, 76, 4}, perm[4] = {2, 0, 1, 3};
  cuttHandle h;
  cuttPlanInfo own = {};
  if (cuttPlan(&h, 4, dim, perm, 8, 0) != CUTT_SUCCESS || cuttGetPlanInfo(h, &own) != CUTT_SUCCESS) return 1;
  cuttDestroy(h);
  std::printf("own policy %d\n", own.cachePolicy);
  gTiledUs = [](const cuttHipTiledArgs&) { return 200.0; };
  gPackedUs = [=](const cuttHipPackedArgs& a) {
    return a.split[0].numSplit == own.numSplit && a.cachePolicy == own.cachePolicy ? 100.0 : othersUs;
  };
  return measure({1544, 426, 76, 4}, {2, 0, 1, 3}, 8);
}

static int groups() {
  setenv("CUTT_MEASURE_NO_PLAYOFF", "1", 1);
  std::map<std::string, int> launches;
  gTiledUs = [&](const cuttHipTiledArgs& a) {
    if (a.order == 7) launches[std::string((const char*)static_cast<const void*>(&a), sizeof(a))]++;
    return a.order == 7 ? 50.0 : 100.0;
  };
  gPackedUs = [](const cuttHipPackedArgs&) { return 100.0; };
  if (measure({1024, 64, 1024, 3}, {2, 1, 0, 3}, 8)) return 1;
  int most = 0;
  for (const auto& l : launches) most = std::max(most, l.second);
  std::printf("most launches of one plan %d\n", most);
  return 0;
}

static int narrow() {
  setenv("CUTT_MEASURE_NO_PLAYOFF", "1", 1);
  std::map<std::string, int> launches;
  gTiledUs = [&](const cuttHipTiledArgs& a) {
    if (a.wide) return 100.0;
    if (a.order != 6) return 60.0;
    const bool first = a.superM == 2 && a.superK == 2;
    if (!first) launches[std::string((const char*)static_cast<const void*>(&a), sizeof(a))]++;
    return first ? 40.0 : 41.0;
  };
  gPackedUs = [](const cuttHipPackedArgs&) { return 100.0; };
  cuttSetMethodOverride(CUTT_METHOD_TILED);
  if (measure({1024, 1024, 96}, {1, 0, 2}, 4)) return 1;
  int most = 0;
  for (const auto& l : launches) most = std::max(most, l.second);
  std::printf("most launches of one plan %d\n", most);
  return 0;
}

static int bits(std::vector<int> dim, std::vector<int> perm, int es, double numbered, double inGroups, double inChunks) {
  cuttSetMethodOverride(CUTT_METHOD_PACKEDSPLIT);
  cuttHandle h;
  cuttPlanInfo own = {};
  if (cuttPlan(&h, (int)dim.size(), dim.data(), perm.data(), es, 0) != CUTT_SUCCESS || cuttGetPlanInfo(h, &own) != CUTT_SUCCESS) return 1;
  cuttDestroy(h);
  std::printf("own numbered %d group %d\n", own.tileDigits[0] != 0, own.xcdGroup);
  // (a numbering by digits leaves no cut ranks; blocks of another size are slower)
  gPackedUs = [=](const cuttHipPackedArgs& a) { return cuttHipPackedLdsBytes(&a) != own.ldsBytes ? 150.0 : oneSlab(a) ? numbered : (a.xcdGroup ? inGroups : inChunks); };
  return measure(dim, perm, es);
}

static int predicted() {
  int dim[7] = {18, 39, 13, 100, 2, 3, 25}, perm[7] = {0, 3, 1, 6, 5, 2, 4};
  for (const char* gather : {"1", "0"}) {
    setenv("CUTT_ROW_GATHER", gather, 1);
    cuttHandle h;
    cuttPlanInfo i = {};
    if (cuttPlan(&h, 7, dim, perm, 4, 0) != CUTT_SUCCESS || cuttGetPlanInfo(h, &i) != CUTT_SUCCESS) return 1;
    std::printf("predicted %.4f gathered %d\n", i.usPredicted, i.rowGather);
    cuttDestroy(h);
  }
  return 0;
}

static int accesses() {
  for (const char* policy : {"", "1"}) {
    if (*policy) setenv("CUTT_CACHE_POLICY", policy, 1);
    for (std::vector<int> dim : {std::vector<int>{772, 586, 304}, std::vector<int>{643, 703, 331}}) {
      int perm[3] = {2, 1, 0};
      cuttHandle h;
      cuttPlanInfo i = {};
      setenv("CUTT_TILED_ALIGNED", "0", 1);
      if (cuttPlan(&h, 3, dim.data(), perm, 4, 0) != CUTT_SUCCESS || cuttGetPlanInfo(h, &i) != CUTT_SUCCESS) return 1;
      std::printf("accesses method %d policy %d grouped %d\n", i.method, i.cachePolicy, i.tiledGrouped);
      cuttDestroy(h);
    }
  }
  return 0;
}

int main(int argc, char** argv) {
  const std::string what = argc > 1 ? argv[1] : "";
  if (what == "cold") return cold();
  if (what == "plain") return otherForm({1201, 30011}, {1, 0}, 8, false);
  if (what == "lines") return otherForm({96001, 407}, {1, 0}, 4, true);
  if (what == "accesses") return accesses();
  if (what == "predicted") return predicted();
  if (what == "drift") return drift();
  if (what == "tie98") return tie(98.0);
  if (what == "tie99") return tie(99.5);
  if (what == "bits") return bits({32, 4096, 2048}, {0, 2, 1}, 4, 50, 100, 100);
  if (what == "nobits") return bits({2, 4096, 512, 64}, {0, 3, 1, 2}, 4, 100, 50, 120);
  if (what == "groups") return groups();
  if (what == "narrow") return narrow();
  return 2;
}
