// Batched multi-view draws: many independent views, one launch per stage.
//
// The reference draws one view per CudaRaster::drawTriangles() call, each
// with its own four launches and a blocking read of the overflow counters
// (CudaRaster.cpp:237-342).  A batch lays the intermediate buffers of all its
// views out in shared allocations (per-view regions, per-view queue depths),
// keeps a device table of per-view Params, and runs each stage as one grid
// over the work of every view: setup+bin over all triangle chunks, coarse
// over all bins, fine over all tile groups of each pipe variant (the
// workgroup -> view lookup is a binary search over a prefix table).  From the
// second draw on the launch sequence is replayed from a captured hipGraph.
//
// Per view the kernels are the plain draw's, with the same Params, so every
// image is bit-identical to a plain draw of that view.  Overflow is per view:
// views whose counters report it are grown and re-drawn alone; the others
// are complete (the fine stage skips a view whose counters overflowed, so
// its surfaces were not touched).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <new>
#include <set>
#include <vector>

#include "cr/cr.h"
#include "cr_device.h"
#include "cr_host.h"

using namespace crhip;
using namespace crhost;

namespace {

struct ViewState {
  cr_view desc;
  Geometry g;
  int32_t numChunks = 0;
  uint32_t clearColor = 0, clearDepth = 0;
  int64_t maxSubtris = 1, maxBin = 1, maxTile = 1;
  // Element offsets of the view's regions in the shared buffers.
  size_t oTri = 0, oSlot = 0, oClip = 0, oBinAddr = 0, oBin = 0, oTile = 0, oTileList = 0;
};

// One launch set: the device Params table of a list of views and, per
// stage, the order in which the stage lists them with its workgroup prefix.
struct Tables {
  struct Stage {
    int variant = -1;          // fine stages: pipe variant
    int n = 0;                 // listed views
    int blocks = 0;            // workgroups (fine: tile groups)
    int64_t tiles = 0;         // fine stages: tiles of the listed views
    int ofs = 0, orderOfs = 0; // prefix (n + 1 entries) and order (n entries) in `starts`
  };
  int n = 0;
  std::vector<int> members;    // the views, in the order of `params`
  Stage setup, coarse;
  std::vector<Stage> fine;
  DevBuf params, starts;
};

size_t align64(size_t x) { return (x + 63) & ~(size_t)63; }

constexpr int kMaxGroups = 4;   // concurrent view groups (streams / graph branches)

}  // namespace

struct cr_batch {
  cr_context* ctx = nullptr;
  int device = 0;
  std::vector<ViewState> views;
  DevBuf triSubtris, triHeader, triData, subtriTri, binAddr, binList;
  DevBuf tileStart, tileCount, tileList, tileSegNext, counters, saved;
  Counters* hostCounters = nullptr;   // pinned, one block per view, written by the draws' finish kernels
  Counters* hostCountersDev = nullptr;   // their device address
  bool countersClean = false;         // every view's last draw has ended: it left its counters cleared
  Tables groups[kMaxGroups];          // views split into cost-balanced groups, one launch chain each
  int numGroups = 1;
  Tables subset;                      // views re-drawn after an overflow
  // Streams and events of the graph's parallel branches, used in captures only:
  // groups 1.. (group 0 on the capturing stream), and every second fine stage
  // of a single group.
  hipStream_t side[kMaxGroups] = {}, fineSide = nullptr;
  hipEvent_t evFork = nullptr, evJoin[kMaxGroups] = {}, evFineFork = nullptr, evFineJoin = nullptr;
  int tilesPerGroup = 4;
  int banded = 0;                     // fine tile groups in XCD bands (1) or round-robin (0)
  int coarseThreads = 256;            // coarse workgroup size
  bool haveCounts = false;            // hostCounters hold every view's demand from a complete draw
  bool moved = false;                 // views' buffers changed since the tables were built
  bool laidOut = false, useGraph = true, graphValid = false, tuned = false;
  bool drawn = false;                 // a draw of these views is behind: their capacities have held
  hipStream_t capStream = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  uint64_t lastTicks = 0;             // GPU time of the last draw, in wall clock ticks
  float tunedMs = 0.0f;
  int64_t retries = 0;
  size_t reserved = 0;
};

namespace {

cr_status layout(cr_batch* b) {
  cr_context* ctx = b->ctx;
  size_t nTri = 0, nSlot = 0, nClip = 0, nBinAddr = 0, nBin = 0, nTile = 0, nTileList = 0;
  for (ViewState& v : b->views) {
    const int64_t nt = v.desc.num_tris;
    v.oTri = nTri;
    nTri += align64((size_t)std::max<int64_t>(nt, 1));
    v.oSlot = nSlot;
    nSlot += align64((size_t)v.maxSubtris);
    v.oClip = nClip;
    nClip += align64((size_t)std::max<int64_t>(v.maxSubtris - nt, 1));
    v.oBinAddr = nBinAddr;
    nBinAddr += align64((size_t)(v.g.nb + 1) * std::max(v.numChunks, 1));
    v.oBin = nBin;
    nBin += align64((size_t)v.maxBin);
    v.oTile = nTile;
    nTile += align64((size_t)v.g.nt);
    v.oTileList = nTileList;
    nTileList += align64((size_t)v.maxTile);
  }
  CR_HIP(ctx, b->triSubtris.ensure(nTri));
  CR_HIP(ctx, b->triHeader.ensure(nSlot * sizeof(Header)));
  CR_HIP(ctx, b->triData.ensure(nSlot * sizeof(TriData)));
  CR_HIP(ctx, b->subtriTri.ensure(nClip * 4));
  CR_HIP(ctx, b->binAddr.ensure(nBinAddr * 4));
  CR_HIP(ctx, b->binList.ensure(nBin * 16));
  CR_HIP(ctx, b->tileStart.ensure(nTile * 4));
  CR_HIP(ctx, b->tileCount.ensure(nTile * 4));
  CR_HIP(ctx, b->tileList.ensure(nTileList * 4));
  CR_HIP(ctx, b->tileSegNext.ensure(std::max<size_t>(nTileList >> kTileSegLog2, 1) * 8));
  const void* before = b->counters.ptr;
  CR_HIP(ctx, b->counters.ensure(b->views.size() * sizeof(Counters)));
  if (b->counters.ptr != before) b->countersClean = false;
  b->reserved = b->triSubtris.bytes + b->triHeader.bytes + b->triData.bytes + b->subtriTri.bytes +
                b->binAddr.bytes + b->binList.bytes + b->tileStart.bytes +
                b->tileCount.bytes + b->tileList.bytes + b->tileSegNext.bytes + b->counters.bytes;
  b->graphValid = false;
  b->laidOut = true;
  return CR_OK;
}

Params viewParams(const cr_batch* b, int i) {
  const ViewState& v = b->views[i];
  const cr_view& d = v.desc;
  Params P;
  memset(&P, 0, sizeof(P));
  P.numTris = d.num_tris;
  P.numVertices = (int32_t)std::min<int64_t>(d.num_vertices, INT32_MAX);
  P.vertexStride = d.pipe.vertex_struct_size;
  P.vertices = static_cast<const uint8_t*>(d.vertices);
  P.indices = static_cast<const int32_t*>(d.indices);
  P.viewportWidth = v.g.vw;
  P.viewportHeight = v.g.vh;
  P.widthPixels = v.g.wp;
  P.heightPixels = v.g.hp;
  P.widthTiles = v.g.wt;
  P.heightTiles = v.g.ht;
  P.numTiles = v.g.nt;
  P.binLog2 = v.g.bl;
  P.widthBins = v.g.wb;
  P.heightBins = v.g.hb;
  P.numBins = v.g.nb;
  P.samplesLog2 = d.pipe.samples_log2;
  P.flags = d.pipe.render_mode_flags & (kFlagDepth | kFlagLerp);
  P.blend = d.pipe.blend_shader;
  P.shader = d.pipe.fragment_shader;
  P.constColor = d.pipe.const_color;
  P.deferredClear = d.deferred_clear ? 1 : 0;
  P.clearColor = v.clearColor;
  P.clearDepth = v.clearDepth;
  P.hiz = 1;
  P.maxSubtris = (int32_t)v.maxSubtris;
  P.triSubtris = b->triSubtris.as<uint8_t>() + v.oTri;
  P.triHeader = b->triHeader.as<Header>() + v.oSlot;
  P.triData = b->triData.as<TriData>() + v.oSlot;
  P.subtriTri = b->subtriTri.as<uint32_t>() + v.oClip;
  P.numChunks = v.numChunks;
  P.binAddr = b->binAddr.as<uint32_t>() + v.oBinAddr;
  P.maxBinEntries = (int32_t)v.maxBin;
  P.binList = b->binList.as<uint4>() + v.oBin;
  P.tileStart = b->tileStart.as<uint32_t>() + v.oTile;
  P.tileCount = b->tileCount.as<uint32_t>() + v.oTile;
  P.maxTileEntries = (int32_t)v.maxTile;
  P.tileList = b->tileList.as<uint32_t>() + v.oTileList;
  P.tileSegNext = b->tileSegNext.as<uint32_t>() + 2 * (v.oTileList >> kTileSegLog2);   // oTileList: a multiple of 64
  P.color = d.color->dev;
  P.depth = d.depth->dev;
  P.triid = d.tri_id ? d.tri_id->dev : nullptr;
  P.counters = b->counters.as<Counters>() + i;
  return P;
}

// Appends one stage: the listed Params indices `list` (in launch order) with
// `blocks[k]` workgroups each.
void appendStage(std::vector<int32_t>& st, Tables::Stage& S, const std::vector<int>& list,
                 const std::vector<int64_t>& blocks, int64_t& most) {
  S.n = (int)list.size();
  S.ofs = (int)st.size();
  int64_t acc = 0;
  for (int k : list) {
    st.push_back((int32_t)acc);
    acc += blocks[k];
  }
  st.push_back((int32_t)acc);
  S.orderOfs = (int)st.size();
  for (int k : list) st.push_back(k);
  S.blocks = (int)std::min<int64_t>(acc, INT32_MAX);
  most = std::max(most, acc);
}

// Params indices sorted by decreasing cost per workgroup, so that the
// longest workgroups start first (ties keep submission order).
std::vector<int> longestFirst(const std::vector<double>& cost, const std::vector<int>& list) {
  std::vector<int> out = list;
  std::stable_sort(out.begin(), out.end(), [&](int a, int c) { return cost[a] > cost[c]; });
  return out;
}

cr_status buildTables(cr_batch* b, Tables& T, const std::vector<int>& idx) {
  cr_context* ctx = b->ctx;
  const int n = (int)idx.size();
  const int W = b->tilesPerGroup;
  std::vector<Params> ps(n);
  for (int k = 0; k < n; k++) ps[k] = viewParams(b, idx[k]);
  // Cost per workgroup: measured entries per bin / per tile once a draw has
  // counted them, else triangles per bin / per tile.
  std::vector<double> binCost(n), tileCost(n);
  std::vector<int64_t> chunks(n), bins(n), groups(n);
  for (int k = 0; k < n; k++) {
    const Params& P = ps[k];
    const Counters& c = b->hostCounters[idx[k]];
    const bool measured = b->haveCounts && !c.overflow;
    binCost[k] = (measured ? (double)c.binEntries : (double)P.numTris) / std::max(P.numBins, 1);
    tileCost[k] = (measured ? (double)c.tileEntries : 2.0 * P.numTris) * (1 << P.samplesLog2) /
                  std::max(P.numTiles, 1);
    chunks[k] = P.numTris > 0 ? P.numChunks : 0;
    bins[k] = coarseBlocks(P);
    groups[k] = ((P.numTiles + W - 1) / W + kFineRounds - 1) / kFineRounds;
  }
  std::vector<int> all(n);
  for (int k = 0; k < n; k++) all[k] = k;
  std::vector<int32_t> st;
  int64_t most = 0;
  appendStage(st, T.setup, all, chunks, most);
  appendStage(st, T.coarse, longestFirst(binCost, all), bins, most);
  T.fine.clear();
  for (int var = 0; var < kFineVariants; var++) {
    std::vector<int> list;
    for (int k = 0; k < n; k++)
      if (fineVariant(ps[k]) == var) list.push_back(k);
    if (list.empty()) continue;
    Tables::Stage S;
    S.variant = var;
    for (int k : list) S.tiles += ps[k].numTiles;
    appendStage(st, S, longestFirst(tileCost, list), groups, most);
    if (S.blocks > 0) T.fine.push_back(S);
  }
  if (most >= (int64_t)1 << 30) return fail(ctx, CR_ERR_OVERFLOW, "batch: more than 2^30 workgroups in one stage");
  CR_HIP(ctx, T.params.ensure((size_t)std::max(n, 1) * sizeof(Params)));
  CR_HIP(ctx, T.starts.ensure(st.size() * sizeof(int32_t)));
  // On a stream of the batch's own, and waited for: whatever stream a draw or
  // its graph's branches run on, the tables are there.
  hipError_t e = hipSuccess;
  if (n > 0)
    e = hipMemcpyAsync(T.params.ptr, ps.data(), (size_t)n * sizeof(Params), hipMemcpyHostToDevice, b->capStream);
  if (e == hipSuccess)
    e = hipMemcpyAsync(T.starts.ptr, st.data(), st.size() * sizeof(int32_t), hipMemcpyHostToDevice, b->capStream);
  const hipError_t waited = hipStreamSynchronize(b->capStream);
  CR_HIP(ctx, e);
  CR_HIP(ctx, waited);
  T.n = n;
  T.members = idx;
  return CR_OK;
}

std::vector<int> allViews(const cr_batch* b) {
  std::vector<int> idx(b->views.size());
  for (size_t i = 0; i < idx.size(); i++) idx[i] = (int)i;
  return idx;
}

// Splits the views into numGroups groups of similar cost (longest first to
// the least loaded group) and builds each group's tables.
cr_status buildAll(cr_batch* b) {
  const int n = (int)b->views.size();
  const int K = std::max(1, std::min(b->numGroups, n));
  std::vector<double> cost(n);
  for (int i = 0; i < n; i++) {
    const Counters& c = b->hostCounters[i];
    const int ns = 1 << b->views[i].desc.pipe.samples_log2;
    cost[i] = (b->haveCounts && !c.overflow) ? (double)c.binEntries + (double)c.tileEntries * ns
                                             : (double)b->views[i].desc.num_tris * (1 + ns);
  }
  std::vector<int> order = allViews(b);
  std::stable_sort(order.begin(), order.end(), [&](int a, int c) { return cost[a] > cost[c]; });
  std::vector<std::vector<int>> members(K);
  std::vector<double> load(K, 0.0);
  for (int i : order) {
    const int g = (int)(std::min_element(load.begin(), load.end()) - load.begin());
    members[g].push_back(i);
    load[g] += cost[i];
  }
  for (int g = 0; g < K; g++) {
    std::sort(members[g].begin(), members[g].end());
    cr_status st = buildTables(b, b->groups[g], members[g]);
    if (st != CR_OK) return st;
  }
  b->numGroups = K;
  b->graphValid = false;
  return CR_OK;
}

// Whether a graph's fine stages of several pipe variants run in two chains side
// by side: a variant's last tiles, one wave each over a list of hundreds of
// entries, leave most of the chip idle, and small views are all last tiles.
// 1x and 4x views: 3.6k tiles 188 -> 145 us a draw, 25k 408 -> 317, 60k 166 ->
// 151, 183k 330 -> 319; with 540k, full of either variant, 767 -> 776.  The
// branch itself costs some 8 us: with 169 tiles on one side 90 -> 98.
bool forksFine(const Tables& T) {
  int64_t chain[2] = {0, 0};
  for (size_t i = 0; i < T.fine.size(); i++) chain[i & 1] += T.fine[i].tiles;
  return std::min(chain[0], chain[1]) >= 512 && chain[0] + chain[1] <= 256 * 1024;
}

// One launch chain, or two for the fine stages.
cr_status launchTables(cr_batch* b, const Tables& T, hipStream_t stream, bool twoFine = false) {
  const Params* pv = T.params.as<Params>();
  const int32_t* s = T.starts.as<int32_t>();
  launchSetupBatch(pv, s + T.setup.ofs, s + T.setup.orderOfs, T.setup.n, T.setup.blocks, stream);
  launchCoarseBatch(b->coarseThreads, pv, s + T.coarse.ofs, s + T.coarse.orderOfs, T.coarse.n, T.coarse.blocks,
                    stream);
  twoFine = twoFine && forksFine(T);
  if (twoFine) {
    CR_HIP(b->ctx, hipEventRecord(b->evFineFork, stream));
    CR_HIP(b->ctx, hipStreamWaitEvent(b->fineSide, b->evFineFork, 0));
  }
  for (size_t i = 0; i < T.fine.size(); i++) {
    const Tables::Stage& f = T.fine[i];
    launchFineBatch(f.variant, b->tilesPerGroup, b->banded, pv, s + f.ofs, s + f.orderOfs, f.n, f.blocks,
                    twoFine && (i & 1) ? b->fineSide : stream);
  }
  if (twoFine) {
    CR_HIP(b->ctx, hipEventRecord(b->evFineJoin, b->fineSide));
    CR_HIP(b->ctx, hipStreamWaitEvent(stream, b->evFineJoin, 0));
  }
  launchFinishBatch(pv, T.n, b->counters.as<Counters>(), b->hostCountersDev, stream);
  CR_HIP(b->ctx, hipGetLastError());
  return CR_OK;
}

// All groups launched one after the other on `stream`.  (Only a graph runs them
// side by side: direct launches of freshly built groups on forked streams have
// faulted the GPU for a cause that was not found.)
cr_status launchAllGroups(cr_batch* b, hipStream_t stream) {
  cr_status st = CR_OK;
  for (int g = 0; g < b->numGroups && st == CR_OK; g++) st = launchTables(b, b->groups[g], stream);
  return st;
}

// All groups as parallel branches of the graph that capStream captures.
cr_status captureGroups(cr_batch* b) {
  hipStream_t stream = b->capStream;
  if (b->numGroups <= 1) return launchTables(b, b->groups[0], stream, true);
  CR_HIP(b->ctx, hipEventRecord(b->evFork, stream));
  for (int g = 1; g < b->numGroups; g++) CR_HIP(b->ctx, hipStreamWaitEvent(b->side[g], b->evFork, 0));
  cr_status st = launchTables(b, b->groups[0], stream);
  for (int g = 1; g < b->numGroups && st == CR_OK; g++) st = launchTables(b, b->groups[g], b->side[g]);
  for (int g = 1; g < b->numGroups; g++) {
    CR_HIP(b->ctx, hipEventRecord(b->evJoin[g], b->side[g]));
    CR_HIP(b->ctx, hipStreamWaitEvent(stream, b->evJoin[g], 0));
  }
  return st;
}

cr_status capture(cr_batch* b) {
  cr_context* ctx = b->ctx;
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  b->exec = nullptr;
  b->graph = nullptr;
  CR_HIP(ctx, hipStreamBeginCapture(b->capStream, hipStreamCaptureModeThreadLocal));
  cr_status st = captureGroups(b);
  hipError_t e = hipStreamEndCapture(b->capStream, &b->graph);
  if (st != CR_OK) return st;
  CR_HIP(ctx, e);
  CR_HIP(ctx, hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0));
  b->graphValid = true;
  return CR_OK;
}

cr_status prepare(cr_batch* b) {
  if (b->laidOut) return CR_OK;
  cr_status st = layout(b);
  if (st != CR_OK) return st;
  return buildAll(b);
}

// Clears the counters of every view unless the draw before left them so.
cr_status clearCounters(cr_batch* b, hipStream_t stream) {
  if (b->countersClean) return CR_OK;
  for (int g = 0; g < b->numGroups; g++)
    launchResetBatch(b->groups[g].params.as<Params>(), b->groups[g].n, stream);
  CR_HIP(b->ctx, hipGetLastError());
  return CR_OK;
}

// Writes the views' current vertex and index buffers into the tables of
// views.  (In a small kernel on the draw's stream, the pointers in its
// arguments: the captured graph stays as it is, and nothing is copied.)
cr_status patchBuffers(cr_batch* b, hipStream_t stream) {
  if (!b->moved) return CR_OK;
  for (int g = 0; g < b->numGroups; g++) {
    const Tables& T = b->groups[g];
    for (int first = 0; first < T.n; first += kPatchViews) {
      PatchTable P = {};
      const int n = std::min(T.n - first, kPatchViews);
      for (int k = 0; k < n; k++) {
        const cr_view& d = b->views[T.members[first + k]].desc;
        P.vertices[k] = static_cast<const uint8_t*>(d.vertices);
        P.indices[k] = static_cast<const int32_t*>(d.indices);
      }
      launchPatchBatch(T.params.as<Params>(), P, first, n, stream);
    }
  }
  CR_HIP(b->ctx, hipGetLastError());
  return CR_OK;
}

// Grows the capacities of every view whose counters overflowed and re-draws
// those views (only) until none does.
cr_status settleOverflow(cr_batch* b, hipStream_t stream) {
  for (;;) {
    std::vector<int> over;
    for (size_t i = 0; i < b->views.size(); i++) {
      const Counters& c = b->hostCounters[i];
      if (!c.overflow) continue;
      ViewState& v = b->views[i];
      if (c.overflow & 1u) v.maxSubtris = std::max<int64_t>(v.maxSubtris, (int64_t)c.numSubtris + kSubtrisSlack);
      if (c.overflow & 2u) v.maxBin = std::max<int64_t>(v.maxBin, (int64_t)c.binEntries + kBinSlack);
      if (c.overflow & 4u) v.maxTile = std::max<int64_t>(v.maxTile, (int64_t)c.tileEntries + kTileSlack);
      if (v.maxSubtris > kMaxSubtris)
        return fail(b->ctx, CR_ERR_OVERFLOW, "batch view %zu: more than 2^28 subtriangles", i);
      if (v.maxBin > kMaxEntries || v.maxTile > kMaxEntries)
        return fail(b->ctx, CR_ERR_OVERFLOW, "batch view %zu: internal queue capacity exceeded (2^31 entries)", i);
      over.push_back((int)i);
    }
    if (over.empty()) {
      b->haveCounts = true;
      return CR_OK;
    }
    b->retries++;
    cr_status st = layout(b);
    if (st == CR_OK) st = buildAll(b);
    if (st == CR_OK) st = buildTables(b, b->subset, over);
    if (st == CR_OK) st = clearCounters(b, stream);
    if (st != CR_OK) return st;
    b->countersClean = false;
    st = launchTables(b, b->subset, stream);
    if (st != CR_OK) return st;
    CR_HIP(b->ctx, hipStreamSynchronize(stream));
    b->countersClean = true;
  }
}

// A batch draw waits for its counters: refused, before anything of the batch
// changes, on a stream that captures (its launches would be recorded instead of
// run, the counters neither cleared nor the moved buffers written).
cr_status refuseCapture(cr_batch* b, hipStream_t stream) {
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  const hipError_t e = hipStreamIsCapturing(stream, &cap);
  if (e != hipSuccess) (void)hipGetLastError();    // (the null stream beside a capturing one; not for the next draw to find)
  CR_HIP(b->ctx, e);
  if (cap != hipStreamCaptureStatusNone)
    return fail(b->ctx, CR_ERR_DEVICE, "batch: the draw waits for its counters, which a capturing stream cannot");
  return CR_OK;
}

cr_status drawBatch(cr_batch* b, hipStream_t stream, bool graph) {
  cr_context* ctx = b->ctx;
  CR_HIP(ctx, hipSetDevice(ctx->device));
  cr_status st = refuseCapture(b, stream);
  if (st == CR_OK) st = prepare(b);
  if (st != CR_OK) return st;
  b->retries = 0;
  // The first draw is launched stage by stage: capturing costs more than the
  // graph saves on it (8 small views, first draw: 585 us captured, 410 launched;
  // later draws: 137 replayed, 143 launched), and queues that turn out too small
  // void the graph.
  graph = graph && b->drawn;
  if (graph && !b->graphValid) {
    st = capture(b);
    if (st != CR_OK) return st;
  }
  st = patchBuffers(b, stream);
  if (st == CR_OK) st = clearCounters(b, stream);
  if (st != CR_OK) return st;
  b->countersClean = false;
  if (graph) {
    CR_HIP(ctx, hipGraphLaunch(b->exec, stream));
  } else {
    st = launchAllGroups(b, stream);
    if (st != CR_OK) return st;
  }
  CR_HIP(ctx, hipStreamSynchronize(stream));
  b->countersClean = true;
  b->moved = false;
  // GPU time: the first stage's start to the last view's end.
  uint64_t first = UINT64_MAX, last = 0;
  for (size_t i = 0; i < b->views.size(); i++) {
    const uint64_t* s = b->hostCounters[i].stamp;
    for (int k = 0; k < kStampCount; k++)
      if (s[k] != 0) first = std::min(first, s[k]);
    last = std::max(last, s[kStampEnd]);
  }
  b->lastTicks = last > first ? last - first : 0;
  st = settleOverflow(b, stream);
  if (st == CR_OK) b->drawn = true;
  return st;
}

// Device-to-device copies of the surfaces of views drawn without deferred
// clear (the autotuner draws the batch several times).
cr_status saveSurfaces(cr_batch* b, hipStream_t stream, bool restore) {
  size_t need = 0;
  for (const ViewState& v : b->views)
    if (!v.desc.deferred_clear)
      need += v.desc.color->bytes + v.desc.depth->bytes + (v.desc.tri_id ? v.desc.tri_id->bytes : 0);
  if (need == 0) return CR_OK;
  if (!restore) CR_HIP(b->ctx, b->saved.ensure(need));
  uint8_t* p = b->saved.as<uint8_t>();
  for (const ViewState& v : b->views) {
    if (v.desc.deferred_clear) continue;
    for (const cr_surface* s : {v.desc.color, v.desc.depth, v.desc.tri_id}) {
      if (!s) continue;
      if (restore) CR_HIP(b->ctx, hipMemcpyAsync(s->dev, p, s->bytes, hipMemcpyDeviceToDevice, stream));
      else CR_HIP(b->ctx, hipMemcpyAsync(p, s->dev, s->bytes, hipMemcpyDeviceToDevice, stream));
      p += s->bytes;
    }
  }
  return CR_OK;
}

cr_status validateView(cr_context* ctx, const cr_view& v, int i) {
  if (!v.color || !v.depth) return fail(ctx, CR_ERR_INVALID, "batch view %d: colour and depth surfaces are required", i);
  if (v.color->format != CR_FORMAT_RGBA8) return fail(ctx, CR_ERR_INVALID, "batch view %d: unsupported color buffer format", i);
  if (v.depth->format != CR_FORMAT_DEPTH32) return fail(ctx, CR_ERR_INVALID, "batch view %d: unsupported depth buffer format", i);
  if (v.color->width != v.depth->width || v.color->height != v.depth->height)
    return fail(ctx, CR_ERR_INVALID, "batch view %d: mismatch in size between surfaces", i);
  if (v.color->samples != v.depth->samples)
    return fail(ctx, CR_ERR_INVALID, "batch view %d: mismatch in multisampling between surfaces", i);
  if (v.tri_id && (v.tri_id->format != CR_FORMAT_TRIANGLE_ID || v.tri_id->width != v.color->width ||
                   v.tri_id->height != v.color->height || v.tri_id->samples != v.color->samples))
    return fail(ctx, CR_ERR_INVALID, "batch view %d: triangle-id surface does not match the colour surface", i);
  cr_status st = validatePipe(ctx, &v.pipe);
  if (st != CR_OK) return st;
  if (v.pipe.fragment_shader == CR_SHADER_TEX_PHONG)
    return fail(ctx, CR_ERR_UNSUPPORTED, "batch view %d: the texPhong shader draws through cr_draw_triangles", i);
  if (v.pipe.samples_log2 != v.color->samplesLog2)
    return fail(ctx, CR_ERR_INVALID, "batch view %d: mismatch in multisampling between pixel pipe and surface", i);
  if (v.num_tris < 0 || v.num_tris > kMaxTris || v.num_vertices < 0)
    return fail(ctx, CR_ERR_INVALID, "batch view %d: bad triangle or vertex count", i);
  if (v.num_tris > 0 && (!v.vertices || !v.indices))
    return fail(ctx, CR_ERR_INVALID, "batch view %d: vertex and index buffers are required", i);
  if (((uintptr_t)v.vertices & 15) || ((uintptr_t)v.indices & 3))
    return fail(ctx, CR_ERR_INVALID, "batch view %d: misaligned vertex or index pointer", i);
  return CR_OK;
}

}  // namespace

extern "C" {

cr_status cr_batch_create(cr_context* ctx, const cr_view* views, int32_t numViews, cr_batch** out) {
  if (!ctx || !out || (!views && numViews > 0) || numViews < 0)
    return fail(ctx, CR_ERR_INVALID, "cr_batch_create: bad arguments");
  *out = nullptr;
  std::set<const cr_surface*> seen;
  for (int i = 0; i < numViews; i++) {
    cr_status st = validateView(ctx, views[i], i);
    if (st != CR_OK) return st;
    for (const cr_surface* s : {views[i].color, views[i].depth, views[i].tri_id})
      if (s && !seen.insert(s).second)
        return fail(ctx, CR_ERR_INVALID, "batch view %d: a surface appears in more than one view", i);
  }
  cr_batch* b = new (std::nothrow) cr_batch();
  if (!b) return fail(ctx, CR_ERR_NOMEM, "out of host memory");
  b->ctx = ctx;
  b->device = ctx->device;
  b->views.resize(numViews);
  for (int i = 0; i < numViews; i++) {
    ViewState& v = b->views[i];
    v.desc = views[i];
    v.g = geometryOf(v.desc.color);
    v.numChunks = (v.desc.num_tris + kSetupChunkTris - 1) / kSetupChunkTris;
    if (v.desc.deferred_clear) clearValues(v.desc.clear_color, v.desc.clear_depth, &v.clearColor, &v.clearDepth);
    initialCapacities(v.desc.num_tris, v.g, v.maxSubtris, v.maxBin, v.maxTile);
  }
  hipError_t e = hipSetDevice(ctx->device);
  if (e == hipSuccess) e = hipHostMalloc((void**)&b->hostCounters, std::max<size_t>(numViews, 1) * sizeof(Counters),
                                         hipHostMallocDefault);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&b->capStream, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipHostGetDevicePointer((void**)&b->hostCountersDev, b->hostCounters, 0);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&b->evFork, hipEventDisableTiming);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&b->evFineFork, hipEventDisableTiming);
  if (e == hipSuccess) e = hipEventCreateWithFlags(&b->evFineJoin, hipEventDisableTiming);
  if (e == hipSuccess) e = hipStreamCreateWithFlags(&b->fineSide, hipStreamNonBlocking);
  for (int g = 1; g < kMaxGroups && e == hipSuccess; g++) {
    e = hipStreamCreateWithFlags(&b->side[g], hipStreamNonBlocking);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&b->evJoin[g], hipEventDisableTiming);
  }
  if (e != hipSuccess) {
    cr_batch_destroy(b);
    return fail(ctx, CR_ERR_DEVICE, "cr_batch_create: %s", hipGetErrorString(e));
  }
  memset(b->hostCounters, 0, std::max<size_t>(numViews, 1) * sizeof(Counters));
  *out = b;
  return CR_OK;
}

cr_status cr_batch_destroy(cr_batch* b) {
  if (!b) return CR_OK;
  (void)hipSetDevice(b->device);
  (void)hipDeviceSynchronize();
  if (b->exec) (void)hipGraphExecDestroy(b->exec);
  if (b->graph) (void)hipGraphDestroy(b->graph);
  for (DevBuf* d : {&b->triSubtris, &b->triHeader, &b->triData, &b->subtriTri, &b->binAddr, &b->binList,
                    &b->tileStart, &b->tileCount, &b->tileList, &b->tileSegNext, &b->counters,
                    &b->saved,
                    &b->subset.params, &b->subset.starts})
    d->release();
  for (Tables& t : b->groups) {
    t.params.release();
    t.starts.release();
  }
  if (b->hostCounters) (void)hipHostFree(b->hostCounters);
  if (b->capStream) (void)hipStreamDestroy(b->capStream);
  for (int g = 1; g < kMaxGroups; g++) {
    if (b->side[g]) (void)hipStreamDestroy(b->side[g]);
    if (b->evJoin[g]) (void)hipEventDestroy(b->evJoin[g]);
  }
  if (b->fineSide) (void)hipStreamDestroy(b->fineSide);
  for (hipEvent_t e : {b->evFork, b->evFineFork, b->evFineJoin})
    if (e) (void)hipEventDestroy(e);
  delete b;
  return CR_OK;
}

cr_status cr_batch_draw(cr_batch* b, void* stream) {
  if (!b) return fail(nullptr, CR_ERR_INVALID, "cr_batch_draw: batch is NULL");
  if (b->views.empty()) return CR_OK;
  return drawBatch(b, static_cast<hipStream_t>(stream), b->useGraph);
}

cr_status cr_batch_autotune(cr_batch* b, void* stream_) {
  if (!b) return fail(nullptr, CR_ERR_INVALID, "cr_batch_autotune: batch is NULL");
  if (b->views.empty()) return CR_OK;
  cr_context* ctx = b->ctx;
  hipStream_t stream = static_cast<hipStream_t>(stream_);
  CR_HIP(ctx, hipSetDevice(ctx->device));
  cr_status st = refuseCapture(b, stream);
  if (st == CR_OK) st = prepare(b);
  if (st == CR_OK) st = saveSurfaces(b, stream, false);
  // 1. Exact per-view queue demand (the draw grows whatever overflows).
  if (st == CR_OK) st = drawBatch(b, stream, false);
  if (st != CR_OK) return st;
  // 2. Queue depths = demand + 1/16 + a small constant margin.
  for (size_t i = 0; i < b->views.size(); i++) {
    const Counters& c = b->hostCounters[i];
    ViewState& v = b->views[i];
    const int64_t sub = std::max<int64_t>(c.numSubtris, v.desc.num_tris);
    v.maxSubtris = std::min<int64_t>(sub + sub / 16 + 1024, kMaxSubtris);
    v.maxBin = std::min<int64_t>((int64_t)c.binEntries + c.binEntries / 16 + 4096, kMaxEntries);
    v.maxTile = std::min<int64_t>((int64_t)c.tileEntries + c.tileEntries / 16 + 4096, kMaxEntries);
  }
  st = layout(b);
  if (st != CR_OK) return st;
  // 3. Fine-stage workgroup shape and placement: the fastest combination of
  //    the compiled shapes and banded / round-robin tile groups (the stages
  //    list views longest-first by the measured entries per bin and tile).
  //    What is timed is what later draws run: the captured graph with its
  //    parallel branches (rep 0 captures it), unless graphs are off.
  int bestW = b->tilesPerGroup, bestBanded = b->banded, bestCoarse = b->coarseThreads;
  float bestMs = 1e30f;
  const double tick = clockTick(b->device) * 1e3;
  for (int banded = 0; banded < 2; banded++) {
    for (int trial = 0; trial < 3 + 1; trial++) {
      // three fine shapes with the current coarse size, then the other
      // coarse size with the best fine shape so far
      const int W = trial < 3 ? kFineBatchShapes[trial] : bestW;
      b->tilesPerGroup = W;
      b->banded = banded;
      b->coarseThreads = trial < 3 ? bestCoarse : (bestCoarse == 256 ? 1024 : 256);
      st = buildAll(b);
      if (st != CR_OK) return st;
      float ms[3];
      for (int rep = 0; rep < 4; rep++) {
        st = saveSurfaces(b, stream, true);
        if (st == CR_OK) st = drawBatch(b, stream, b->useGraph);
        if (st != CR_OK) return st;
        if (rep > 0) ms[rep - 1] = (float)((double)b->lastTicks * tick);
      }
      std::sort(ms, ms + 3);
      if (ms[1] < bestMs) {
        bestMs = ms[1];
        bestW = W;
        bestBanded = banded;
        bestCoarse = b->coarseThreads;
      }
      b->coarseThreads = bestCoarse;
    }
  }
  b->tilesPerGroup = bestW;
  b->banded = bestBanded;
  b->coarseThreads = bestCoarse;
  // 4. Concurrent view groups: the views split into K cost-balanced groups
  //    whose launch chains run side by side (K = 1, 2 or 4) in the graph.
  int bestK = 1;
  for (int K : {2, 4}) {
    if (K > (int)b->views.size() || !b->useGraph) break;
    b->numGroups = K;
    st = buildAll(b);
    if (st != CR_OK) return st;
    float ms[3];
    for (int rep = 0; rep < 4; rep++) {
      st = saveSurfaces(b, stream, true);
      if (st == CR_OK) st = drawBatch(b, stream, b->useGraph);
      if (st != CR_OK) return st;
      if (rep > 0) ms[rep - 1] = (float)((double)b->lastTicks * tick);
    }
    std::sort(ms, ms + 3);
    if (ms[1] < bestMs) {
      bestMs = ms[1];
      bestK = K;
    }
  }
  b->numGroups = bestK;
  st = buildAll(b);
  if (st == CR_OK) st = saveSurfaces(b, stream, true);
  if (st != CR_OK) return st;
  CR_HIP(ctx, hipStreamSynchronize(stream));
  b->saved.release();
  b->graphValid = false;
  b->tuned = true;
  b->tunedMs = bestMs;
  return CR_OK;
}

cr_status cr_batch_reserve(cr_batch* b, int32_t view, int64_t maxSubtris, int64_t maxBin, int64_t maxTile) {
  if (!b) return fail(nullptr, CR_ERR_INVALID, "cr_batch_reserve: batch is NULL");
  if (view < 0 || view >= (int32_t)b->views.size()) return fail(b->ctx, CR_ERR_INVALID, "cr_batch_reserve: bad view");
  if (maxSubtris < 1 || maxBin < 1 || maxTile < 1 || maxSubtris > kMaxEntries || maxBin > kMaxEntries ||
      maxTile > kMaxEntries)
    return fail(b->ctx, CR_ERR_INVALID, "cr_batch_reserve: capacities must be in 1 .. 2^31-2");
  ViewState& v = b->views[view];
  // Slot t holds triangle t: at least one slot per input triangle.
  v.maxSubtris = std::max<int64_t>(maxSubtris, v.desc.num_tris);
  v.maxBin = maxBin;
  v.maxTile = maxTile;
  b->laidOut = false;
  b->graphValid = false;
  return CR_OK;
}

cr_status cr_batch_set_buffers(cr_batch* b, const void* const* vertices, const void* const* indices,
                               int32_t numViews) {
  if (!b || (numViews > 0 && (!vertices || !indices)))
    return fail(b ? b->ctx : nullptr, CR_ERR_INVALID, "cr_batch_set_buffers: NULL argument");
  if (numViews != (int32_t)b->views.size())
    return fail(b->ctx, CR_ERR_INVALID, "cr_batch_set_buffers: %d views, the batch has %zu", numViews, b->views.size());
  for (int i = 0; i < numViews; i++) {
    cr_view v = b->views[i].desc;
    v.vertices = vertices[i];
    v.indices = indices[i];
    const cr_status st = validateView(b->ctx, v, i);
    if (st != CR_OK) return st;
  }
  for (int i = 0; i < numViews; i++) {
    b->views[i].desc.vertices = vertices[i];
    b->views[i].desc.indices = indices[i];
  }
  b->moved = true;
  return CR_OK;
}

cr_status cr_batch_configure(cr_batch* b, const cr_batch_config* c) {
  if (!b || !c) return fail(nullptr, CR_ERR_INVALID, "cr_batch_configure: NULL argument");
  if ((c->fine_tiles_per_group != 2 && c->fine_tiles_per_group != 4 && c->fine_tiles_per_group != 8) ||
      (c->fine_banded != 0 && c->fine_banded != 1) || (c->coarse_threads != 256 && c->coarse_threads != 1024) ||
      c->view_groups < 1 || c->view_groups > kMaxGroups)
    return fail(b->ctx, CR_ERR_INVALID, "cr_batch_configure: fine tiles 2/4/8, banded 0/1, coarse 256/1024, groups 1..4");
  b->tilesPerGroup = c->fine_tiles_per_group;
  b->banded = c->fine_banded;
  b->coarseThreads = c->coarse_threads;
  b->numGroups = c->view_groups;
  b->laidOut = false;                 // tables are rebuilt on the next draw
  b->graphValid = false;
  return CR_OK;
}

cr_status cr_batch_use_graph(cr_batch* b, int32_t enable) {
  if (!b) return fail(nullptr, CR_ERR_INVALID, "cr_batch_use_graph: batch is NULL");
  b->useGraph = enable != 0;
  return CR_OK;
}

cr_status cr_batch_get_info(const cr_batch* b, cr_batch_info* out) {
  if (!b || !out) return fail(nullptr, CR_ERR_INVALID, "cr_batch_get_info: NULL argument");
  memset(out, 0, sizeof(*out));
  out->num_views = (int32_t)b->views.size();
  out->fine_tiles_per_group = b->tilesPerGroup;
  out->fine_banded = b->banded;
  out->coarse_threads = b->coarseThreads;
  out->view_groups = b->numGroups;
  out->uses_graph = b->useGraph ? 1 : 0;
  out->tuned = b->tuned ? 1 : 0;
  out->retries = b->retries;
  out->reserved_bytes = (int64_t)b->reserved;
  out->last_gpu_ms = (float)((double)b->lastTicks * clockTick(b->device) * 1e3);
  out->tuned_gpu_ms = b->tunedMs;
  return CR_OK;
}

cr_status cr_batch_get_view_counters(const cr_batch* b, int32_t view, cr_counters* out) {
  if (!b || !out) return fail(nullptr, CR_ERR_INVALID, "cr_batch_get_view_counters: NULL argument");
  if (view < 0 || view >= (int32_t)b->views.size())
    return fail(b->ctx, CR_ERR_INVALID, "cr_batch_get_view_counters: bad view");
  const Counters& c = b->hostCounters[view];
  memset(out, 0, sizeof(*out));
  out->num_tris = b->views[view].desc.num_tris;
  out->num_subtris = c.numSubtris;
  out->bin_entries = c.binEntries;
  out->tile_entries = c.tileEntries;
  out->tile_list_entries = c.tileListEntries;
  out->retries = b->retries;
  return CR_OK;
}

}  // extern "C"
