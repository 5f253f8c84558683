// Moment-table form of the strip MLEM iteration (host interface).
//
// Along an image row an event's kernel is a Gaussian of one fixed width (sigma_z
// alone sets it) around the row's vertex c = cz + tan dy, cut to the row's
// in-ellipse run [lo, hi].  About a nearby line X that many events share,
// with u = x - X and delta = c - X,
//   exp(-(C/2)(x - c)^2) = exp(-(C/2) u^2) exp(C u delta) exp(-(C/2) delta^2),
// and where |C u delta| <= 1 the middle factor is a degree-7 polynomial in
// (C s delta)(u / s) to 5e-7 (where it is <= 0.42 a degree-5 one, to 8e-7), its
// error averaging to nothing over a run.  Events are therefore split into
// (event, band) pairs (a band = 16 image rows) and the pairs binned by band, by
// the vertex at the band's middle and by tan: all pairs of a bin share one
// sheared line X(row) from which no vertex strays further than 0.214 sigma_z.
// Then
//   forward          a workgroup tabulates, per row and side of the line, the
//                    running sums over columns outward from the line of
//                    rho exp(-(C/2) u^2) (u / s)^m, m = 0..7; a row's sum over
//                    its run is 2 x 8 table words and a Horner evaluation,
//                    whatever the run's length;
//   back-projection  the transpose: a row adds weight x eta^m at the two cells
//                    its run ends in; per task the cells are summed inward
//                    and expanded back to pixels.
// Sums run outward from the line, so no difference of large numbers is
// formed and a pixel outside an event's run never enters its sums (an infinity
// or NaN there stays away from it, as in the pixel-by-pixel kernels).  A run
// that misses the line's column (a short run at an ellipse's tip) is walked
// pixel by pixel.
#pragma once

#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "strip_device.hpp"

namespace strip {

constexpr int kMomentRows = 16;  // image rows of a band

// One workgroup's (forward) or wavefront's (back-projection) share of a bin.
struct MomentTask {
  float xc, tc;  // the bin's line: z at the band's middle row, slope
  int band;
  int instance;  // index of its MomentInstance
  int group;     // first 16-pair group
  int pairs;
  int first_column;  // merged tasks (`pairs` counts groups): see the kernel
  int pad;
};

// 16 pairs (fewer at a bin's end) of one bin.
struct MomentGroup {
  float xc, tc;
  int bin;
  int pairs;
};

// What the kernels need of one reconstruction (device array; a task names its
// entry).
struct MomentInstance {
  DeviceGeometry g;
  // bins: band-major, then the vertex at the band's middle row, then tan
  int nx, nt;
  float x_lo, dx;  // lower edge of bin 0 and bin width, z coordinate
  float t_lo, dt;  // the same of tan
  int positions;   // table cells per row and side, besides the empty one
  int merged_columns;  // pixel columns of a merged back-projection task
  int max_bands;
  float inv_s;     // 1 / s
  float cs;        // C s
  const uint32_t* blocks;  // 1 KiB per 16 pairs (moment_pack_kernel)
  const MomentGroup* groups;
  const float* rhoT;       // image the forward pass reads (column-major)
  float* rho_next;
  float* partial;          // per (band of the record, record)
  const int* counts;       // bands of each record
  float* inv;
  float* bpT;              // bp_images images, n_pixels apart
  int bp_images;
  int64_t n_events;
};

// The row-band tiling that a plan's events would have as lists.
struct ListTiling {
  bool known = false;
  int forward_group = 0, backward_group = 0;
  int forward_rows = 0, backward_rows = 0;
  int window_columns = 0;
  int64_t forward_pairs = 0, backward_pairs = 0;
};

struct MomentPlan {
  bool ready = false;
  ListTiling tiling;  // looked up when a caller first asks for it
  int64_t n_events = 0, n_pairs = 0;
  int n_bins = 0, n_groups = 0;
  int n_fwd = 0, n_bwd = 0;
  int terms = 8;      // of the polynomial: 8, or 6 about closer lines
  int fwd_waves = 4;  // wavefronts per forward workgroup
  bool merged = false;  // back-projection tasks of several bins
  size_t fwd_lds = 0, bwd_lds = 0;
  MomentInstance inst;  // host copy (image 0)
  void* arena = nullptr;  // per-event arrays and descriptors
  void* lists = nullptr;  // pair groups and tasks
  // pieces of them
  uint32_t* blocks = nullptr;
  float* partial = nullptr;
  float* inv = nullptr;
  // where the back-projection adds: the caller's image, or several images of
  // the plan's own, zero between uses, whose sum it is
  float* bpT = nullptr;
  int bp_images = 1;
  int* counts = nullptr;
  int* order = nullptr;     // record -> caller's event
  MomentTask* fwd_tasks = nullptr;
  MomentTask* bwd_tasks = nullptr;
  MomentInstance* desc = nullptr;  // images 0 / 1
};

// Whether the geometry suits the moment form at all.
bool moment_supported(const DeviceGeometry& g);

// Builds the plan for the events.  *built = false (and 0) where the row-band
// lists are the better choice (batch: among the members of a batch) or the plan
// does not fit.  max_extent: the widest clamped bbox and the most rows of a
// span-table slot, for the lists' plan; left alone where the events were not
// looked at.
int moment_prepare(MomentPlan& plan, const DeviceGeometry& g,
                   const EventSoA& ev, int64_t n_events, float* const rhoT[2],
                   float* bpT, bool batch, hipStream_t stream, bool* built,
                   int max_extent[2], std::string* err);
void moment_release(MomentPlan& plan);

// The passes of an iteration reading image `cur`.
int moment_forward(MomentPlan& plan, int cur, hipStream_t stream,
                   std::string* err);
// D_e = sum of the record's partials; inv (guarded or not) and / or D
int moment_inverse(MomentPlan& plan, int guard, float* inv, float* denominators,
                   hipStream_t stream, std::string* err);
// Adds to the plan's bpT images, whose sum the caller takes and clears.
int moment_backward(MomentPlan& plan, int cur, hipStream_t stream,
                    std::string* err);
// The same with the caller's weights (record order), added to the column-major
// image `into`, or put there.
int moment_backward_into(MomentPlan& plan, const float* weights, float* into,
                         bool add, hipStream_t stream, std::string* err);
// The sum of the plan's images added to `into`, or put there, and the images
// cleared (nothing where `into` is where the back-projection adds).
int moment_fold(MomentPlan& plan, float* into, bool add, hipStream_t stream,
                std::string* err);
// out[stride * (band of the record * n_events + record) + {0, 1, 2}] = sum K x,
// sum K x Q, sum K x (w - Qd) of the column-major image xT (strip_adjoint.hip)
int moment_gradient(MomentPlan& plan, const float* xT, int stride, float* out,
                    hipStream_t stream, std::string* err);
// The plans of many reconstructions, iterated together: one launch per pass and
// kind of task (terms, wavefronts, merged, workgroups that share a CU).
struct MomentBatch {
  struct Launch {
    bool backward;
    int terms, waves;
    bool merged;
    size_t lds;
    int first, n;  // tasks
  };
  std::vector<Launch> launches;
  MomentInstance* desc[2] = {nullptr, nullptr};  // image parity 0 / 1
  MomentTask* tasks = nullptr;
};
void moment_batch_release(MomentBatch& batch);
int moment_batch_build(MomentBatch& batch,
                       const std::vector<const MomentPlan*>& plans,
                       hipStream_t stream, std::string* err);
// the forward or back-projection launches, image parity c
int moment_batch_launch(const MomentBatch& batch, int c, bool backward,
                        hipStream_t stream, std::string* err);
// *total += kernel evaluations of the stored runs
int moment_count(MomentPlan& plan, unsigned long long* total,
                 hipStream_t stream, std::string* err);

}  // namespace strip
