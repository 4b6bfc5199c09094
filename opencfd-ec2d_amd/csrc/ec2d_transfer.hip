// What the host reads and writes between launches: the caller's arrays (in
// the reference's layouts: i fastest after the component, sub_init.f90:20-60)
// and a mailbox with the error words, norms and forces.
//
// A kernel reads and writes pinned host memory itself.  Array traffic is then
// one launch and one wait per chunk instead of, for every component, a copy of
// the whole padded plane each way and a strided loop on the host.  257 x 65
// cells of five equations (0.7 MB): put 163 -> 39 us, get 121 -> 44 us; norms of
// the last residual 79 -> 17 us, forces 26 -> 17 us (before: four copies and
// three waits, one copy and one wait).  The host's own copy takes most of what
// is left of a put or get.
//   Threads run along the host array, so that transfers over the link are
// whole lines; the planes' side is strided by components within a few
// lines, which the caches merge.
#include "ec2d_device.h"

namespace ec2d {

// elements [e0, e0 + n) of a caller's array a[j][i][m], i = lo .. lo + ni - 1,
// j from lo, m < nc, and their places in the block's planes
struct MoveArgs {
  BlockDesc b;
  double* planes;  // plane of component 0
  double* host;    // staging: element e0 first
  int64_t e0;
  int n, nc, ni, lo;
};

template <bool PUT>
__global__ __launch_bounds__(256) void k_move(MoveArgs a) {
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (t >= a.n) return;
  const int64_t e = a.e0 + t, cell = e / a.nc;
  const int m = (int)(e - cell * a.nc), j = (int)(cell / a.ni), i = (int)(cell - (int64_t)j * a.ni);
  double* p = a.planes + m * a.b.plane + pidx(a.b, a.lo + i, a.lo + j);
  if (PUT) *p = a.host[t];
  else a.host[t] = *p;
}

// Pinned; the host reads it once the stream has drained.
struct Mail {
  double norms[12];         // ec2d_res_norms: maxima, then rms, of one case
  double forces[4];         // k_forces
  unsigned long long derr;  // the device's error words (device_errors)
  int sweep_err;
};

__device__ inline void mail_errors(Mail* mail, const unsigned long long* derr, const int* sweep_err) {
  mail->derr = *derr;
  mail->sweep_err = *sweep_err;
}

__global__ void k_mail(Mail* mail, const double* norms, const unsigned long long* derr, const int* sweep_err) {
  if (norms && threadIdx.x < 12) mail->norms[threadIdx.x] = norms[threadIdx.x];
  if (threadIdx.x == 0) mail_errors(mail, derr, sweep_err);
}

}  // namespace ec2d
