// domain.cpp -- host side of a device-resident lattice domain.
#include "domain.hpp"
#include "host_pipe.hpp"

#include <algorithm>
#include <cmath>
#include <cstring>
#include <functional>
#include <limits>
#include <mutex>

#include "lattice.hpp"

namespace wake_hip {

// A failed runtime call also stays the thread's "last error" until read,
// and kernel launches are checked with hipGetLastError(); reset it here so
// a handled failure (e.g. an allocation refused for lack of HBM) is not
// reported again by the next launch.
void check(hipError_t e, const char* what) {
  if (e != hipSuccess) {
    (void)hipGetLastError();
    throw HipError(std::string(what) + ": " + hipGetErrorString(e));
  }
}

namespace {

struct LatTab {
  int Q;
  const int *cx, *cy, *cz, *opp;
  const float* w;
};

template <class L>
LatTab tab_of() {
  return {L::Q, L::cx, L::cy, L::cz, L::opp, L::w};
}

LatTab tab(int lattice) {
  if (lattice == 9) return tab_of<D2Q9>();
  if (lattice == 27) return tab_of<D3Q27>();
  return tab_of<D3Q19>();
}

// Round a float to the population storage format (bits of the element).
uint16_t to_half_bits(float v) {
  _Float16 h = static_cast<_Float16>(v);
  uint16_t b;
  std::memcpy(&b, &h, 2);
  return b;
}
uint16_t to_bf16_bits(float v) {
  uint32_t b;
  std::memcpy(&b, &v, 4);
  return static_cast<uint16_t>((b + 0x7FFFu + ((b >> 16) & 1u)) >> 16);
}
float from_half_bits(uint16_t b) {
  _Float16 h;
  std::memcpy(&h, &b, 2);
  return static_cast<float>(h);
}
float from_bf16_bits(uint16_t b) {
  uint32_t u = static_cast<uint32_t>(b) << 16;
  float f;
  std::memcpy(&f, &u, 4);
  return f;
}

size_t elem_size(int storage) { return storage == kStoreF32 ? 4 : 2; }

}  // namespace

// Live domains, for device_copy_of_host_populations().
namespace {
std::mutex g_live_mutex;
std::vector<const Domain*> g_live;
}  // namespace

const float* device_copy_of_host_populations(const float* host, size_t count) {
  if (!host) return nullptr;
  std::lock_guard<std::mutex> lock(g_live_mutex);
  for (const Domain* d : g_live)
    if (d->fsrc_valid_ && d->sout_is_fsrc_ && d->d_sout_ && host == d->h_fsrc_.data() &&
        count == static_cast<size_t>(d->Q_) * d->N_)
      return d->d_sout_;
  return nullptr;
}

Domain::Domain(int dim, int lattice, int nx, int ny, int nz, float tau, int storage, long long plane_pad)
    : dim_(dim), lattice_(lattice), nx_(nx), ny_(ny), nz_(dim == 2 ? 1 : nz), storage_(storage), tau_(tau) {
  if (dim != 2 && dim != 3) throw HipError("dimension must be 2 or 3");
  // 0 picks the default lattice of the dimension (D2Q9, D3Q19)
  if (dim == 2 && lattice != 0 && lattice != 9) throw HipError("a 2D domain uses D2Q9 (lattice 9)");
  if (dim == 3 && lattice != 0 && lattice != 19 && lattice != 27) throw HipError("a 3D domain uses lattice 19 or 27");
  if (dim == 2) lattice_ = 9;
  else if (lattice == 0) lattice_ = 19;
  if (storage < kStoreF32 || storage > kStoreBF16) throw HipError("unknown population storage format");
  if (nx_ < 2 || ny_ < 1 || nz_ < 1) throw HipError("grid dimensions must be positive (nx >= 2)");
  Q_ = lattice_;
  N_ = static_cast<size_t>(nx_) * ny_ * nz_;
  if (N_ >= (1ull << 31)) throw HipError("grid larger than 2^31 nodes");
  elem_ = elem_size(storage);
  const long long base = static_cast<long long>((N_ + 255) / 256 * 256);
  stride_ = base + (plane_pad >= 0 ? plane_pad : (N_ >= (1u << 20) ? 1024 : 0));
  is_periodic_ = (dim == 3);
  try {
    allocate_and_initialize();
  } catch (...) {
    release();  // the destructor does not run for a constructor that throws
    throw;
  }
  std::lock_guard<std::mutex> lock(g_live_mutex);
  g_live.push_back(this);
}

void Domain::allocate_and_initialize() {
  check(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking), "hipStreamCreate");
  for (int b = 0; b < 2; ++b) buf_[b] = alloc(static_cast<size_t>(Q_) * stride_ * elem_);
  d_flags_ = static_cast<uint8_t*>(alloc(N_));
  d_cls_ = static_cast<uint8_t*>(alloc(N_));
  d_aux_ = static_cast<int*>(alloc(N_ * sizeof(int)));
  d_bmask_ = static_cast<uint32_t*>(alloc(N_ * sizeof(uint32_t)));
  d_prev_ = static_cast<float*>(alloc(static_cast<size_t>(prev_stride(Q_)) * ny_ * nz_ * sizeof(float)));
  d_rho_ = static_cast<float*>(alloc(N_ * 4));
  d_ux_ = static_cast<float*>(alloc(N_ * 4));
  d_uy_ = static_cast<float*>(alloc(N_ * 4));
  d_uz_ = static_cast<float*>(alloc(N_ * 4));
  d_speed_ = static_cast<float*>(alloc(N_ * 4));
  d_partial_ = static_cast<double*>(alloc(3 * 1024 * sizeof(double)));
  d_out_ = static_cast<double*>(alloc(8 * sizeof(double)));
  d_nonfinite_ = static_cast<int*>(alloc(sizeof(int)));
  d_nfcount_ = static_cast<unsigned long long*>(alloc(2 * sizeof(unsigned long long)));
  flags_.assign(N_, kFluid);
  initialize(1.0f, 0.0f, 0.0f, 0.0f);
}

Domain::~Domain() { release(); }

void Domain::release() noexcept {
  bool last = false;
  {
    std::lock_guard<std::mutex> lock(g_live_mutex);
    g_live.erase(std::remove(g_live.begin(), g_live.end(), this), g_live.end());
    last = g_live.empty();
  }
  if (last) trim_host_pipe();
  if (stream_) (void)hipStreamSynchronize(stream_);
  for (hipEvent_t e : kev_) (void)hipEventDestroy(e);
  kev_.clear();
  if (kev_marker_) (void)hipEventDestroy(kev_marker_);
  kev_marker_ = nullptr;
  for (void* p : allocations_) (void)hipFree(p);
  allocations_.clear();
  if (stream_) (void)hipStreamDestroy(stream_);
  stream_ = nullptr;
  (void)hipGetLastError();  // nothing of the teardown reaches the next launch check
}

void* Domain::alloc(size_t bytes) {
  void* p = nullptr;
  check(hipMalloc(&p, bytes ? bytes : 1), "hipMalloc");
  allocations_.push_back(p);
  device_bytes_ += bytes;
  return p;
}

// The convective outlet store: one record of prev_stride(Q) floats per
// (y, z) row, value(row, q) for q < Q, zero padding.
void Domain::upload_prev(const std::function<float(size_t, int)>& value) {
  const int QP = prev_stride(Q_);
  const size_t rows = static_cast<size_t>(ny_) * nz_;
  h_prev_.assign(rows * QP, 0.0f);
  for (size_t r = 0; r < rows; ++r)
    for (int q = 0; q < Q_; ++q) h_prev_[r * QP + q] = value(r, q);
  check(hipMemcpyAsync(d_prev_, h_prev_.data(), h_prev_.size() * sizeof(float), hipMemcpyHostToDevice, stream_),
        "upload outlet store");
  check(hipStreamSynchronize(stream_), "upload outlet store");
}

void Domain::release(void* p) {
  if (!p) return;
  (void)hipFree(p);
  allocations_.erase(std::remove(allocations_.begin(), allocations_.end(), p), allocations_.end());
}

const void* Domain::state_buffer() const { return buf_[s_buf_ >= 0 ? s_buf_ : a_buf_]; }

// ------------------------------------------------------------ initialisation
// lattice_grid_3d.cpp:66-93: feq of uniform fields in both buffers, macro
// fields set, every cell type reset to Fluid.
void Domain::initialize(float rho, float ux, float uy, float uz) {
  ++version_;
  const LatTab L = tab(lattice_);
  const int slot = state_slot();
  if (dim_ == 2) uz = 0.0f;
  step_count_ = 0;
  const float u_sq = dim_ == 2 ? ux * ux + uy * uy : ux * ux + uy * uy + uz * uz;
  std::vector<float> fe_q(Q_);
  for (int q = 0; q < Q_; ++q) {
    const float ci_u = dim_ == 2 ? static_cast<float>(L.cx[q]) * ux + static_cast<float>(L.cy[q]) * uy
                                 : static_cast<float>(L.cx[q]) * ux + static_cast<float>(L.cy[q]) * uy +
                                       static_cast<float>(L.cz[q]) * uz;
    const float fe = L.w[q] * rho * (1.0f + 3.0f * ci_u + 4.5f * ci_u * ci_u - 1.5f * u_sq);
    void* plane = static_cast<char*>(buf_[slot]) + static_cast<size_t>(q) * stride_ * elem_;
    if (storage_ == kStoreF32) {
      uint32_t bits;
      std::memcpy(&bits, &fe, 4);
      check(hipMemsetD32Async(static_cast<hipDeviceptr_t>(plane), bits, stride_, stream_), "fill");
    } else {
      const uint16_t bits = storage_ == kStoreF16 ? to_half_bits(fe - L.w[q]) : to_bf16_bits(fe - L.w[q]);
      check(hipMemsetD16Async(static_cast<hipDeviceptr_t>(plane), bits, stride_, stream_), "fill");
    }
    fe_q[q] = fe;
  }
  upload_prev([&](size_t, int q) { return fe_q[q]; });
  s_buf_ = slot;
  a_buf_ = -1;
  unclosed_ = false;
  std::fill(flags_.begin(), flags_.end(), static_cast<uint8_t>(kFluid));
  moving_cells_ = false;
  flags_dirty_ = cls_dirty_ = true;
  ++flags_version_;
  const float sp = std::sqrt(u_sq);
  const float vals[5] = {rho, ux, uy, uz, sp};
  float* dst[5] = {d_rho_, d_ux_, d_uy_, d_uz_, d_speed_};
  for (int k = 0; k < 5; ++k) {
    uint32_t b;
    std::memcpy(&b, &vals[k], 4);
    check(hipMemsetD32Async(static_cast<hipDeviceptr_t>(dst[k]), b, N_, stream_), "fill");
  }
  invalidate_mirrors();
  dfields_valid_ = true;
  clear_nonfinite();
  check(hipStreamSynchronize(stream_), "initialize");
  if (probe_) probe_restart();
  refresh_held();
}

// The buffer a new state is written to.  A temperature goes on from where it
// is: a materialised S of it lies in that slot when this returns.
int Domain::state_slot() {
  if (!thermal_) return 0;
  if (s_buf_ >= 0) return s_buf_;
  sync_device_config();
  const int out = 1 - a_buf_;
  check(launch_materialize_thermal(args(false), gbuf_[a_buf_], gbuf_[out], stream_), "materialize temperature");
  return out;
}

// The state now is a materialised S in buffer `slot`, formed on the device.
void Domain::state_set(int slot) {
  ++version_;
  clear_nonfinite();
  s_buf_ = slot;
  a_buf_ = -1;
  unclosed_ = false;
  fsrc_valid_ = fdst_valid_ = sout_is_fsrc_ = false;
  if (probe_) probe_restart();  // the state the samples were taken of is gone
}

// After a state was set: whatever of it was handed out before.
void Domain::refresh_held() {
  refresh_mirrors(0);
  if (!h_fsrc_.empty()) f_src();
}

float* Domain::planes_scratch() {
  if (!d_sout_) d_sout_ = static_cast<float*>(alloc(static_cast<size_t>(Q_) * N_ * sizeof(float)));
  return d_sout_;
}

// lattice_grid_3d.cpp:95-131 with the per-node values as arrays; cell types
// are left untouched.
void Domain::initialize_fields(const float* rho, const float* ux, const float* uy, const float* uz) {
  const int slot = state_slot();
  step_count_ = 0;
  float* dst[4] = {d_rho_, d_ux_, d_uy_, d_uz_};
  const float* src[4] = {rho, ux, uy, dim_ == 2 ? nullptr : uz};
  for (int k = 0; k < 4; ++k) {
    if (src[k]) check(hipMemcpyAsync(dst[k], src[k], N_ * sizeof(float), hipMemcpyHostToDevice, stream_), "upload");
    else check(hipMemsetAsync(dst[k], 0, N_ * sizeof(float), stream_), "upload");
  }
  check(launch_init_fields(lattice_, storage_, d_rho_, d_ux_, d_uy_, d_uz_, d_speed_, buf_[slot], stride_, d_prev_,
                           nx_, static_cast<int>(N_), stream_),
        "initialize");
  state_set(slot);
  check(hipStreamSynchronize(stream_), "upload");  // the caller's arrays are free again
  drop_fields();
  dfields_valid_ = true;  // the fields given, not the moments of their equilibria
  refresh_held();
}

// The planes go up through the moment arrays, five at a time: they hold
// nothing after this, and a scratch of Q planes would double what a domain
// with 16-bit storage takes.
void Domain::set_populations(const float* f_ref) {
  before_config_change();
  const int slot = state_slot();
  invalidate_mirrors();
  float* const stage[5] = {d_rho_, d_ux_, d_uy_, d_uz_, d_speed_};
  for (int q = 0; q < Q_; q += 5) {
    const int count = std::min(5, Q_ - q);
    for (int k = 0; k < count; ++k)
      check(hipMemcpyAsync(stage[k], f_ref + static_cast<size_t>(q + k) * N_, N_ * sizeof(float),
                           hipMemcpyHostToDevice, stream_),
            "upload");
    check(launch_init_planes(lattice_, storage_, stage, q, count, 0.0f, 0, buf_[slot], stride_, d_prev_, nx_,
                             static_cast<int>(N_), stream_),
          "set populations");
  }
  state_set(slot);
  check(hipStreamSynchronize(stream_), "upload");
  planes_given_ = storage_ == kStoreF32;
  refresh_held();
}

// Seeded uniform noise U(-a, a) on every population, counter = node * Q + q.
// The fields stay those of the state without it until the next step, except
// right after set_populations() with FP32 storage: no field of those planes
// has been formed, and they are then the noisy ones.
void Domain::add_noise(float amplitude, uint64_t seed) {
  form_planes();
  const int slot = state_slot();
  const float* planes[27];
  for (int q = 0; q < Q_; ++q) planes[q] = d_sout_ + static_cast<size_t>(q) * N_;
  check(launch_init_planes(lattice_, storage_, planes, 0, Q_, amplitude, seed, buf_[slot], stride_, d_prev_, nx_,
                           static_cast<int>(N_), stream_),
        "noise");
  state_set(slot);
  check(hipStreamSynchronize(stream_), "noise");
  refresh_held();
}

// ------------------------------------------------------------- cell types
void Domain::before_config_change() {
  ++version_;
  if (s_buf_ < 0 && a_buf_ >= 0) materialize();
}

void Domain::set_cell_type(int x, int y, int z, uint8_t type) {
  if (x < 0 || x >= nx_ || y < 0 || y >= ny_ || z < 0 || z >= nz_) return;
  before_config_change();
  flags_[(static_cast<size_t>(z) * ny_ + y) * nx_ + x] = type;
  if (type != kFluid) is_periodic_ = false;
  // (noted here: looking for one over all cell types took 1.5 ms of the first
  // run after a change at 256^3)
  if (type == kMovingWall) moving_cells_ = true;
  flags_dirty_ = cls_dirty_ = true;
  ++flags_version_;
}

uint8_t Domain::get_cell_type(int x, int y, int z) const {
  if (x >= 0 && x < nx_ && y >= 0 && y < ny_ && z >= 0 && z < nz_)
    return flags_[(static_cast<size_t>(z) * ny_ + y) * nx_ + x];
  return kSolid;
}

void Domain::set_periodic(bool p) {
  before_config_change();
  is_periodic_ = p;
  cls_dirty_ = true;
}

void Domain::set_periodic_axes(bool py, bool pz) {
  before_config_change();
  ext_axes_ = true;
  per_y_ = py;
  per_z_ = pz;
  cls_dirty_ = true;
}

// lattice_grid_3d.cpp:149-158
void Domain::set_solid_box(int x0, int y0, int z0, int x1, int y1, int z1) {
  before_config_change();
  is_periodic_ = false;
  for (int z = std::max(0, z0); z <= std::min(nz_ - 1, z1); ++z)
    for (int y = std::max(0, y0); y <= std::min(ny_ - 1, y1); ++y)
      for (int x = std::max(0, x0); x <= std::min(nx_ - 1, x1); ++x) set_cell_type(x, y, z, kSolid);
}

// naca_airfoil.cpp:23-41 (digits -> camber, camber position, thickness) and
// :113-150 (contains_point), statement for statement in FP32 so the flags are
// bit-exact: the query point is turned into the unrotated chord frame and
// tested against the 4-digit thickness and camber lines.
namespace {
struct Naca {
  float camber, camber_pos, thickness, chord, aoa_deg;
  bool contains(float x, float y, float lead_x, float lead_y) const {
    const float kPi = 3.14159265358979323846f;
    const float dx = x - lead_x;
    const float dy = y - lead_y;
    const float alpha_rad = -aoa_deg * (kPi / 180.0f);
    const float cos_a = std::cos(-alpha_rad);
    const float sin_a = std::sin(-alpha_rad);
    const float x_chord = dx * cos_a - dy * sin_a;
    const float y_chord = dx * sin_a + dy * cos_a;
    if (x_chord < 0.0f || x_chord > chord) return false;
    const float xc = x_chord / chord;
    const float yt = 5.0f * thickness *
                     (0.2969f * std::sqrt(xc) - 0.1260f * xc - 0.3516f * xc * xc + 0.2843f * xc * xc * xc -
                      0.1036f * xc * xc * xc * xc) *
                     chord;
    float yc = 0.0f;
    if (camber_pos > 1e-6f) {
      if (xc < camber_pos) {
        yc = (camber / (camber_pos * camber_pos)) * (2.0f * camber_pos * xc - xc * xc) * chord;
      } else {
        const float one_minus_p = 1.0f - camber_pos;
        yc = (camber / (one_minus_p * one_minus_p)) * ((1.0f - 2.0f * camber_pos) + 2.0f * camber_pos * xc - xc * xc) *
             chord;
      }
    }
    return std::abs(y_chord - yc) <= yt;
  }
};
}  // namespace

// naca_airfoil.cpp:152-190: rasterize (2D) / voxelize_extruded over z0..z1 (3D).
void Domain::set_solid_naca(int digits, float chord, float aoa_deg, float lead_x, float lead_y, int z0, int z1) {
  if (digits < 0 || digits > 9999) throw HipError("NACA designation must be 4 digits");
  before_config_change();
  is_periodic_ = false;
  const int m_digit = digits / 1000, p_digit = (digits / 100) % 10, t_digits = digits % 100;
  Naca a{static_cast<float>(m_digit) / 100.0f, static_cast<float>(p_digit) / 10.0f,
         static_cast<float>(t_digits) / 100.0f, chord, aoa_deg};
  const float rad_bound = chord * 1.5f;
  const int min_x = std::max(0, static_cast<int>(lead_x - rad_bound));
  const int max_x = std::min(nx_ - 1, static_cast<int>(lead_x + rad_bound));
  const int min_y = std::max(0, static_cast<int>(lead_y - rad_bound));
  const int max_y = std::min(ny_ - 1, static_cast<int>(lead_y + rad_bound));
  const int za = dim_ == 2 ? 0 : std::max(0, z0), zb = dim_ == 2 ? 0 : std::min(nz_ - 1, z1);
  for (int y = min_y; y <= max_y; ++y)
    for (int x = min_x; x <= max_x; ++x)
      if (a.contains(static_cast<float>(x), static_cast<float>(y), lead_x, lead_y))
        for (int z = za; z <= zb; ++z) set_cell_type(x, y, z, kSolid);
}

// primitives.cpp:73-100: FP32 ellipsoid test, bit-exact flags.  With axes
// (rows = body axes in world coordinates) the point is first projected on
// the body axes and the box is bounded by the largest semi-axis.
void Domain::set_solid_ellipsoid(float cx, float cy, float cz, float rx, float ry, float rz, const float* axes) {
  before_config_change();
  is_periodic_ = false;
  float ex = rx, ey = ry, ez = rz;
  if (axes) ex = ey = ez = std::max(rx, std::max(ry, rz));
  const int min_x = std::max(0, static_cast<int>(cx - ex - 1.0f)), max_x = std::min(nx_ - 1, static_cast<int>(cx + ex + 1.0f));
  const int min_y = std::max(0, static_cast<int>(cy - ey - 1.0f)), max_y = std::min(ny_ - 1, static_cast<int>(cy + ey + 1.0f));
  const int min_z = std::max(0, static_cast<int>(cz - ez - 1.0f)), max_z = std::min(nz_ - 1, static_cast<int>(cz + ez + 1.0f));
  const float irx = 1.0f / (rx * rx), iry = 1.0f / (ry * ry), irz = 1.0f / (rz * rz);
  for (int z = min_z; z <= max_z; ++z)
    for (int y = min_y; y <= max_y; ++y)
      for (int x = min_x; x <= max_x; ++x) {
        float dx = static_cast<float>(x) - cx, dy = static_cast<float>(y) - cy, dz = static_cast<float>(z) - cz;
        if (axes) {
          const float b0 = axes[0] * dx + axes[1] * dy + axes[2] * dz;
          const float b1 = axes[3] * dx + axes[4] * dy + axes[5] * dz;
          const float b2 = axes[6] * dx + axes[7] * dy + axes[8] * dz;
          dx = b0;
          dy = b1;
          dz = b2;
        }
        if (dx * dx * irx + dy * dy * iry + dz * dz * irz <= 1.0f) set_cell_type(x, y, z, kSolid);
      }
}

// obj_loader.cpp:208-400 on the device.  The host mirror of the cell types
// is refreshed from the device afterwards; set_cell_type's rule applies: a
// Solid write clears the all-periodic mode.
void Domain::voxelize_mesh(const float* tris, long long ntri, bool fill_interior) {
  if (ntri < 0 || (ntri > 0 && !tris)) throw HipError("voxelize_mesh: bad triangle array");
  for (long long i = 0; i < 9 * ntri; ++i)
    if (!std::isfinite(tris[i])) throw HipError("voxelize_mesh: mesh vertices must be finite");
  before_config_change();
  if (flags_dirty_) {
    check(hipMemcpyAsync(d_flags_, flags_.data(), N_, hipMemcpyHostToDevice, stream_), "upload flags");
    flags_dirty_ = false;
  }
  bool any = false;
  check(launch_voxelize_mesh(tris, ntri, fill_interior, d_flags_, nx_, ny_, nz_, stream_, &any), "voxelize mesh");
  check(hipMemcpyAsync(flags_.data(), d_flags_, N_, hipMemcpyDeviceToHost, stream_), "download flags");
  check(hipStreamSynchronize(stream_), "voxelize mesh");
  if (any) is_periodic_ = false;
  cls_dirty_ = true;
  ++flags_version_;
}

// lattice_grid_3d.cpp:160-182 (FP32 ball test, bit-exact flags)
void Domain::set_solid_sphere(float cx, float cy, float cz, float radius) {
  before_config_change();
  is_periodic_ = false;
  const float r_sq = radius * radius;
  const int min_x = std::max(0, static_cast<int>(cx - radius - 1)), max_x = std::min(nx_ - 1, static_cast<int>(cx + radius + 1));
  const int min_y = std::max(0, static_cast<int>(cy - radius - 1)), max_y = std::min(ny_ - 1, static_cast<int>(cy + radius + 1));
  const int min_z = std::max(0, static_cast<int>(cz - radius - 1)), max_z = std::min(nz_ - 1, static_cast<int>(cz + radius + 1));
  for (int z = min_z; z <= max_z; ++z)
    for (int y = min_y; y <= max_y; ++y)
      for (int x = min_x; x <= max_x; ++x) {
        const float dx = static_cast<float>(x) - cx, dy = static_cast<float>(y) - cy, dz = static_cast<float>(z) - cz;
        if (dx * dx + dy * dy + dz * dz <= r_sq) set_cell_type(x, y, z, kSolid);
      }
}

// lattice_grid_2d.cpp:143-159
void Domain::set_solid_circle(float cx, float cy, float radius) {
  before_config_change();
  const float r_sq = radius * radius;
  const int min_x = std::max(0, static_cast<int>(cx - radius - 1)), max_x = std::min(nx_ - 1, static_cast<int>(cx + radius + 1));
  const int min_y = std::max(0, static_cast<int>(cy - radius - 1)), max_y = std::min(ny_ - 1, static_cast<int>(cy + radius + 1));
  for (int y = min_y; y <= max_y; ++y)
    for (int x = min_x; x <= max_x; ++x) {
      const float dx = static_cast<float>(x) - cx, dy = static_cast<float>(y) - cy;
      if (dx * dx + dy * dy <= r_sq) set_cell_type(x, y, 0, kSolid);
    }
}

// lattice_grid_3d.cpp:184-203
void Domain::set_solid_cylinder_z(float cx, float cy, float radius) {
  before_config_change();
  is_periodic_ = false;
  const float r_sq = radius * radius;
  const int min_x = std::max(0, static_cast<int>(cx - radius - 1)), max_x = std::min(nx_ - 1, static_cast<int>(cx + radius + 1));
  const int min_y = std::max(0, static_cast<int>(cy - radius - 1)), max_y = std::min(ny_ - 1, static_cast<int>(cy + radius + 1));
  for (int z = 0; z < nz_; ++z)
    for (int y = min_y; y <= max_y; ++y)
      for (int x = min_x; x <= max_x; ++x) {
        const float dx = static_cast<float>(x) - cx, dy = static_cast<float>(y) - cy;
        if (dx * dx + dy * dy <= r_sq) set_cell_type(x, y, z, kSolid);
      }
}

// lattice_grid_3d.cpp:205-215 (3D top wall) and lattice_grid_2d.cpp:178-184
// (2D north wall).
void Domain::set_moving_wall_top(float uwx, float uwz) {
  before_config_change();
  is_periodic_ = false;
  has_moving_wall_ = true;
  uwx_ = uwx;
  uwz_ = dim_ == 2 ? 0.0f : uwz;
  for (int z = 0; z < nz_; ++z)
    for (int x = 0; x < nx_; ++x) set_cell_type(x, ny_ - 1, z, kMovingWall);
}

// lattice_grid_2d.cpp:161-168 (3D: the x = 0 plane)
void Domain::set_inflow_west(float ux, float uy) {
  before_config_change();
  has_inflow_ = true;
  inflow_parabolic_ = false;
  uin_x_ = ux;
  uin_y_ = uy;
  for (int z = 0; z < nz_; ++z)
    for (int y = 0; y < ny_; ++y) set_cell_type(0, y, z, kInflow);
  cls_dirty_ = true;
}

void Domain::set_inflow_parabolic(float u_max) {
  set_inflow_west(u_max, 0.0f);
  inflow_parabolic_ = true;
  umax_ = u_max;
}

void Domain::set_inflow_turbulence(float amplitude, uint64_t seed) {
  before_config_change();
  turb_amp_ = amplitude;
  turb_seed_ = seed;
}

// lattice_grid_2d.cpp:170-176
void Domain::set_outflow_east(float rho_out) {
  before_config_change();
  outflow_ = 1;
  rho_out_ = rho_out;
  for (int z = 0; z < nz_; ++z)
    for (int y = 0; y < ny_; ++y) set_cell_type(nx_ - 1, y, z, kOutflow);
  cls_dirty_ = true;
}

void Domain::set_convective_outflow_east(float u_conv) {
  // the outlet blends in its upstream neighbour x = nx - 2
  if (nx_ < 2) throw HipError("wake: convective outflow needs nx >= 2");
  before_config_change();
  outflow_ = 2;
  u_conv_ = u_conv;
  for (int z = 0; z < nz_; ++z)
    for (int y = 0; y < ny_; ++y) set_cell_type(nx_ - 1, y, z, kOutflow);
  // the outlet store starts from the current post-stream state (S is
  // materialised by before_config_change)
  check(launch_prev_from_s(lattice_, storage_, args(false), buf_[s_buf_], stream_), "outlet store");
  cls_dirty_ = true;
}

// lattice_grid_3d.cpp:217-290: links in z -> y -> x -> q order from Fluid
// nodes to Solid neighbours (x periodic, y/z in range or wrapped on a
// periodic axis), FP32 ray-sphere quadratic, delta clamped to [0.01, 0.99];
// built on the device from the device cell types (geometry.hip).
int Domain::build_curved_sphere_links(float cx, float cy, float cz, float radius) {
  before_config_change();
  is_periodic_ = false;
  if (flags_dirty_) {
    check(hipMemcpyAsync(d_flags_, flags_.data(), N_, hipMemcpyHostToDevice, stream_), "upload flags");
    flags_dirty_ = false;
    cls_dirty_ = true;
  }
  CurvedLinks k;
  check(launch_build_sphere_links(lattice_, d_flags_, nx_, ny_, nz_, ext_axes_ && per_y_, ext_axes_ && per_z_, cx, cy,
                                  cz, radius, stream_, k.fluid_index, k.q_dir, k.delta),
        "build curved links");
  k.uw_x.assign(k.fluid_index.size(), 0.0f);
  k.uw_y.assign(k.fluid_index.size(), 0.0f);
  k.uw_z.assign(k.fluid_index.size(), 0.0f);
  set_curved_links(k);
  return static_cast<int>(links_.fluid_index.size());
}

void Domain::set_curved_links(const CurvedLinks& links) {
  before_config_change();
  links_ = links;
  bfl_dirty_ = cls_dirty_ = true;
}

// ------------------------------------------------------------ device sync
StepArgs Domain::args(bool commit) const {
  StepArgs a;
  std::memset(&a, 0, sizeof(a));
  a.nx = nx_;
  a.ny = ny_;
  a.nz = nz_;
  a.stride = stride_;
  a.periodic_mode = (is_periodic_ && !has_moving_wall_) ? 1 : 0;
  a.per_y = ext_axes_ && per_y_;
  a.per_z = ext_axes_ && per_z_;
  a.bfl_per_y = a.per_y;
  a.bfl_per_z = a.per_z;
  a.tau = tau_;
  a.uw[0] = has_moving_wall_ ? uwx_ : 0.0f;
  a.uw[1] = 0.0f;
  a.uw[2] = has_moving_wall_ && dim_ == 3 ? uwz_ : 0.0f;
  a.inflow = has_inflow_ ? 1 : 0;
  a.inflow_parabolic = inflow_parabolic_ ? 1 : 0;
  a.uin_x = uin_x_;
  a.uin_y = uin_y_;
  a.umax = umax_;
  a.turb_amp = turb_amp_;
  a.turb_seed = turb_seed_;
  a.s_step = step_count_;
  int outflow = outflow_;
  if (outflow == 1 && (dim_ != 2 || a.per_y)) outflow = 0;  // the pressure outlet exists in 2D only
  a.outflow = outflow;
  a.rho_out = rho_out_;
  a.u_conv = u_conv_;
  a.conv_alpha = u_conv_ / (1.0f + u_conv_);
  a.conv_beta = 1.0f / (1.0f + u_conv_);
  a.by0 = a.per_y ? 0 : 1;
  a.by1 = a.per_y ? ny_ : ny_ - 1;
  a.bz0 = dim_ == 2 ? 0 : (a.per_z ? 0 : 1);
  a.bz1 = dim_ == 2 ? 1 : (a.per_z ? nz_ : nz_ - 1);
  a.commit_prev = commit ? 1 : 0;
  a.keep_stores = keep_stores_for(2ull * Q_ * stride_ * elem_) ? 1 : 0;
  a.global_addr = buffer_addressing_ ? 0 : 1;
  a.f_prev = d_prev_;
  a.flags = d_flags_;
  a.cls = d_cls_;
  a.aux = d_aux_;
  a.bmask = d_bmask_;
  a.mmask = d_mmask_;
  a.bfl = d_bfl_;
  a.gx = g_last_[0];
  a.gy = g_last_[1];
  a.gz = g_last_[2];
  a.tau_g = tau_g_;
  a.gbeta = gbeta_;
  a.t_ref = t_ref_;
  a.t_wall = d_twall_;
  a.nonfinite = d_nonfinite_;
  return a;
}

void Domain::sync_device_config() {
  if (twall_dirty_) {
    check(hipMemcpyAsync(d_twall_, h_twall_.data(), N_ * sizeof(float), hipMemcpyHostToDevice, stream_),
          "upload wall temperatures");
    twall_dirty_ = false;
  }
  if (flags_dirty_) {
    check(hipMemcpyAsync(d_flags_, flags_.data(), N_, hipMemcpyHostToDevice, stream_), "upload flags");
    flags_dirty_ = false;
    cls_dirty_ = true;
  }
  if (bfl_dirty_) {
    // group the links (z -> y -> x -> q order) into one record per fluid node
    const LatTab L = tab(lattice_);
    std::vector<BflNode> recs;
    std::vector<int> nodes;
    for (size_t i = 0; i < links_.fluid_index.size(); ++i) {
      const int n = links_.fluid_index[i];
      if (nodes.empty() || nodes.back() != n) {
        nodes.push_back(n);
        BflNode r;
        std::memset(&r, 0, sizeof(r));
        recs.push_back(r);
      }
      BflNode& r = recs.back();
      const int q = links_.q_dir[i];
      r.mask |= 1u << q;
      r.delta[q] = links_.delta[i];
      r.ciuw[q] = static_cast<float>(L.cx[q]) * links_.uw_x[i] + static_cast<float>(L.cy[q]) * links_.uw_y[i] +
                  static_cast<float>(L.cz[q]) * links_.uw_z[i];
    }
    if (d_bfl_) {
      (void)hipStreamSynchronize(stream_);
      (void)hipFree(d_bfl_);
      (void)hipFree(d_bfl_nodes_);
      allocations_.erase(std::remove(allocations_.begin(), allocations_.end(), static_cast<void*>(d_bfl_)),
                         allocations_.end());
      allocations_.erase(std::remove(allocations_.begin(), allocations_.end(), static_cast<void*>(d_bfl_nodes_)),
                         allocations_.end());
      d_bfl_ = nullptr;
      d_bfl_nodes_ = nullptr;
    }
    n_bfl_nodes_ = static_cast<int>(nodes.size());
    if (n_bfl_nodes_ > 0) {
      d_bfl_ = static_cast<BflNode*>(alloc(recs.size() * sizeof(BflNode)));
      d_bfl_nodes_ = static_cast<int*>(alloc(nodes.size() * sizeof(int)));
      check(hipMemcpyAsync(d_bfl_, recs.data(), recs.size() * sizeof(BflNode), hipMemcpyHostToDevice, stream_), "bfl");
      check(hipMemcpyAsync(d_bfl_nodes_, nodes.data(), nodes.size() * sizeof(int), hipMemcpyHostToDevice, stream_),
            "bfl");
      check(hipStreamSynchronize(stream_), "bfl");
    }
    bfl_dirty_ = false;
    cls_dirty_ = true;
  }
  if (cls_dirty_) {
    all_fluid_ = std::all_of(flags_.begin(), flags_.end(), [](uint8_t t) { return t == kFluid; });
    if (!d_mmask_ && moving_cells_) d_mmask_ = static_cast<uint32_t*>(alloc(N_ * sizeof(uint32_t)));
    const StepArgs a = args(false);
    check(launch_build_class(lattice_, a, d_cls_, d_bmask_, d_mmask_, stream_), "build class");
    check(launch_mark_bfl(d_bfl_nodes_, n_bfl_nodes_, d_cls_, d_aux_, stream_), "mark bfl");
    cls_dirty_ = false;
    ++cls_epoch_;
  }
}

// Solid nodes in the inlet and outlet rows as single steps leave them.
void Domain::close_solids() {
  if (unclosed_ && dim_ == 2 && (has_inflow_ || outflow_ == 1)) {
    StepArgs a = args(false);
    a.s_step = step_count_ - 1;
    check(launch_close_solid(storage_, a, buf_[a_buf_], stream_), "solid nodes");
  }
  unclosed_ = false;
}

void Domain::materialize() {
  sync_device_config();
  close_solids();  // f_dst may be read after the change this comes before
  if (probe_) {
    // the force sample of S_k is taken from the unrounded S, as a pull
    // launch would take it, before the state is stored
    probe_sync();
    probe_sample_current();
  }
  const StepArgs a = args(true);
  const int out = 1 - a_buf_;
  check(launch_materialize(lattice_, storage_, a, buf_[a_buf_], buf_[out], stream_), "materialize");
  if (thermal_) check(launch_materialize_thermal(a, gbuf_[a_buf_], gbuf_[out], stream_), "materialize temperature");
  s_buf_ = out;
}

// ------------------------------------------------------------------ step
bool Domain::tile_kind() const {
  if (dim_ != 2 || !tile_enabled_) return false;
  // curved links and the convective outlet read past the tile's halo
  if (n_bfl_nodes_ > 0 || outflow_ == 2) return false;
  // (the temperature kernels with BF16 storage round some products otherwise
  // in a step loop than in a single step)
  return !(thermal_ && storage_ == kStoreBF16);
}

bool Domain::tiles_pay(int storage, bool thermal, uint64_t nodes) {
  // Measured, us a step of single launches / tiles without forces: FP32
  // channels 4.6 / 1.8 at 240 x 80, 12.8 / 8.6 at 1500 x 403, 202 / 147 at
  // 4096^2; FP32 temperature 6.0 / 2.2 at 240 x 80, 36 / 31 at 1536 x 1024, 341 / 326 at 4096^2.  With
  // 16-bit storage a single launch moves half the bytes, so the largest
  // domains do without: TRT channels 19.2 / 19.7 at 1536 x 1024, 151 / 153 at
  // 4096^2 (MRT 135 / 130); temperature 14.3 / 13.7 at 1024 x 512, 30 / 37 at
  // 1536 x 1024.
  if (storage == kStoreF32) return true;
  return nodes <= (thermal ? 1u << 19 : 1u << 23);
}

bool Domain::tile_eligible() const { return tile_kind() && tiles_pay(storage_, thermal_, N_); }

bool Domain::batch_tiles() {
  sync_device_config();
  return tile_kind();
}

bool Domain::plain_periodic() const {
  return all_fluid_ && is_periodic_ && !has_moving_wall_ && !has_inflow_ && outflow_ == 0 && !thermal_;
}

void Domain::step_tile(int nsteps, int collision, float gx, float gy, bool use_les, float smag) {
  version_ += static_cast<uint64_t>(nsteps);
  const bool from_s = s_buf_ >= 0;
  TileForces mf{};
  // samples follow one another: after steps that took none (a batch's) the
  // history stays where it ended
  const bool sampling = probe_ && fh_next_ >= step_count_;
  if (sampling) {
    probe_sync();
    // a launch from a materialised S forms S_{k+1} first
    if (from_s) probe_sample_current();
    mf = probe_tile(nsteps);
  }
  StepArgs a = args(true);
  a.tau = tau_;
  a.gx = gx;
  a.gy = gy;
  a.gz = 0.0f;
  a.cs = smag;
  for (int k = 0; k < 3; ++k) a.mem_c[k] = probe_c_[k];
  a.mem_rmax = probe_rmax_;
  const int in = from_s ? s_buf_ : a_buf_, out = 1 - in;
  check(launch_tile2d(storage_, collision, use_les && les_coupled_, thermal_, from_s, !plain_periodic() || mf.index, nsteps, a,
                      buf_[in], buf_[out], gbuf_[in], gbuf_[out], mf, stream_),
        "tile steps");
  a_buf_ = out;
  s_buf_ = -1;
  unclosed_ = nsteps > (from_s ? 1 : 0);
  g_last_[0] = gx;
  g_last_[1] = gy;
  g_last_[2] = 0.0f;
  step_count_ += static_cast<uint64_t>(nsteps);
  if (sampling) fh_next_ = tile_end_ = step_count_;
  invalidate_mirrors();
}

void Domain::step(int collision, float gx, float gy, float gz, bool use_les, float smag) {
  ++version_;
  sync_device_config();
  if (probe_) probe_sync();
  if (dim_ == 2) gz = 0.0f;
  StepArgs a = args(true);
  a.tau = tau_;
  a.gx = gx;
  a.gy = gy;
  a.gz = gz;
  a.cs = smag;
  const bool les = use_les && les_coupled_;
  if (thermal_) {
    // coupled flow + temperature: one kernel, open boundaries inline
    const bool pull = s_buf_ < 0;
    const int in = pull ? a_buf_ : s_buf_;
    const int out = 1 - in;
    check(launch_step_thermal(storage_, collision, pull, a, buf_[in], buf_[out], gbuf_[in], gbuf_[out], stream_),
          "thermal step");
    a_buf_ = out;
    s_buf_ = -1;
  } else if (s_buf_ >= 0) {
    // S_k is materialised: the collide-only launch forms no S, so the force
    // sample of S_k is taken from the materialised state
    if (probe_) probe_sample_current();
    const int out = 1 - s_buf_;
    check(launch_step(lattice_, storage_, collision, les, false, a, buf_[s_buf_], buf_[out], block_x_, stream_),
          "step");
    a_buf_ = out;
    s_buf_ = -1;
  } else {
    const int out = 1 - a_buf_;
    // the pull forms S_k: its force sample is taken inside the launch
    if (probe_ && fh_next_ == step_count_) {
      a = with_mem(a, probe_rows_, probe_slot(step_count_), probe_c_, probe_rmax_);
      if (probe_rows_.nrows == 0) a.mem_rows = nullptr;
      fh_next_ = step_count_ + 1;
    }
    // A timed run brackets every kTimingStride-th pull launch with events:
    // a pair around every launch costs about 8 us (1.7% of a 256^3 FP32
    // step), which the sampled average no longer pays.
    // The start event is recorded after a plain marker: recorded straight
    // after the previous (unsampled) kernel it read the launch gap as part
    // of the kernel (462 vs 459 us per 256^3 FP32 step, rocprof 459 us).
    const bool sample = time_kernels_ && (timed_launches_++ % kTimingStride == 0);
    if (sample) {
      if (kev_used_ + 2 > kev_.size()) {
        for (int e = 0; e < 2; ++e) {
          hipEvent_t ev;
          check(hipEventCreate(&ev), "event");
          kev_.push_back(ev);
        }
      }
      if (!kev_marker_) check(hipEventCreate(&kev_marker_), "event");
      check(hipEventRecord(kev_marker_, stream_), "event");
      check(hipEventRecord(kev_[kev_used_], stream_), "event");
    }
    check(launch_step(lattice_, storage_, collision, les, true, a, buf_[a_buf_], buf_[out], block_x_, stream_),
          "step");
    if (sample) {
      check(hipEventRecord(kev_[kev_used_ + 1], stream_), "event");
      kev_used_ += 2;
    }
    a_buf_ = out;
  }
  g_last_[0] = gx;
  g_last_[1] = gy;
  g_last_[2] = gz;
  unclosed_ = false;
  ++step_count_;
  invalidate_mirrors();
}

float Domain::run(int steps, int collision, float gx, float gy, float gz, bool use_les, float smag, bool timed) {
  sync_device_config();
  hipEvent_t e0 = nullptr, e1 = nullptr;
  if (timed) {
    check(hipEventCreate(&e0), "event");
    check(hipEventCreate(&e1), "event");
    check(hipEventRecord(e0, stream_), "event");
  }
  time_kernels_ = timed;
  kev_used_ = 0;
  timed_launches_ = 0;
  try {
    int s = 0;
    // 2D domains: up to kTbSteps steps per launch (an untimed run only: the
    // kernel timer samples single-step launches)
    if (!timed && steps >= 2 && tile_eligible() && probe_lists(steps)) {
      const int most = tile2d_steps_of(nx_, ny_, thermal_ && storage_ == kStoreF32);
      while (steps - s >= 2) {
        const int k = std::min(steps - s, most);
        step_tile(k, collision, gx, gy, use_les, smag);
        s += k;
      }
    }
    for (; s < steps; ++s) step(collision, gx, gy, gz, use_les, smag);
  } catch (...) {
    time_kernels_ = false;
    throw;
  }
  time_kernels_ = false;
  float ms = 0.0f;
  if (timed) {
    check(hipEventRecord(e1, stream_), "event");
    check(hipEventSynchronize(e1), "event");
    check(hipEventElapsedTime(&ms, e0, e1), "event");
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    double sum = 0.0;
    for (size_t k = 0; k + 1 < kev_used_; k += 2) {
      float t = 0.0f;
      check(hipEventElapsedTime(&t, kev_[k], kev_[k + 1]), "event");
      sum += t;
    }
    last_kernel_ms_ = kev_used_ ? static_cast<float>(sum / (kev_used_ / 2)) : 0.0f;
  }
  return ms;
}

void Domain::synchronize() { check(hipStreamSynchronize(stream_), "synchronize"); }

// ------------------------------------------------------------- read-back
void Domain::ensure_device_fields() {
  if (dfields_valid_) return;
  sync_device_config();
  StepArgs a = args(false);
  a.rho = d_rho_;
  a.ux = d_ux_;
  a.uy = d_uy_;
  a.uz = d_uz_;
  a.speed = d_speed_;
  const bool from_s = s_buf_ >= 0;
  const int b = from_s ? s_buf_ : a_buf_;
  if (thermal_) {
    a.temp = d_temp_;
    check(launch_readback_thermal(storage_, from_s, a, buf_[b], gbuf_[b], stream_), "readback");
  } else {
    check(launch_readback(lattice_, storage_, from_s, a, buf_[b], stream_), "readback");
  }
  dfields_valid_ = true;
}

float* Domain::device_array(int which) {
  float* d[6] = {d_rho_, d_ux_, d_uy_, d_uz_, d_speed_, d_temp_};
  return d[which];
}

const float* Domain::mirror(int which) {
  if (!(mirrors_.load(std::memory_order_acquire) & (1u << which))) refresh_mirrors(1u << which);
  return h_field_[which].data();
}

void Domain::refresh_mirrors(unsigned want) {
  std::lock_guard<std::mutex> lock(mirror_mutex_);
  held_ |= want;
  const unsigned stale = held_ & ~mirrors_.load(std::memory_order_relaxed);
  if (stale == 0) return;
  ensure_device_fields();
  for (int k = 0; k < 6; ++k) {
    if (!(stale & (1u << k))) continue;
    h_field_[k].resize(N_);
    device_to_host(h_field_[k].data(), device_array(k), N_ * sizeof(float), stream_);
  }
  mirrors_.fetch_or(stale, std::memory_order_release);
}

void Domain::read_field(int which, float* out) {
  if (which == 5 && !thermal_) throw HipError("temperature is not enabled on this domain");
  if (mirrors_.load(std::memory_order_acquire) & (1u << which)) {
    std::memcpy(out, h_field_[which].data(), N_ * sizeof(float));
    return;
  }
  ensure_device_fields();
  device_to_host(out, device_array(which), N_ * sizeof(float), stream_);
}

// lattice_grid_3d.cpp:292-299: unforced moments of f_src, then |u|.
void Domain::update_macroscopic() {
  const float keep[3] = {g_last_[0], g_last_[1], g_last_[2]};
  g_last_[0] = g_last_[1] = g_last_[2] = 0.0f;
  drop_fields();
  ensure_device_fields();
  refresh_mirrors(0);
  g_last_[0] = keep[0];
  g_last_[1] = keep[1];
  g_last_[2] = keep[2];
}

void Domain::ensure_analytics(int which) {
  if (which < 0 || which > 3) throw HipError("unknown analytics field");
  if (dim_ == 2 && which != 2) throw HipError("a 2D domain has only the z vorticity");
  if (an_valid_) return;
  ensure_device_fields();
  const int k0 = dim_ == 2 ? 2 : 0, k1 = dim_ == 2 ? 2 : 3;
  for (int k = k0; k <= k1; ++k)
    if (!d_an_[k]) d_an_[k] = static_cast<float*>(alloc(N_ * sizeof(float)));
  if (dim_ == 2)
    check(launch_vorticity_2d(d_ux_, d_uy_, d_an_[2], nx_, ny_, stream_), "vorticity");
  else
    check(launch_vorticity_q_3d(d_ux_, d_uy_, d_uz_, d_an_[0], d_an_[1], d_an_[2], d_an_[3], nx_, ny_, nz_, stream_),
          "vorticity");
  an_valid_ = true;
  an_mirrors_ = 0;
}

const float* Domain::analytics(int which) {
  ensure_analytics(which);
  refresh_mirrors(0);
  if (!(an_mirrors_ & (1u << which))) {
    h_an_[which].resize(N_);
    device_to_host(h_an_[which].data(), d_an_[which], N_ * sizeof(float), stream_);
    an_mirrors_ |= 1u << which;
  }
  return h_an_[which].data();
}

void Domain::read_analytics(int which, float* out) {
  ensure_analytics(which);
  if (an_mirrors_ & (1u << which)) std::memcpy(out, h_an_[which].data(), N_ * sizeof(float));
  else device_to_host(out, d_an_[which], N_ * sizeof(float), stream_);
}

const float* Domain::device_field(int which) {
  if (which < 0 || which > 4) throw HipError("unknown device field");
  ensure_device_fields();
  const float* d[5] = {d_rho_, d_ux_, d_uy_, d_uz_, d_speed_};
  return d[which];
}

const uint8_t* Domain::device_cell_types() {
  sync_device_config();
  return d_flags_;
}

const float* Domain::rho() { return mirror(0); }
const float* Domain::ux() { return mirror(1); }
const float* Domain::uy() { return mirror(2); }
const float* Domain::uz() { return mirror(3); }
const float* Domain::speed() { return mirror(4); }

// S_k in the reference layout (FP32 planes of N) in d_sout_, and with it the
// moments where they are not current: those of this S, also when a change of
// the configuration rounds it to 16-bit storage later, and the planes read
// again are then these too.  (Planes just given have no moments yet; a
// temperature's come from its own read-back.)
void Domain::form_planes() {
  if (sout_is_fsrc_) return;
  sync_device_config();
  StepArgs a = args(false);
  a.s_out = planes_scratch();
  const bool moments = !dfields_valid_ && !planes_given_;
  if (moments && thermal_) ensure_device_fields();
  if (moments && !thermal_) {
    a.rho = d_rho_;
    a.ux = d_ux_;
    a.uy = d_uy_;
    a.uz = d_uz_;
    a.speed = d_speed_;
  }
  const bool from_s = s_buf_ >= 0;
  check(launch_readback(lattice_, storage_, from_s, a, buf_[from_s ? s_buf_ : a_buf_], stream_), "readback");
  if (moments) dfields_valid_ = true;
  sout_is_fsrc_ = true;
}

const float* Domain::f_src() {
  if (fsrc_valid_) return h_fsrc_.data();
  form_planes();
  h_fsrc_.resize(static_cast<size_t>(Q_) * N_);
  device_to_host(h_fsrc_.data(), d_sout_, h_fsrc_.size() * sizeof(float), stream_);
  fsrc_valid_ = true;
  refresh_mirrors(0);
  return h_fsrc_.data();
}

void Domain::read_f_src(float* out) {
  const size_t bytes = static_cast<size_t>(Q_) * N_ * sizeof(float);
  if (fsrc_valid_) {
    std::memcpy(out, h_fsrc_.data(), bytes);
    return;
  }
  form_planes();
  device_to_host(out, d_sout_, bytes, stream_);
}

// After step k the reference's f_dst holds A_{k-1}; before any step it holds
// the initial state.
bool Domain::form_dst_planes() {
  if (a_buf_ < 0) return false;
  close_solids();
  StepArgs a = args(false);
  a.s_out = planes_scratch();
  // planes only: read the buffer as-is (no moments written)
  check(launch_readback(lattice_, storage_, true, a, buf_[a_buf_], stream_), "readback");
  fsrc_valid_ = sout_is_fsrc_ = false;  // d_sout_ now holds f_dst
  return true;
}

const float* Domain::f_dst() {
  if (fdst_valid_) return h_fdst_.data();
  if (form_dst_planes()) {
    h_fdst_.resize(static_cast<size_t>(Q_) * N_);
    device_to_host(h_fdst_.data(), d_sout_, h_fdst_.size() * sizeof(float), stream_);
  } else {
    h_fdst_.assign(f_src(), f_src() + static_cast<size_t>(Q_) * N_);
  }
  fdst_valid_ = true;
  return h_fdst_.data();
}

void Domain::read_f_dst(float* out) {
  const size_t bytes = static_cast<size_t>(Q_) * N_ * sizeof(float);
  if (fdst_valid_) std::memcpy(out, h_fdst_.data(), bytes);
  else if (form_dst_planes()) device_to_host(out, d_sout_, bytes, stream_);
  else read_f_src(out);
}

void Domain::diagnostics(double out[3]) {
  ensure_device_fields();
  refresh_mirrors(0);
  sync_device_config();  // the reduction reads the device cell types
  check(launch_diagnostics(d_flags_, d_rho_, d_speed_, static_cast<long long>(N_), d_partial_, 1024, d_out_, stream_),
        "diagnostics");
  check(hipMemcpyAsync(out, d_out_, 3 * sizeof(double), hipMemcpyDeviceToHost, stream_), "d2h");
  check(hipStreamSynchronize(stream_), "diagnostics");
}

double Domain::total_mass() {
  double d[3];
  diagnostics(d);
  return d[0];
}

double Domain::total_kinetic_energy() {
  double d[3];
  diagnostics(d);
  return d[1];
}

double Domain::max_speed() {
  double d[3];
  diagnostics(d);
  return d[2];
}

// ------------------------------------------------------ momentum exchange
// Linked rows of (centre, r_max) from the device cell types: the rows are
// marked on the device, numbered here in (z, y) order, each given
// mem_waves_per_row(nx) partial slots.
Domain::MemRows Domain::build_mem_rows(float ccx, float ccy, float ccz, float r_max) {
  const size_t rows = static_cast<size_t>(ny_) * nz_;
  MemRows r;
  r.d_rows = static_cast<int*>(alloc(rows * sizeof(int)));
  StepArgs a = args(false);
  a.mem_c[0] = ccx;
  a.mem_c[1] = ccy;
  a.mem_c[2] = ccz;
  a.mem_rmax = r_max;
  check(hipMemsetAsync(r.d_rows, 0, rows * sizeof(int), stream_), "mark rows");
  check(launch_mem_mark_rows(lattice_, a, r.d_rows, stream_), "mark rows");
  std::vector<int> has(rows);
  check(hipMemcpyAsync(has.data(), r.d_rows, rows * sizeof(int), hipMemcpyDeviceToHost, stream_), "mark rows");
  check(hipStreamSynchronize(stream_), "mark rows");
  const int W = mem_waves_per_row(nx_);
  std::vector<int> list;
  for (size_t i = 0; i < rows; ++i) {
    if (has[i]) {
      has[i] = static_cast<int>(list.size()) * W;
      list.push_back(static_cast<int>(i));
    } else {
      has[i] = -1;
    }
  }
  r.nrows = static_cast<int>(list.size());
  r.nslots = r.nrows * W;
  r.d_list = static_cast<int*>(alloc(std::max<size_t>(1, list.size()) * sizeof(int)));
  check(hipMemcpyAsync(r.d_rows, has.data(), rows * sizeof(int), hipMemcpyHostToDevice, stream_), "rows");
  if (!list.empty())
    check(hipMemcpyAsync(r.d_list, list.data(), list.size() * sizeof(int), hipMemcpyHostToDevice, stream_), "rows");
  check(hipStreamSynchronize(stream_), "rows");  // the host vectors go out of scope
  return r;
}

// Per-row counts, their prefix on the host, then the nodes.
int* Domain::build_mem_nodes(const MemRows& rows, float ccx, float ccy, float ccz, float r_max, int* count) {
  *count = 0;
  const int nr = rows.nrows;
  if (nr == 0) return nullptr;
  StepArgs a = args(false);
  a.mem_c[0] = ccx;
  a.mem_c[1] = ccy;
  a.mem_c[2] = ccz;
  a.mem_rmax = r_max;
  int* d_cnt = static_cast<int*>(alloc(2 * static_cast<size_t>(nr) * sizeof(int)));
  int* d_nodes = nullptr;
  try {
    check(launch_mem_row_nodes(lattice_, a, rows.d_list, nr, d_cnt, nullptr, nullptr, stream_), "link nodes");
    std::vector<int> cnt(nr), off(nr);
    check(hipMemcpyAsync(cnt.data(), d_cnt, nr * sizeof(int), hipMemcpyDeviceToHost, stream_), "link nodes");
    check(hipStreamSynchronize(stream_), "link nodes");
    for (int r = 0; r < nr; ++r) {
      off[r] = *count;
      *count += cnt[r];
    }
    d_nodes = static_cast<int*>(alloc(std::max(1, *count) * sizeof(int)));
    check(hipMemcpyAsync(d_cnt + nr, off.data(), nr * sizeof(int), hipMemcpyHostToDevice, stream_), "link nodes");
    check(launch_mem_row_nodes(lattice_, a, rows.d_list, nr, d_cnt, d_cnt + nr, d_nodes, stream_), "link nodes");
    check(hipStreamSynchronize(stream_), "link nodes");
  } catch (...) {
    (void)hipStreamSynchronize(stream_);
    release(d_nodes);
    release(d_cnt);
    *count = 0;
    throw;
  }
  release(d_cnt);
  return d_nodes;
}

void Domain::free_mem_rows(MemRows& r) {
  if (r.d_rows || r.d_list) check(hipStreamSynchronize(stream_), "free rows");
  release(r.d_rows);
  release(r.d_list);
  r = MemRows{};
}

const Domain::MemRows& Domain::cached_mem_rows(float ccx, float ccy, float ccz, float r_max) {
  const auto key = std::make_tuple(ccx, ccy, ccz, r_max, cls_epoch_);
  auto it = mem_rows_cache_.find(key);
  if (it != mem_rows_cache_.end()) return it->second;
  if (mem_rows_cache_.size() >= 4) {
    for (auto& kv : mem_rows_cache_) free_mem_rows(kv.second);
    mem_rows_cache_.clear();
  }
  return mem_rows_cache_.emplace(key, build_mem_rows(ccx, ccy, ccz, r_max)).first->second;
}

StepArgs Domain::with_mem(StepArgs a, const MemRows& r, double* part, const float c[3], float r_max) const {
  a.mem_rows = r.d_rows;
  a.mem_part = part;
  a.mem_c[0] = c[0];
  a.mem_c[1] = c[1];
  a.mem_c[2] = c[2];
  a.mem_rmax = r_max;
  return a;
}

// Forces on the current S_k: the partials of the linked rows (S_k formed at
// the nodes next to a wall, or read from a materialised state), summed in
// slot order.  The same kernels and order as the per-step history.
void Domain::momentum_exchange(float ccx, float ccy, float ccz, float r_max, double out[3]) {
  sync_device_config();
  const MemRows& r = cached_mem_rows(ccx, ccy, ccz, r_max);
  if (r.nrows == 0) {
    out[0] = out[1] = out[2] = 0.0;
    return;
  }
  const size_t need = 3 * static_cast<size_t>(r.nslots);
  if (need > mempart_cap_) {
    if (d_mempart_) {
      check(hipStreamSynchronize(stream_), "momentum exchange");
      release(d_mempart_);
    }
    d_mempart_ = static_cast<double*>(alloc(need * sizeof(double)));
    mempart_cap_ = need;
  }
  const float c[3] = {ccx, ccy, ccz};
  const StepArgs a = with_mem(args(false), r, d_mempart_, c, r_max);
  const bool from_s = s_buf_ >= 0;
  check(launch_mem_rows(lattice_, storage_, from_s, a, buf_[from_s ? s_buf_ : a_buf_], r.d_list, r.nrows, stream_),
        "momentum exchange");
  check(launch_mem_fold(d_mempart_, r.nslots, 1, 0, 1, d_out_, 0, stream_), "momentum exchange");
  check(hipMemcpyAsync(out, d_out_, 3 * sizeof(double), hipMemcpyDeviceToHost, stream_), "d2h");
  check(hipStreamSynchronize(stream_), "momentum exchange");
}

// -------------------------------------------------------------- divergence
void Domain::clear_nonfinite() { check(hipMemsetAsync(d_nonfinite_, 0, sizeof(int), stream_), "clear flag"); }

bool Domain::nonfinite_seen() {
  int v = 0;
  check(hipMemcpyAsync(&v, d_nonfinite_, sizeof(int), hipMemcpyDeviceToHost, stream_), "d2h");
  check(hipStreamSynchronize(stream_), "divergence flag");
  return v != 0;
}

long long Domain::count_nonfinite(long long* first) {
  ensure_device_fields();
  unsigned long long h[2] = {0ull, ~0ull};
  check(hipMemcpyAsync(d_nfcount_, h, sizeof(h), hipMemcpyHostToDevice, stream_), "non-finite count");
  check(launch_count_nonfinite(d_rho_, d_speed_, static_cast<long long>(N_), d_nfcount_, stream_),
        "non-finite count");
  check(hipMemcpyAsync(h, d_nfcount_, sizeof(h), hipMemcpyDeviceToHost, stream_), "d2h");
  check(hipStreamSynchronize(stream_), "non-finite count");
  if (first) *first = h[0] ? static_cast<long long>(h[1]) : -1;
  return static_cast<long long>(h[0]);
}

// ------------------------------------------------------------- force probe
void Domain::set_force_probe(float ccx, float ccy, float ccz, float r_max) {
  if (thermal_) throw HipError("the force history is not available on temperature-coupled domains");
  // the linked rows and nodes belong to the centre, the radius and the
  // geometry (probe_epoch_): a restart of the same probe keeps them
  if (!probe_ || probe_c_[0] != ccx || probe_c_[1] != ccy || probe_c_[2] != ccz || probe_rmax_ != r_max) {
    if (probe_rows_.d_rows) free_mem_rows(probe_rows_);
    probe_epoch_ = tile_epoch_ = wait_epoch_ = ~0ull;
  }
  probe_ = true;
  probe_c_[0] = ccx;
  probe_c_[1] = ccy;
  probe_c_[2] = ccz;
  probe_rmax_ = r_max;
  if (!d_fhist_) d_fhist_ = static_cast<double*>(alloc(3 * static_cast<size_t>(kForceHistCap) * sizeof(double)));
  probe_restart();
}

void Domain::clear_force_probe() {
  probe_ = false;
  if (probe_rows_.d_rows) free_mem_rows(probe_rows_);
  probe_epoch_ = tile_epoch_ = ~0ull;
  h_fhist_.clear();
}

void Domain::probe_restart() {
  fh_first_ = fh_next_ = fh_folded_ = fh_dbase_ = fh_host_ = step_count_;
  tile_first_ = tile_end_ = step_count_;
  h_fhist_.clear();
}

// Rows for the current class bytes; samples written with the previous rows
// are folded first (their slot layout goes with those rows).
void Domain::probe_sync() {
  if (probe_epoch_ == cls_epoch_) return;
  probe_fold(fh_next_);
  if (probe_rows_.d_rows) free_mem_rows(probe_rows_);
  probe_rows_ = build_mem_rows(probe_c_[0], probe_c_[1], probe_c_[2], probe_rmax_);
  probe_epoch_ = cls_epoch_;
  // one slot at least: a geometry without links has all-zero samples
  const size_t need = 3 * static_cast<size_t>(kForceRing) * std::max(1, probe_rows_.nslots);
  if (need > ring_cap_) {
    if (d_ring_) {
      check(hipStreamSynchronize(stream_), "force ring");
      release(d_ring_);
    }
    d_ring_ = static_cast<double*>(alloc(need * sizeof(double)));
    ring_cap_ = need;
  }
  if (probe_rows_.nrows == 0) check(hipMemsetAsync(d_ring_, 0, need * sizeof(double), stream_), "force ring");
}

void Domain::probe_fold(uint64_t upto) {
  if (upto <= fh_folded_) return;
  probe_flush_tiles();
  if (upto - fh_dbase_ > static_cast<uint64_t>(kForceHistCap)) {
    // the device history is full: move what is folded to the host
    const size_t n = static_cast<size_t>(fh_folded_ - fh_host_);
    const size_t at = h_fhist_.size();
    h_fhist_.resize(at + 3 * n);
    if (n)
      check(hipMemcpyAsync(h_fhist_.data() + at, d_fhist_ + 3 * (fh_host_ - fh_dbase_), 3 * n * sizeof(double),
                           hipMemcpyDeviceToHost, stream_),
            "force history");
    check(hipStreamSynchronize(stream_), "force history");
    fh_host_ = fh_dbase_ = fh_folded_;
  }
  const int count = static_cast<int>(upto - fh_folded_);
  check(launch_mem_fold(d_ring_, std::max(1, probe_rows_.nslots), kForceRing, static_cast<long long>(fh_folded_),
                        count, d_fhist_, static_cast<long long>(fh_folded_ - fh_dbase_), stream_),
        "force fold");
  fh_folded_ = upto;
}

double* Domain::probe_slot(uint64_t k) {
  if (k - fh_folded_ >= static_cast<uint64_t>(kForceRing)) probe_fold(k);
  return d_ring_ + 3 * static_cast<size_t>(std::max(1, probe_rows_.nslots)) * (k % kForceRing);
}

// Whether the next `steps` steps may leave their samples through tile
// launches: the list of the nodes holding links, and the sums of a ring of
// steps for each.
bool Domain::probe_lists(int steps) {
  if (!probe_ || fh_next_ < step_count_) return true;  // no samples are taken
  probe_sync();
  if (tile_epoch_ == probe_epoch_) return tile_lists_;
  // Building them takes 60 us (240 x 80) to 90 us (1500 x 403 nodes), a tile
  // launch saves 3.6 to 4.6 us a step: they pay after 15 to 27 steps.  Until
  // then a geometry or a probe that changes from run to run takes single
  // steps.  (A domain's first lists are built at once: they are paid once, and
  // a new domain's first 20 steps take 226 us against 240, 449 against 475.)
  if (wait_epoch_ != probe_epoch_) wait_steps_ = 0;
  wait_epoch_ = probe_epoch_;
  if (lists_built_ && steps < kListSteps - wait_steps_) {
    wait_steps_ += steps;
    return false;
  }
  if (d_findex_ || d_fnode_) check(hipStreamSynchronize(stream_), "force nodes");
  free_tile_lists();
  tile_epoch_ = probe_epoch_;
  lists_built_ = true;
  int* d_nodes = nullptr;
  try {
    d_nodes = build_mem_nodes(probe_rows_, probe_c_[0], probe_c_[1], probe_c_[2], probe_rmax_, &n_fnodes_);
    // (a porous body can hold a link in every other node: past the size of
    // the state itself its samples are left to single steps)
    const size_t sums = 3 * sizeof(double) * kForceRing * static_cast<size_t>(n_fnodes_);
    tile_lists_ = sums <= std::max<size_t>(64u << 20, 2 * static_cast<size_t>(Q_) * stride_ * elem_);
    if (tile_lists_ && n_fnodes_ > 0) {
      d_findex_ = static_cast<int*>(alloc(N_ * sizeof(int)));
      d_fnode_ = static_cast<double*>(alloc(sums));
      check(hipMemsetAsync(d_findex_, 0xff, N_ * sizeof(int), stream_), "force nodes");
      check(launch_index_nodes(d_nodes, n_fnodes_, d_findex_, stream_), "force nodes");
      check(hipStreamSynchronize(stream_), "force nodes");
    }
  } catch (const HipError&) {
    tile_lists_ = false;  // no memory for them: single steps take the samples
  }
  release(d_nodes);
  if (!tile_lists_) free_tile_lists();
  return tile_lists_;
}

void Domain::free_tile_lists() {
  release(d_findex_);
  release(d_fnode_);
  d_findex_ = nullptr;
  d_fnode_ = nullptr;
  n_fnodes_ = 0;
}

// Samples a tile launch of nsteps steps from step_count_ takes: S_{fh_next_}
// up to S_{step_count_ + nsteps - 1}, as per-node sums in d_fnode_ until
// probe_flush_tiles() turns them into the ring's partials.
TileForces Domain::probe_tile(int nsteps) {
  if (tile_end_ != fh_next_) {
    probe_flush_tiles();
    tile_first_ = tile_end_ = fh_next_;
  }
  if (step_count_ + nsteps - fh_folded_ > static_cast<uint64_t>(kForceRing)) probe_fold(fh_next_);
  return TileForces{d_findex_, d_fnode_, n_fnodes_, kForceRing};
}

void Domain::probe_flush_tiles() {
  if (tile_first_ < tile_end_ && n_fnodes_ > 0)
    check(launch_mem_slots(TileForces{d_findex_, d_fnode_, n_fnodes_, kForceRing}, probe_rows_.d_list,
                           probe_rows_.nrows, nx_, static_cast<long long>(tile_first_),
                           static_cast<int>(tile_end_ - tile_first_), d_ring_, stream_),
          "force partials");
  tile_first_ = tile_end_;
}

// The sample of S_{step_count_} when no launch has formed it yet: read from
// a materialised state or formed from the post-collision buffer.
void Domain::probe_sample_current() {
  if (fh_next_ != step_count_) return;
  double* part = probe_slot(step_count_);
  if (probe_rows_.nrows > 0) {
    const StepArgs a = with_mem(args(false), probe_rows_, part, probe_c_, probe_rmax_);
    const bool from_s = s_buf_ >= 0;
    check(launch_mem_rows(lattice_, storage_, from_s, a, buf_[from_s ? s_buf_ : a_buf_], probe_rows_.d_list,
                          probe_rows_.nrows, stream_),
          "force sample");
  }
  fh_next_ = step_count_ + 1;
}

const std::vector<double>& Domain::force_history(uint64_t* first_step) {
  if (!probe_) throw HipError("no force probe is set on this domain");
  sync_device_config();
  probe_sync();
  probe_sample_current();
  probe_fold(fh_next_);
  const size_t n = static_cast<size_t>(fh_folded_ - fh_host_);
  if (n) {
    const size_t at = h_fhist_.size();
    h_fhist_.resize(at + 3 * n);
    check(hipMemcpyAsync(h_fhist_.data() + at, d_fhist_ + 3 * (fh_host_ - fh_dbase_), 3 * n * sizeof(double),
                         hipMemcpyDeviceToHost, stream_),
          "force history");
    check(hipStreamSynchronize(stream_), "force history");
    fh_host_ = fh_folded_;
  }
  if (first_step) *first_step = fh_first_;
  return h_fhist_;
}

// ------------------------------------------------------------- temperature
void Domain::enable_thermal(float tau_g, float gbeta, float t_ref, float t_init) {
  if (dim_ != 2) throw HipError("the temperature coupling is 2D (D2Q9 + D2Q5) only");
  if (probe_) throw HipError("clear the force probe before enabling the temperature coupling");
  if (!(tau_g > 0.5f)) throw HipError("temperature relaxation time must exceed 1/2");
  before_config_change();
  if (!thermal_) {
    for (int k = 0; k < 2; ++k) gbuf_[k] = static_cast<float*>(alloc(5 * static_cast<size_t>(stride_) * sizeof(float)));
    d_twall_ = static_cast<float*>(alloc(N_ * sizeof(float)));
    d_temp_ = static_cast<float*>(alloc(N_ * sizeof(float)));
    check(hipMemsetAsync(d_temp_, 0, N_ * sizeof(float), stream_), "temperature");
  }
  h_twall_.assign(N_, std::numeric_limits<float>::quiet_NaN());
  twall_dirty_ = true;
  thermal_ = true;
  tau_g_ = tau_g;
  gbeta_ = gbeta;
  t_ref_ = t_ref;
  std::vector<float> t(N_, t_init);
  set_temperature_field(t.data());
}

void Domain::set_temperature_field(const float* t) {
  if (!thermal_) throw HipError("temperature is not enabled on this domain");
  before_config_change();
  std::vector<float> host(5 * static_cast<size_t>(stride_), 0.0f);
  for (int q = 0; q < 5; ++q)
    for (size_t i = 0; i < N_; ++i) host[q * static_cast<size_t>(stride_) + i] = D2Q5::w[q] * t[i];
  for (int k = 0; k < 2; ++k)
    check(hipMemcpyAsync(gbuf_[k], host.data(), host.size() * sizeof(float), hipMemcpyHostToDevice, stream_),
          "upload temperature");
  check(hipStreamSynchronize(stream_), "upload temperature");
  drop_fields();
}

void Domain::set_wall_temperature(int x0, int y0, int x1, int y1, float t_wall) {
  if (!thermal_) throw HipError("temperature is not enabled on this domain");
  before_config_change();
  for (int y = std::max(0, y0); y <= std::min(ny_ - 1, y1); ++y)
    for (int x = std::max(0, x0); x <= std::min(nx_ - 1, x1); ++x) h_twall_[static_cast<size_t>(y) * nx_ + x] = t_wall;
  twall_dirty_ = true;
}

const float* Domain::temperature() {
  if (!thermal_) throw HipError("temperature is not enabled on this domain");
  return mirror(5);
}

// ------------------------------------------------------------ batched steps
void Domain::batch_prepare(float gx, float gy, float gz, float smag, StepArgs& a, void* buf[2], float* gbuf[2],
                           int& parity, bool& s_state) {
  sync_device_config();
  if (dim_ == 2) gz = 0.0f;
  a = args(true);
  a.gx = gx;
  a.gy = gy;
  a.gz = gz;
  a.cs = smag;
  buf[0] = buf_[0];
  buf[1] = buf_[1];
  gbuf[0] = gbuf_[0];
  gbuf[1] = gbuf_[1];
  s_state = s_buf_ >= 0;
  parity = s_state ? s_buf_ : a_buf_;
  // uploads were issued on the domain's stream; the batch runs on its own
  check(hipStreamSynchronize(stream_), "batch prepare");
}

void Domain::batch_advance(uint64_t k, int parity_after, float gx, float gy, float gz) {
  if (k == 0) return;
  unclosed_ = k > (s_buf_ >= 0 ? 1u : 0u);
  a_buf_ = parity_after;
  s_buf_ = -1;
  step_count_ += k;
  g_last_[0] = gx;
  g_last_[1] = gy;
  g_last_[2] = dim_ == 2 ? 0.0f : gz;
  invalidate_mirrors();
}

const int* Domain::batch_mem_nodes(float ccx, float ccy, float ccz, float r_max, int* count) {
  sync_device_config();
  const auto key = std::make_tuple(ccx, ccy, ccz, r_max, cls_epoch_);
  if (key != batch_rows_key_ || !batch_rows_.d_list) {
    if (batch_rows_.d_rows) free_mem_rows(batch_rows_);
    if (d_batch_nodes_) {
      check(hipStreamSynchronize(stream_), "batch nodes");
      release(d_batch_nodes_);
      d_batch_nodes_ = nullptr;
    }
    if (d_batch_index_ || d_batch_sums_) check(hipStreamSynchronize(stream_), "batch nodes");
    release(d_batch_index_);
    release(d_batch_sums_);
    d_batch_index_ = nullptr;
    d_batch_sums_ = nullptr;
    batch_rows_ = build_mem_rows(ccx, ccy, ccz, r_max);
    batch_rows_key_ = {0.0f, 0.0f, 0.0f, 0.0f, ~0ull};  // (none, should the next line throw)
    d_batch_nodes_ = build_mem_nodes(batch_rows_, ccx, ccy, ccz, r_max, &n_batch_nodes_);
    batch_rows_key_ = key;
  }
  *count = n_batch_nodes_;
  return d_batch_nodes_;
}

TileForces Domain::batch_tile_forces() {
  if (n_batch_nodes_ > 0 && !d_batch_index_) {
    int* index = static_cast<int*>(alloc(N_ * sizeof(int)));
    double* sums = nullptr;
    try {
      sums = static_cast<double*>(alloc(3 * sizeof(double) * kTbSteps * static_cast<size_t>(n_batch_nodes_)));
      check(hipMemsetAsync(index, 0xff, N_ * sizeof(int), stream_), "batch nodes");
      check(launch_index_nodes(d_batch_nodes_, n_batch_nodes_, index, stream_), "batch nodes");
      check(hipStreamSynchronize(stream_), "batch nodes");  // the batch runs on its own stream
    } catch (...) {
      (void)hipStreamSynchronize(stream_);
      release(sums);
      release(index);
      throw;
    }
    d_batch_index_ = index;  // both or neither: the tiles write the sums of every indexed node
    d_batch_sums_ = sums;
  }
  return TileForces{d_batch_index_, d_batch_sums_, n_batch_nodes_, kTbSteps};
}

size_t Domain::bytes_needed(int dim, int lattice, int nx, int ny, int nz, int storage, long long plane_pad,
                            bool thermal) {
  const int Q = dim == 2 ? 9 : (lattice == 27 ? 27 : 19);
  const size_t N = static_cast<size_t>(nx) * ny * (dim == 2 ? 1 : nz);
  const long long base = static_cast<long long>((N + 255) / 256 * 256);
  const long long stride = base + (plane_pad >= 0 ? plane_pad : (N >= (1u << 20) ? 1024 : 0));
  const size_t yz = static_cast<size_t>(ny) * (dim == 2 ? 1 : nz);
  const size_t t = thermal ? 2 * 5 * static_cast<size_t>(stride) * 4 + N * 8 : 0;
  return 2 * static_cast<size_t>(Q) * stride * elem_size(storage) + N * (1 + 1 + 4 + 4 + 5 * 4) + prev_stride(Q) * yz * 4 +
         3 * 1024 * 8 + 64 + t;
}

}  // namespace wake_hip
