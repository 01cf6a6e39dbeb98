// transfer.hip -- copies between a caller's (pageable) host memory and the
// device, through pinned memory of the library's own.
//
// hipMemcpyAsync on pageable memory is slow in two places: below 1 MiB (128 KiB
// down 62 us, 512 KiB 230 us, against 14 and 29 us through a pinned buffer) and
// for large downloads, where one thread copies out of the runtime's staging
// buffer (8 MiB 480 us, 64 MiB into pages not touched before 15.6 ms, against
// 300 us and 3.6 ms with two and eight threads copying as the pieces arrive).
// Uploads above 1.5 MiB are left to the runtime, which is as fast there.
//
// Whole increments (steps, mass, download), before and after: 128^2 FP64 49.7
// and 47.4 us, 1024^2 FP64 2007 and 1877 us, 150x203x97 FP32 5013 and 4667 us.
// The server's transfers, which run beside its steps, were no faster this way
// (22.0 and 22.8 ms for 16 requests) and stay with the runtime.
//
// Memory of the caller's that the runtime knows already (pinned, managed, of a
// device) takes one direct copy: a pinned destination of 8 MiB 156 us, through
// the area 337.
//
// The pinned memory is one area per process: at most 16 MiB, made when a
// transfer first needs it, grown once, given back when the last state or
// batch is destroyed. Making it and giving it back takes 20 us (2 MiB) to 75, more
// than one small transfer saves, and a program that makes a state for each solve
// would pay it each time (create, upload, ten steps, download, destroy: 128^2
// 153 us plain, 171 to 186 with the area; 700^2 555 and 630; 1024^2 925 and 900,
// 128^3 1690 and 1470): downloads of 8 MiB and more make it at once, smaller
// transfers when eight of them have asked for it. One transfer holds it at a
// time; another thread's transfer that finds it taken uses hipMemcpyAsync.
#include <algorithm>
#include <cstring>
#include <mutex>
#include <thread>

#include "core.hpp"

namespace mmspx {

namespace {

constexpr size_t kSlotBytes = (size_t)1 << 20;
constexpr int kSlots = 16;
constexpr size_t kAtOnce = 8 * kSlotBytes;
constexpr int kAsk = 8;
constexpr size_t kStagedDown = 2 * kSlotBytes, kStagedUp = kSlotBytes + kSlotBytes / 2;

struct Staging {
	std::mutex busy;     // held by the transfer that uses the area
	std::mutex mu;       // users
	int users = 0;
	char* base = nullptr;
	size_t bytes = 0;
	int asked = 0;       // transfers that found no area of their size
	int device = -1;
	hipEvent_t ev[kSlots] = {};
};
Staging g_staging;

void give_back(Staging& s)
{
	for (auto& e : s.ev)
		if (e) {
			(void)hipEventDestroy(e);
			e = nullptr;
		}
	if (s.base) (void)hipHostFree(s.base);
	s.base = nullptr;
	s.bytes = 0;
	s.asked = 0;
	s.device = -1;
}

// The area, at least `need` bytes of it and with its events; the caller holds
// `busy`. False: use the plain copy (also on a device other than the area's).
bool ready(Staging& s, size_t need, bool events, hipStream_t st)
{
	int dev = -1, own = -1;
	if (hipGetDevice(&dev) != hipSuccess || hipStreamGetDevice(st, &own) != hipSuccess || own != dev ||
	    (s.device >= 0 && s.device != dev)) {
		(void)hipGetLastError();
		return false;
	}
	const size_t want = need <= 2 * kSlotBytes ? 2 * kSlotBytes : kSlots * kSlotBytes;
	if (s.bytes < want) {
		if (need < kAtOnce && ++s.asked <= kAsk) return false;
		// relaxed: another thread's stream capture is not ours to disturb
		hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
		(void)hipThreadExchangeStreamCaptureMode(&mode);
		if (s.base) (void)hipHostFree(s.base);
		s.base = nullptr;
		s.bytes = 0;
		const hipError_t e = hipHostMalloc((void**)&s.base, want, 0);
		(void)hipThreadExchangeStreamCaptureMode(&mode);
		if (e != hipSuccess) {
			(void)hipGetLastError();
			s.base = nullptr;
			return false;
		}
		s.bytes = want;
		s.asked = 0;
		s.device = dev;
	}
	for (int k = 0; events && k < kSlots; k++)
		if (!s.ev[k] && hipEventCreateWithFlags(&s.ev[k], hipEventDisableTiming) != hipSuccess) {
			(void)hipGetLastError();
			s.ev[k] = nullptr;
			return false;
		}
	return true;
}

// The pieces of a large download: piece c goes through slot c % kSlots and is
// copied out by thread c % T, which sends the piece that takes the slot next
// (kSlots is a multiple of T, so that piece is its own).
int download_pieces(Staging& s, char* dst, const char* src, size_t bytes, hipStream_t st, int T)
{
	const int n = (int)((bytes + kSlotBytes - 1) / kSlotBytes);
	auto len = [&](int c) { return std::min(kSlotBytes, bytes - (size_t)c * kSlotBytes); };
	auto send = [&](int c) {
		hipError_t e = hipMemcpyAsync(s.base + (size_t)(c % kSlots) * kSlotBytes, src + (size_t)c * kSlotBytes, len(c),
		                              hipMemcpyDeviceToHost, st);
		return e == hipSuccess ? hipEventRecord(s.ev[c % kSlots], st) : e;
	};
	hipError_t err[8] = {};
	for (int c = 0; c < std::min(n, kSlots) && err[0] == hipSuccess; c++) err[0] = send(c);
	if (err[0] == hipSuccess) {
		auto work = [&](int k) {
			hipError_t e = k ? hipSetDevice(s.device) : hipSuccess;
			for (int c = k; c < n && e == hipSuccess; c += T) {
				e = hipEventSynchronize(s.ev[c % kSlots]);
				if (e != hipSuccess) break;
				std::memcpy(dst + (size_t)c * kSlotBytes, s.base + (size_t)(c % kSlots) * kSlotBytes, len(c));
				if (c + kSlots < n) e = send(c + kSlots);
			}
			err[k] = e;
		};
		std::thread th[8];
		int started = 1;
		try {
			for (; started < T; started++) th[started] = std::thread(work, started);
		} catch (...) {  // no more threads: their pieces are done here
		}
		work(0);
		for (int k = 1; k < started; k++) th[k].join();
		for (int k = started; k < T; k++) work(k);
	}
	const hipError_t last = hipStreamSynchronize(st);
	for (const hipError_t& e : err)
		if (e != hipSuccess) return fail(MMSPX_EDEVICE, std::string("download: ") + hipGetErrorString(e));
	if (last != hipSuccess) return fail(MMSPX_EDEVICE, std::string("download: ") + hipGetErrorString(last));
	return 0;
}

}  // namespace

void staging_retain()
{
	std::lock_guard<std::mutex> lk(g_staging.mu);
	g_staging.users += 1;
}

void staging_release()
{
	std::lock_guard<std::mutex> lk(g_staging.mu);
	if (--g_staging.users > 0) return;
	std::lock_guard<std::mutex> area(g_staging.busy);
	give_back(g_staging);
}

// pageable: memory the runtime does not know
static bool pageable(const void* p)
{
	hipPointerAttribute_t a;
	if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeUnregistered;
	(void)hipGetLastError();
	return true;
}

int copy_to_host(void* dst, const void* src, size_t bytes, hipStream_t st)
{
	std::unique_lock<std::mutex> area(g_staging.busy, std::defer_lock);
	if (bytes > 0 && pageable(dst) && area.try_lock() && ready(g_staging, bytes, bytes > kStagedDown, st)) {
		if (bytes > kStagedDown)
			return download_pieces(g_staging, (char*)dst, (const char*)src, bytes, st,
			                       bytes < ((size_t)16 << 20) ? 2 : bytes < ((size_t)48 << 20) ? 4 : 8);
		MMSPX_HIP(hipMemcpyAsync(g_staging.base, src, bytes, hipMemcpyDeviceToHost, st));
		MMSPX_HIP(hipStreamSynchronize(st));
		std::memcpy(dst, g_staging.base, bytes);
		return 0;
	}
	if (area.owns_lock()) area.unlock();
	MMSPX_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st));
	MMSPX_HIP(hipStreamSynchronize(st));
	return 0;
}

int copy_to_device(void* dst, const void* src, size_t bytes, hipStream_t st)
{
	std::unique_lock<std::mutex> area(g_staging.busy, std::defer_lock);
	if (bytes > 0 && bytes <= kStagedUp && pageable(src) && area.try_lock() && ready(g_staging, bytes, false, st)) {
		// in pieces, so that the copy into pinned memory overlaps the transfer
		constexpr size_t piece = kSlotBytes / 2;
		hipError_t e = hipSuccess;
		for (size_t o = 0; o < bytes && e == hipSuccess; o += piece) {
			const size_t n = std::min(piece, bytes - o);
			std::memcpy(g_staging.base + o, (const char*)src + o, n);
			e = hipMemcpyAsync((char*)dst + o, g_staging.base + o, n, hipMemcpyHostToDevice, st);
		}
		const hipError_t last = hipStreamSynchronize(st);  // also before an error leaves the area to others
		if (e == hipSuccess) e = last;
		return e == hipSuccess ? 0 : fail(MMSPX_EDEVICE, std::string("upload: ") + hipGetErrorString(e));
	}
	if (area.owns_lock()) area.unlock();
	MMSPX_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st));
	MMSPX_HIP(hipStreamSynchronize(st));
	return 0;
}

}  // namespace mmspx
