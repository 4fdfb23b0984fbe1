// The error codes and status of every host call (the reference's
// lrt::ErrorCode and Result, modules/core/include/lrt/core/Error.h:14-53,
// Result.h:14-95): never thrown, returned.
#pragma once

#include <cstdint>
#include <string>
#include <utility>

namespace lrt {

enum class ErrorCode : int {   // modules/core/include/lrt/core/Error.h:14-26
    Ok = 0,
    Unknown,
    NotFound,
    InvalidArgument,
    Unsupported,
    IoFailure,
    DeviceFailure,
    ShaderFailure,
    PluginFailure,
    OutOfMemory,
    Cancelled,
    InternalError,
};

struct Status {
    ErrorCode code = ErrorCode::Ok;
    std::string message;
    [[nodiscard]] bool ok() const noexcept { return code == ErrorCode::Ok; }
    static Status error(ErrorCode c, std::string m) { return Status{c, std::move(m)}; }
};

// The counter words of a frame or batch that the kernels flag failures in.
constexpr unsigned kPairsDropped = 2, kSortGaveUp = 4, kScanGaveUp = 5, kDepthOutside = 10;
constexpr const char* kScanGaveUpMessage = "the scan's look-back gave up";

// What those words, read back once all of its launches are done, say went
// wrong; depthOutside: the message for a depth key outside its range. A frame
// that sorts by depth first scans twice, so the scan's word is checked here too
// and not only where the host waits for the counts.
inline Status binningStatus(const uint32_t* counters, const char* depthOutside) {
    const char* message = counters[kScanGaveUp] != 0     ? kScanGaveUpMessage
                          : counters[kPairsDropped] != 0 ? "the duplication overran its pairs"
                          : counters[kDepthOutside] != 0 ? depthOutside
                          : counters[kSortGaveUp] != 0   ? "the sort's look-back gave up"
                                                         : nullptr;
    return message != nullptr ? Status::error(ErrorCode::InternalError, message) : Status{};
}

}   // namespace lrt
