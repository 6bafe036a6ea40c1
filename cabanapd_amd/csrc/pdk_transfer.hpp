// pdk_transfer.hpp -- copies from the device to the caller's (pageable) arrays
// through pinned slots of the context and a few host threads.
//
// The runtime's own path for pageable memory reached 10 to 17 GB/s of the
// link's 54 (one thread copies, and the first touch of a fresh result array
// faults its pages in on the same thread).  Here the chunks of a copy are
// taken in turn by the calling thread and the context's workers, each with a
// pinned slot of its own: its DMA, then its memcpy, while the other chunks are
// on the link.  (34.6 MB field of a 1.44M-particle specimen into a new array:
// 3.4 -> 1.2 ms.)  The caller waits for chunks, not for workers: one that
// wakes late (a scheduler tick, 4 ms, on a busy host) finds nothing left.
// (uploads keep the runtime's path: it pins the caller's filled pages and was
// within 15 % of this one)
#ifndef PDK_TRANSFER_HPP
#define PDK_TRANSFER_HPP

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

#include "pdk_internal.hpp"

namespace pdk
{
class HostTransfer
{
  public:
    explicit HostTransfer( int device ) : device_( device ) {}
    HostTransfer( const HostTransfer& ) = delete;
    HostTransfer& operator=( const HostTransfer& ) = delete;
    ~HostTransfer()
    {
        {
            std::lock_guard<std::mutex> g( job_mu_ );
            stop_ = true;
        }
        wake_.notify_all();
        for ( std::thread& t : workers_ )
            t.join();
        for ( Slot& s : slots_ )
        {
            if ( s.done )
            {
                (void)hipEventSynchronize( s.done );
                (void)hipEventDestroy( s.done );
            }
            if ( s.mem )
                (void)hipHostFree( s.mem );
        }
    }

    // dst (host) <- src (device) after the work queued on st; complete on return.
    // That work is waited for here, before the context's slots are taken and
    // before a chunk is queued: a queued copy holds its DMA engine until its
    // stream gets there, and other specimens' copies with it.  The workers are
    // woken meanwhile (waiting first made a 34.6 MB copy 20 us longer without).
    void out( void* dst, const void* src, size_t bytes, hipStream_t st )
    {
        if ( bytes >= kDirect )
        {
            rouse();
            PDK_HIP( hipStreamSynchronize( st ) );
        }
        if ( bytes < kDirect || !run( bytes, [=]( Slot& s, size_t off, size_t len ) {
            hipError_t e = hipMemcpyAsync( s.mem, static_cast<const char*>( src ) + off, len, hipMemcpyDeviceToHost, st );
            if ( e == hipSuccess )
                e = hipEventRecord( s.done, st );
            if ( e == hipSuccess )
                e = hipEventSynchronize( s.done );
            if ( e == hipSuccess )
                std::memcpy( static_cast<char*>( dst ) + off, s.mem, len );
            return e;
        } ) )
        {
            PDK_HIP( hipMemcpyAsync( dst, src, bytes, hipMemcpyDeviceToHost, st ) );
            PDK_HIP( hipStreamSynchronize( st ) );
        }
    }

  private:
    static constexpr size_t kChunk = size_t( 1 ) << 20;
    // below, the runtime's own staging is as fast (1.65 MB: 0.12 ms either way)
    static constexpr size_t kDirect = size_t( 4 ) << 20;
    static constexpr int kSlots = 6; // the caller's and five workers'; 6 MiB pinned per context, released with it
    struct Slot
    {
        char* mem = nullptr;
        hipEvent_t done = nullptr; // the slot's last DMA
    };
    struct Job
    {
        std::function<hipError_t( Slot&, size_t, size_t )> chunk;
        size_t bytes = 0, nchunks = 0;
        std::atomic<size_t> next{ 0 };
        std::atomic<int> err{ 0 };
        size_t done = 0; // under job_mu_
    };

    // Chunks of a job until none is left.
    void take( Job& j, Slot& s )
    {
        for ( ;; )
        {
            const size_t c = j.next.fetch_add( 1 );
            if ( c >= j.nchunks )
                return;
            hipError_t e = static_cast<hipError_t>( j.err.load() );
            if ( e == hipSuccess )
                e = hipEventSynchronize( s.done ); // (success if never recorded)
            const size_t off = c * kChunk;
            if ( e == hipSuccess )
                e = j.chunk( s, off, j.bytes - off < kChunk ? j.bytes - off : kChunk );
            if ( e != hipSuccess )
                j.err.store( static_cast<int>( e ) );
            std::lock_guard<std::mutex> g( job_mu_ );
            if ( ++j.done == j.nchunks )
                finished_.notify_all();
        }
    }

    void work( int t )
    {
        if ( hipSetDevice( device_ ) != hipSuccess )
            return;
        uint64_t seen = 0, roused = 0;
        for ( ;; )
        {
            std::shared_ptr<Job> j;
            bool soon = false;
            {
                std::unique_lock<std::mutex> g( job_mu_ );
                wake_.wait( g, [&] { return stop_ || generation_ != seen || roused_ != roused; } );
                if ( stop_ )
                    return;
                soon = generation_ == seen;
                roused = roused_;
                if ( !soon )
                {
                    seen = generation_;
                    j = job_;
                }
            }
            if ( soon ) // stay awake for it, for 100 us at most
            {
                const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds( 100 );
                while ( generation_ == seen && std::chrono::steady_clock::now() < until )
                    std::this_thread::yield();
            }
            if ( j )
                take( *j, slots_[t] );
        }
    }

    // The pinned slots and their events; false where they cannot be had.
    bool ready()
    {
        for ( Slot& s : slots_ )
        {
            hipError_t e = hipSuccess;
            if ( !s.mem )
                e = hipHostMalloc( reinterpret_cast<void**>( &s.mem ), kChunk, hipHostMallocDefault );
            if ( e != hipSuccess )
                s.mem = nullptr;
            else if ( !s.done )
            {
                e = hipEventCreateWithFlags( &s.done, hipEventDisableTiming );
                if ( e != hipSuccess )
                    s.done = nullptr;
            }
            if ( e != hipSuccess )
            {
                (void)hipGetLastError();
                return false;
            }
        }
        return true;
    }

    // A copy is about to come.
    void rouse()
    {
        {
            std::lock_guard<std::mutex> g( job_mu_ );
            roused_++;
        }
        wake_.notify_all();
    }

    // False, with nothing copied, where there are no slots.
    bool run( size_t bytes, std::function<hipError_t( Slot&, size_t, size_t )> chunk )
    {
        std::lock_guard<std::mutex> one( mu_ ); // one copy at a time
        if ( !ready() )
            return false;
        try
        {
            while ( workers_.size() + 1 < kSlots )
            {
                const int t = static_cast<int>( workers_.size() ) + 1;
                workers_.emplace_back( [this, t] { work( t ); } );
            }
        }
        catch ( const std::exception& )
        {
            // no more threads: the others take their chunks
        }
        auto j = std::make_shared<Job>();
        j->chunk = std::move( chunk );
        j->bytes = bytes;
        j->nchunks = ( bytes + kChunk - 1 ) / kChunk;
        {
            std::lock_guard<std::mutex> g( job_mu_ );
            job_ = j;
            generation_++;
        }
        wake_.notify_all();
        take( *j, slots_[0] );
        {
            std::unique_lock<std::mutex> g( job_mu_ );
            finished_.wait( g, [&] { return j->done == j->nchunks; } );
            job_.reset();
        }
        PDK_HIP( static_cast<hipError_t>( j->err.load() ) );
        return true;
    }

    int device_;
    std::mutex mu_;
    Slot slots_[kSlots];
    std::vector<std::thread> workers_;
    std::mutex job_mu_; // job_, generation_, roused_, stop_ and the jobs' done counts
    std::condition_variable wake_, finished_;
    std::shared_ptr<Job> job_;
    std::atomic<uint64_t> generation_{ 0 }; // written under job_mu_
    uint64_t roused_ = 0;
    bool stop_ = false;
};
} // namespace pdk

#endif
