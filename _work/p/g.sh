# g.sh <name> <timeout> <cmd>
cd /root/repo
timeout 2300 /usr/local/graft/bin/gpurun --timeout $2 -- "mkdir -p gpurun_out; ($3) > gpurun_out/$1.log 2>&1; rc=\$?; tail -25 gpurun_out/$1.log; exit \$rc" > /tmp/$1.out 2>&1; echo rc $?; grep -E "status=|left" /tmp/$1.out; tail -${4:-30} gpurun_out/$1.log
